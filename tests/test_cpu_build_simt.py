"""Whole kernels on the CPU: translation units of the library compiled with g++ against cpu_build/simt (workgroups as fibers) and
run through their own entry points under AddressSanitizer and UBSan, results against the oracle.  An index outside a buffer, a
barrier that not every thread reaches or a wrong launch shape fails here and not on the GPU."""
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
DIR = os.path.join(HERE, "cpu_build")


def _build(unit, folder):
    so = os.path.join(folder, f"simt_{unit}.so")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-fno-extern-tls-init", "-fsanitize=address,undefined",
                           "-fno-sanitize-recover=undefined", "-I", os.path.join(DIR, "simt"), "-o", so, os.path.join(DIR, f"simt_{unit}.cpp")])
    return so


@pytest.fixture(scope="module")
def built(tmp_path_factory):
    """One build per translation unit, made when a test first asks for it."""
    made, folder = {}, str(tmp_path_factory.mktemp("simt"))
    return lambda unit: made[unit] if unit in made else made.setdefault(unit, _build(unit, folder))


@pytest.mark.parametrize("unit,what,switches", [("lookup", "lookup", {}), ("ntt", "ntt", {}), ("ntt", "ntt", {"VI_NTT_ROW": "0"}), ("ntt", "lde", {}), ("ntt", "tables", {}),
                                                ("matmul", "matmul", {}), ("sumcheck", "sumcheck", {}), ("sumcheck", "sumcheck", {"SIMT_CUS": "1"}),
                                                ("sumcheck", "sumcheck", {"SIMT_CUS": "2"}), ("sumcheck", "sumcheck", {"SIMT_CUS": "3"}), ("mle", "mle", {}), ("blake3", "blake3", {})])
def test_kernels_on_the_cpu(built, unit, what, switches):
    asan = subprocess.check_output(["g++", "-print-file-name=libasan.so"], text=True).strip()
    env = dict(os.environ, LD_PRELOAD=asan, ASAN_OPTIONS="detect_leaks=0,verify_asan_link_order=0", OPENBLAS_NUM_THREADS="1", **switches)
    res = subprocess.run([sys.executable, os.path.join(DIR, "simt_checks.py"), what, built(unit)], stdout=subprocess.PIPE, stderr=subprocess.STDOUT,
                         text=True, env=env, timeout=600)
    assert res.returncode == 0 and res.stdout.strip().endswith("OK"), res.stdout[-4000:]
