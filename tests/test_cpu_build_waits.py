"""Loads straight into LDS are outside the compiler's count of loads in flight, and loads end in order: where it waits for a load of its
own behind them, it waits for them too.  The listing of the long sumcheck pass is looked through for such waits."""
import os
import re
import shutil
import subprocess

import pytest

from verinf_amd.build import FLAGS

HERE = os.path.dirname(os.path.abspath(__file__))
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


@pytest.mark.skipif(not shutil.which(HIPCC), reason="no hipcc")
def test_nothing_waits_for_words_on_their_way_to_lds(tmp_path):
    listing = str(tmp_path / "pass.s")
    flags = [f for f in FLAGS if f != "-fPIC"]
    subprocess.check_call([HIPCC] + flags + ["--cuda-device-only", "-S", "-o", listing, os.path.join(HERE, "cpu_build", "pass_waits.hip")])
    kernels = re.findall(r"^(\S*k_pass3_long\S*):[^\n]*\n(.*?)\.Lfunc_end", open(listing).read(), re.S | re.M)
    assert len(kernels) == 2
    for name, body in kernels:
        requests, flying = 0, False
        for line in body.splitlines():
            line = line.strip()
            if line.startswith("global_load_lds"):
                requests, flying = requests + 1, True
            elif line.startswith("global_store"):          # the end of a piece: the next one's start waits for everything
                flying = False
            assert not (flying and line.startswith("s_waitcnt") and "vmcnt" in line), (name, line)
        tables = int(re.search(r"k_pass3_longILi(\d)", name).group(1))
        assert requests == 2 * 12 * tables                 # in front of the loop and in it
