"""ctypes binding of libverinf_hip.so (C ABI: include/verinf_hip.h).

The library is built ahead of time by `python -m verinf_amd.build`; loading fails
loudly if it is missing.  torch is imported first on purpose: its bundled HIP
runtime must be the one the library binds to, so that tensor pointers and stream
handles mean the same thing on both sides.
"""
import array
import contextlib
import ctypes
import functools
import os
import threading
from ctypes import POINTER, c_char_p, c_double, c_int, c_int64, c_size_t, c_uint64, c_void_p

import numpy as np
import torch  # noqa: F401  (must precede the CDLL below)

_HERE = os.path.dirname(os.path.abspath(__file__))
# VERINF_HIP_LIB points at an alternative build of the same library (e.g. one compiled
# with different tuning flags); the default is the in-tree build.
LIB_PATH = os.environ.get("VERINF_HIP_LIB") or os.path.join(_HERE, "libverinf_hip.so")

EXPORTS = [
    "vi_last_error", "vi_version",
    "vi_read_back", "vi_wait_words", "vi_upload_words",
    "vi_gl_binop", "vi_gl_binop_bcast", "vi_gl_unop", "vi_gl_axpy", "vi_gl_probe",
    "vi_gl_sum_workspace_bytes", "vi_gl_sum",
    "vi_gl_matmul_workspace_bytes", "vi_gl_matmul", "vi_gl_matvec", "vi_poly_eval",
    "vi_ntt_workspace_bytes", "vi_ntt_best_workspace_bytes", "vi_ntt_batched",
    "vi_coset_lde_workspace_bytes", "vi_coset_lde_min_workspace_bytes", "vi_coset_lde_launches",
    "vi_coset_lde", "vi_coset_lde_coeffs", "vi_coset_extend",
    "vi_kquant_to_field",
    "vi_kquant_to_field_transposed",
    "vi_sumcheck_workspace_bytes", "vi_sumcheck_eval", "vi_sumcheck_eval_static", "vi_sumcheck_fold_eval",
    "vi_sumcheck_prove", "vi_sumcheck_prove_coins_workspace_bytes", "vi_sumcheck_prove_coins",
    "vi_hash_columns_workspace_bytes", "vi_hash_columns", "vi_hash_columns_update", "vi_hash_columns_finalize",
    "vi_merkle_level", "vi_merkle_tree_nodes", "vi_merkle_tree", "vi_row_prg", "vi_pad_rows",
    "vi_eq_vector", "vi_mle_eval_workspace_bytes", "vi_mle_eval",
    "vi_challenge", "vi_gl_spmv", "vi_lookup_multiplicities",
    "vi_lookup_histogram_workspace_bytes", "vi_lookup_histogram",
    "vi_valu_probe_count", "vi_valu_probe_name", "vi_wall_clock_khz", "vi_valu_probe",
]

COIN_FN = ctypes.CFUNCTYPE(c_int, c_int, POINTER(c_uint64), c_int, POINTER(c_uint64), c_void_p)

_lib = None


class VerinfHipError(RuntimeError):
    pass


def lib():
    """The loaded library with argument types declared."""
    global _lib
    if _lib is not None:
        return _lib
    if not os.path.exists(LIB_PATH):
        raise VerinfHipError(
            f"{LIB_PATH} is missing: build it with `python -m verinf_amd.build` "
            "(there is no CPU fallback)")
    L = ctypes.CDLL(LIB_PATH)
    vp, i64, u64, sz = c_void_p, c_int64, c_uint64, c_size_t
    ip = POINTER(c_int)
    L.vi_last_error.restype = c_char_p
    L.vi_version.restype = c_char_p
    L.vi_gl_binop.argtypes = [c_int, vp, vp, vp, i64, vp]
    L.vi_gl_binop_bcast.argtypes = [c_int, vp, vp, i64, vp, i64, vp]
    L.vi_gl_unop.argtypes = [c_int, vp, u64, vp, i64, vp]
    L.vi_gl_axpy.argtypes = [vp, u64, vp, i64, vp]
    L.vi_gl_probe.argtypes = [c_int, vp, vp, vp, i64, vp]
    L.vi_gl_sum_workspace_bytes.restype = sz
    L.vi_gl_sum_workspace_bytes.argtypes = [i64]
    L.vi_gl_sum.argtypes = [vp, i64, vp, vp, sz, vp]
    L.vi_gl_matmul_workspace_bytes.restype = sz
    L.vi_gl_matmul_workspace_bytes.argtypes = [i64, i64, i64]
    L.vi_gl_matmul.argtypes = [vp, vp, vp, i64, i64, i64, vp, sz, vp]
    L.vi_gl_matvec.argtypes = [vp, vp, vp, i64, i64, vp]
    L.vi_poly_eval.argtypes = [vp, i64, i64, vp, i64, vp, vp]
    L.vi_ntt_workspace_bytes.restype = sz
    L.vi_ntt_workspace_bytes.argtypes = [i64, i64]
    L.vi_ntt_best_workspace_bytes.restype = sz
    L.vi_ntt_best_workspace_bytes.argtypes = [i64, i64]
    L.vi_ntt_batched.argtypes = [vp, i64, i64, c_int, vp, sz, vp]
    L.vi_coset_lde_workspace_bytes.restype = sz
    L.vi_coset_lde_workspace_bytes.argtypes = [i64, i64, i64]
    L.vi_coset_lde_min_workspace_bytes.restype = sz
    L.vi_coset_lde_min_workspace_bytes.argtypes = [i64, i64]
    L.vi_coset_lde_launches.restype = i64
    L.vi_coset_lde_launches.argtypes = [i64, i64, i64, sz]
    L.vi_coset_lde.argtypes = [vp, i64, i64, i64, i64, i64, u64, vp, i64, vp, sz, vp]
    L.vi_coset_lde_coeffs.argtypes = [vp, i64, i64, i64, i64, i64, u64, vp, i64, vp, i64, vp, sz, vp]
    L.vi_coset_extend.argtypes = [vp, i64, i64, i64, i64, i64, u64, vp, i64, vp, sz, vp]
    L.vi_kquant_to_field.argtypes = [c_int, vp, i64, c_double, vp, vp]
    L.vi_kquant_to_field_transposed.argtypes = [c_int, vp, i64, i64, c_double, vp, vp]
    L.vi_sumcheck_workspace_bytes.restype = sz
    L.vi_sumcheck_workspace_bytes.argtypes = []
    L.vi_sumcheck_eval.argtypes = [POINTER(vp), c_int, i64, ip, ip, POINTER(u64), c_int, vp, vp, sz, vp]
    L.vi_sumcheck_eval_static.argtypes = [POINTER(vp), c_int, i64, ip, ip, POINTER(u64), c_int, vp, vp]
    L.vi_sumcheck_fold_eval.argtypes = [POINTER(vp), POINTER(vp), c_int, i64, u64, ip, ip,
                                        POINTER(u64), c_int, POINTER(u64), vp, vp, sz, vp]
    L.vi_sumcheck_prove.argtypes = [POINTER(vp), POINTER(vp), c_int, i64, ip, ip, POINTER(u64), c_int,
                                    COIN_FN, vp, vp, sz, POINTER(u64), POINTER(u64), vp, sz, vp]
    L.vi_sumcheck_prove.restype = c_int
    L.vi_sumcheck_prove_coins_workspace_bytes.restype = sz
    L.vi_sumcheck_prove_coins_workspace_bytes.argtypes = [i64]
    L.vi_sumcheck_prove_coins.argtypes = [POINTER(vp), POINTER(vp), c_int, i64, ip, ip, POINTER(u64), c_int,
                                          POINTER(u64), vp, vp, sz, vp]
    L.vi_sumcheck_prove_coins.restype = c_int
    L.vi_hash_columns_workspace_bytes.restype = sz
    L.vi_hash_columns_workspace_bytes.argtypes = [i64, i64]
    L.vi_hash_columns.argtypes = [vp, i64, i64, i64, vp, vp, sz, vp]
    L.vi_hash_columns_update.argtypes = [vp, i64, i64, i64, i64, i64, vp, sz, vp]
    L.vi_hash_columns_finalize.argtypes = [i64, i64, vp, sz, vp, vp]
    L.vi_merkle_level.argtypes = [vp, i64, vp, vp]
    L.vi_merkle_tree_nodes.restype = i64
    L.vi_merkle_tree_nodes.argtypes = [i64]
    L.vi_merkle_tree.argtypes = [vp, i64, vp, vp]
    L.vi_row_prg.argtypes = [vp, vp, i64, i64, i64, vp, i64, vp]
    L.vi_pad_rows.argtypes = [vp, i64, vp, i64, i64, i64, i64, vp, vp]
    L.vi_pad_rows.restype = c_int
    L.vi_challenge.argtypes = [vp, vp, c_int, vp, i64, vp, vp]
    L.vi_gl_spmv.argtypes = [vp, vp, vp, i64, i64, vp, vp, vp, c_int, vp, vp]
    L.vi_lookup_multiplicities.argtypes = [vp, i64, vp, i64, c_int, vp, vp]
    L.vi_lookup_histogram_workspace_bytes.restype = sz
    L.vi_lookup_histogram_workspace_bytes.argtypes = [i64, i64, c_int]
    L.vi_lookup_histogram.argtypes = [vp, i64, vp, i64, c_int, c_int, vp, vp, sz, vp]
    L.vi_lookup_histogram.restype = c_int
    L.vi_read_back.argtypes = [vp, i64, vp, sz, vp]
    L.vi_read_back.restype = c_int
    L.vi_wait_words.argtypes = [vp, i64, i64, i64, vp]
    L.vi_wait_words.restype = c_int
    L.vi_upload_words.argtypes = [vp, i64, vp, vp]
    L.vi_upload_words.restype = c_int
    L.vi_eq_vector.argtypes = [POINTER(u64), c_int, c_int, vp, vp]
    L.vi_mle_eval_workspace_bytes.restype = sz
    L.vi_mle_eval_workspace_bytes.argtypes = [i64]
    L.vi_mle_eval.argtypes = [vp, i64, i64, POINTER(u64), c_int, vp, vp, sz, vp]
    L.vi_valu_probe_name.restype = c_char_p
    L.vi_valu_probe_name.argtypes = [c_int]
    L.vi_valu_probe.argtypes = [c_int, c_int, c_int, vp, vp, POINTER(i64), vp]
    for name in EXPORTS:
        getattr(L, name)                     # AttributeError here = stale build
    for name in ("vi_gl_binop", "vi_gl_binop_bcast", "vi_gl_unop", "vi_gl_axpy", "vi_gl_probe", "vi_gl_sum",
                 "vi_gl_matmul", "vi_gl_matvec", "vi_poly_eval",
                 "vi_ntt_batched", "vi_coset_lde", "vi_coset_lde_coeffs", "vi_coset_extend", "vi_kquant_to_field", "vi_kquant_to_field_transposed", "vi_sumcheck_eval", "vi_sumcheck_eval_static",
                 "vi_sumcheck_fold_eval", "vi_hash_columns", "vi_hash_columns_update", "vi_hash_columns_finalize",
                 "vi_merkle_level", "vi_merkle_tree_nodes", "vi_merkle_tree", "vi_row_prg", "vi_eq_vector", "vi_mle_eval",
                 "vi_challenge", "vi_gl_spmv", "vi_lookup_multiplicities", "vi_valu_probe"):
        getattr(L, name).restype = c_int
    _lib = L
    return L


def check(rc: int) -> None:
    """Turn a negative C-ABI return code into an exception carrying vi_last_error()."""
    if rc != 0:
        msg = lib().vi_last_error().decode("utf-8", "replace")
        raise VerinfHipError(f"libverinf_hip error {rc}: {msg}")


# The handle of torch's current stream and the current device as plain integers, straight from torch's bindings: the
# Stream object of torch.cuda.current_stream() costs 2.8 us and a torch.cuda.device() block 1.3 us per call, more than
# the kernels of a small call take (0.08 and 0.13 us this way).
_raw_stream = torch._C._cuda_getCurrentRawStream
_get_device = torch._C._cuda_getDevice
_capturing = torch._C._cuda_isCurrentStreamCapturing


def stream_ptr() -> int:
    """hipStream_t of torch's current stream (kernels are queued behind torch's own work)."""
    return _raw_stream(_get_device())


_NO_GUARD = contextlib.nullcontext()


def on_device(dev):
    """Context that makes `dev` current; nothing to do (and nothing paid) when it already is."""
    return _NO_GUARD if dev.index is None or dev.index == _get_device() else torch.cuda.device(dev)


@functools.lru_cache(maxsize=1024)
def workspace_bytes(entry: str, *sizes: int) -> int:
    """vi_<entry>_workspace_bytes(*sizes), which depends on nothing else (0.1 us where the call through ctypes takes 0.5)."""
    return getattr(lib(), f"vi_{entry}_workspace_bytes")(*sizes)


_ws_cache = {}
_stream_locks = {}


def stream_lock(stream_ptr: int):
    """The lock of the current device's stream with this handle, which a call that uses workspace() holds from there to its
    last launch.

    Host threads that share a stream share its scratch buffers: what one call leaves in them for its next launch has to
    stay there until that launch is queued, and a buffer that another thread outgrows must not be dropped before.  The
    lock is held while work is queued, not while the host waits for a result or runs a caller's code."""
    key = (_get_device(), stream_ptr)
    lock = _stream_locks.get(key)
    return lock if lock is not None else _stream_locks.setdefault(key, threading.RLock())


def workspace(nbytes: int, tag: str, stream_ptr: int):
    """A cached uint8 device buffer of at least nbytes for a stream of the current device; the caller holds stream_lock().

    One buffer per (purpose, device, stream): the wrappers launch on torch's current stream, so two streams
    (or two host threads on their own streams) never share scratch, and a buffer is only ever used on the
    stream it was allocated on -- when it is outgrown and dropped, the caching allocator may reuse its memory
    in stream order without further bookkeeping.  Buffers grow and are kept; release_workspaces() drops them.
    A call under stream capture gets a buffer of its own from the graph's memory: the graph keeps its address, and a
    cached one may be outgrown and given back while the graph lives."""
    index = _get_device()
    if stream_ptr and _capturing():              # the default stream (0) cannot be captured; asking costs 0.35 us
        return torch.empty(max(int(nbytes), 256), dtype=torch.uint8, device=torch.device("cuda", index))
    key = (tag, index, stream_ptr)
    buf = _ws_cache.get(key)
    if buf is None or buf.numel() < nbytes:
        buf = _ws_cache[key] = torch.empty(max(int(nbytes), 256), dtype=torch.uint8, device=torch.device("cuda", index))
    return buf


_pinned = threading.local()
NO_WORD = 0xFFFFFFFFFFFFFFFF    # VI_NO_WORD: no field element


class _Words:
    """Pinned host words and a numpy view of the same memory.  As a context: a call's kernels write the words and the call
    polls them.  Left by an exception, those kernels may still be on their way, and words they write later would pass for the
    results of the next call, so the stream is waited for."""
    __slots__ = ("host", "view", "polled")

    def __init__(self, words):
        self.host = torch.zeros(words, dtype=torch.uint64).pin_memory()
        self.view = self.host.numpy()
        self.polled = False

    def __enter__(self):
        self.polled = True
        return self

    def __exit__(self, kind, value, trace):
        if kind is not None:
            torch.cuda.current_stream().synchronize()
        self.polled = False


def _words(words: int, stream_ptr: int):
    bufs = getattr(_pinned, "bufs", None)
    if bufs is None:
        bufs = _pinned.bufs = {}
    key = (_get_device(), stream_ptr)
    buf = bufs.get(key)
    if buf is not None and buf.polled:
        # the context was left without its wait (a second interrupt), or a call runs inside another one's: what is queued is
        # waited for before the buffer may go, and its words are left to whoever still reads them
        torch.cuda.current_stream().synchronize()
        buf = None
    if buf is None or buf.host.numel() < words:
        buf = bufs[key] = _Words(max(words, 512))
    return buf


def pinned_words(words: int, stream_ptr: int):
    """Pinned host words that kernels of a call write results into and the call reads them from, with a numpy view of
    the same memory; stream_ptr is torch's current stream.  One buffer per host thread and stream: a call has read its
    results before the next one on that stream starts, and two threads (or two streams) never see each other's.  Buffers
    grow and are kept for the life of the thread (a few KiB each)."""
    buf = _words(words, stream_ptr)
    return buf.host, buf.view


def polled_words(words: int, stream_ptr: int):
    """The same buffer for results that vi_wait_words() waits for: a context around launches and wait, with `words` words
    set to NO_WORD."""
    buf = _words(words, stream_ptr)
    buf.view[:words] = NO_WORD
    return buf


def read_back_ptr(src: int, nbytes: int, sp: int) -> bytes:
    """`nbytes` (a multiple of 4) at device address `src`, once the stream `sp` has reached this point.

    A kernel writes the bytes and then a tag into pinned memory and the host polls the tag: 6 us less than a copy
    and a stream synchronisation."""
    words = (nbytes + 7) // 8
    host, view = pinned_words(words + 1, sp)
    check(lib().vi_read_back(src, nbytes, host.data_ptr(), host.numel() * 8, sp))
    return view[:words].tobytes()[:nbytes]


def read_back(t, nbytes: int) -> bytes:
    """The first `nbytes` of a contiguous device tensor, through the current stream."""
    with on_device(t.device):
        return read_back_ptr(t.data_ptr(), nbytes, stream_ptr())


_UPLOAD_WORDS = 448         # VI_UPLOAD_WORDS
_P = (1 << 64) - (1 << 32) + 1


def field_words(values):
    """Python integers as an array('Q') of residues mod p."""
    if not isinstance(values, (list, tuple)):    # array() takes the bytes of a bytes object for memory, and a generator runs once
        return array.array("Q", [int(v) % _P for v in values])
    try:
        words = array.array("Q", values)         # 20 ns per entry, ten times less than int(v) % p one by one
    except (OverflowError, TypeError):
        return array.array("Q", [int(v) % _P for v in values])
    if len(words) and (max(words) if len(words) < 64 else int(np.frombuffer(words, dtype=np.uint64).max())) >= _P:
        return array.array("Q", [v % _P for v in words])
    return words


def upload_words(words):
    """An array('Q') as a (1, n) uint64 tensor on the current device.  Short ones travel in a kernel's arguments (one
    launch); a copy from pageable memory waits for the stream first (15 us with nothing to wait for)."""
    n = len(words)
    if n > _UPLOAD_WORDS or n == 0:
        return torch.from_numpy(np.frombuffer(words, dtype=np.uint64).reshape(1, n).copy()).cuda()
    out = torch.empty((1, n), dtype=torch.uint64, device="cuda")
    check(lib().vi_upload_words(words.buffer_info()[0], n, out.data_ptr(), stream_ptr()))
    return out


def release_workspaces() -> None:
    """Drop every cached scratch buffer (they come back on demand).  Call it with the device idle: a buffer
    still in use by queued kernels must not be handed back to the allocator from another stream."""
    for key in list(_ws_cache):
        with _stream_locks.get(key[1:], _NO_GUARD):          # not between a call's look-up and its launches
            _ws_cache.pop(key, None)
