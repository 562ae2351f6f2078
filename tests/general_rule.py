"""Which kernel a call of the general entry point runs on, asked of csrc/fa2_general_rule.h."""
import ctypes
import functools
import tempfile
from pathlib import Path

from host_rules import rules

STAGED, SPLIT, DIMS, DIMS_SMALL = range(4)
BODY = """
int kernel(const int64_t* n, int d, int dv, int bits16, float scale, int n_cus, int xcd_log2) {
  using namespace mi_fa2;
  return general_kernel({n[0], n[1], n[2], n[3], n[4], n[5], n[6], d, dv, bits16 != 0, scale, n_cus,
                         xcd_log2});
}
"""


@functools.lru_cache(None)
def _library():
    with tempfile.TemporaryDirectory() as tmp:
        fn = rules(Path(tmp), "fa2_general_rule.h", BODY).kernel
    fn.argtypes = [ctypes.POINTER(ctypes.c_int64)] + [ctypes.c_int] * 3 + [ctypes.c_float] + [ctypes.c_int] * 2
    return fn


def kernel(B, Hq, Hkv, T, S, d, dv=None, bits16=True, scale=0.1, strides=None, n_cus=256,
           xcd_log2=3):
    dv = d if dv is None else dv
    sizes = (ctypes.c_int64 * 7)(B, Hq, Hkv, T, S, *(strides or (d, dv)))
    return _library()(sizes, d, dv, bits16, scale, n_cus, xcd_log2)


def on_this_device(*sizes, **kw):
    """The kernel a call of these sizes takes on the current GPU."""
    from kernels import _lib
    plan = _lib.launch_plan()
    return kernel(*sizes, **kw, n_cus=plan["num_cus"], xcd_log2=plan["xcds_mapped"].bit_length() - 1)
