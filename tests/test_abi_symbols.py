"""The C-ABI library loads without a GPU and exports every function include/*.h declares."""
import ctypes
import glob
import os
import re

import pytest

from gpuhelp import pkg
from zkhelp import ROOT


def declared_functions():
    names = []
    for h in glob.glob(os.path.join(ROOT, "include", "*.h")):
        text = re.sub(r"/\*.*?\*/", "", open(h).read(), flags=re.S)
        names += re.findall(r"\b(zk_[a-z0-9_]+)\s*\(", text)
    return sorted(set(names))


def test_every_declared_symbol_is_exported():
    lib = pkg.load_hip()
    names = declared_functions()
    assert len(names) > 40
    missing = [n for n in names if not hasattr(lib, n)]
    assert not missing, f"declared in include/ but not exported: {missing}"


def test_init_fails_loudly_without_gpu_or_succeeds_with_one():
    lib = pkg.load_hip()
    rc = lib.zk_init(ctypes.c_int(0))
    if rc != 0:
        assert b"no HIP device" in lib.zk_last_error() or len(lib.zk_last_error()) > 0


@pytest.mark.parametrize("null", range(9))
def test_matmul_sumcheck_refuses_null_operands_challenges_and_outputs(null):
    """Each of the nine pointers alone: the claim, the polynomials, the folded values; X, W, Y; the three lists of challenges."""
    lib = pkg.load_hip()
    words = (ctypes.c_uint32 * 64)()
    p = [None if i == null else words for i in range(9)]
    two, one = ctypes.c_uint32(2), ctypes.c_int(1)
    assert lib.zk_matmul_sumcheck(*p[:6], two, two, two, p[6], one, p[7], one, p[8], one, None) == 10001
    assert b"zk_matmul_sumcheck: null" in lib.zk_last_error()
