"""Where the KN loop in one launch is taken: its workgroups (16 rows of M each) wait for each other, so
never with more of them than the device has CUs.  The rule is host arithmetic, compiled here."""
import ctypes
import os
import subprocess

import pytest

from conftest import ROOT


@pytest.fixture(scope="module")
def fits(tmp_path_factory):
    d = tmp_path_factory.mktemp("kn_rule")
    src = d / "rule.cpp"
    src.write_text('#include "kn_rule.hpp"\nextern "C" int fits(int elem, long long l, long long Nl, '
                   'int cus) { return isvd::kn_loop_fits(elem, l, Nl, cus); }\n')
    subprocess.run(["g++", "-std=c++20", "-shared", "-fPIC", "-I",
                    os.path.join(ROOT, "isvd_amd", "csrc"), str(src), "-o", str(d / "rule.so")],
                   check=True)
    f = ctypes.CDLL(str(d / "rule.so")).fits
    f.argtypes = [ctypes.c_int, ctypes.c_longlong, ctypes.c_longlong, ctypes.c_int]
    return f


@pytest.mark.parametrize("cus", [8, 32, 64, 127, 128, 256])
@pytest.mark.parametrize("elem,most", [(8, 64), (4, 80)])
def test_workgroups_fit_the_device(fits, elem, most, cus):
    for l in (1, 16, 47, most):
        for Nl in (l, 16 * 7, 16 * 32, 16 * 32 + 1, 16 * 64, 16 * 127 + 1, 2048):
            if Nl >= l:
                assert fits(elem, l, Nl, cus) == ((Nl + 15) // 16 <= cus)
        assert not fits(elem, l, 2049, cus)
    assert not fits(elem, most + 1, 1024, 256)
    assert not fits(elem, 0, 16, 256) and not fits(elem, 17, 16, 256)
