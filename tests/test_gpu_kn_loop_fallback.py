"""The KN loop in one launch where it hands over: a wait that times out (every one does, with a limit
of no polls) leaves the integration to the separate launches, and the state between two launches of the
loop (after 512 iterations) carries on where it was."""
import numpy as np
import pytest

from isvd_amd import capi, pipeline
from test_gpu_kn_loop import bases, check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("l,N", [(16, 65), (47, 11), (64, 32)])
def test_timeout(torch_cuda, monkeypatch, l, N, dtype):
    monkeypatch.setenv("ISVD_KN_LOOP", "2")
    check(torch_cuda, 300, l, N, 0.7, dtype, 10 * l + N)


def test_several_launches(torch_cuda, monkeypatch):
    """600 iterations in launches of 512 against the separate launches."""
    its = 600
    qs = torch_cuda.from_numpy(bases(200, 20, 6, 0.7, 1)).cuda()
    prm = capi.create_param(200, 40, 20, 0, 6)
    q, it, _ = pipeline.integrate(prm, qs, "KN", argv=[its, 0.0])
    monkeypatch.setenv("ISVD_KN_LOOP", "0")
    r, rit, _ = pipeline.integrate(prm, qs, "KN", argv=[its, 0.0])
    assert it == rit == its + 1
    # a few rounding errors per iteration
    assert (q - r).abs().max().item() <= 8 * its * np.sqrt(20) * np.finfo(float).eps
