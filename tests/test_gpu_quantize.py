"""The e4m3 quantizer on views that are not 16-byte aligned and at the edges of its 128 x 128 blocks,
bit for bit against the oracle, and with infinities and NaN in the matrix."""
import numpy as np
import pytest

from isvd_amd import pipeline
from oracle import fp8

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ordera", ["R", "C"])
@pytest.mark.parametrize("off", [0, 1])
@pytest.mark.parametrize("m,n", [(1, 1), (127, 129), (128, 128), (129, 127), (256, 131), (387, 512)])
def test_quantize_views(torch_cuda, ordera, off, m, n):
    torch = torch_cuda
    rng = np.random.default_rng(m * n)
    a = (rng.standard_normal((m, n)) * np.exp2(rng.uniform(-9, 9, size=(m, n)))).astype(np.float32)
    store = np.ascontiguousarray(a if ordera == "R" else a.T)
    buf = torch.empty(store.size + off, device="cuda")
    a_in = buf[off:].view(store.shape)
    a_in.copy_(torch.from_numpy(store))
    a8, scale = pipeline.quantize_e4m3(a_in, ordera=ordera)
    codes, s_ref = fp8.quantize(a.astype(np.float64))
    assert np.array_equal(scale.cpu().numpy().astype(np.float64), s_ref)
    assert np.array_equal(a8.cpu().numpy()[:, :n], codes)
    assert not a8.cpu().numpy()[:, n:].any()


@pytest.mark.parametrize("ordera", ["R", "C"])
def test_quantize_special_values(torch_cuda, ordera):
    a = np.random.default_rng(0).standard_normal((256, 256)).astype(np.float32)
    a[3, 200] = np.nan   # block (0, 1): the NaN takes no part in the scale
    a[200, 7] = np.inf   # block (1, 0): the largest scale
    a[201, 8] = -np.inf
    clean = np.where(np.isfinite(a), a, 0).astype(np.float64)
    codes, s_ref = fp8.quantize(clean)
    x = torch_cuda.from_numpy(np.ascontiguousarray(a if ordera == "R" else a.T)).cuda()
    a8, scale = (t.cpu().numpy() for t in pipeline.quantize_e4m3(x, ordera=ordera))
    assert a8[3, 200] & 0x7F == 0x7F
    assert a8[200, 7] == 0x7E and a8[201, 8] == 0xFE
    assert scale[1, 0] == 2.0 ** 127
    keep = np.isfinite(a)
    keep[128:, :128] = False
    assert np.array_equal(a8[keep], codes[keep])
    assert np.array_equal(scale.ravel()[[0, 1, 3]].astype(np.float64), s_ref.ravel()[[0, 1, 3]])
