"""Split overlap in parts of chunks: states whose digits, products and sums are
all exact, so every depth of the split must give the exact S.  Entries are
integers of at most 100 over 128: one digit holds them, the sums stay below
2^53 and every scale is a power of two, hence equality."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"


# one to several tiles, whole and ragged; a part of a chunk short of the others,
# fewer parts than 8 and chunks of one stage
@pytest.mark.parametrize("prec", ["int8x3", "int8x5", "int8x6a", "fp16x4"])
@pytest.mark.parametrize("n,npw,nkx0", [(1, 16, 0), (96, 301, 1), (128, 8192, 1), (129, 2048, 0),
                                        (300, 16001, 1), (512, 16384, 1), (640, 5000, 1)])
def test_parts_sum_exactly(handle, n, npw, nkx0, prec):
    g = torch.Generator(device=DEV)
    g.manual_seed(n + npw)
    psi = torch.randint(-100, 101, (n, 2 * npw), generator=g, device=DEV).double() / 128.0
    # light chunks at the end, as in plane waves of growing |G|
    psi[:, npw:] = torch.round(psi[:, npw:] * 4.0) / 128.0
    S = handle.overlap_sym(psi, nkx0=nkx0, alpha=2.0, prec=prec)
    p = psi.cpu()
    ref = 2.0 * (p @ p.T) - p[:, :2 * nkx0] @ p[:, :2 * nkx0].T
    assert torch.equal(S.cpu(), ref)
