"""H += X^T X (gpuq_hessian_accumulate_dev) where its tiling can go wrong: triangles of 2 to 18 tiles (whole groups of
eight row tiles, a ragged one, one beside it) and row counts around the chunk of 16. X and H hold small whole numbers,
so every sum is exact and the result has to be equal."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ne0", [256, 1024, 1280, 2304])
@pytest.mark.parametrize("nrows", [1, 15, 16, 17, 50])
def test_tiles(ne0, nrows):
    import torch
    torch.cuda.init()
    import gpuq
    gq = gpuq.load_gpuq(0)
    g = torch.Generator(device="cuda").manual_seed(ne0 + nrows)
    buf = torch.randint(-9, 10, (nrows * ne0 + 1,), device="cuda", generator=g).float()
    X = buf[1:].view(nrows, ne0)                      # (4-byte aligned)
    A = torch.randint(-50, 50, (ne0, ne0), device="cuda", generator=g).double()
    H = A + A.T
    want = H.cpu() + X.cpu().double().T @ X.cpu().double()
    assert gq.gpuq_hessian_accumulate_dev(X.data_ptr(), nrows, ne0, H.data_ptr(),
                                          torch.cuda.current_stream().cuda_stream) == 0
    assert torch.equal(H.cpu(), want)
