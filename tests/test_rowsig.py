"""The row-wide sigma2 of the fallback types' imatrix rules where its split can go wrong: rows of one round of 12 blocks,
a little more, two and many, row counts around a workgroup's 16, and one past the count from which a lane takes a row;
through the blocks, byte for byte against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

Q4_0, BF16, F32 = 2, 30, 0


def run(oracle_lib, src, nrow, ncol):
    import torch
    torch.cuda.init()
    import gpuq
    gq = gpuq.load_gpuq(0)
    rng = np.random.default_rng(nrow + ncol)
    x = (rng.standard_normal((nrow, ncol)) * rng.uniform(0.001, 1, (nrow, 1))).astype(np.float32)
    raw = x
    if src == BF16:
        raw = (x.view(np.uint32) >> 16).astype(np.uint16)
        x = (raw.astype(np.uint32) << 16).view(np.float32)
    im = rng.lognormal(0, 1.5, ncol).astype(np.float32)
    raw = np.ascontiguousarray(raw)
    print("case rowsig %d %dx%d" % (src, nrow, ncol), flush=True)
    d_raw = torch.from_numpy(raw.view(np.uint8).reshape(-1)).cuda()
    d_im = torch.from_numpy(im).cuda()
    out = torch.zeros(nrow * ncol // 32 * 18, dtype=torch.uint8, device="cuda")
    assert gq.gpuq_requantize_dev(src, d_raw.data_ptr(), Q4_0, out.data_ptr(), 1, nrow, ncol, d_im.data_ptr(),
                                  torch.cuda.current_stream().cuda_stream) == out.numel()
    torch.cuda.synchronize()
    # (rows stand alone: of many, the first, the last and some between)
    rows = np.arange(nrow) if nrow < 500 else np.r_[0:40, nrow - 40:nrow, rng.integers(0, nrow, 200)]
    got = out.cpu().numpy().reshape(nrow, -1)
    assert np.array_equal(got[rows], oracle_lib.quantize(Q4_0, x[rows], im).reshape(len(rows), -1))


@pytest.mark.parametrize("src", [F32, BF16], ids=["f32", "bf16"])
@pytest.mark.parametrize("ncol", [352, 384, 416, 768, 1184])
@pytest.mark.parametrize("nrow", [1, 15, 16, 17, 33])
def test_rows(oracle_lib, src, nrow, ncol):
    run(oracle_lib, src, nrow, ncol)


@pytest.mark.parametrize("ncol", [384, 480, 512])
@pytest.mark.parametrize("past", [0, 1])
@pytest.mark.parametrize("a_cu", [32, 64])
def test_many_rows(oracle_lib, a_cu, past, ncol):
    """the row counts from which a lane takes a row: 32 a CU under 512 values, 64 from there (BF16)"""
    import torch
    run(oracle_lib, BF16, a_cu * torch.cuda.get_device_properties(0).multi_processor_count + past, ncol)
