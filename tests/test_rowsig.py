"""The row-wide sigma2 of the fallback types' imatrix rules where its split can go wrong: rows of one round of 12 blocks,
a little more, two and many, row counts around a workgroup's 16, and both sides of the counts from which a lane takes a
row; every source encoding, one matrix and two; through the blocks, byte for byte against the oracle."""
import numpy as np
import pytest

from test_gpu_fallback import BF16, F16, F32, MXFP4, Q4_0, Q5_0, Q5_1, Q8_0, SNAME, TNAME, source

pytestmark = pytest.mark.gpu

BLOCK_BYTES = {Q4_0: 18, Q5_0: 22, Q5_1: 24}
SOURCES = [F32, F16, BF16, Q8_0, MXFP4]


def run(oracle_lib, src, typ, nmat, nrow, ncol):
    import torch
    torch.cuda.init()
    import gpuq
    gq = gpuq.load_gpuq(0)
    rng = np.random.default_rng(nrow + ncol)
    x = (rng.standard_normal((nmat, nrow, ncol)) * rng.uniform(0.001, 1, (nmat, nrow, 1))).astype(np.float32)
    raw, x = source(oracle_lib, src, x, rng)
    im = rng.lognormal(0, 1.5, (nmat, ncol)).astype(np.float32)
    print("case rowsig %s %s %dx%dx%d" % (SNAME[src], TNAME[typ], nmat, nrow, ncol), flush=True)
    d_raw = torch.from_numpy(np.ascontiguousarray(raw)).cuda()
    d_im = torch.from_numpy(im).cuda()
    out = torch.zeros(x.size // 32 * BLOCK_BYTES[typ], dtype=torch.uint8, device="cuda")
    assert gq.gpuq_requantize_dev(src, d_raw.data_ptr(), typ, out.data_ptr(), nmat, nrow, ncol, d_im.data_ptr(),
                                  torch.cuda.current_stream().cuda_stream) == out.numel()
    torch.cuda.synchronize()
    # (rows stand alone: of many, the first, the last and some between)
    rows = np.arange(nrow) if nrow < 500 else np.r_[0:40, nrow - 40:nrow, rng.integers(0, nrow, 200)]
    got = out.cpu().numpy().reshape(nmat, nrow, -1)
    for m in range(nmat):
        assert np.array_equal(got[m, rows], oracle_lib.quantize(typ, x[m, rows], im[m]).reshape(len(rows), -1)), m


@pytest.mark.parametrize("src", SOURCES, ids=[SNAME[s] for s in SOURCES])
@pytest.mark.parametrize("ncol", [352, 384, 416, 768, 1184])
@pytest.mark.parametrize("nrow", [1, 15, 16, 17, 33])
def test_rows(oracle_lib, src, nrow, ncol):
    run(oracle_lib, src, Q4_0, 1, nrow, ncol)


@pytest.mark.parametrize("src", SOURCES, ids=[SNAME[s] for s in SOURCES])
@pytest.mark.parametrize("typ", [Q4_0, Q5_0, Q5_1], ids=["q4_0", "q5_0", "q5_1"])
def test_two_matrices(oracle_lib, src, typ):
    run(oracle_lib, src, typ, 2, 21, 800)


@pytest.mark.parametrize("src,ncol,a_cu", [(BF16, 384, 32), (BF16, 480, 32), (BF16, 512, 64), (F32, 384, 64),
                                           (F16, 384, 64), (Q8_0, 480, 64), (Q8_0, 512, 128), (MXFP4, 384, 128)])
@pytest.mark.parametrize("past", [0, 1])
def test_many_rows(oracle_lib, src, ncol, a_cu, past):
    """the row counts from which a lane takes a row"""
    import torch
    run(oracle_lib, src, Q4_0, 1, a_cu * torch.cuda.get_device_properties(0).multi_processor_count + past, ncol)
