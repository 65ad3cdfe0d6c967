"""The search types' calls of few super-blocks, whose tiles hold fewer of them (kernels of their own): every count around
the places where the tile's size, the workgroup's or the kernel change gives the bytes that the same blocks get inside a
call large enough for whole tiles, and those are the oracle's in sampled blocks; every source encoding."""
import numpy as np
import pytest

from test_gpu_fallback import BF16, F16, F32, MXFP4, Q8_0, SNAME, source

pytestmark = pytest.mark.gpu

TYPES = {16: "iq2_xxs", 17: "iq2_xs", 22: "iq2_s", 18: "iq3_xxs", 21: "iq3_s"}
SOURCES = [F32, F16, BF16, Q8_0, MXFP4]


@pytest.mark.parametrize("src", SOURCES, ids=[SNAME[s] for s in SOURCES])
@pytest.mark.parametrize("typ", list(TYPES), ids=list(TYPES.values()))
def test_counts(oracle_lib, typ, src):
    import torch
    torch.cuda.init()
    import gpuq
    gq = gpuq.load_gpuq(0)
    rng = np.random.default_rng(typ)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    n = 72 * cus
    x = rng.standard_normal((n, 256), dtype=np.float32) * np.float32(0.02)
    x[::37] = 0                                             # zero blocks, a zero sub-block, a spike
    x[5::41, 32:64] = 0
    x[7::43, 100] = 3.0
    raw, x = source(oracle_lib, src, x, rng)
    raw = torch.from_numpy(np.ascontiguousarray(raw)).cuda()
    im = rng.lognormal(0, 1, 256).astype(np.float32)
    d_im = torch.from_numpy(im).cuda()
    st = torch.cuda.current_stream().cuda_stream
    bb = gq.gpuq_block_bytes(typ)

    def quantize(first, count):
        r = raw.view(n, -1)[first:first + count].contiguous()
        out = torch.full((count * bb + 16,), 0xA5, dtype=torch.uint8, device="cuda")
        assert gq.gpuq_requantize_dev(src, r.data_ptr(), typ, out.data_ptr(), 1, count, 256, d_im.data_ptr(),
                                      st) == count * bb
        assert bool((out[count * bb:] == 0xA5).all())
        return out[:count * bb].view(count, bb)

    print("case thin tiles %s %s" % (TYPES[typ], SNAME[src]), flush=True)
    want = quantize(0, n)
    some = np.r_[0:8, 5 + 41 * 7, 7 + 43 * 9, 37 * 11, rng.integers(0, n, 40), n - 4:n]
    assert np.array_equal(want[some].cpu().numpy(), oracle_lib.quantize(typ, x[some], im).reshape(len(some), bb))
    for count in (1, 2, 3, 5, 9, 31, 2 * cus + 1, 4 * cus, 8 * cus + 1, 16 * cus - 1, 16 * cus + 1, 32 * cus, 32 * cus + 3):
        first = n - count if count % 2 else 0
        assert torch.equal(quantize(first, count), want[first:first + count]), count
