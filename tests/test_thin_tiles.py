"""The search types' calls of few super-blocks, whose tiles hold fewer of them: every count around the places where the
tile's size, the workgroup's or the tile queue change gives the bytes that the same blocks get inside a call large enough
for whole tiles (those are compared with the oracle elsewhere)."""
import pytest

pytestmark = pytest.mark.gpu

TYPES = {16: "iq2_xxs", 17: "iq2_xs", 22: "iq2_s", 18: "iq3_xxs", 21: "iq3_s"}
BF16, MXFP4 = 30, 39


@pytest.mark.parametrize("src", [BF16, MXFP4], ids=["bf16", "mxfp4"])
@pytest.mark.parametrize("typ", list(TYPES), ids=list(TYPES.values()))
def test_counts(typ, src):
    import torch
    torch.cuda.init()
    import gpuq
    gq = gpuq.load_gpuq(0)
    g = torch.Generator(device="cuda").manual_seed(typ)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    n = 72 * cus
    if src == BF16:
        x = torch.randn(n, 256, device="cuda", generator=g) * 0.02
        x[::37] = 0                                             # zero blocks, a zero sub-block, a spike
        x[5::41, 32:64] = 0
        x[7::43, 100] = 3.0
        raw = x.to(torch.bfloat16).reshape(-1).view(torch.uint8)
    else:
        raw = torch.randint(0, 256, (n * 8, 17), dtype=torch.uint8, device="cuda", generator=g)
        raw[:, 0] = 127 - 8 + raw[:, 0] % 5
        raw = raw.reshape(-1)
    im = torch.exp(torch.randn(256, device="cuda", generator=g))
    st = torch.cuda.current_stream().cuda_stream
    bb = gq.gpuq_block_bytes(typ)

    def quantize(first, count):
        r = raw.view(n, -1)[first:first + count].contiguous()
        out = torch.full((count * bb + 16,), 0xA5, dtype=torch.uint8, device="cuda")
        assert gq.gpuq_requantize_dev(src, r.data_ptr(), typ, out.data_ptr(), 1, count, 256, im.data_ptr(),
                                      st) == count * bb
        assert bool((out[count * bb:] == 0xA5).all())
        return out[:count * bb].view(count, bb)

    print("case thin tiles %s" % TYPES[typ], flush=True)
    want = quantize(0, n)
    for count in (1, 2, 3, 5, 9, 31, 2 * cus + 1, 4 * cus, 8 * cus + 1, 16 * cus - 1, 16 * cus + 1, 32 * cus, 32 * cus + 3):
        first = n - count if count % 2 else 0
        assert torch.equal(quantize(first, count), want[first:first + count]), count
