"""The LDLQ solve where its split can go wrong: groups of 16 rows that are ragged or nearly empty, both sides of the row
count from which 64 rows go to a wave, matrices with factors of their own; and the values that its short division does
not take: zero errors, a factor far from 1, infinities in the weights."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

Q4_K = 12
LDLQ_TYPES = {16: "iq2_xxs", 17: "iq2_xs", 22: "iq2_s", 18: "iq3_xxs", 21: "iq3_s", 19: "iq1_s", 29: "iq1_m", 23: "iq4_xs",
              10: "q2_k", 11: "q3_k", 12: "q4_k", 13: "q5_k", 14: "q6_k"}


@pytest.fixture(scope="module")
def env():
    import torch
    torch.cuda.init()
    import gpuq
    return torch, gpuq.load_gpuq(0)


def factor(rng, n, scale=1.0):
    U = np.triu(rng.standard_normal((n, n)) / 40, 1)
    U[np.diag_indices(n)] = 0.7 + 0.7 * rng.random(n)
    return np.ascontiguousarray(U * scale)


def check(env, oracle_lib, typ, W, U, own=False):
    torch, gq = env
    from gpuq import ldlq
    nmat, ne1, ne0 = W.shape
    perm = np.arange(ne0)
    qw = np.ones((nmat, ne0), dtype=np.float32)
    slots = ldlq.slot_order(perm)
    if own:
        want = np.concatenate([oracle_lib.ldlq(typ, W[m:m + 1], U[m], qw[m:m + 1], slots)[0] for m in range(nmat)])
    else:
        want = oracle_lib.ldlq(typ, W, U, qw, slots)[0]
    print("case ldlq solve %s own=%s" % (W.shape, own), flush=True)
    got = ldlq.quantize_matrix_dev(gq, typ, torch.from_numpy(W).cuda(), torch.from_numpy(U).cuda(), perm,
                                   torch.from_numpy(qw).cuda(), u_per_matrix=own)
    torch.cuda.synchronize()
    assert np.array_equal(got.cpu().numpy().reshape(-1), want.reshape(-1))


@pytest.mark.parametrize("nmat,ne1,own", [(1, 1, False), (1, 15, False), (1, 16, False), (1, 17, False), (2, 33, True),
                                          (3, 100, False)])
def test_rows(env, oracle_lib, nmat, ne1, own):
    rng = np.random.default_rng(ne1)
    W = (rng.standard_normal((nmat, ne1, 768)) * 0.05).astype(np.float32)
    U = np.stack([factor(rng, 768) for _ in range(nmat)]) if own else factor(rng, 768)
    check(env, oracle_lib, Q4_K, W, U, own)


@pytest.mark.parametrize("typ", list(LDLQ_TYPES), ids=list(LDLQ_TYPES.values()))
def test_rows_either_side(env, oracle_lib, typ):
    """a stack of ragged matrices with more than five groups of 16 rows a CU (64 rows a wave, 128 x 128 update tiles), one
    matrix fewer (16 rows a workgroup) and few enough for 64 x 64 tiles: the same bytes, and the oracle's in sampled rows"""
    torch, gq = env
    from gpuq import ldlq
    rng = np.random.default_rng(5)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    nmat, ne1, ne0 = 5 * cus // 6 + 1, 90, 768                # 6 groups of 16 rows a matrix: just over 5 a CU
    few = cus // 4                                            # 4 tiles of 128 x 128 in two blocks, 2 in one
    U = factor(rng, ne0)
    dU = torch.from_numpy(U).cuda()
    W = torch.randn(nmat, ne1, ne0, device="cuda", generator=torch.Generator("cuda").manual_seed(1)) * 0.05
    qw = rng.lognormal(0, 1, (nmat, ne0)).astype(np.float32)
    dqw = torch.from_numpy(qw).cuda()
    perm = np.arange(ne0)
    print("case ldlq either side %s" % LDLQ_TYPES[typ], flush=True)
    many = ldlq.quantize_matrix_dev(gq, typ, W, dU, perm, dqw).clone()
    for n in (nmat - 1, few - 1):
        fewer = ldlq.quantize_matrix_dev(gq, typ, W[:n].contiguous(), dU, perm, dqw[:n].contiguous())
        assert torch.equal(many[:n], fewer), n
    rows = [0, 15, 63, 64, 80, 89]
    for m in (0, nmat // 2, nmat - 1):
        want = oracle_lib.ldlq(typ, W[m:m + 1, rows].cpu().numpy(), U, qw[m:m + 1], ldlq.slot_order(perm))[0]
        assert np.array_equal(many[m, rows].cpu().numpy().reshape(-1), want.reshape(-1)), m


@pytest.mark.parametrize("what", ["zero rows", "large factor", "small factor", "zero diagonal", "infinite weight"])
def test_division_range(env, oracle_lib, what):
    rng = np.random.default_rng(7)
    W = (rng.standard_normal((1, 20, 512)) * 0.05).astype(np.float32)
    U = factor(rng, 512)
    if what == "zero rows":
        W[0, 3:7] = 0
    elif what == "large factor":
        U = np.ldexp(U, 560)
    elif what == "small factor":
        U = np.ldexp(U, -560)
    elif what == "zero diagonal":
        U[77, 77] = 0
    else:
        W[0, 5, 40] = np.inf
        W[0, 6, 300] = -np.inf
    check(env, oracle_lib, Q4_K, W, U)
