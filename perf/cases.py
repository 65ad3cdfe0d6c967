"""The framework's performance cases: what its users have it do, through the C ABI and the Python package.

A user re-quantizes a model: tensor by tensor the stored bytes (F32, F16, BF16, Q8_0 or MXFP4) become ggml blocks,
from device memory (gpuq_requantize_dev) or from host buffers (gpuq_requantize_batch, the route of the reference's
drivers); the blocks are read back (gpuq_dequantize_dev); and for the best quality the LDLQ path sums a Hessian
(gpuq_hessian_accumulate_dev), factors it (gpuq_prepare_hessian_dev) and quantizes with error feedback
(gpuq.ldlq.quantize_matrix_dev). Sizes are the configurations of the benchmark (2048 x 7168 experts, a 4096 x 4096
dense tensor), the tests' (1536 columns, fallback rows of 7200) and their neighbours.

`listed()` are the fixed cases, `draw(rng)` one more of the same ranges; `prepare(case, seed)` makes what the user's
program has in hand, `run(state)` is one pass, `work(case)` what the pass cannot do without, `tolerance(case)` and
`exact(case, seed)` how its outputs are judged.
"""
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "trench-gguf_amd"))
# the repository's table file holds stand-in IQ codebooks, loaded only where a program asks for them
os.environ.setdefault("GPUQ_ALLOW_SYNTHETIC_TABLES", "1")

import gpuq  # noqa: E402
from gpuq import ldlq  # noqa: E402

SOURCES = {"f32": gpuq.F32, "f16": gpuq.F16, "bf16": gpuq.BF16, "q8_0": gpuq.Q8_0, "mxfp4": gpuq.MXFP4}
TYPES = {gpuq.TYPE_NAMES[t].lower(): t for t in gpuq.TYPE_NAMES}
BLOCK_BYTES = {"q8_0": 34, "q2_k": 84, "q3_k": 110, "q4_k": 144, "q5_k": 176, "q6_k": 210, "iq2_xxs": 66,
               "iq2_xs": 74, "iq3_xxs": 98, "iq1_s": 50, "iq4_nl": 18, "iq3_s": 110, "iq2_s": 82, "iq4_xs": 136,
               "iq1_m": 56, "q4_0": 18, "q5_0": 22, "q5_1": 24, "f16": 2}
# arithmetic operations a weight of ggml's sequential search with an imatrix (each add, multiply, compare, select or
# conversion one; the search types' depend a little on the data: means over normal weights)
OPS = {"q8_0": 5, "q2_k": 868, "q3_k": 281, "q4_k": 810, "q5_k": 810, "q6_k": 254, "iq2_xxs": 1020, "iq2_xs": 1002,
       "iq3_xxs": 1042, "iq1_s": 842, "iq4_nl": 230, "iq3_s": 854, "iq2_s": 492, "iq4_xs": 229, "iq1_m": 706,
       "q4_0": 250, "q5_0": 250, "q5_1": 800, "f16": 1}
NEED_IMATRIX = ("iq2_xxs", "iq2_xs", "iq2_s", "iq1_s", "iq1_m", "iq3_xxs", "iq3_s")
NO_IMATRIX = ("q8_0", "f16")
LDLQ_TYPES = ("iq2_xxs", "iq2_xs", "iq2_s", "iq3_xxs", "iq3_s", "iq1_s", "iq1_m", "iq4_xs", "q2_k", "q3_k", "q4_k",
              "q5_k", "q6_k")

_lib = []


def lib():
    """the library, initialised on the GPU once a process"""
    if not _lib:
        torch.cuda.init()
        _lib.append(gpuq.load_gpuq(0))
    return _lib[0]


def stream():
    return torch.cuda.current_stream().cuda_stream


def block(typ):
    return gpuq.BLOCK[TYPES[typ]]


def quantize_case(name, op, src, typ, nmat, nrow, ncol, imatrix):
    case = {"op": op, "src": src, "type": typ, "nmat": nmat, "nrow": nrow, "ncol": ncol, "imatrix": imatrix}
    return dict({"name": name}, **case) if name else case


def listed():
    return [
        # the smallest calls: a narrow projection of a few rows, one launch that fills a fraction of the GPU
        quantize_case("small_iq3_s_f16", "device", "f16", "iq3_s", 1, 64, 1536, True),
        # a dense tensor at the bandwidth-bound type (the benchmark's first configuration)
        quantize_case("dense_q8_0_f32", "device", "f32", "q8_0", 1, 4096, 4096, False),
        # one attention / dense tensor with an imatrix at the usual k-quant (the second configuration)
        quantize_case("tensor_q4_k_bf16", "device", "bf16", "q4_k", 1, 2048, 7168, True),
        # stacked experts at the usual i-quant (the headline's experts, 16 of them)
        quantize_case("experts_iq2_xxs_bf16", "device", "bf16", "iq2_xxs", 16, 2048, 7168, True),
        # stacked experts stored as MXFP4 at the smallest i-quant (the fourth configuration, 16 experts)
        quantize_case("experts_iq1_m_mxfp4", "device", "mxfp4", "iq1_m", 16, 2048, 7168, True),
        # rows that are not whole super-blocks get a fallback type, weighted over the whole row
        quantize_case("ragged_q5_1_bf16", "device", "bf16", "q5_1", 1, 2048, 7200, True),
        # reading blocks back as floats: eight experts' worth
        {"name": "to_float_iq2_s", "op": "to_float", "type": "iq2_s", "nblocks": 8 * 2048 * 28},
        # error feedback on an expert's gate and up matrices, which share a factor
        {"name": "ldlq_pair_iq2_s", "op": "ldlq", "type": "iq2_s", "nmat": 2, "ne1": 2048, "ne0": 7168, "own": False},
        # error feedback on a stack of down projections, each with its own factor
        {"name": "ldlq_down_iq2_xxs", "op": "ldlq", "type": "iq2_xxs", "nmat": 8, "ne1": 7168, "ne0": 2048,
         "own": True},
        # collecting a Hessian: one chunk of activation rows
        {"name": "hessian_add_4096", "op": "hessian_add", "nrows": 4096, "ne0": 7168},
        # the factor of one expert's Hessian
        {"name": "hessian_factor_7168", "op": "hessian_factor", "ne0": 7168, "order": "act", "dead": 0},
        # the reference drivers' route: host buffers in and out, four experts
        quantize_case("host_q4_k_bf16", "host", "bf16", "q4_k", 4, 2048, 7168, True),
    ]


def between(rng, lo, hi):
    """a whole number of [lo, hi], spread over its logarithm, odd ones among them"""
    return min(hi, max(lo, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    op = rng.choice(["device"] * 6 + ["blocks", "host", "host", "to_float", "src_to_float", "ldlq", "ldlq", "ldlq",
                                      "hessian_add", "hessian_add", "hessian_factor", "hessian_factor", "schur"])
    if op in ("device", "host"):
        typ = rng.choice(sorted(OPS))
        src = rng.choice(sorted(SOURCES))
        # rows are whole blocks of the type and, for the packed sources, whole 32-value blocks
        if typ == "f16" and src in ("f32", "f16", "bf16"):
            ncol = between(rng, 96, 7200)
        elif block(typ) == 256:
            ncol = 256 * between(rng, 1, 28)
        else:
            ncol = 32 * between(rng, 2, 225)
        nrow = between(rng, 1, 4096)
        # at most a quarter of the listed experts' weights
        nmat = between(rng, 1, max(1, min(16, 4 * 2048 * 7168 // (nrow * ncol))))
        im = typ in NEED_IMATRIX or (typ not in NO_IMATRIX and rng.random() < 0.7)
        return quantize_case(None, op, src, typ, nmat, nrow, ncol, im)
    if op == "blocks":
        typ = rng.choice(sorted(t for t in OPS if block(t) == 256))
        return {"op": op, "type": typ, "nblocks": between(rng, 1, 100000),
                "imatrix": typ in NEED_IMATRIX or rng.random() < 0.7}
    if op == "to_float":
        return {"op": op, "type": rng.choice(LDLQ_TYPES), "nblocks": between(rng, 1, 8 * 2048 * 28)}
    if op == "src_to_float":
        return {"op": op, "src": rng.choice(sorted(SOURCES)), "n": 32 * between(rng, 1, 1 << 21)}
    if op == "ldlq":
        ne0 = 256 * between(rng, 2, 28)
        ne1 = between(rng, 16, 7168)
        nmat = between(rng, 1, max(1, min(8, (4096 * 7168) // (ne1 * ne0))))
        return {"op": op, "type": rng.choice(LDLQ_TYPES), "nmat": nmat, "ne1": ne1, "ne0": ne0,
                "own": nmat > 1 and rng.random() < 0.5}
    if op == "hessian_add":
        return {"op": op, "nrows": between(rng, 16, 4096), "ne0": 256 * between(rng, 2, 28)}
    if op == "hessian_factor":
        ne0 = 256 * between(rng, 1, 28)
        return {"op": op, "ne0": ne0, "order": rng.choice(["seq", "act"]), "dead": rng.choice([0, 0, between(rng, 1, 40)])}
    return {"op": op, "ne0": 256 * between(rng, 1, 28), "nrep": between(rng, 1, 8)}


def src_bytes(src, n):
    return {"f32": 4 * n, "f16": 2 * n, "bf16": 2 * n, "q8_0": n // 32 * 34, "mxfp4": n // 32 * 17}[src]


def work(case):
    op = case["op"]
    if op in ("device", "host"):
        n = case["nmat"] * case["nrow"] * case["ncol"]
        im = 4 * case["nmat"] * case["ncol"] if case["imatrix"] else 0
        # (without importances the k-quants and IQ4 search a little less; the fallback types take a single pass)
        ops = 8 if case["type"] in ("q4_0", "q5_0", "q5_1") and not case["imatrix"] else OPS[case["type"]]
        return {"bytes": src_bytes(case["src"], n) + im + n // block(case["type"]) * BLOCK_BYTES[case["type"]],
                "flops": n * ops}
    if op == "blocks":
        n = 256 * case["nblocks"]
        return {"bytes": 4 * n + case["nblocks"] * BLOCK_BYTES[case["type"]], "flops": n * OPS[case["type"]]}
    if op == "to_float":
        return {"bytes": case["nblocks"] * (1024 + BLOCK_BYTES[case["type"]]), "flops": 2 * 256 * case["nblocks"]}
    if op == "src_to_float":
        return {"bytes": src_bytes(case["src"], case["n"]) + 4 * case["n"], "flops": case["n"]}
    if op == "ldlq":
        rows, ne0 = case["nmat"] * case["ne1"], case["ne0"]
        nblk = ne0 // 256
        # the weights in, the blocks out, the factor's upper triangle; a multiply-add for every later column of every
        # block's 256 errors, the triangular solve of all but the last block, and the search
        return {"bytes": rows * (4 * ne0 + nblk * BLOCK_BYTES[case["type"]])
                + (case["nmat"] if case["own"] else 1) * 4 * ne0 * (ne0 + 1),
                "flops": rows * (2 * 256 * 256 * (nblk * (nblk - 1) // 2) + 256 * 256 * (nblk - 1)
                                 + ne0 * OPS[case["type"]])}
    if op == "hessian_add":
        d = case["ne0"]
        return {"bytes": 4 * case["nrows"] * d + 8 * d * d, "flops": case["nrows"] * d * (d + 1)}
    if op == "hessian_factor":
        d = case["ne0"]
        return {"bytes": 16 * d * d, "flops": 2 * d ** 3 // 3}
    d = case["ne0"]       # schur: the inverse of each 256-column diagonal block's triangle, its rows' norms
    return {"bytes": d // 256 * 8 * 256 * 257 // 2 + 4 * d * case["nrep"], "flops": d // 256 * (256 ** 3 // 3 + 256 ** 2)}


def generator(seed, device="cuda"):
    return torch.Generator(device=device).manual_seed(int(seed))


def values(gen, nmat, nrow, ncol):
    """expert weights: N(0, s_e) with s_e in [0.01, 0.03], 0.1% outliers at 8 sigma"""
    sig = torch.rand(nmat, 1, 1, device="cuda", generator=gen) * 0.02 + 0.01
    x = torch.randn(nmat, nrow, ncol, device="cuda", generator=gen)
    out = torch.rand(nmat, nrow, ncol, device="cuda", generator=gen) < 1e-3
    return torch.where(out, 8 * torch.sign(x), x) * sig


def source(gen, src, nmat, nrow, ncol):
    """the tensor's stored bytes (uint8, device)"""
    n = nmat * nrow * ncol
    if src == "mxfp4":      # e8m0 exponents of [-8, -4], uniform e2m1 codes
        raw = torch.randint(0, 256, (n // 32, 17), dtype=torch.uint8, device="cuda", generator=gen)
        raw[:, 0] = 127 + torch.randint(-8, -3, (n // 32,), device="cuda", generator=gen)
        return raw.reshape(-1)
    x = values(gen, nmat, nrow, ncol)
    if src == "q8_0":       # fp16 scales, int8 values
        b = x.reshape(-1, 32)
        d = (b.abs().amax(1, keepdim=True) / 127).to(torch.float16)
        q = torch.round(b / d.float().clamp_min(1e-7)).clamp(-127, 127).to(torch.int8)
        return torch.cat([d.view(torch.uint8), q.view(torch.uint8)], 1).reshape(-1)
    return x.to({"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}[src]).reshape(-1).view(torch.uint8)


def importances(gen, nmat, ncol):
    return torch.exp(torch.randn(nmat, ncol, device="cuda", generator=gen) * 1.5).contiguous()


def activations(gen, nrows, ne0):
    """heavy-tailed activations (Student-t, four degrees of freedom), each column with its own scale"""
    z = torch.randn(nrows, ne0, device="cuda", generator=gen)
    chi = torch.randn(nrows, ne0, device="cuda", generator=gen) ** 2
    for _ in range(3):
        chi += torch.randn(nrows, ne0, device="cuda", generator=gen) ** 2
    return z / torch.sqrt(chi / 4) * (0.5 + torch.rand(ne0, device="cuda", generator=gen))


def hessian(case, seed):
    """the f64 sum of x x^T over ne0 + 512 activation rows, with the case's dead columns"""
    gen = generator(seed)
    x = activations(gen, case["ne0"] + 512, case["ne0"]).double()
    if case["dead"]:
        x[:, torch.randperm(case["ne0"], device="cuda", generator=gen)[:case["dead"]]] = 0
    return x.T.contiguous() @ x, case["ne0"] + 512


def prepare(case, seed):
    gq, gen, op = lib(), generator(seed), case["op"]
    s = {"case": case, "gq": gq}
    if op in ("device", "host"):
        nmat, nrow, ncol = case["nmat"], case["nrow"], case["ncol"]
        s["raw"] = source(gen, case["src"], nmat, nrow, ncol)
        s["imatrix"] = importances(gen, nmat, ncol) if case["imatrix"] else None
        nbytes = nmat * nrow * ncol // block(case["type"]) * BLOCK_BYTES[case["type"]]
        if op == "device":
            s["out"] = torch.empty(nbytes, dtype=torch.uint8, device="cuda")
        else:               # a program on the host: pageable buffers
            s["raw"] = s["raw"].cpu().numpy()
            s["imatrix"] = s["imatrix"].cpu().numpy() if case["imatrix"] else None
            s["out"] = np.zeros(nbytes, dtype=np.uint8)
    elif op == "blocks":
        # a column of blocks of one matrix: all weighted by a row of eight blocks' importances
        s["x"] = values(gen, 1, case["nblocks"], 256).reshape(-1).contiguous()
        s["imatrix"] = importances(gen, 1, 2048) if case["imatrix"] else None
        s["out"] = torch.empty(case["nblocks"] * BLOCK_BYTES[case["type"]], dtype=torch.uint8, device="cuda")
    elif op == "to_float":
        # blocks as the quantizer writes them: up to 4096 of them made from weights, repeated
        typ, nb = TYPES[case["type"]], min(case["nblocks"], 4096)
        x = values(gen, 1, nb, 256).reshape(-1).contiguous()
        im = importances(gen, 1, 256)
        q = torch.empty((nb, BLOCK_BYTES[case["type"]]), dtype=torch.uint8, device="cuda")
        assert gq.gpuq_quantize_dev(typ, x.data_ptr(), q.data_ptr(), nb, im.data_ptr(), 1, 1, stream()) == q.numel()
        s["q"] = q.repeat((case["nblocks"] + nb - 1) // nb, 1)[:case["nblocks"]].contiguous()
        s["out"] = torch.empty(case["nblocks"] * 256, dtype=torch.float32, device="cuda")
    elif op == "src_to_float":
        s["raw"] = source(gen, case["src"], 1, case["n"] // 32, 32)
        s["out"] = torch.empty(case["n"], dtype=torch.float32, device="cuda")
    elif op == "ldlq":
        nmat, ne1, ne0 = case["nmat"], case["ne1"], case["ne0"]
        s["W"] = values(gen, nmat, ne1, ne0)
        # a factor with the entries that a Hessian of a few thousand activation rows gives
        u = torch.randn(nmat if case["own"] else 1, ne0, ne0, dtype=torch.float64, device="cuda", generator=gen) / 90
        u = torch.triu(u, 1)
        u.diagonal(dim1=1, dim2=2).copy_(0.7 + 0.7 * torch.rand(u.shape[:2], dtype=torch.float64, device="cuda",
                                                                generator=gen))
        s["U"] = u if case["own"] else u[0]
        # the blocks in an order of descending energy: here any order
        order = torch.randperm(ne0 // 256, generator=generator(seed, "cpu")).numpy()
        s["perm"] = (order[:, None] * 256 + np.arange(256)[None]).reshape(-1)
        s["qw"] = importances(gen, nmat, ne0)
    elif op == "hessian_add":
        s["X"] = activations(gen, case["nrows"], case["ne0"])
    elif op == "hessian_factor":
        s["H"], s["n"] = hessian(case, seed)
        s["U"] = torch.empty_like(s["H"])
    else:
        ne0 = case["ne0"]
        u = torch.triu(torch.randn(ne0, ne0, dtype=torch.float64, device="cuda", generator=gen) / 90, 1)
        u.diagonal().copy_(0.7 + 0.7 * torch.rand(ne0, dtype=torch.float64, device="cuda", generator=gen))
        s["U"] = u
    return s


def done(got, want):
    if got != want:
        raise RuntimeError("the library answered %d, not %d" % (got, want))


def run(s):
    gq, case, op = s["gq"], s["case"], s["case"]["op"]
    if op == "device":
        im = s["imatrix"]
        done(gq.gpuq_requantize_dev(SOURCES[case["src"]], s["raw"].data_ptr(), TYPES[case["type"]],
                                    s["out"].data_ptr(), case["nmat"], case["nrow"], case["ncol"],
                                    None if im is None else im.data_ptr(), stream()), s["out"].numel())
        return s["out"]
    if op == "host":
        im = s["imatrix"]
        done(gq.gpuq_requantize_batch(SOURCES[case["src"]], s["raw"].ctypes.data, TYPES[case["type"]],
                                      s["out"].ctypes.data, case["nmat"], case["nrow"], case["ncol"],
                                      None if im is None else im.ctypes.data), s["out"].nbytes)
        return s["out"]
    if op == "blocks":
        im = s["imatrix"]
        done(gq.gpuq_quantize_dev(TYPES[case["type"]], s["x"].data_ptr(), s["out"].data_ptr(), case["nblocks"],
                                  None if im is None else im.data_ptr(), 8, 1, stream()), s["out"].numel())
        return s["out"]
    if op == "to_float":
        done(gq.gpuq_dequantize_dev(TYPES[case["type"]], s["q"].data_ptr(), s["out"].data_ptr(), case["nblocks"],
                                    stream()), s["out"].numel() * 4)
        return s["out"]
    if op == "src_to_float":
        done(gq.gpuq_dequantize_src_dev(SOURCES[case["src"]], s["raw"].data_ptr(), s["out"].data_ptr(), case["n"],
                                        stream()), case["n"] * 4)
        return s["out"]
    if op == "ldlq":
        return ldlq.quantize_matrix_dev(gq, TYPES[case["type"]], s["W"], s["U"], s["perm"], s["qw"],
                                        u_per_matrix=case["own"])
    if op == "hessian_add":     # a Hessian's first chunk
        H = torch.zeros(case["ne0"], case["ne0"], dtype=torch.float64, device="cuda")
        done(gq.gpuq_hessian_accumulate_dev(s["X"].data_ptr(), case["nrows"], case["ne0"], H.data_ptr(), stream()), 0)
        return H
    if op == "hessian_factor":
        ne0 = case["ne0"]
        perm, diag_n = np.empty(ne0, dtype=np.int64), np.empty(ne0, dtype=np.float64)
        dead = np.empty(ne0, dtype=np.uint8)
        done(gq.gpuq_prepare_hessian_dev(s["H"].data_ptr(), ne0, float(s["n"]), 0.01,
                                         1 if case["order"] == "act" else 0, s["U"].data_ptr(), perm.ctypes.data,
                                         diag_n.ctypes.data, dead.ctypes.data, stream()), 0)
        return {"U": s["U"], "perm": perm, "diag_n": diag_n, "dead": dead}
    return ldlq.schur_weights_dev(gq, s["U"], nrep=case["nrep"])


def tolerance(case):
    if case["op"] == "hessian_add":      # f64 sums over the rows in another order (measured 5e-16, 6e-15)
        return {"rel": 2e-15, "max": 2.5e-14}
    if case["op"] == "hessian_factor":   # the factor by way of the inverse against one without (1.6e-14, 2.5e-13)
        return {"rel": 6e-14, "max": 1e-12}
    return "exact"          # ggml's bytes, its floats bit for bit, and the LDLQ loop's fixed-order sums


def exact(case, seed):
    if case["op"] == "hessian_add":
        x = activations(generator(seed), case["nrows"], case["ne0"]).double().cpu()
        return x.T.contiguous() @ x
    if case["op"] == "hessian_factor":
        H, n = hessian(case, seed)
        H = H.cpu().numpy() / float(n)
        ne0 = case["ne0"]
        d = np.diag(H).copy()
        dead = d <= 0
        d[dead] = 1.0
        H[dead, :] = 0
        H[:, dead] = 0
        H[np.diag_indices(ne0)] = d
        order = np.arange(ne0 // 256)
        if case["order"] == "act":
            order = np.argsort(-d.reshape(-1, 256).sum(1), kind="stable")
        perm = (order[:, None] * 256 + np.arange(256)[None]).reshape(-1)
        Hp = H[np.ix_(perm, perm)]
        Hp[np.diag_indices(ne0)] += 0.01 * d[perm].mean()
        # Hp = V V^T with V upper: the Cholesky factor of the matrix read backwards; U = V^-1 (no inverse is formed)
        L = torch.linalg.cholesky(torch.from_numpy(np.ascontiguousarray(Hp[::-1, ::-1])))
        V = torch.flip(L, (0, 1))
        U = torch.linalg.solve_triangular(V, torch.eye(ne0, dtype=torch.float64), upper=True)
        return {"U": U, "perm": perm, "diag_n": d[perm], "dead": dead.astype(np.uint8)}
    return None
