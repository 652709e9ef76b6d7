"""The work whose speed counts: calls of the public entry points as a program
that keeps FP8 tensors compressed makes them (add two encodings, decode one,
multiply by an encoded matrix, encode a tensor or a matrix).

listed() holds named cases, draw() more of the same ranges; prepare() makes
what such a program holds before the call, run() is one call, work() what the
call cannot do without, exact() the result in 64 bits by plain torch.

Data: N(0, 0.02) scaled so that |max| maps to 448 and cast to E4M3FN (the
benchmark's inputs), encoded with a table of the data's own exponent
histogram.  Products and decodes take data drawn for each seed; the encoders'
inputs differ by seed in the order of their rows and in their signs.
"""
import math
import os
import sys

import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(_ROOT, "tans-vectoradd_amd"))

import rans_vectoradd as R  # noqa: E402
from rans_vectoradd import tans_codec as T  # noqa: E402

HIST_SAMPLE = 1 << 24   # elements the exponent histogram is taken from


def listed():
    return [
        # -- fused add: K lanes of N elements per operand -----------------
        # the smallest call of the test programs: latency and launches
        {"name": "add_256x256", "op": "add", "K": 256, "N": 256, "alphabet": "pair"},
        # one ordinary tensor of 16 Mi elements in the default lane length
        {"name": "add_16mi", "op": "add", "K": 16384, "N": 1024, "alphabet": "pair"},
        # the headline: 512 Mi elements per operand, 64 Ki-element streams
        {"name": "add_512mi", "op": "add", "K": 524288, "N": 1024, "alphabet": "pair"},
        # the shortest streams of the benchmark's sweep, an odd lane count
        {"name": "add_short_odd", "op": "add", "K": 1500007, "N": 16, "alphabet": "pair"},
        # -- standalone decode --------------------------------------------
        # a mid-size tensor whose lanes fill no whole tiles and no whole
        # group, the 16-symbol alphabet
        {"name": "decode_odd_nibble", "op": "decode", "K": 10007, "N": 1000, "alphabet": "nibble"},
        # the benchmark's decode: 1 Gi elements
        {"name": "decode_1gi", "op": "decode", "K": 1 << 20, "N": 1024, "alphabet": "pair"},
        # -- matrix times a few rows of activations ------------------------
        # one token through the up projection of the benchmark's layers
        {"name": "gemv_up", "op": "gemm", "R": 17408, "C": 5120, "B": 1, "alphabet": "pair"},
        # eight tokens through the down projection
        {"name": "gemm_down_b8", "op": "gemm", "R": 5120, "C": 17408, "B": 8, "alphabet": "pair"},
        # a small projection, three tokens, the 16-symbol alphabet
        {"name": "gemm_small", "op": "gemm", "R": 2176, "C": 1280, "B": 3, "alphabet": "nibble"},
        # -- encode on the GPU ----------------------------------------------
        # a large tensor in the default lane length
        {"name": "encode_512mi", "op": "encode", "K": 524288, "N": 1024, "alphabet": "pair"},
        # a weight matrix of a checkpoint (layout and encoding)
        {"name": "encode_matrix_up", "op": "encode_matrix", "R": 17408, "C": 5120,
         "alphabet": "pair"},
        # short streams (64 elements per lane), an odd lane count
        {"name": "encode_short_odd", "op": "encode", "K": 262147, "N": 64, "alphabet": "pair"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(("add", "add", "decode", "decode", "gemm", "gemm", "encode", "encode",
                     "encode_matrix"))
    alphabet = rng.choice(("pair", "pair", "nibble"))
    if op in ("gemm", "encode_matrix"):
        rows = _log_int(rng, 256, 17408)
        cols = _log_int(rng, 256, 17408)
        cols = min(cols, 17408 * 5120 // rows)
        case = {"op": op, "R": rows, "C": cols, "alphabet": alphabet}
        if op == "gemm":
            case["B"] = rng.randint(1, 8)
        return case
    # lanes of 16 to 4096 elements; whole 16-element tiles for the add (its
    # entry point takes no others) and for half of the other calls
    n = _log_int(rng, 16, 4096)
    n = n // 16 * 16 if op == "add" or rng.random() < 0.5 else n // 2 * 2
    most = {"add": 1 << 28, "decode": 1 << 28, "encode": 1 << 26}[op]
    total = _log_int(rng, 1 << 16, most)
    return {"op": op, "K": max(1, total // n), "N": n, "alphabet": alphabet}


# ---------------------------------------------------------------------------


def _bytes(n, seed):
    """n E4M3FN bytes on the GPU and the scale that brings them back."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn(n, generator=g, device="cuda").mul_(0.02)
    amax = x.abs().max()
    q = x.mul_(448.0 / amax).clamp_(-448.0, 448.0).to(torch.float8_e4m3fn)
    return q.view(torch.uint8), float(amax) / 448.0


def _hist(*qs):
    """Exponent histogram (every exponent counted once more, so that none
    the sample lacks is left without a code)."""
    h = torch.ones(16, dtype=torch.float64, device="cuda")
    for q in qs:
        e = (q[:HIST_SAMPLE] >> 3) & 15
        h += torch.bincount(e.to(torch.int32), minlength=16).to(torch.float64)
    return h.cpu()


def _lane_bytes(case, seed, count):
    n = case["K"] * case["N"]
    return [_bytes(n, 2 * seed + i)[0] for i in range(count)]


def _matrix(case, seed):
    q, scale = _bytes(case["R"] * case["C"], 2 * seed)
    return q.view(case["R"], case["C"]), scale


def _rolled(q, rows, cols, block, seed):
    """The bytes to encode, [rows, cols], and their histogram: one fixed draw
    whose whole blocks of `block` rows (the rows that share a stream) are
    rolled by a distance from the seed, with sign bits from the seed.  Every
    seed's streams then have the same lengths in another order, so that the
    outputs of all seeds have the same shapes."""
    h = _hist(q)
    g = torch.Generator(device="cuda").manual_seed(2 * seed)
    sign = torch.randint(0, 2, (rows * cols,), generator=g, device="cuda", dtype=torch.uint8)
    q = (q ^ sign.mul_(128)).view(rows, cols)
    whole = rows // block * block
    if whole > block:
        blocks = whole // block
        q[:whole] = torch.roll(q[:whole], block * (1 + seed % (blocks - 1)), 0)
    return q, h


def _x(case, seed):
    g = torch.Generator(device="cuda").manual_seed(2 * seed + 1)
    return torch.randn(case["B"], case["C"], generator=g, device="cuda").to(torch.bfloat16)


def _table(enc):
    return T.build_decode_table(enc[6].cpu().numpy(), enc[5].cpu().numpy()).cuda()


def prepare(case, seed):
    op = case["op"]
    if op == "add":
        qa, qb = _lane_bytes(case, seed, 2)
        h = _hist(qa, qb)
        ea, eb = (T.encode_gpu(q.view(case["K"], case["N"]), h, alphabet=case["alphabet"])
                  for q in (qa, qb))
        order = (0, 2, 1, 3, 4)   # comp, offsets, states, partial, sign/mantissa
        return op, [ea[i] for i in order] + [eb[i] for i in order] + [_table(ea), case["N"]]
    if op == "decode":
        (q,) = _lane_bytes(case, seed, 1)
        e = T.encode_gpu(q.view(case["K"], case["N"]), _hist(q), alphabet=case["alphabet"])
        return op, [e[i] for i in (0, 2, 1, 3, 4, 6, 5)] + [case["N"]]
    if op == "gemm":
        w, scale = _matrix(case, seed)
        m = T.encode_matrix(w, _hist(w.view(-1)), alphabet=case["alphabet"])
        return op, [m, m.decode_table().cuda(), _x(case, seed), scale]
    if op == "encode":
        K, N = case["K"], case["N"]
        return op, [*_rolled(_bytes(K * N, 1)[0], K, N, 64, seed), case["alphabet"]]
    R_, C = case["R"], case["C"]
    return op, [*_rolled(_bytes(R_ * C, 1)[0], R_, C, 16, seed), case["alphabet"]]


def run(state):
    op, a = state
    if op == "add":
        return R.fp8_vecadd_fused_tans(*a)
    if op == "decode":
        return R.gpu_tans_decode(*a)
    if op == "gemm":
        return R.fp8_gemm_fused_tans(*a)
    if op == "encode":
        return list(T.encode_gpu(a[0], a[1], alphabet=a[2]))
    m = T.encode_matrix(a[0], a[1], alphabet=a[2])
    return [m.comp, m.states, m.offsets, m.partial, m.sm, m.freqs, m.spread]


# ---------------------------------------------------------------------------

# bits per FP8 byte of this data: half a byte of sign and mantissa and the
# exponent's entropy (2.55 bits)
BITS = 6.55


def work(case):
    """Bytes: the raw side at one byte per element, the encoded side at the
    data's entropy, activations and results; operations: two per product."""
    op = case["op"]
    if op in ("gemm", "encode_matrix"):
        n = case["R"] * case["C"]
        if op == "encode_matrix":
            return {"bytes": n + n * BITS / 8, "flops": 0}
        io = 2 * case["B"] * (case["R"] + case["C"])
        return {"bytes": n * BITS / 8 + io, "flops": 2 * n * case["B"]}
    n = case["K"] * case["N"]
    if op == "add":
        return {"bytes": 2 * n * BITS / 8 + n, "flops": n}
    return {"bytes": n + n * BITS / 8, "flops": 0}


def tolerance(case):
    """Bytes are bytes.  A product is rounded to bf16 (relative step 2^-8,
    error against 64 bits about 1.7e-3 in the 2-norm); sums in another order
    move some results by one step."""
    if case["op"] == "gemm":
        return {"rel": 6e-3, "max": 0.02}
    return "exact"


def exact(case, seed):
    op = case["op"]
    if op == "gemm":
        w, scale = _matrix(case, seed)
        x = _x(case, seed).double()
        parts = [x @ w[r:r + 4096].view(torch.float8_e4m3fn).to(torch.float32).double().t()
                 .contiguous() for r in range(0, case["R"], 4096)]
        return torch.cat(parts, dim=1) * scale
    if op == "add":
        K, N = case["K"], case["N"]
        qa, qb = _lane_bytes(case, seed, 2)
        out = torch.empty(K * N, dtype=torch.uint8, device="cuda")
        step = 1 << 26
        for i in range(0, K * N, step):
            a, b = (q[i:i + step].view(torch.float8_e4m3fn).to(torch.float32).double()
                    for q in (qa, qb))
            s = (a + b).clamp_(-448.0, 448.0).to(torch.float32)
            out[i:i + step] = s.to(torch.float8_e4m3fn).view(torch.uint8)
        return out.view(K, N // 16, 16).permute(1, 0, 2).contiguous().view(-1)
    if op == "decode":
        (q,) = _lane_bytes(case, seed, 1)
        return q.view(case["K"], case["N"]).t().contiguous()
    return None
