"""The launch rule that spreads groups over the CUs (spread_waves in
kernels.hip): tensors of one group, of about one group per CU, around whole
rounds of 16 waves per CU, and of two uneven rounds.  The outputs are bytes
(fused add == raw add, decode == input) or, for the GEMM, the raw kernel's
product to a bf16 step."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _say(msg):
    print(msg, flush=True)


@pytest.fixture(scope="module")
def R():
    import rans_vectoradd
    assert torch.cuda.is_available(), "GPU tests need a GPU"
    return rans_vectoradd


def _bytes(R, n, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return R.random_fp8_bytes(n, device="cuda", generator=g)


# groups of 64 lanes against 256 CUs: one, fewer than CUs, one more than CUs
# (two waves on one), a whole round of 16 and one group more or less, two
# rounds of 10 waves; the lane count ragged in each.  Up to 4 and up to 8
# waves per CU have kernels of their own for streams of any length (1500
# groups: 6 waves), whose tiles overlap: every tile count mod 4
@pytest.mark.parametrize("alphabet,N", [("pair", 16), ("pair", 48), ("pair", 80), ("pair", 96),
                                        ("pair", 112), ("pair", 128), ("pair", 144),
                                        ("nibble", 48), ("nibble", 64), ("nibble", 80),
                                        ("nibble", 96)])
@pytest.mark.parametrize("groups", [1, 100, 257, 1500, 4095, 4096, 4097, 5000])
def test_groups_spread_over_cus(R, alphabet, N, groups):
    from rans_vectoradd import tans_codec as T
    K = groups * 64 - 3
    _say(f"case: spread {groups} groups x {N} {alphabet}")
    hist = torch.tensor(R.QWEN3_14B_FP8_EXP)
    a, b = _bytes(R, K * N, groups).view(K, N), _bytes(R, K * N, groups + 1).view(K, N)
    ea, eb = (T.encode_gpu(q, hist, alphabet=alphabet) for q in (a, b))
    tbl = T.build_decode_table(ea[6].cpu().numpy(), ea[5].cpu().numpy()).cuda()
    order = (0, 2, 1, 3, 4)
    out = R.fp8_vecadd_fused_tans(*[ea[i] for i in order], *[eb[i] for i in order], tbl, N)
    raw = R.fp8_vecadd_raw(a.view(-1), b.view(-1)).view(K, N // 16, 16).permute(1, 0, 2).reshape(-1)
    assert torch.equal(out, raw)
    dec = R.gpu_tans_decode(ea[0], ea[2], ea[1], ea[3], ea[4], ea[6], ea[5], N)
    assert torch.equal(dec, a.t())


# the fused add's kernels for streams loaded whole at their start (refill
# schedule: pair up to 4 tiles, nibble up to 2), whose group switches step by
# the waves of a workgroup: 2 to 11 waves, one round, and several rounds
@pytest.mark.parametrize("alphabet,N", [("pair", 16), ("pair", 48), ("pair", 64), ("nibble", 16),
                                        ("nibble", 32)])
@pytest.mark.parametrize("groups", [257, 1500, 2600, 4096, 4097, 5000, 12300])
def test_resident_streams_spread_over_cus(R, alphabet, N, groups):
    from rans_vectoradd import tans_codec as T
    K = groups * 64 - 3
    _say(f"case: spread resident {groups} groups x {N} {alphabet}")
    hist = torch.tensor(R.QWEN3_14B_FP8_EXP)
    a, b = _bytes(R, K * N, groups).view(K, N), _bytes(R, K * N, groups + 1).view(K, N)
    ea, eb = (T.encode_gpu(q, hist, alphabet=alphabet, layout="words") for q in (a, b))
    tbl = T.build_decode_table(ea[6].cpu().numpy(), ea[5].cpu().numpy()).cuda()
    order = (0, 2, 1, 3, 4)
    out = R.fp8_vecadd_fused_tans(*[ea[i] for i in order], *[eb[i] for i in order], tbl, N)
    raw = R.fp8_vecadd_raw(a.view(-1), b.view(-1)).view(K, N // 16, 16).permute(1, 0, 2).reshape(-1)
    assert torch.equal(out, raw)


# the decoder's kernels for few waves (one group per wave up to 8 waves per CU,
# then two): rows of whole 16-byte columns (K % 16 == 0, through the staging
# rows) and others, whole and partial last groups, ragged last tiles of every
# tile count mod 4
@pytest.mark.parametrize("alphabet,N", [("pair", 82), ("pair", 104), ("pair", 128), ("pair", 130),
                                        ("nibble", 34), ("nibble", 56), ("nibble", 64),
                                        ("nibble", 90)])
@pytest.mark.parametrize("K", [64, 6400, 6384, 6397, 96000, 95997, 192000 - 48, 192001])
def test_decode_with_few_waves(R, alphabet, N, K):
    from rans_vectoradd import tans_codec as T
    _say(f"case: decode few waves {K} x {N} {alphabet}")
    a = _bytes(R, K * N, K + N).view(K, N)
    e = T.encode_gpu(a, torch.tensor(R.QWEN3_14B_FP8_EXP), alphabet=alphabet)
    dec = R.gpu_tans_decode(e[0], e[2], e[1], e[3], e[4], e[6], e[5], N)
    assert torch.equal(dec, a.t())


# row groups of 16 rows per segment: one, an odd number, more than the CUs
# of a segment's share hold in one round
@pytest.mark.parametrize("rows,cols,segments", [(16, 512, 1), (1000, 2048, 8), (8272, 288, 1),
                                                (140000, 64, 1)])
def test_gemm_row_groups_spread_over_cus(R, rows, cols, segments):
    from rans_vectoradd import tans_codec as T
    _say(f"case: spread gemm {rows}x{cols} S={segments}")
    w = _bytes(R, rows * cols, rows).view(rows, cols)
    g = torch.Generator(device="cuda").manual_seed(cols)
    x = torch.randn(3, cols, generator=g, device="cuda").to(torch.bfloat16)
    m = T.encode_matrix(w, torch.tensor(R.QWEN3_14B_FP8_EXP), segments=segments)
    y = R.fp8_gemm_fused_tans(m, m.decode_table().cuda(), x, 2.0 ** -9).float()
    y_raw = R.fp8_gemm_raw(w, x, 2.0 ** -9).float()
    # both round an fp32 sum (whose order differs by at most cols * 2^-24 of
    # the terms' magnitude) to bf16: one bf16 step (2^-7 relative) apart
    mag = (x.abs().float() @ w.view(torch.float8_e4m3fn).float().nan_to_num(0).abs().t()) * 2.0 ** -9
    same_nan = torch.isnan(y) == torch.isnan(y_raw)
    ok = (y - y_raw).abs() <= 2.0 ** -7 * y_raw.abs() + cols * 2.0 ** -23 * mag
    assert bool((same_nan & (ok | torch.isnan(y_raw))).all())


# one workgroup per row block holding every segment (B small enough for x in
# LDS) against one workgroup per segment and the separate sum (B = 8): the
# same products in the same order, so equal to the bit.  Segments 5, 7, 8, 13
# and 16, half tiles (width 32 mod 64), one to three pairs of row groups per
# workgroup, ragged rows and columns, an odd pair count
@pytest.mark.parametrize("alphabet", ["pair", "nibble"])
@pytest.mark.parametrize("rows,cols,segments,batch", [(200, 2040, 8, 5), (48, 4096, 16, 2),
                                                      (16, 1555, 5, 6), (1000, 1540, 16, 7),
                                                      (17000, 1600, 5, 3), (8300, 1537, 7, 1)])
def test_gemm_whole_rows_equal_the_segment_sums(R, alphabet, rows, cols, segments, batch):
    from rans_vectoradd import tans_codec as T
    _say(f"case: gemm whole rows {rows}x{cols} S={segments} B={batch} {alphabet}")
    w = _bytes(R, rows * cols, rows + cols).view(rows, cols)
    g = torch.Generator(device="cuda").manual_seed(cols)
    x = torch.randn(8, cols, generator=g, device="cuda").to(torch.bfloat16)
    m = T.encode_matrix(w, torch.tensor(R.QWEN3_14B_FP8_EXP), segments=segments, alphabet=alphabet)
    tbl = m.decode_table().cuda()
    y8 = R.fp8_gemm_fused_tans(m, tbl, x, 2.0 ** -9)
    y = R.fp8_gemm_fused_tans(m, tbl, x[:batch].contiguous(), 2.0 ** -9)
    assert torch.equal(y.view(torch.int16), y8[:batch].view(torch.int16))


# one segment (whose sum is no sum) with one, an odd and several pairs of row
# groups per workgroup, and the two-kernel form (140000 rows): products whose
# sums are whole numbers below 2^24, exact in any order
@pytest.mark.parametrize("alphabet", ["pair", "nibble"])
@pytest.mark.parametrize("rows,cols", [(16, 1024), (100, 95), (17000, 1000), (140000, 96)])
@pytest.mark.parametrize("batch", [1, 8])
def test_gemm_of_one_segment_is_exact(R, alphabet, rows, cols, batch):
    from rans_vectoradd import tans_codec as T
    _say(f"case: gemm one segment {rows}x{cols} B={batch} {alphabet}")
    g = torch.Generator(device="cuda").manual_seed(rows + batch)
    w = torch.randint(-4, 5, (rows, cols), generator=g, device="cuda").float()
    x = torch.randint(-8, 9, (batch, cols), generator=g, device="cuda").float()
    wq = w.to(torch.float8_e4m3fn).view(torch.uint8)
    m = T.encode_matrix(wq, torch.tensor(R.QWEN3_14B_FP8_EXP) + 1e-3, segments=1,
                        alphabet=alphabet)
    y = R.fp8_gemm_fused_tans(m, m.decode_table().cuda(), x.to(torch.bfloat16), 0.5)
    want = (x.cpu().double() @ w.cpu().double().t() * 0.5).to(torch.float32).to(torch.bfloat16)
    assert torch.equal(y.cpu(), want)


# an infinity in one row of x and a NaN in another, at the ends of segments, in
# half tiles and in the last column: those rows give infinities of W's signs
# (NaN where W is zero) and NaN, and the other rows are what they are without
# them, in one workgroup per row block (B = 3) and with the separate sum (B = 8)
@pytest.mark.parametrize("alphabet", ["pair", "nibble"])
@pytest.mark.parametrize("batch", [3, 8])
@pytest.mark.parametrize("rows,cols,segments,at", [(200, 2040, 8, 2039), (200, 2040, 8, 255),
                                                   (200, 2040, 8, 256), (100, 1537, 7, 223),
                                                   (100, 1537, 7, 1536), (33, 96, 1, 95)])
def test_gemm_infinities_and_nan_stay_in_their_row(R, alphabet, batch, rows, cols, segments, at):
    from rans_vectoradd import data as D, tans_codec as T
    _say(f"case: gemm inf/nan {rows}x{cols} S={segments} B={batch} at {at} {alphabet}")
    q, _ = D.gaussian_fp8_bytes(rows * cols, seed=rows + cols)
    q[::97] &= 0x80                       # zeros of both signs
    w = q.view(rows, cols)
    m = T.encode_matrix(w.cuda(), D.exp_histogram(q) + 1, segments=segments, alphabet=alphabet)
    tbl = m.decode_table().cuda()
    g = torch.Generator(device="cuda").manual_seed(at)
    x = torch.randn(batch, cols, generator=g, device="cuda").to(torch.bfloat16)
    clean = R.fp8_gemm_fused_tans(m, tbl, x, 0.25)
    x[0, at] = float("inf")
    x[2, at] = float("nan")
    y = R.fp8_gemm_fused_tans(m, tbl, x, 0.25)
    col = w[:, at].cuda().view(torch.float8_e4m3fn).float()
    want = torch.where(col == 0, torch.nan, torch.sign(col) * torch.inf)
    assert torch.equal(torch.isnan(y[0]), torch.isnan(want))
    ok = ~torch.isnan(want)
    assert torch.equal(y[0].float()[ok], want[ok])
    assert bool(torch.isnan(y[2]).all())
    rest = [b for b in range(batch) if b not in (0, 2)]
    assert torch.equal(y[rest].view(torch.int16), clean[rest].view(torch.int16))


# the table built in each workgroup (tans_decode_spread) against a host-built
# one (tans_decode): every decoder kernel, by alphabet, layout, tiles and waves
@pytest.mark.parametrize("alphabet,layout,N,groups", [
    ("pair", "auto", 16, 40), ("pair", "auto", 32, 40), ("pair", "auto", 48, 40),
    ("pair", "auto", 64, 40), ("pair", "words", 16, 40), ("pair", "words", 64, 40),
    ("pair", "words", 96, 40), ("pair", "words", 96, 1500), ("pair", "words", 96, 3000),
    ("pair", "words", 96, 6000), ("nibble", "words", 16, 40), ("nibble", "words", 40, 40),
    ("nibble", "words", 40, 1500), ("nibble", "words", 40, 3000), ("nibble", "words", 40, 6000)])
def test_decode_builds_the_host_table(R, alphabet, layout, N, groups):
    from rans_vectoradd import tans_codec as T
    from rans_vectoradd._lib import lib
    K = 64 * groups - 5
    _say(f"case: decode_spread {K} x {N} {alphabet} {layout}")
    a = _bytes(R, K * N, K + N).view(K, N)
    comp, st, off, _, sm, fr, sp = T.encode_gpu(a, torch.tensor(R.QWEN3_14B_FP8_EXP),
                                                alphabet=alphabet, layout=layout)
    tbl = T.build_decode_table(sp.cpu().numpy(), fr.cpu().numpy()).cuda()
    log2L = 12 if alphabet == "pair" else 11
    stream = torch.cuda.current_stream().cuda_stream
    outs = [torch.zeros((N, K), dtype=torch.uint8, device="cuda") for _ in range(2)]
    args = (comp.data_ptr(), comp.numel(), off.data_ptr(), st.data_ptr() if st.numel() else None,
            sm.data_ptr())
    assert lib.tans_decode(*args, tbl.data_ptr(), log2L, K, N, outs[0].data_ptr(), stream) == 0
    assert lib.tans_decode_spread(*args, sp.data_ptr(), fr.data_ptr(), log2L, K, N,
                                  outs[1].data_ptr(), stream) == 0
    assert torch.equal(outs[0], a.t()) and torch.equal(outs[1], a.t())
