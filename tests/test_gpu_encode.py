"""GPU encoder (tans_codec.encode_gpu) against the CPU encoder, byte for byte:
compressed words, offsets, states and sign/mantissa tiles, at the reference's
test shapes (test_gpu_decode_tans.py:69-74, seed 42, Qwen3 histogram) and
ragged ones, then GPU encode -> GPU decode round trips on config data."""
import pytest
import torch

pytestmark = pytest.mark.gpu

ALPHABETS = ["pair", "nibble"]


def _say(msg):
    print(msg, flush=True)


@pytest.fixture(scope="module")
def R():
    import rans_vectoradd
    assert torch.cuda.is_available(), "GPU tests need a GPU"
    return rans_vectoradd


def _compare(T, fp8, hist, alphabet, layout="auto"):
    cpu = T.encode(fp8, hist, alphabet=alphabet, layout=layout)
    gpu = T.encode_gpu(fp8.cuda(), hist, alphabet=alphabet, layout=layout)
    names = ("comp", "states", "offsets", "partial", "sm", "freqs", "spread")
    for name, c, g in zip(names, cpu, gpu):
        assert g.is_cuda, name
        assert torch.equal(c, g.cpu()), f"{name} differs"
    return gpu


SHAPES = [(128, 128), (1024, 128), (10000, 128), (100000, 128), (64, 2), (65, 18), (200, 130),
          (3, 1000), (1, 16), (127, 4096), (130, 30), (4096, 14), (300, 208), (70, 48),
          (2000, 20), (2000, 36), (1000, 34)]
# every shape with both alphabets; pair shapes of N <= 64 once more in the
# refill-schedule layout ("auto" gives them the packed one)
CASES = ([(a, K, N, "auto") for a in ALPHABETS for K, N in SHAPES]
         + [("pair", K, N, "words") for K, N in SHAPES if N <= 64])


@pytest.mark.parametrize("alphabet,K,N,layout", CASES)
def test_gpu_encode_matches_cpu(R, alphabet, K, N, layout):
    """The walk reads rows in 8-tile blocks (whole blocks at N = 128, 4096; a
    partial last block at 208, 48, 16); N % 16 != 0 reads unaligned tiles and
    a masked last one.  K % 64 != 0 and
    K < 64 give groups with lanes out of range; N = 2 (pair) is one step.
    N = 18, 20, 34, 36 end in a tile of one refill segment (18, 34 with both
    alphabets, 20, 36 with pairs), where the check before it is the plain
    one.  With the pair alphabet and N <= 64, layout "auto" is the packed
    layout of short streams (its own place pass)."""
    from rans_vectoradd import tans_codec as T
    _say(f"case: encode_gpu K={K} N={N} {alphabet} {layout}")
    torch.manual_seed(42)
    fp8 = R.random_fp8_bytes(K * N, device="cpu").reshape(K, N)
    _compare(T, fp8, torch.tensor(R.QWEN3_14B_FP8_EXP), alphabet, layout)


@pytest.mark.parametrize("alphabet", ALPHABETS)
@pytest.mark.parametrize("dist", ["gaussian", "laplace"])
def test_gpu_encode_config_data_roundtrip(R, alphabet, dist):
    """2^24 config data (own histogram, 1024 per lane): GPU encode == CPU
    encode, and GPU decode of the GPU encoding == the input."""
    from rans_vectoradd import data as D, tans_codec as T
    _say(f"case: encode_gpu {dist} 2^24 {alphabet}")
    n, N = 1 << 24, 1024
    gen = D.gaussian_fp8_bytes if dist == "gaussian" else D.laplace_fp8_bytes
    q, _ = gen(n, seed=9)
    fp8 = q.reshape(n // N, N)
    comp, st, off, part, sm, fr, sp = _compare(T, fp8, D.exp_histogram(q), alphabet)
    dec = R.gpu_tans_decode(comp, off, st, part, sm, sp, fr, N)
    assert torch.equal(dec.cpu(), fp8.t())


@pytest.mark.parametrize("N", [16, 64, 30])
def test_gpu_encode_packed_config_data(R, N):
    """Config-1 data (own histogram) in the packed layout of short streams,
    2^22 elements at 16, 64 and 30 elements per lane (several rounds of the
    place pass' workgroups; a ragged last tile at 30): GPU encode == CPU
    encode, and the GPU decode of it == the input."""
    from rans_vectoradd import data as D, tans_codec as T
    _say(f"case: encode_gpu packed 2^22, {N} per lane")
    K = (1 << 22) // N
    q, _ = D.gaussian_fp8_bytes(K * N, seed=N)
    fp8 = q.reshape(K, N)
    comp, st, off, part, sm, fr, sp = _compare(T, fp8, D.exp_histogram(q), "pair")
    assert st.numel() == 0
    dec = R.gpu_tans_decode(comp, off, st, part, sm, sp, fr, N)
    assert torch.equal(dec.cpu(), fp8.t())


@pytest.mark.parametrize("alphabet", ALPHABETS)
@pytest.mark.parametrize("steep", [1.0, 14.0])
@pytest.mark.parametrize("K,N", [(300, 16), (130, 64), (65, 30), (70, 130), (200, 400),
                                 (64, 128), (127, 1042), (100, 4096)])
def test_gpu_encode_tiles_past_64_bits(R, alphabet, K, N, steep):
    """Rows that cost up to the table's longest codes (uniform bytes, steep
    histogram) beside rows that cost almost nothing (one exponent): tiles
    of more than 64 bits, whose records overflow, and lanes that cross word
    boundaries in every segment or in hardly any, in one group.  With the
    steeper histogram a row of one exponent costs almost no bits, so its
    words' places fall thousands of words behind the others'.  Whole and
    ragged last tiles, one and several 8-tile blocks.  Bytes equal the CPU
    encoder's."""
    from rans_vectoradd import tans_codec as T
    _say(f"case: encode_gpu overflowing tiles K={K} N={N} {alphabet}")
    torch.manual_seed(K + N)
    hist = 2.0 ** -torch.arange(16, dtype=torch.float64)
    hist[1:] *= 2.0 ** -(steep - 1.0)
    fp8 = torch.randint(0, 256, (K, N), dtype=torch.uint8)
    fp8[::3] &= 0x87                                  # exponent 0: the shortest code
    half = torch.arange(K) % 5 == 1                   # rows that change halfway
    fp8[half, : N // 2] &= 0x87
    for layout in ("auto", "words"):
        _compare(T, fp8, hist, alphabet, layout)


@pytest.mark.parametrize("alphabet", ALPHABETS)
@pytest.mark.parametrize("groups,N", [(3072, 128), (4096, 256), (3071, 128)])
def test_gpu_encode_rows_of_whole_lines(R, alphabet, groups, N):
    """Tensors that fill the chip with 16-wave workgroups and whose rows are
    whole 128-byte lines (one and two blocks of 8 tiles, a partial last
    group), and one group fewer, which takes the other kernel: the bytes equal
    the CPU encoder's."""
    _say(f"case: encode_gpu whole lines {groups} groups x {N} {alphabet}")
    from rans_vectoradd import tans_codec as T
    K = groups * 64 - 7
    torch.manual_seed(N)
    fp8 = R.random_fp8_bytes(K * N, device="cpu").reshape(K, N)
    _compare(T, fp8, torch.tensor(R.QWEN3_14B_FP8_EXP), alphabet)


def test_gpu_encode_edge_cases(R):
    from rans_vectoradd import tans_codec as T
    exp = torch.tensor(R.QWEN3_14B_FP8_EXP)
    comp, st, off, part, sm, fr, sp = T.encode_gpu(torch.zeros((0, 16), dtype=torch.uint8).cuda(), exp)
    assert st.numel() == 0 and off.cpu().tolist() == [0] and comp.numel() == 1024
    assert int(comp.sum()) == 0
    # a symbol whose frequency is 0 is reported, as by the CPU encoder
    hist = torch.zeros(16)
    hist[7] = 1.0
    fp8 = torch.full((64, 32), 7 << 3, dtype=torch.uint8)
    fp8[5, 3] = 9 << 3
    with pytest.raises(RuntimeError, match="frequency is 0"):
        T.encode_gpu(fp8.cuda(), hist, alphabet="nibble")
    # a misaligned view (row offset of 2 bytes) encodes like a fresh copy
    torch.manual_seed(5)
    big = R.random_fp8_bytes(65 * 34, device="cpu").reshape(65, 34)
    view = big.cuda().reshape(-1)[2:2 + 64 * 34].reshape(64, 34)
    assert view.data_ptr() % 16 != 0
    a = T.encode_gpu(view, exp)
    b = T.encode(view.cpu().contiguous(), exp)
    assert torch.equal(a[0].cpu(), b[0]) and torch.equal(a[4].cpu(), b[4])
    with pytest.raises(ValueError):
        T.encode_gpu(torch.zeros((4, 16), dtype=torch.uint8), exp)       # CPU tensor
    with pytest.raises(ValueError):
        T.encode_gpu(torch.zeros((4, 15), dtype=torch.uint8).cuda(), exp)


@pytest.mark.parametrize("alphabet", ["pair", "nibble"])
@pytest.mark.parametrize("rows,cols,segments", [(17408, 5120, None), (5120, 17408, None),
                                                (100, 70, None), (130, 1000, 3), (1, 32, None)])
def test_encode_matrix_on_gpu_equals_cpu(R, alphabet, rows, cols, segments):
    """encode_matrix of a GPU tensor (padding, lane layout and encoder on the
    GPU) gives the CPU encoder's bytes, at config 3/4's shapes and ragged
    ones."""
    from rans_vectoradd import data as D, tans_codec as T
    _say(f"case: encode_matrix on GPU {rows}x{cols} S={segments} {alphabet}")
    q, _ = D.gaussian_fp8_bytes(rows * cols, seed=rows + cols)
    w = q.reshape(rows, cols)
    hist = D.exp_histogram(q)
    a = T.encode_matrix(w.cuda(), hist, segments=segments, alphabet=alphabet)
    b = T.encode_matrix(w, hist, segments=segments, alphabet=alphabet)
    assert a.comp.is_cuda and (a.segments, a.seg_cols) == (b.segments, b.seg_cols)
    for part in ("comp", "states", "offsets", "sm", "freqs", "spread"):
        assert torch.equal(getattr(a, part).cpu(), getattr(b, part)), part


@pytest.mark.parametrize("alphabet", ALPHABETS)
@pytest.mark.parametrize("rows,cols,segments", [(16, 16, 1), (17, 17, 1), (65, 95, 2), (64, 96, 1),
                                                (63, 1033, None), (200, 4100, None), (3, 40, 2),
                                                (64, 2048, 2), (10, 8, 1)])
def test_encode_matrix_reads_w_in_place(R, alphabet, rows, cols, segments):
    """The walk reads W's rows where they lie: columns that end inside a
    16-column chunk, a half tile or a segment, odd row lengths (unaligned
    rows), rows past R, a segment whose width is one half tile, fewer columns
    than a chunk, and a matrix that starts at an odd address and ends with its
    storage.  Bytes equal the CPU encoder's."""
    from rans_vectoradd import data as D, tans_codec as T
    _say(f"case: encode_matrix in place {rows}x{cols} S={segments} {alphabet}")
    q, _ = D.gaussian_fp8_bytes((rows + 1) * cols, seed=rows * cols)
    w = q[cols:].reshape(rows, cols)
    hist = D.exp_histogram(q) + 1
    big = q.cuda()
    for wg in (w.cuda(), big[cols:].view(rows, cols), w.t().contiguous().cuda().t()):
        a = T.encode_matrix(wg, hist, segments=segments, alphabet=alphabet)
        b = T.encode_matrix(w, hist, segments=segments, alphabet=alphabet)
        for part in ("comp", "states", "offsets", "sm", "freqs", "spread"):
            assert torch.equal(getattr(a, part).cpu(), getattr(b, part)), part


def test_checkpoint_container_on_gpu(R, tmp_path):
    """A checkpoint encoded with the GPU encoder into a container, loaded on
    the GPU: the lane tensor decodes to its bytes and the matrix gives the
    same product as the raw FP8 kernel."""
    import os
    from safetensors.torch import save_file
    from rans_vectoradd import container, data as D, ingest
    _say("case: checkpoint -> container -> GPU")
    w, scale = D.gaussian_fp8_bytes(1024 * 512, seed=21)
    v, _ = D.laplace_fp8_bytes(1 << 16, seed=22)
    src = os.path.join(tmp_path, "ckpt.safetensors")
    dst = os.path.join(tmp_path, "ckpt.tans.safetensors")
    save_file({"w": w.reshape(1024, 512).view(torch.float8_e4m3fn),
               "v": v.view(torch.float8_e4m3fn)}, src)
    ingest.encode_checkpoint(src, dst, device="cuda")
    got = container.load(dst, device="cuda")
    vec = got["v"]
    dec = R.gpu_tans_decode(vec.comp, vec.offsets, vec.states, vec.partial, vec.sm, vec.spread,
                            vec.freqs, vec.N)
    assert torch.equal(dec.t().reshape(-1).cpu(), v)
    m = got["w"]
    x = torch.randn(3, 512, generator=torch.Generator().manual_seed(3)).to(torch.bfloat16).cuda()
    y = R.fp8_gemm_fused_tans(m, m.decode_table().cuda(), x, scale).float()
    y_raw = R.fp8_gemm_raw(w.reshape(1024, 512).cuda(), x, scale).float()
    assert bool(((y - y_raw).abs() <= 2.0 ** -7 * y_raw.abs() + 1e-6).all())


def _tables(T, lib, hist, alphabet):
    freqs = T.symbol_freqs(hist.numpy(), alphabet)
    spread = T.build_spread(freqs)
    nsym, L, _ = T.ALPHABETS[alphabet]
    tab, nxt = torch.empty(nsym, dtype=torch.int32), torch.empty(L, dtype=torch.int16)
    assert lib.tans_build_encode_table(spread.ctypes.data, freqs.ctypes.data, nsym,
                                       L.bit_length() - 1, tab.data_ptr(), nxt.data_ptr()) == 0
    return tab.cuda(), nxt.cuda(), L.bit_length() - 1


@pytest.mark.parametrize("alphabet,layout", [("pair", "words"), ("pair", "packed"),
                                             ("nibble", "words")])
def test_gpu_encode_begin_reports_through_status(R, alphabet, layout):
    """tans_gpu_encode_begin and tans_gpu_encode_packed_begin with their
    finish: the bytes of encode_gpu; the status word stays 0 on good data and
    becomes TANS_ESYMBOL (-3) for a symbol of frequency 0; no lanes give
    offsets {0}."""
    from rans_vectoradd import tans_codec as T
    from rans_vectoradd._lib import lib
    packed = layout == "packed"
    K, N = 517, 64
    _say(f"case: encode begin with status {alphabet} {layout}")
    hist = torch.tensor(R.QWEN3_14B_FP8_EXP)
    hist[0] = 0.0
    torch.manual_seed(3)
    good = R.random_fp8_bytes(K * N, device="cpu").reshape(K, N)
    good[((good >> 3) & 15) == 0] |= 1 << 3       # (no exponent 0)
    want = T.encode_gpu(good.cuda(), hist, alphabet=alphabet, layout=layout)
    bad = good.clone()
    bad[516, 63] &= 0x87                          # the last lane's last element
    tab, nxt, log2L = _tables(T, lib, hist, alphabet)
    stream = torch.cuda.current_stream().cuda_stream
    ws = torch.empty(1 << 20, dtype=torch.uint8, device="cuda")
    off = torch.empty(-(-K // 64) + 1, dtype=torch.int64, device="cuda")
    st = torch.empty(0 if packed else K, dtype=torch.uint16, device="cuda")
    sm = torch.empty_like(want[4])

    def begin(x, status, lanes=K):
        args = (x.data_ptr(), lanes, N, tab.data_ptr(), nxt.data_ptr(), log2L, ws.data_ptr(),
                ws.numel(), off.data_ptr())
        out = (sm.data_ptr(), status.data_ptr(), stream)
        if packed:
            return lib.tans_gpu_encode_packed_begin(*args, *out)
        return lib.tans_gpu_encode_begin(*args, st.data_ptr(), *out)

    status = torch.zeros(1, dtype=torch.int32, device="cuda")
    x = good.cuda()
    assert begin(x, status) == 0 and status.item() == 0
    comp = torch.empty((int(off[-1]) + 256) * 4, dtype=torch.uint8, device="cuda")
    finish = lib.tans_gpu_encode_packed_finish if packed else lib.tans_gpu_encode_finish
    assert finish(K, N, log2L, ws.data_ptr(), off.data_ptr(), comp.data_ptr(), comp.numel(),
                  stream) == 0
    for a, b in zip((comp, st, off, sm), (want[0], want[1], want[2], want[4])):
        assert torch.equal(a.cpu(), b.cpu())
    x = bad.cuda()
    assert begin(x, status) == 0 and status.item() == -3
    status.zero_()
    off.fill_(9)
    assert begin(x, status, 0) == 0 and status.item() == 0 and off[0].item() == 0


# every walk that marks a symbol of frequency 0: a tensor's rows per lane and
# as whole lines, with both alphabets, ragged rows, the packed layout; the mark
# is set by the first and by the last lane, in the walk's first tile (the row's
# last) and in its last one, and cleared for the same data without the symbol
@pytest.mark.parametrize("alphabet,K,N,layout", [
    ("pair", 300, 208, "words"), ("pair", 65, 18, "words"), ("pair", 300, 64, "packed"),
    ("pair", 130, 2, "packed"), ("pair", 3072 * 64 - 7, 128, "words"), ("nibble", 130, 90, "words"),
    ("nibble", 3072 * 64 - 7, 128, "words")])
def test_gpu_encode_marks_frequency_zero(R, alphabet, K, N, layout):
    from rans_vectoradd import tans_codec as T
    _say(f"case: frequency 0 K={K} N={N} {alphabet} {layout}")
    hist = torch.zeros(16)
    hist[5:9] = torch.tensor([1.0, 2.0, 3.0, 4.0])
    g = torch.Generator().manual_seed(K)
    x = torch.randint(0, 256, (K, N), dtype=torch.uint8, generator=g)
    x = ((x & 0x87) | (5 + ((x >> 3) & 3)) << 3).cuda()
    want = [t.cpu() for t in T.encode_gpu(x, hist, alphabet=alphabet, layout=layout)]
    for k, n in ((0, 0), (K - 1, N - 1), (K // 2, N // 2), (K - 1, 0)):
        kept = x[k, n].clone()
        x[k, n] = 12 << 3
        with pytest.raises(RuntimeError, match="frequency is 0"):
            T.encode_gpu(x, hist, alphabet=alphabet, layout=layout)
        x[k, n] = kept
    for a, b in zip(want, T.encode_gpu(x, hist, alphabet=alphabet, layout=layout)):
        assert torch.equal(a, b.cpu())


# the same for a matrix: its corners and the last column of a segment, where
# rows and columns are padded and the last block is a half tile
@pytest.mark.parametrize("alphabet", ALPHABETS)
@pytest.mark.parametrize("rows,cols,segments", [(70, 95, 1), (64, 256, 2), (10, 8, 1)])
def test_encode_matrix_marks_frequency_zero(R, alphabet, rows, cols, segments):
    from rans_vectoradd import tans_codec as T
    _say(f"case: matrix frequency 0 {rows}x{cols} {alphabet}")
    hist = torch.zeros(16)
    hist[5:9] = torch.tensor([1.0, 2.0, 3.0, 4.0])
    g = torch.Generator().manual_seed(rows)
    w = torch.randint(0, 256, (rows, cols), dtype=torch.uint8, generator=g)
    w = ((w & 0x87) | (5 + ((w >> 3) & 3)) << 3).cuda()
    want = T.encode_matrix(w, hist, segments=segments, alphabet=alphabet)
    for r, c in ((0, 0), (rows - 1, cols - 1), (0, want.seg_cols - 1), (rows - 1, cols // 2)):
        if c >= cols:
            continue
        kept = w[r, c].clone()
        w[r, c] = 12 << 3
        with pytest.raises(RuntimeError, match="frequency is 0"):
            T.encode_matrix(w, hist, segments=segments, alphabet=alphabet)
        w[r, c] = kept
    again = T.encode_matrix(w, hist, segments=segments, alphabet=alphabet)
    for part in ("comp", "states", "offsets", "sm"):
        assert torch.equal(getattr(want, part).cpu(), getattr(again, part).cpu()), part
