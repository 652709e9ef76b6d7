"""The product's CPU codec (libtans_amd.so: split, tables, encoder) checked
against the oracle, CPU only.

The wave64 lane layout the encoder writes is decoded by the oracle's
independent C checker (oracle.c section 3), which shares no code with the
product and also verifies the layout invariants (final states, stream
padding, unread bits)."""
import os

import numpy as np
import pytest
import torch

from oracle import oracle as O
from gemm_layout import gemm_lane_coords

GOLDEN = np.load(os.path.join(os.path.dirname(__file__), "golden", "reference_vectors.npz"))
ALPHABETS = {"pair": (12, 2), "nibble": (11, 1)}


@pytest.fixture(scope="module")
def T():
    from rans_vectoradd import tans_codec
    return tans_codec


# (alphabet, layout): the refill-schedule layout of both alphabets and, for
# lanes of at most 64 elements, the packed layout ("auto" picks it there)
CODECS = [("pair", "words"), ("pair", "auto"), ("nibble", "auto")]


def _encode_check(T, fp8, exp_freqs, alphabet, layout="auto"):
    K, N = fp8.shape
    log2L, sps = ALPHABETS[alphabet]
    enc = T.encode(fp8, exp_freqs, alphabet=alphabet, layout=layout)
    assert (enc[1].numel() == 0) == (K > 0 and T.packed_layout(N, alphabet, layout))
    dec = O.layout_decode(enc, K, N, log2L, sps)
    assert np.array_equal(dec, fp8.numpy())
    return enc


def test_quantize_freqs_matches_reference_golden(T):
    assert np.array_equal(T.quantize_freqs(GOLDEN["qf_pair_qwen_in"], 4096), GOLDEN["qf_pair_qwen_out"])
    invalid = 0
    for i in range(7):
        probs = GOLDEN[f"qf_case{i}_in"]
        want = GOLDEN[f"qf_case{i}_out"]
        tgt = int(GOLDEN[f"qf_case{i}_target"][0])
        got = T.quantize_freqs(probs, target=tgt)
        if want.min() >= 0:
            assert np.array_equal(got, want), f"case {i}"
        else:
            # the reference returned a negative frequency for a p == 0
            # symbol; the product keeps it at 0 and shrinks a live symbol
            invalid += 1
            assert got.sum() == tgt and np.array_equal(got == 0, probs == 0), f"case {i}"
            assert (got[probs > 0] >= 1).all()
    assert invalid == 1                     # golden case 3


@pytest.mark.parametrize("alphabet", list(ALPHABETS))
def test_symbol_freqs_and_spread_match_oracle(T, alphabet):
    from rans_vectoradd import data as D
    f = T.symbol_freqs(D.QWEN3_14B_FP8_EXP, alphabet)
    L = 1 << ALPHABETS[alphabet][0]
    p = np.asarray(D.QWEN3_14B_FP8_EXP, dtype=np.float32)
    p = p / p.sum()
    if alphabet == "pair":
        p = (p[:, None] * p[None, :]).reshape(-1)
    q = O.quantize_freqs(p, L).astype(np.int64)
    if alphabet == "nibble":
        # the floor of the 3-3-2 refill schedule: the two frequency-1
        # exponents go to 2, and the two units come off the largest (556)
        assert sorted(np.flatnonzero(q == 1).tolist()) == [0, 1]
        q[q == 1] = 2
        q[int(np.argmax(q))] -= 2
    assert np.array_equal(f, q)
    assert np.array_equal(T.build_spread(f), O.build_spread(f, L))


def test_floor_freqs(T):
    """Present symbols below the floor are raised to it; the units come off
    the largest frequencies one at a time (lowest index on ties), absent
    symbols stay absent, and the total is kept."""
    assert T.floor_freqs([1, 1, 5, 5], 2).tolist() == [2, 2, 4, 4]
    assert T.floor_freqs([0, 1, 7, 8], 2).tolist() == [0, 2, 7, 7]
    assert T.floor_freqs([3, 0, 2, 11], 2).tolist() == [3, 0, 2, 11]
    assert T.floor_freqs([1, 1, 1, 13], 4).tolist() == [4, 4, 4, 4]
    with pytest.raises(ValueError):
        T.floor_freqs([1, 1, 1, 1], 2)


def test_absent_exponent_gives_valid_pair_table(T):
    """An exponent that never occurs makes 31 pair symbols impossible.  The
    reference's fix-up rule can then shrink one of them to -1 (the oracle,
    restating it, does); the product never shrinks a zero-probability
    symbol, and agrees with the oracle whenever the oracle's result is
    valid."""
    from rans_vectoradd import data as D
    torch.manual_seed(3)
    fp8 = D.random_fp8_bytes(64 * 256, device="cpu")
    e = (fp8 >> 3) & 0xF
    fp8 = torch.where(e == 0, fp8 | (1 << 3), fp8)          # exponent 0 -> 1
    hist = D.exp_histogram(fp8)
    assert hist[0] == 0
    p = hist.numpy().astype(np.float32)
    p = p / p.sum()
    pp = (p[:, None] * p[None, :]).reshape(-1)
    ref = O.quantize_freqs(pp, 4096)
    got = T.symbol_freqs(hist, "pair")
    assert got.sum() == 4096 and got.min() >= 0
    assert np.array_equal(got == 0, pp == 0)
    if ref.min() >= 0:
        assert np.array_equal(got, ref)
    else:                                   # the reference's rule failed here
        assert np.array_equal(got[pp > 0] >= 1, np.ones((pp > 0).sum(), bool))
    _encode_check(T, fp8.reshape(64, 256), hist, "pair")
    # cases where the reference's result is valid are unchanged
    for i in range(7):
        probs = GOLDEN[f"qf_case{i}_in"]
        tgt = int(GOLDEN[f"qf_case{i}_target"][0])
        ref_i = O.quantize_freqs(probs, tgt)
        if ref_i.min() >= 0:
            assert np.array_equal(T.quantize_freqs(probs, tgt), ref_i)


@pytest.mark.parametrize("alphabet", list(ALPHABETS))
def test_decode_table_matches_oracle_slot_table(T, alphabet):
    from rans_vectoradd import data as D
    log2L, sps = ALPHABETS[alphabet]
    L = 1 << log2L
    f = T.symbol_freqs(D.QWEN3_14B_FP8_EXP, alphabet)
    sp = T.build_spread(f)
    tbl = T.build_decode_table(sp, f).numpy().view(np.uint32).reshape(L, 2)
    sym, nb, base = O.slot_table(sp, f, L)
    assert np.array_equal(tbl[:, 0] & 0xFF, nb)
    assert np.array_equal(tbl[:, 1], (base - L) * 8)
    e0 = sym >> 4 if sps == 2 else sym
    assert np.array_equal((tbl[:, 0] >> 11) & 0xF, e0)
    if sps == 2:
        assert np.array_equal((tbl[:, 0] >> 19) & 0xF, sym & 0xF)


@pytest.mark.parametrize("alphabet,layout", CODECS)
@pytest.mark.parametrize("K,N", [(128, 128), (1024, 128), (10000, 128), (64, 2), (65, 18),
                                 (200, 130), (3, 1000), (1, 16), (127, 4096), (130, 64),
                                 (63, 46)])
def test_encode_roundtrip_reference_test_cases(T, alphabet, layout, K, N):
    """Cases of the reference's test_gpu_decode_tans.py:69-74 (seed 42, Qwen3
    histogram) plus ragged shapes: K not a multiple of 64, N not a multiple of
    16, a single lane, N = 2."""
    from rans_vectoradd import data as D
    torch.manual_seed(42)
    fp8 = D.random_fp8_bytes(K * N, device="cpu").reshape(K, N)
    comp, st, off, part, sm, fr, sp = _encode_check(T, fp8, torch.tensor(D.QWEN3_14B_FP8_EXP),
                                                    alphabet, layout)
    off = off.numpy()
    assert off[0] == 0 and (np.diff(off) >= 0).all() and (off % 4 == 0).all()
    words = comp.numpy().view(np.uint32)
    assert (words[off[-1]:] == 0).all() and words.size - off[-1] == 256   # zero tail
    assert part.numel() == 0
    assert sm.shape == ((N + 15) // 16, K, 8)


@pytest.mark.parametrize("alphabet,N", [("pair", 18), ("pair", 20), ("pair", 36),
                                         ("nibble", 18), ("nibble", 34), ("pair", 22),
                                         ("nibble", 20)])
def test_encode_roundtrip_last_tile_of_one_segment(T, alphabet, N):
    """Streams whose last 16-element tile holds a single segment (pair: N %
    16 = 2 or 4, nibble: N % 16 = 2), where the check after the
    second-to-last segment is the plain one, and two neighbours where it is
    the final one; uniformly random bytes with the (mismatched) Qwen3
    table, so lanes end that segment holding every number of bits.  The
    oracle's checker decodes the CPU encoder's streams, consuming every
    word and bit."""
    from rans_vectoradd import data as D
    K = 2000
    g = torch.Generator().manual_seed(N)
    fp8 = torch.randint(0, 256, (K, N), dtype=torch.uint8, generator=g)
    _encode_check(T, fp8, torch.tensor(D.QWEN3_14B_FP8_EXP), alphabet, "words")


def test_config0_cpu_roundtrip_bits_per_byte(T):
    """2^24 values N(0, 0.02) scaled to |max| = 448 and
    RNE-cast; 16-symbol alphabet, 2^11-state table from the data's own
    histogram; encode, decode on the CPU, bit-exact, and the size."""
    from rans_vectoradd import data as D
    n, lane = 1 << 24, 1024
    q, _ = D.gaussian_fp8_bytes(n, seed=0)
    hist = D.exp_histogram(q)
    fp8 = q.reshape(n // lane, lane)
    enc = _encode_check(T, fp8, hist, "nibble")
    bits = T.compressed_bytes(*enc[:5]) * 8 / n
    p = hist.numpy() / hist.numpy().sum()
    entropy = float(-(p[p > 0] * np.log2(p[p > 0])).sum())
    # exponent entropy + 4 raw sign/mantissa bits is the floor; the layout's
    # states, offsets and word padding cost well under 0.1 bit
    assert 4 + entropy < bits < 4 + entropy + 0.1
    assert bits < 7.0


def test_encoder_rejects_zero_frequency_symbol(T):
    from rans_vectoradd import _C
    syms = torch.zeros((3, 8), dtype=torch.uint8)
    syms[1, 2] = 5
    freqs = torch.zeros(16, dtype=torch.int32)
    freqs[0] = 2048
    spread = torch.from_numpy(T.build_spread(freqs.numpy()))
    with pytest.raises(RuntimeError, match="frequency 0"):
        _C.tans_encode_interleaved(syms, freqs, spread)


def test_encoder_rejects_symbol_outside_the_alphabet(T):
    """Pair symbols coded with a 16-symbol table: the encoder reports
    TANS_ESYMBOL instead of reading past its per-symbol tables."""
    from rans_vectoradd import _C
    syms = torch.full((64, 8), 200, dtype=torch.uint8)
    freqs = torch.from_numpy(T.symbol_freqs(np.ones(16), "nibble"))
    spread = torch.from_numpy(T.build_spread(freqs.numpy()))
    with pytest.raises(RuntimeError, match="outside the alphabet"):
        _C.tans_encode_interleaved(syms, freqs, spread)


def test_encoder_rejects_bad_tables(T):
    from rans_vectoradd import _C
    syms = torch.zeros((2, 4), dtype=torch.uint8)
    freqs = torch.full((16,), 128, dtype=torch.int32)
    spread = torch.from_numpy(T.build_spread(freqs.numpy()))
    bad = freqs.clone()
    bad[0] += 1
    with pytest.raises(RuntimeError, match="sum"):
        _C.tans_encode_interleaved(syms, bad, spread)
    sp2 = spread.clone()
    sp2[0] = 99
    with pytest.raises(RuntimeError, match="spread"):
        _C.tans_encode_interleaved(syms, freqs, sp2)
    sp3 = spread.clone()
    sp3[0] = (int(sp3[0]) + 1) % 16
    with pytest.raises(RuntimeError, match="spread"):
        _C.tans_encode_interleaved(syms, freqs, sp3)


def test_encode_argument_checks(T):
    from rans_vectoradd import data as D
    exp = D.QWEN3_14B_FP8_EXP
    with pytest.raises(ValueError):
        T.encode(torch.zeros(16, dtype=torch.uint8), exp)            # not 2-D
    with pytest.raises(ValueError):
        T.encode(torch.zeros((4, 3), dtype=torch.uint8), exp)        # odd N
    with pytest.raises(ValueError):
        T.encode(torch.zeros((4, 4), dtype=torch.int32), exp)        # dtype
    with pytest.raises(ValueError):
        T.encode(torch.zeros((4, 4), dtype=torch.uint8), exp, tile=3)     # 3 does not divide 2
    with pytest.raises(ValueError):
        T.encode(torch.zeros((4, 4), dtype=torch.uint8), exp, tile=-1)
    with pytest.raises(ValueError):
        T.encode(torch.zeros((4, 4), dtype=torch.uint8), exp, alphabet="triple")


def test_encode_accepts_the_references_tiles(T):
    """Any tile dividing N / 2 is accepted, as by the reference
    (tans_codec.py:115-120), and gives the same encoding: the sign/mantissa
    layout is the decoders' 16-element tiles whatever the tile."""
    from rans_vectoradd import data as D
    q, _ = D.gaussian_fp8_bytes(70 * 48, seed=3)
    x = q.reshape(70, 48)
    ref = T.encode(x, D.exp_histogram(q))
    for tile in (1, 2, 3, 4, 6, 8, 12, 24):
        got = T.encode(x, D.exp_histogram(q), tile=tile)
        assert all(torch.equal(a, b) for a, b in zip(ref, got)), tile


def test_empty_input(T):
    from rans_vectoradd import data as D
    comp, st, off, part, sm, fr, sp = T.encode(torch.zeros((0, 16), dtype=torch.uint8),
                                               D.QWEN3_14B_FP8_EXP)
    assert st.numel() == 0 and off.tolist() == [0] and comp.numel() == 1024


def test_untile_inverts_the_tiled_layout(T):
    K, N = 70, 48
    x = torch.arange(K * N, dtype=torch.int64).reshape(K, N)
    tiled = x.reshape(K, N // 16, 16).permute(1, 0, 2).reshape(-1)
    assert torch.equal(T.untile(tiled, K, N), x)


@pytest.mark.parametrize("alphabet", list(ALPHABETS))
@pytest.mark.parametrize("R,C,S", [(17408 // 16, 5120 // 16, None), (100, 70, None), (64, 512, 1),
                                   (130, 1000, 3), (5, 17, 2), (70, 96, 1), (64, 2048, None)])
def test_encode_matrix_slab_layout(T, alphabet, R, C, S):
    """encode_matrix: rows padded to 64, columns to S * Nc (Nc a multiple of
    32, at most 1024), lanes in the 16-row group layout; the oracle decodes
    the encoding back to exactly the padded matrix at each lane's
    coordinates."""
    from rans_vectoradd import data as D
    q, _ = D.gaussian_fp8_bytes(R * C, seed=R + C)
    w = q.reshape(R, C)
    hist = D.exp_histogram(q)
    m = T.encode_matrix(w, hist, segments=S, alphabet=alphabet)
    Rp = -(-R // 64) * 64
    Nc = m.seg_cols
    assert Nc % 32 == 0 and Nc <= 1024
    assert (m.segments - 1) * Nc < C <= m.segments * Nc
    if S is not None:
        assert m.segments <= S
    log2L, sps = ALPHABETS[alphabet]
    K = m.segments * Rp * 4
    assert m.states.numel() == K       # the GEMM reads the refill-schedule layout
    dec = O.w64_decode(m.comp.numpy(), m.offsets.numpy(), m.states.numpy(), m.sm.numpy(),
                       m.spread.numpy(), m.freqs.numpy(), log2L, sps, K, Nc // 4)
    pad = int(np.argmax(hist.numpy())) << 3
    full = np.full((Rp, m.segments * Nc), pad, np.uint8)
    full[:R, :C] = w.numpy()
    rows, cols = gemm_lane_coords(m.segments, Rp, Nc)
    assert np.array_equal(dec, full[rows, cols])
    # every padded-matrix element is held by exactly one lane slot
    seen = np.zeros(full.shape, np.int64)
    np.add.at(seen, (rows, cols), 1)
    assert (seen == 1).all()


def test_gemm_segments_fill_one_round():
    """Config 3/4 shapes: one workgroup per CU at most (<= 256), segment
    widths multiples of 32."""
    from rans_vectoradd import tans_codec as T
    for R, C in ((17408, 5120), (5120, 17408)):
        S = T.gemm_segments(R, C)
        Nc = -(-C // (S * 32)) * 32
        blocks = -(-(R // 16) // 32) * S
        assert blocks <= 256 and blocks > 200, (R, C, S, blocks)
        assert (S - 1) * Nc < C <= S * Nc


def test_encode_matrix_rejects_bad_input(T):
    from rans_vectoradd import data as D
    with pytest.raises(ValueError):
        T.encode_matrix(torch.zeros(16, dtype=torch.uint8), D.QWEN3_14B_FP8_EXP)
    with pytest.raises(ValueError):
        T.encode_matrix(torch.zeros((4, 2000), dtype=torch.uint8), D.QWEN3_14B_FP8_EXP, segments=1)
    with pytest.raises(ValueError):
        T.encode_matrix(torch.zeros((0, 16), dtype=torch.uint8), D.QWEN3_14B_FP8_EXP)


def test_encode_tables_of_several_threads_stay_bounded(monkeypatch):
    """Threads that encode with more histograms than are kept: each gets its
    tables, and no more than the limit stay."""
    import contextlib
    import sys
    import threading

    from rans_vectoradd import tans_codec as T
    f = T.symbol_freqs([1.0] * 16, "nibble")
    sp = T.build_spread(f)
    monkeypatch.setattr(T, "_ENC_TABLES", {})
    monkeypatch.setattr(T, "symbol_freqs", lambda *a: f)   # (the same tables, quickly)
    monkeypatch.setattr(T, "build_spread", lambda *a: sp)
    monkeypatch.setattr(torch.cuda, "device", lambda d: contextlib.nullcontext())
    failed = []

    def work(i):
        try:
            for j in range(400):
                got = T._encode_tables([i + 1.0] + [j + 1.0] * 15, "nibble", torch.device("cpu"))
                assert torch.equal(got[0], torch.from_numpy(f))
        except BaseException as e:   # noqa: BLE001  (reported by the main thread)
            failed.append(repr(e)[:80])

    interval = sys.getswitchinterval()
    sys.setswitchinterval(1e-6)
    try:
        threads = [threading.Thread(target=work, args=(i,)) for i in range(8)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
    finally:
        sys.setswitchinterval(interval)
    assert not failed and len(T._ENC_TABLES) == T._ENC_TABLES_MAX
