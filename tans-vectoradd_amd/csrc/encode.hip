// gfx950 tANS encoder into the wave64 lane layout (include/tans_amd.h).
// It writes the same bytes as the CPU encoder in codec.cpp: the same
// backward tANS construction (csrc/tans_codec.cpp:22-60 of the reference:
// walk the symbols backwards from x = L, emit the low nb bits that bring x
// into [f_s, 2 f_s), then x = L + slot of the rank-th occurrence of s), the
// same per-step bit chunks written forwards LSB-first, and the same refill
// schedule ordering the words of a group's 64 lanes.
//
// Passes (all on the caller's stream):
//   enc_walk_kernel      one wave per 64-lane group, one lane per row: the
//                        backward walk, a 16-element tile at a time.  Each
//                        tile of a lane becomes a 12-byte record (its
//                        segments' bit counts and its first 64 bits; the
//                        bits past 64 go to an overflow array, written
//                        where a lane has any).  Also the sign/mantissa
//                        tiles, the initial decoder states, and the number
//                        of stream words the lane takes (a closed form of
//                        the refill schedule in the lane's bit counts),
//                        summed per group (padded to 4)
//   enc_scan_kernel      exclusive prefix of the group counts -> offsets
//   enc_place_kernel     one wave per group: replays the schedule from the
//                        records' counts while each lane joins its tiles'
//                        bits into words; a word's place (offset + handed +
//                        rank) is fixed when the lane takes it, and the
//                        word is stored there when its last bit is known
//
// The packed layout of short streams (pair alphabet, at most 32 steps per
// lane; schedule.h, tans_pack) reuses the walk, which then records each
// lane's bit count and state in the workspace and sums the group's bits
// into its stream size; enc_place_packed_kernel assembles each group's
// stream (header of lane-pair counts, bit area) in LDS and copies it out.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <string>
#include <type_traits>

#include "../../include/tans_amd.h"
#include "launch.h"
#include "schedule.h"

extern "C" void tans_internal_set_error(const char* msg);  // codec.cpp

namespace {

constexpr int kLanes = 64;
constexpr int kTile = 16;
constexpr int64_t kTailWords = 256;
constexpr int kEncBlock = 256;
static_assert(kTailWords <= kEncBlock, "one workgroup zeroes the tail");

int fail(int code, const std::string& msg) {
    tans_internal_set_error(msg.c_str());
    return code;
}

int hip_check(hipError_t e, const char* what) {
    if (e == hipSuccess) return TANS_OK;
    return fail(TANS_EHIP, std::string(what) + ": " + hipGetErrorString(e));
}

int64_t align256(int64_t b) { return (b + 255) / 256 * 256; }

// Compile-time loop: f(std::integral_constant<int, I>) for I in [B, E).
template <int B, int E, class F>
__device__ __forceinline__ void static_for(F&& f) {
    if constexpr (B < E) {
        f(std::integral_constant<int, B>{});
        static_for<B + 1, E>(f);
    }
}

// Workspace: the tile records u32 [tiles][K][3], their overflow words
// u32 [tiles][overflow words][K], group lengths u32 [G], and for the packed
// layout each lane's bit count and initial state (u16 [K] each).
constexpr int kRecWords = 3;       // counts, bits 0-31, bits 32-63
constexpr uint32_t kRecBits = 64;  // bits of a tile the record holds

// A tile of 16 elements: 8 steps in four segments of 2 (pair alphabet) or 16
// steps in six of 3, 3, 2, 3, 3, 2 (schedule.h).  A segment's bit count
// (at most 24 or 30) takes 5 bits of the record's first word; a tile holds
// at most 96 or 160 bits.
template <int SPS>
struct TileFmt {
    static constexpr bool kTriple = SPS == 1;
    static constexpr int kSteps = kTile / SPS;
    static constexpr int kSegs = kTriple ? 6 : 4;
    static constexpr int kOvf = kTriple ? 3 : 1;   // overflow words
    static constexpr int seg_first(int q) { return kTriple ? 8 * (q / 3) + 3 * (q % 3) : 2 * q; }
    static constexpr int seg_len(int q) { return kTriple ? (q % 3 == 2 ? 2 : 3) : 2; }
    static_assert(kSteps == (int)tans_sched::tile_steps(kTriple), "the schedule's tile");
};

struct WsLayout {
    int64_t rec, ovf, glen, plen, pstate, total;
};

WsLayout ws_layout(int64_t K, int64_t N, int32_t log2L) {
    const int64_t G = (K + kLanes - 1) / kLanes;
    const int64_t tiles = (N + kTile - 1) / kTile;
    const int64_t n_ovf = log2L == TANS_PAIR_LOG2L ? TileFmt<2>::kOvf : TileFmt<1>::kOvf;
    WsLayout l;
    l.rec = 0;
    l.ovf = align256(tiles * K * kRecWords * 4);
    l.glen = l.ovf + align256(tiles * K * n_ovf * 4);
    l.plen = l.glen + align256(G * 4);
    l.pstate = l.plen + align256(K * 2);
    l.total = l.pstate + align256(K * 2);
    return l;
}

typedef uint32_t v4u __attribute__((ext_vector_type(4)));
typedef uint32_t v3u __attribute__((ext_vector_type(3)));
typedef uint32_t v2u __attribute__((ext_vector_type(2)));
typedef __amdgpu_buffer_rsrc_t Rsrc;
typedef uint64_t Mask;   // a lane mask of the wave
constexpr int kNT = 2;   // cache policy: non-temporal

// A buffer resource of `bytes` from a wave-uniform base: loads past it
// return zero, stores past it are dropped.
__device__ __forceinline__ Rsrc rsrc(const void* base, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, (int)bytes,
                                             0x00020000);
}

// Per-symbol step constants (the FSE formulation of the same construction).
// For x in [L, 2L) the step emits the nb low bits of x with x >> nb in
// [f, 2f): nb = (x + x.dnb) >> 16 with maxb = log2L - floor(log2(f - 1))
// (log2L for f = 1) and dnb = (maxb << 16) - (f << maxb); then x = next[idx]
// with idx = start + (x >> nb) - f, kept as a byte offset: y = 2 (start - f).
// This gives the same nb as floor(log2 x) - floor(log2 f), less one when
// x >> nb < f, for every f in [1, L] and x in [L, 2L), and idx is in [start,
// start + f).  f and start are clamped so that it is inside the table
// whatever enc_tab holds.  A symbol of frequency 0 takes nb = log2L plus
// kBadNb, a multiple of 32: shifts and field widths see log2L (so x >> nb is
// 1 and idx = start), and the tile's bit count shows it.
constexpr uint32_t kBadNb = 1024;
constexpr uint32_t kBadGroup = 0x80000000u;   // in glen: the group holds such a symbol

__device__ __forceinline__ uint2 enc_consts(uint32_t e, int log2L) {
    const uint32_t L = 1u << log2L;
    uint32_t f = e & 0xFFFFu;
    uint32_t start = e >> 16;
    f = f > L ? L : f;
    const bool bad = f == 0;
    if (bad) f = 1;
    start = start > L - f ? L - f : start;
    const uint32_t maxb = f == 1 ? (uint32_t)log2L
                                 : (uint32_t)log2L - (31u - (uint32_t)__builtin_clz(f - 1u));
    const uint32_t dnb = bad ? ((uint32_t)log2L + kBadNb) << 16 : (maxb << 16) - (f << maxb);
    return uint2{dnb, 2u * (start - f)};
}

// LDS tables of the walk.  tab is indexed by the symbol's bits as they lie
// in the FP8 bytes: entry e (nibble) or e1 * 16 + e0 (pair), so an entry's
// byte offset is a shift and a mask away (sym_offsets).  nx holds the next
// states, each brought into [L, 2L).
template <int SPS>
struct EncTab {
    uint2 tab[SPS == 2 ? 256 : 16];
    uint16_t nx[1 << TANS_PAIR_LOG2L];
};

template <int SPS>
__device__ __forceinline__ void load_tables(EncTab<SPS>& t, const uint32_t* __restrict__ enc_tab,
                                            const uint16_t* __restrict__ next, int log2L) {
    constexpr int NSYM = SPS == 2 ? 256 : 16;
    const uint32_t L = 1u << log2L;
    for (int i = threadIdx.x; i < NSYM; i += blockDim.x)
        t.tab[SPS == 2 ? ((i & 15) << 4 | i >> 4) : i] = enc_consts(enc_tab[i], log2L);
    for (uint32_t i = threadIdx.x; i < L; i += blockDim.x)
        t.nx[i] = (uint16_t)(L + (next[i] & (L - 1u)));
}

// Byte offset in tab of step Q's symbol of a tile (16 FP8 bytes in c): the
// exponents of bytes 2Q, 2Q + 1 (bits 6:3 of each) as e1 << 7 | e0 << 3, or
// of byte Q as e << 3.
template <int SPS, int Q>
__device__ __forceinline__ uint32_t sym_offset(const v4u& c) {
    const uint32_t w = c[Q * SPS / 4];
    constexpr uint32_t sh = (uint32_t)((Q * SPS) % 4) * 8u;
    if constexpr (SPS == 2) {
        const uint32_t u = w & 0x78787878u;
        return ((u | u >> 4) >> sh) & 0x7F8u;   // (u is shared by the word's two symbols)
    } else {
        return (w >> sh) & 0x78u;
    }
}

// The two sign/mantissa words of a 16-byte tile: sign and mantissa bits
// (mask 0x87 of each byte) of bytes 0-3 in place and of bytes 4-7 rotated
// by 4 bits into the exponent positions, the same for bytes 8-15.
__device__ __forceinline__ v2u sm_words(const v4u& b) {
    const uint32_t m = 0x87878787u;
    return v2u{(b.x & m) | __builtin_amdgcn_alignbit(b.y & m, b.y & m, 28u),
               (b.z & m) | __builtin_amdgcn_alignbit(b.w & m, b.w & m, 28u)};
}

// The bits of one tile of a lane, in decode order (LSB first).
template <int SPS>
struct TileBits {
    uint32_t cnt[TileFmt<SPS>::kSegs];   // bits of each segment
    uint32_t total;                      // their sum
    uint64_t lo;                         // bits 0 .. 63
    uint32_t ovf[TileFmt<SPS>::kOvf];    // the bits past 64 (only when total > 64)
};

// Walk one tile backwards from state x (steps steps - 1 .. 0; GUARD false: all
// kSteps).  A step emits the nb low bits of x above the bits of the steps
// before it; the segments are then joined, and the bits past 64 are formed
// only when a lane of the wave has some.
template <int SPS, bool GUARD>
__device__ __forceinline__ void enc_tile(const v4u& c, int steps, const EncTab<SPS>& t,
                                         uint32_t& x, TileBits<SPS>& o) {
    using F = TileFmt<SPS>;
    uint32_t val[F::kSegs];
    static_for<0, F::kSegs>([&](auto I) {
        constexpr int s = F::kSegs - 1 - decltype(I)::value;
        val[s] = 0u;
        o.cnt[s] = 0u;
        static_for<0, F::seg_len(s)>([&](auto J) {
            constexpr int q = F::seg_first(s) + F::seg_len(s) - 1 - decltype(J)::value;
            if (GUARD && q >= steps) return;   // wave-uniform
            const uint2 e = *reinterpret_cast<const uint2*>(
                reinterpret_cast<const char*>(t.tab) + sym_offset<SPS, q>(c));
            const uint32_t nb = (x + e.x) >> 16;
            val[s] = (val[s] << (nb & 31u)) | __builtin_amdgcn_ubfe(x, 0u, nb);
            o.cnt[s] += nb;
            x = *reinterpret_cast<const uint16_t*>(reinterpret_cast<const char*>(t.nx) +
                                                   (((x >> (nb & 31u)) << 1) + e.y));
        });
    });
    if constexpr (!F::kTriple) {
        const uint32_t n01 = o.cnt[0] + o.cnt[1];
        o.total = n01 + o.cnt[2] + o.cnt[3];
        const uint64_t b01 = (uint64_t)val[1] << (o.cnt[0] & 63u) | val[0];
        const uint64_t b23 = (uint64_t)val[3] << (o.cnt[2] & 63u) | val[2];
        o.lo = b23 << (n01 & 63u) | b01;   // n01 <= 48
        o.ovf[0] = 0u;
        if (__any(o.total > kRecBits))     // (n01 > 0 in the lanes that keep it)
            o.ovf[0] = o.total > kRecBits ? (uint32_t)(b23 >> ((64u - n01) & 63u)) : 0u;
    } else {
        // two halves of three segments (at most 30 + 30 + 20 bits)
        uint64_t lo[2];
        uint32_t hi[2], n[2];
        #pragma unroll
        for (int h = 0; h < 2; h++) {
            const uint32_t n01 = o.cnt[3 * h] + o.cnt[3 * h + 1];
            n[h] = n01 + o.cnt[3 * h + 2];
            lo[h] = (uint64_t)val[3 * h + 2] << (n01 & 63u) |
                    (uint64_t)val[3 * h + 1] << (o.cnt[3 * h] & 63u) | val[3 * h];
            // bits 64 .. 79 (n01 > 44 where there are any)
            hi[h] = n[h] > 64u ? val[3 * h + 2] >> ((64u - n01) & 31u) : 0u;
        }
        o.total = n[0] + n[1];
        o.lo = n[0] < 64u ? lo[1] << (n[0] & 63u) | lo[0] : lo[0];
        o.ovf[0] = o.ovf[1] = o.ovf[2] = 0u;
        if (__any(o.total > kRecBits)) {
            const unsigned __int128 h1 = (unsigned __int128)hi[1] << 64 | lo[1];
            unsigned __int128 up = 0;
            if (o.total > kRecBits)
                up = n[0] >= 64u ? h1 << ((n[0] - 64u) & 63u) | hi[0] : h1 >> ((64u - n[0]) & 127u);
            o.ovf[0] = (uint32_t)up;
            o.ovf[1] = (uint32_t)(up >> 32);
            o.ovf[2] = (uint32_t)(up >> 64);
        }
    }
}

// The refill schedule (schedule.h): every lane in range starts with two
// words (64 bits); each segment of steps (2 steps, or 3, 3, 2 per 8 with
// 2^11-state tables) consumes its nb bits, and after a segment that is not
// the last, a lane holding at most 32 bits takes the next word (+32 bits);
// after the second-to-last segment only a lane holding fewer bits than the
// last segment can read (final_below) does.  A segment consumes at most 30
// bits, so after every check but the final one a lane holds 33..64 bits:
// with c the bits consumed so far it has taken floor(c / 32) + 2 words.
// The words a lane takes in all are therefore fixed by its bit count up to
// the third-to-last segment (c3) and up to the second-to-last (c2):
// t = floor(c3 / 32) + 2, plus one when 32 t - c2 < final_below (t = 2,
// c3 = 0 with two segments; 2 words with one segment; none for S = 0).  The
// walk records its bit count after the last segment (b1: bits of the last
// segment's steps) and after the second-to-last (b2: the last two
// segments'), so c2 = bits - b1 and c3 = bits - b2.
__device__ __forceinline__ uint32_t lane_words(int64_t S, bool triple, uint32_t bits,
                                               uint32_t b1, uint32_t b2) {
    if (S == 0) return 0u;
    const int64_t n = tans_sched::segments(S, triple);
    if (n == 1) return 2u;
    const uint32_t c2 = bits - b1;
    const uint32_t c3 = n >= 3 ? bits - b2 : 0u;
    const uint32_t t = c3 / 32u + 2u;
    return t + (32u * t - c2 < (uint32_t)tans_sched::final_below(S, triple) ? 1u : 0u);
}

// The rows of an FP8 tensor [K, N].  Rows of whole 16-byte tiles start
// 16-byte aligned; others start on any even byte, and their tiles are
// unaligned 16-byte loads (gfx950 takes any alignment).
typedef v4u v4u_any __attribute__((aligned(1)));
typedef v2u v2u_any __attribute__((aligned(1)));

struct RowSrc {
    const uint8_t* fp8;
    int64_t K, N;

    const uint8_t* row;   // the lane's row
    int64_t left;         // bytes from it to the tensor's end

    __device__ __forceinline__ void start(int64_t k) {
        row = fp8 + k * N;
        left = K * N - k * N;
    }
    __device__ __forceinline__ v4u tile(int64_t t) const {
        return *reinterpret_cast<const v4u_any*>(row + t * kTile);
    }
    // the last tile's n < 16 bytes (zeros after them): one load where the
    // tensor goes on past it, else byte by byte
    __device__ __forceinline__ v4u last(int64_t t, int n) const {
        v4u v = {0u, 0u, 0u, 0u};
        const uint8_t* p = row + t * kTile;
        if (left >= t * kTile + kTile) {
            v = *reinterpret_cast<const v4u_any*>(p);
        } else {
            #pragma unroll
            for (int i = 0; i < kTile; i++)
                if (i < n) v[i / 4] |= (uint32_t)p[i] << (8 * (i % 4));
        }
        #pragma unroll
        for (int w = 0; w < 4; w++) {
            const int b = n - 4 * w;   // bytes of this word (wave-uniform)
            v[w] &= b >= 4 ? 0xFFFFFFFFu : b <= 0 ? 0u : (1u << (8 * b)) - 1u;
        }
        return v;
    }
};

// The lanes of a matrix W [R, C] in the decode-GEMM's layout (the lane streams
// of rans_vectoradd.tans_codec.gemm_slab, read where they lie): lane ((s *
// n_rg + g) * 4 + q) * 16 + r holds row 16 g + r of segment s (columns s Nc
// on): its tile t is columns 16 q .. 16 q + 15 of the segment's 64-column
// block t, and of a last block of 32 columns it has the 8 columns 8 q on.
// Rows past R and columns past C read as the byte `pad`.  C >= 16.
struct MatSrc {
    const uint8_t* w;
    int64_t R, C;
    int n_rg, Nc;
    uint32_t pad4;        // `pad` in each byte

    const uint8_t* p;     // the lane's columns of block 0
    const uint8_t* p8;    // its columns of a last 32-column block
    int lim, lim8;        // columns of W from p, p8 on (0 in rows past R)
    bool inside;          // every whole tile of the wave's lanes lies in W

    __device__ __forceinline__ void start(int64_t k) {
        const uint32_t grp = __builtin_amdgcn_readfirstlane((uint32_t)(k / kLanes));
        const int j = (int)(k % kLanes), q = j >> 4;
        const uint32_t s = grp / (uint32_t)n_rg;
        const int64_t row = (int64_t)(grp % (uint32_t)n_rg) * 16 + (j & 15);
        const int64_t col0 = (int64_t)s * Nc;
        const int blocks = Nc / 64;
        p = w + (row < R ? row * C : 0) + col0 + 16 * q;
        p8 = p + 64 * blocks - 8 * q;
        const int64_t left = row < R ? C - col0 : 0;
        auto clamp = [](int64_t v) { return (int)(v < 0 ? 0 : v > kMaxCols ? kMaxCols : v); };
        lim = clamp(left - 16 * q);
        lim8 = clamp(left - 64 * blocks - 8 * q);
        inside = __all(lim >= 64 * (blocks - 1) + 16);
    }
    // the n bytes (8 or 16) at a, of which `avail` lie in W: loaded as the
    // n bytes that end with them (inside the row, as C >= 16), shifted down
    // and padded
    template <int n>
    __device__ __forceinline__ v4u edge(const uint8_t* a, int avail) const {
        avail = avail < 0 ? 0 : avail > n ? n : avail;
        const uint8_t* from = avail ? a - (n - avail) : w;
        unsigned __int128 v = 0, fill = 0;
        if constexpr (n == 16) {
            v = __builtin_bit_cast(unsigned __int128, *reinterpret_cast<const v4u_any*>(from));
            fill = __builtin_bit_cast(unsigned __int128, v4u{pad4, pad4, pad4, pad4});
        } else {
            v = __builtin_bit_cast(uint64_t, *reinterpret_cast<const v2u_any*>(from));
            fill = __builtin_bit_cast(unsigned __int128, v4u{pad4, pad4, 0u, 0u});
        }
        const uint32_t up = (uint32_t)avail * 8u, down = (uint32_t)(n - avail) * 8u;
        const unsigned __int128 kept = avail ? v >> (down & 127u) : 0;
        // the pad bytes sit above the kept ones, below byte n
        const unsigned __int128 above = avail < n ? (fill >> (up & 127u)) << (up & 127u) : 0;
        return __builtin_bit_cast(v4u, kept | above);
    }
    __device__ __forceinline__ v4u tile(int64_t t) const {
        if (inside) return *reinterpret_cast<const v4u_any*>(p + 64 * t);   // wave-uniform
        return edge<16>(p + 64 * t, lim - 64 * (int)t);
    }
    __device__ __forceinline__ v4u last(int64_t, int) const { return edge<8>(p8, lim8); }
    static constexpr int kMaxCols = 1 << 20;   // more than any segment's columns
};

// One wave per 64-lane group; each lane walks its row backwards, a tile at a
// time, and stores per tile its 12-byte record (768 contiguous bytes per
// wave) and its sign/mantissa words (512).  A lane loads its row 128 bytes
// (8 tiles) at a time and the next 128 while it encodes the current ones: a
// step then waits on LDS only, not on a global load, and each line of the
// row is fetched in one go (the lanes' rows are N bytes apart, so a line
// read piecewise over many steps could leave the cache in between).
//
// What bounds it: memory.  2^29 elements at 1024 per lane, 1.21 GB read and
// written, take 202 us (6.0 TB/s) with the whole-line loads below.  Without them
// it was 251 us (284 us with 2-byte chunks stored per step, 0.54 GB of them): the
// same accesses without the walk took 230 us, the walk without its loads and
// stores 97 us, conflict-free table reads changed nothing, and non-temporal
// records cost this kernel 16 us and gave the place pass 11.  The sign/mantissa
// stores are non-temporal: nothing here reads them again, and the place pass
// finds more of the records still cached (142 instead of 149 us before its LDS
// ring).
//
// The lanes' word counts are summed into glen[group], padded to a multiple
// of 4.  PACKED (the packed layout): plen[k] gets the lane's bits (12 for
// the state + its steps' nb), and glen[group] the words of the group's
// stream (header, bits, padding to 16 bytes); `states` is then the
// workspace's state array.
constexpr int kBlockTiles = 8;   // tiles per 128-byte block of a row

// LINES (rows of whole 128-byte lines, RowSrc): a load instruction takes 8 rows'
// lines, 8 lanes each, not 16 bytes of 64 lines; the wave turns them over
// through 8 KiB of LDS (a row's chunks permuted by its index, so that neither
// side conflicts).  Each line is then touched once, and the loads can be
// non-temporal, which leaves the cache to the records.  Workgroups of 16
// waves, so that they share the tables beside 128 KiB of rows.  2^29 elements at
// 1024 per lane: 251 -> 204 us.
constexpr int kLinesBlock = (int)tans_launch::kLineWaves * kLanes;
static_assert(kBlockTiles * kTile == tans_launch::kLineBytes, "a block of tiles is a line");

template <int SPS, bool PACKED, class Src, bool LINES>
__global__ __launch_bounds__(LINES ? kLinesBlock : kEncBlock) void enc_walk_kernel(
    Src src, int64_t K, int64_t N, const uint32_t* __restrict__ enc_tab,
    const uint16_t* __restrict__ next, int log2L, uint32_t* __restrict__ rec,
    uint32_t* __restrict__ ovf, uint16_t* __restrict__ states, uint32_t* __restrict__ glen,
    uint32_t* __restrict__ sm, uint16_t* __restrict__ plen) {
    using F = TileFmt<SPS>;
    constexpr int kWaves = (LINES ? kLinesBlock : kEncBlock) / kLanes;
    static_assert(kEncBlock % kLanes == 0, "blocks hold whole groups");
    static_assert(!LINES || std::is_same_v<Src, RowSrc>, "lines of a tensor's rows");
    __shared__ alignas(16) v4u lines[LINES ? kWaves : 1][LINES ? kBlockTiles * kLanes : 1];
    __shared__ EncTab<SPS> tab;
    load_tables<SPS>(tab, enc_tab, next, log2L);
    __syncthreads();
    const int lane = threadIdx.x & (kLanes - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kLanes);
    const int64_t g = (int64_t)blockIdx.x * kWaves + wave;
    const int64_t k0 = g * kLanes;
    if (k0 >= K) return;
    const uint32_t lanes = (uint32_t)(K - k0 < kLanes ? K - k0 : kLanes);
    const bool active = (uint32_t)lane < lanes;
    src.start(active ? k0 + lane : K - 1);   // lanes out of range repeat the last row, unstored
    const int64_t S = N / SPS;
    const int nt = (int)((N + kTile - 1) / kTile);   // S <= 2^24 (checked by the launcher)
    const int rag = (int)(N % kTile);
    const int last_steps = (rag ? rag : kTile) / SPS;
    const int last_segs = (int)tans_sched::last_tile_segments(S, F::kTriple);
    uint32_t x = 1u << log2L;
    uint32_t bits = 0;          // the lane's stream bits
    uint32_t bad = 0;           // kBadNb or more: a symbol of frequency 0
    uint32_t b1 = 0, b2 = 0;    // bits of the last segment, of the last two (lane_words)
    // the group's part of tile t's records, overflow words and sm rows (wave-uniform)
    const char* rec_t = reinterpret_cast<const char*>(rec) +
                        ((int64_t)(nt - 1) * K + k0) * (kRecWords * 4);
    const char* ovf_t = reinterpret_cast<const char*>(ovf) +
                        ((int64_t)(nt - 1) * F::kOvf * K + k0) * 4;
    const char* sm_t = reinterpret_cast<const char*>(sm) + ((int64_t)(nt - 1) * K + k0) * 8;
    // tiles 8 b .. 8 b + 7 of the row
    auto load = [&](v4u (&buf)[kBlockTiles], int b) {
        #pragma unroll
        for (int c = kBlockTiles - 1; c >= 0; c--) buf[c] = src.tile(b * kBlockTiles + c);
    };
    // tile t; FIRST: it may be the row's last (the walk's first)
    auto tile = [&](const v4u& c, int t, auto FIRST) {
        constexpr bool kFirst = decltype(FIRST)::value;
        TileBits<SPS> o;
        enc_tile<SPS, kFirst>(c, kFirst && t == nt - 1 ? last_steps : F::kSteps, tab, x, o);
        uint32_t counts = o.cnt[0];
        #pragma unroll
        for (int s = 1; s < F::kSegs; s++) counts |= o.cnt[s] << (5 * s);
        const v3u r = {counts, (uint32_t)o.lo, (uint32_t)(o.lo >> 32)};
        __builtin_amdgcn_raw_buffer_store_b96(r, rsrc(rec_t, lanes * (kRecWords * 4)),
                                              (uint32_t)lane * (kRecWords * 4), 0, 0);
        if (__any(o.total > kRecBits)) {
            #pragma unroll
            for (int i = 0; i < F::kOvf; i++)
                if (o.total > kRecBits + 32u * i)
                    __builtin_amdgcn_raw_buffer_store_b32(o.ovf[i],
                                                          rsrc(ovf_t + (int64_t)i * K * 4, lanes * 4),
                                                          (uint32_t)lane * 4, 0, 0);
        }
        __builtin_amdgcn_raw_buffer_store_b64(sm_words(c), rsrc(sm_t, lanes * 8),
                                              (uint32_t)lane * 8, 0, kNT);
        rec_t -= K * (kRecWords * 4);
        ovf_t -= K * (F::kOvf * 4);
        sm_t -= K * 8;
        bits += o.total;
        bad |= o.total;
        if (kFirst && t == nt - 1) {
            #pragma unroll
            for (int s = 0; s < F::kSegs; s++) {
                if (s == last_segs - 1) b1 = o.cnt[s];
                if (s == last_segs - 2) b2 = o.cnt[s];
            }
            b2 += b1;
        } else if (t == nt - 2 && last_segs == 1) {
            b2 += o.cnt[F::kSegs - 1];
        }
    };
    v4u cur[kBlockTiles], nxt[kBlockTiles];
    int b = (nt - 1) / kBlockTiles;
    if constexpr (LINES) {
        // load i of a block: rows 8 i .. 8 i + 7; lane l takes the chunk of row
        // 8 i + l / 8 that belongs at LDS place l of those rows, chunk c of
        // row r being at place c ^ (r mod 8) of its 8
        const int rsub = lane >> 3, chunk = (lane & 7) ^ rsub;
        const uint8_t* first = src.fp8 + k0 * N + chunk * kTile;
        auto load_lines = [&](int blk) {
            #pragma unroll
            for (int i = 0; i < kBlockTiles; i++) {
                const uint32_t r = (uint32_t)(8 * i + rsub);
                nxt[i] = __builtin_nontemporal_load(reinterpret_cast<const v4u*>(
                    first + (int64_t)(r < lanes ? r : lanes - 1) * N + blk * (kBlockTiles * kTile)));
            }
        };
        v4u* stage = lines[wave];
        auto turn = [&]() {   // the wave's LDS accesses execute in order
            #pragma unroll
            for (int i = 0; i < kBlockTiles; i++) stage[i * kLanes + lane] = nxt[i];
        };
        auto get = [&](int c) { return stage[lane * kBlockTiles + (c ^ (lane & 7))]; };
        load_lines(b);
        turn();
        if (b > 0) load_lines(b - 1);
        #pragma unroll
        for (int c = kBlockTiles - 1; c >= 0; c--)
            tile(get(c), b * kBlockTiles + c, std::true_type{});
        for (b--; b >= 0; b--) {
            turn();
            if (b > 0) load_lines(b - 1);
            #pragma unroll
            for (int c = kBlockTiles - 1; c >= 0; c--)
                tile(get(c), b * kBlockTiles + c, std::false_type{});
        }
    } else {
        const int full = nt - (rag ? 1 : 0);   // whole tiles
        #pragma unroll
        for (int c = kBlockTiles - 1; c >= 0; c--)
            if (b * kBlockTiles + c < full) cur[c] = src.tile(b * kBlockTiles + c);   // wave-uniform
        v4u ragged = {0u, 0u, 0u, 0u};
        if (rag) ragged = src.last(nt - 1, rag);
        if (b > 0) load(nxt, b - 1);
        #pragma unroll
        for (int c = kBlockTiles - 1; c >= 0; c--) {
            const int t = b * kBlockTiles + c;
            if (t < nt) tile(rag && t == nt - 1 ? ragged : cur[c], t, std::true_type{});
        }
        for (b--; b >= 0; b--) {
            #pragma unroll
            for (int c = 0; c < kBlockTiles; c++) cur[c] = nxt[c];
            if (b > 0) load(nxt, b - 1);
            #pragma unroll
            for (int c = kBlockTiles - 1; c >= 0; c--)
                tile(cur[c], b * kBlockTiles + c, std::false_type{});
        }
    }
    uint32_t words = 0;
    if (active) {
        states[k0 + lane] = (uint16_t)x;
        if (bad >= kBadNb) bits = b1 = b2 = 0;   // its bit counts mean nothing
        if constexpr (PACKED) {
            words = (uint32_t)tans_pack::kStateBits + bits;   // the lane's bits
            plen[k0 + lane] = (uint16_t)words;
        } else {
            words = lane_words(S, F::kTriple, bits, b1, b2);
        }
    }
    #pragma unroll
    for (int m = 32; m >= 1; m >>= 1) words += __shfl_xor(words, m, kLanes);
    if constexpr (PACKED)   // header + bits, padded to 16 bytes
        words = ((uint32_t)tans_pack::hdr_total(S) + (words + 7u) / 8u + 15u) / 16u * 4u;
    else
        words = (words + 3u) & ~3u;
    if (__any(bad >= kBadNb)) words |= kBadGroup;
    if (lane == 0) glen[g] = words;
}

// offsets[g] = sum of glen[0..g), offsets[G] = total.  One workgroup takes
// kScanItems groups per thread and round; a round's loads are issued before
// the previous round is summed.  A thread's items are a contiguous run, the
// waves scan their threads' sums by shuffles and the 16 wave totals meet in
// LDS.  (8192 groups: 12.9 us with one contiguous run per thread, read word
// by word, 8.9 us now.)  It also reports: *status = TANS_ESYMBOL if a group
// is marked kBadGroup, and result = {total, 1 if any is}, which may be host
// memory, so that a caller waiting for the stream needs no copy.  Either may
// be null.
constexpr int kScanBlock = 1024;
constexpr int kScanItems = 8;

__global__ __launch_bounds__(kScanBlock) void enc_scan_kernel(const uint32_t* __restrict__ glen,
                                                              int64_t G,
                                                              int64_t* __restrict__ offsets,
                                                              int* __restrict__ status,
                                                              int64_t* __restrict__ result) {
    constexpr int kWaves = kScanBlock / kLanes;
    constexpr int64_t kRound = (int64_t)kScanBlock * kScanItems;
    __shared__ int64_t wave_sum[2][kWaves];
    const int lane = threadIdx.x & (kLanes - 1);
    const int wave = threadIdx.x / kLanes;
    auto load = [&](int64_t base, uint32_t (&v)[kScanItems]) {
        const int64_t i0 = base + (int64_t)threadIdx.x * kScanItems;
        #pragma unroll
        for (int i = 0; i < kScanItems; i++) v[i] = i0 + i < G ? glen[i0 + i] : 0u;
    };
    uint32_t v[kScanItems], n[kScanItems];
    load(0, v);
    int64_t carry = 0;
    uint32_t marks = 0;
    int buf = 0;
    for (int64_t base = 0; base < G; base += kRound) {
        load(base + kRound, n);
        int64_t sum = 0;
        #pragma unroll
        for (int i = 0; i < kScanItems; i++) {
            marks |= v[i];
            v[i] &= ~kBadGroup;
            sum += v[i];
        }
        int64_t inc = sum;   // inclusive scan over the wave
        #pragma unroll
        for (int d = 1; d < kLanes; d <<= 1) {
            const int64_t y = __shfl_up(inc, d, kLanes);
            if (lane >= d) inc += y;
        }
        if (lane == kLanes - 1) wave_sum[buf][wave] = inc;
        __syncthreads();
        int64_t run = carry + inc - sum;
        #pragma unroll
        for (int w = 0; w < kWaves; w++) {
            const int64_t s = wave_sum[buf][w];
            if (w < wave) run += s;
            carry += s;
        }
        const int64_t i0 = base + (int64_t)threadIdx.x * kScanItems;
        #pragma unroll
        for (int i = 0; i < kScanItems; i++) {
            if (i0 + i < G) offsets[i0 + i] = run;
            run += v[i];
            v[i] = n[i];
        }
        buf ^= 1;   // the next round writes the other buffer: one barrier per round
    }
    const bool bad = __syncthreads_or((int)(marks & kBadGroup)) != 0;
    if (threadIdx.x == 0) {
        offsets[G] = carry;
        if (bad && status) *status = TANS_ESYMBOL;
        if (result) {
            result[0] = carry;
            result[1] = bad ? 1 : 0;
        }
    }
}

// Zero n words (a kernel rather than hipMemsetAsync, so a caller may
// capture the encoder in a graph).
__global__ __launch_bounds__(kEncBlock) void zero_words_kernel(uint32_t* __restrict__ p, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * kEncBlock + threadIdx.x;
    if (i < n) p[i] = 0u;
}

// x += y with the carry out of every lane as a lane mask (v_add_co_u32 with
// an SGPR carry).
__device__ __forceinline__ Mask add_carry(uint32_t& x, uint32_t y) {
    Mask c;
    asm("v_add_co_u32 %0, %1, %2, %3" : "=v"(x), "=s"(c) : "v"(x), "v"(y));
    return c;
}

// m's lanes take if_set, the others if_clear (v_cndmask_b32 on the mask).
__device__ __forceinline__ uint32_t select(Mask m, uint32_t if_set, uint32_t if_clear) {
    return __builtin_amdgcn_inverse_ballot_w64(m) ? if_set : if_clear;
}

// Place in the lane's mask order (how many of m's lanes come before it).
__device__ __forceinline__ uint32_t rank_in(Mask m) {
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                     __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

// One wave per group replays the refill schedule from the tile records while
// each lane joins its tiles' bits into 32-bit words, LSB first.  A word's
// place in the stream is fixed when the lane takes it: the first two words
// of every lane are the first 2 x lanes words (first words in lane order,
// then the second), and a word taken after a segment goes to handed + rank
// (in lane order, as the decoders read it).  A lane takes a word whenever
// its consumed bits cross a multiple of 32, which is also when its oldest
// word is complete: it then stores that word at the place it took for it
// (f0), and the newly taken place becomes the younger of its two (f1).  The
// position in the oldest word is kept in the top 5 bits of `pos`, so adding
// a segment's count there carries out exactly at a crossing.
//
// A tile's bits are appended to the unfinished word by one 64-bit shift per
// word; the words come out of them in order, one at most per segment.  Words
// taken past the lane's bits, and the group's padding to 4 words, are zero.
//
// Words go to a ring of kRingBytes in LDS that holds the stream from byte
// `flushed` on, and whole KiBs of it are stored 16 bytes per lane.  A place is
// filled two crossings of its lane after it was taken, so by the time the
// ring moves on, hundreds of words later, it is nearly always full.  A lane so
// far behind that its place has left the ring stores the word itself, after
// the wave's earlier stores have completed (they wrote what the ring held
// there).  The stores go through a buffer resource bounded by the group's
// length.
//
// What bounds it: memory and the vector-memory path.  2^29 elements at 1024 per
// lane, 0.58 GB: 128 us, 142 us with one scattered store per segment (201 us
// with a 2-byte load per step and the bits joined step by step).  Records and
// words are non-temporal, as nothing reads them again: with cached words this
// kernel takes 124 us, and the next call's walk, which then has to write them
// back, 267 instead of 251.
constexpr int kRingBytes = 4096;
constexpr int kFlushBytes = 16 * kLanes;
constexpr int kPlaceAhead = 4;   // tiles whose records are in flight

template <int SPS>
__global__ __launch_bounds__(kEncBlock) void enc_place_kernel(
    const uint32_t* __restrict__ rec, const uint32_t* __restrict__ ovf, int64_t K, int64_t N,
    const int64_t* __restrict__ offsets, uint32_t* __restrict__ comp, int64_t words_total) {
    using F = TileFmt<SPS>;
    constexpr int NQ = (F::kTriple ? 160 : 96) / 32 + 1;   // words a tile's bits can touch
    constexpr uint32_t kTileBytes = F::kSegs * kLanes * 4;   // the most a tile can hand out
    static_assert(kRingBytes >= (int)kTileBytes + 2 * kFlushBytes && kRingBytes % kFlushBytes == 0,
                  "a tile's words fit in the ring beside a flush");
    __shared__ alignas(16) unsigned char rings[kEncBlock / kLanes][kRingBytes];
    const int lane = threadIdx.x & (kLanes - 1);
    // the group (wave-uniform, so the output resource stays in SGPRs)
    const int64_t g = (int64_t)blockIdx.x * (kEncBlock / kLanes) +
                      __builtin_amdgcn_readfirstlane(threadIdx.x / kLanes);
    const int64_t k0 = g * kLanes;
    if (blockIdx.x == 0 && threadIdx.x < kTailWords) comp[words_total + threadIdx.x] = 0u;
    if (k0 >= K) return;
    const uint32_t lanes = (uint32_t)(K - k0 < kLanes ? K - k0 : kLanes);
    const bool active = (uint32_t)lane < lanes;
    const int64_t base = offsets[g];
    const int64_t glen = offsets[g + 1] - base;
    // the stream's bytes (a multiple of 16, as every length is of 4 words)
    const uint32_t end = glen < 0 ? 0u : glen > 0x1FFFFFF0 ? 0x7FFFFFC0u : (uint32_t)(glen * 4);
    const Rsrc out = rsrc(comp + base, end);
    const int64_t S = N / SPS;
    const int nt = (int)((N + kTile - 1) / kTile);   // S <= 2^24 (checked by the launcher)
    const int last_segs = (int)tans_sched::last_tile_segments(S, F::kTriple);
    // the final check: a lane that crossed takes a word when it then holds
    // 32 - position < final_below bits
    const uint32_t fin_pos = (uint32_t)(32 - tans_sched::final_below(S, F::kTriple));   // may be -1
    uint32_t pos = 0;     // bits of the oldest word already known, in bits 31:27
    uint32_t acc = 0;     // those bits
    uint32_t f0 = (uint32_t)lane * 4u, f1 = (lanes + (uint32_t)lane) * 4u;   // places (bytes)
    uint32_t handed = 8u * lanes;   // bytes handed out
    uint32_t flushed = 0;           // bytes of the stream that have left the ring
    bool unwaited = false;          // a flush's stores may still be on their way
    unsigned char* ring = rings[__builtin_amdgcn_readfirstlane(threadIdx.x / kLanes)];
    // the calling lane's word for place f (STALE: the place may have left the ring)
    auto put = [&](uint32_t v, uint32_t f, auto STALE) {
        if constexpr (decltype(STALE)::value) {
            if (f < flushed) {
                __builtin_amdgcn_raw_buffer_store_b32(v, out, f, 0, 0);
                return;
            }
        }
        *reinterpret_cast<uint32_t*>(ring + (f & (uint32_t)(kRingBytes - 1))) = v;
    };
    // the next KiB of the ring (bytes past the stream's end are dropped)
    auto flush = [&]() {
        const uint32_t at = flushed + (uint32_t)lane * 16u;
        // (compiler barriers: the ring is written as words and read as
        // vectors, which type-based alias analysis would let it reorder)
        asm volatile("" ::: "memory");
        const v4u v = *reinterpret_cast<const v4u*>(ring + (at & (uint32_t)(kRingBytes - 1)));
        asm volatile("" ::: "memory");
        __builtin_amdgcn_raw_buffer_store_b128(v, out, at, 0, kNT);
        flushed += (uint32_t)kFlushBytes;
        unwaited = true;
    };
    // before a tile: room in the ring for all it can hand out; true if a lane
    // of the wave holds a place that has left the ring
    auto make_room = [&]() {
        while (handed + kTileBytes > flushed + (uint32_t)kRingBytes) flush();   // wave-uniform
        const bool stale = __any(active && f0 < flushed);
        if (stale && unwaited) {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            unwaited = false;
        }
        return stale;
    };
    // tile t's record (zero past the last tile and in lanes out of range)
    const int64_t rec_stride = K * (kRecWords * 4);
    auto load = [&](int t) {
        const int tt = t < nt ? t : nt - 1;
        return __builtin_amdgcn_raw_buffer_load_b96(
            rsrc(reinterpret_cast<const char*>(rec) + (int64_t)tt * rec_stride +
                     k0 * (kRecWords * 4),
                 t < nt ? lanes * (kRecWords * 4) : 0u),
            (uint32_t)lane * (kRecWords * 4), 0, kNT);
    };
    // the words tile t's bits make, the unfinished one first
    auto words_of = [&](const v3u& r, int t, uint32_t (&q)[NQ]) {
        const uint32_t n = pos >> 27;
        const uint64_t a = (uint64_t)r.y << n;
        const uint64_t b = ((uint64_t)r.z << 32 | r.y) << n;
        q[0] = (uint32_t)a | acc;
        q[1] = (uint32_t)(b >> 32);
        q[2] = (uint32_t)(((uint64_t)r.z << n) >> 32);
        #pragma unroll
        for (int i = 3; i < NQ; i++) q[i] = 0u;
        uint32_t total = 0;
        #pragma unroll
        for (int s = 0; s < F::kSegs; s++) total += (r.x >> (5 * s)) & 31u;
        if (__any(total > kRecBits)) {
            uint32_t prev = r.z;
            #pragma unroll
            for (int i = 0; i < F::kOvf; i++) {
                // words past the lane's bits were not written: zero
                const uint32_t v = __builtin_amdgcn_raw_buffer_load_b32(
                    rsrc(ovf + ((int64_t)t * F::kOvf + i) * K + k0,
                         lanes * 4),
                    (uint32_t)lane * 4, 0, 0);
                const uint32_t w = total > kRecBits + 32u * i ? v : 0u;
                q[2 + i] = (uint32_t)((((uint64_t)w << 32 | prev) << n) >> 32);
                prev = w;
            }
            q[2 + F::kOvf] = (uint32_t)(((uint64_t)prev << n) >> 32);
        }
    };
    auto steps = [&](const v3u& r, uint32_t (&q)[NQ], auto STALE) {
        static_for<0, F::kSegs>([&](auto I) {
            constexpr int s = decltype(I)::value;
            const Mask m = add_carry(pos, (r.x << (27 - 5 * s)) & 0xF8000000u);
            if (__builtin_amdgcn_inverse_ballot_w64(m)) put(q[0], f0, STALE);
            f0 = select(m, f1, f0);
            f1 = select(m, rank_in(m) * 4u + handed, f1);
            handed += 4u * (uint32_t)__popcll(m);
            // (the words left can be no more than the segments left, plus one)
            #pragma unroll
            for (int i = 0; i < F::kSegs - s && i + 1 < NQ; i++) q[i] = select(m, q[i + 1], q[i]);
        });
        acc = q[0];
    };
    auto tile = [&](const v3u& r, int t) {
        uint32_t q[NQ];
        words_of(r, t, q);
        if (make_room()) steps(r, q, std::true_type{});
        else steps(r, q, std::false_type{});
    };
    v3u r[kPlaceAhead];
    #pragma unroll
    for (int i = 0; i < kPlaceAhead; i++) r[i] = load(i);
    int t = 0;
    for (; t + kPlaceAhead < nt; t += kPlaceAhead) {
        #pragma unroll
        for (int i = 0; i < kPlaceAhead; i++) {
            tile(r[i], t + i);
            r[i] = load(t + i + kPlaceAhead);
        }
    }
    // the last 1 .. kPlaceAhead tiles; the last one ends the streams
    uint32_t fc = active ? 2u : 0u;   // places held
    #pragma unroll
    for (int i = 0; i < kPlaceAhead; i++) {
        if (t + i >= nt) break;   // wave-uniform
        if (t + i < nt - 1) {
            tile(r[i], t + i);
            continue;
        }
        uint32_t q[NQ];
        words_of(r[i], nt - 1, q);
        make_room();
        #pragma unroll
        for (int s = 0; s < F::kSegs; s++) {
            if (s >= last_segs) break;   // wave-uniform
            const Mask m = add_carry(pos, (r[i].x << (27 - 5 * s)) & 0xF8000000u);
            // after the last segment no word is taken, after the one before
            // it only by the lanes that the final check names
            const Mask take = s == last_segs - 1 ? Mask(0)
                              : s == last_segs - 2
                                  ? m & __ballot((int32_t)(pos >> 27) > (int32_t)fin_pos)
                                  : m;
            if (__builtin_amdgcn_inverse_ballot_w64(m)) put(q[0], f0, std::true_type{});
            f0 = select(m, f1, f0);
            f1 = select(take, rank_in(take) * 4u + handed, f1);
            fc -= select(m & ~take, 1u, 0u);
            handed += 4u * (uint32_t)__popcll(take);
            #pragma unroll
            for (int j = 0; j + 1 < NQ; j++) q[j] = select(m, q[j + 1], q[j]);
        }
        acc = q[0];
    }
    if (active) {
        if (pos >> 27) {   // the last, partial word
            put(acc, f0, std::true_type{});
            f0 = f1;
            fc--;
        }
        if (fc >= 1) put(0u, f0, std::true_type{});
        if (fc >= 2) put(0u, f1, std::true_type{});
    }
    // padding up to the 4-word boundary, which the ring has room for: the last
    // tile handed out no word after its last segment
    if (lane < 4 && handed + 4u * (uint32_t)lane < end)
        put(0u, handed + 4u * (uint32_t)lane, std::true_type{});
    while (flushed < end) flush();   // wave-uniform
}

// The packed layout: one wave per group.  Each lane reads its bit count
// (plen), the pair's count is the two lanes' sum, and a scan of the counts
// over the wave gives each pair's end; the wave then ORs the header and
// every lane's bits (state minus L, then each tile's; even lanes forwards
// from the pair's start, odd lanes bit-reversed backwards from its end) into
// its LDS buffer, which holds the longest possible stream, and copies the
// group's stream words out (zeros past the bits).  A tile goes in as up to
// three 32-bit fields, not step by step.
constexpr int kPackWords = (int)(tans_pack::max_stream_bytes(tans_pack::kMaxSteps) / 4);
constexpr int kPackTiles = (int)(2 * tans_pack::kMaxSteps / kTile);

__global__ __launch_bounds__(kEncBlock) void enc_place_packed_kernel(
    const uint32_t* __restrict__ rec, const uint32_t* __restrict__ ovf,
    const uint16_t* __restrict__ pstate, const uint16_t* __restrict__ plen, int64_t K, int64_t N,
    uint32_t L, const int64_t* __restrict__ offsets, uint32_t* __restrict__ comp,
    int64_t words_total) {
    using F = TileFmt<2>;
    __shared__ uint32_t bufs[kEncBlock / kLanes][kPackWords];
    const int lane = threadIdx.x & (kLanes - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kLanes);
    const int64_t g = (int64_t)blockIdx.x * (kEncBlock / kLanes) + wave;
    if (blockIdx.x == 0 && threadIdx.x < kTailWords) comp[words_total + threadIdx.x] = 0u;
    const int64_t k0 = g * kLanes;
    if (k0 >= K) return;
    const uint32_t lanes = (uint32_t)(K - k0 < kLanes ? K - k0 : kLanes);
    const bool active = (uint32_t)lane < lanes;
    const int nt = (int)((N + kTile - 1) / kTile);   // at most kPackTiles (checked by the launcher)
    v3u r[kPackTiles];
    #pragma unroll
    for (int t = 0; t < kPackTiles; t++)
        r[t] = __builtin_amdgcn_raw_buffer_load_b96(
            rsrc(rec + ((int64_t)(t < nt ? t : nt - 1) * K + k0) * kRecWords,
                 t < nt ? lanes * (kRecWords * 4) : 0u),
            (uint32_t)lane * (kRecWords * 4), 0, 0);
    uint32_t* b = bufs[wave];
    for (int i = lane; i < kPackWords; i += kLanes) b[i] = 0u;
    const uint32_t len = active ? plen[k0 + lane] : 0u;
    const uint32_t st = active ? (uint32_t)pstate[k0 + lane] - L : 0u;
    const uint32_t cnt = len + (uint32_t)__shfl_xor((int)len, 1, kLanes);   // the pair's bits
    uint32_t v = (lane & 1) ? 0u : cnt;
    #pragma unroll
    for (int d = 1; d < kLanes; d <<= 1) {
        const uint32_t y = (uint32_t)__shfl_up((int)v, d, kLanes);
        if (lane >= d) v += y;
    }
    const int64_t S = N / 2;
    const int hb = tans_pack::hdr_bytes(S);
    const uint32_t end = (uint32_t)tans_pack::hdr_total(S) * 8u + v;
    const uint32_t start = end - cnt;
    // (the wave's LDS accesses execute in order: the zeroing above lands first)
    if (!(lane & 1)) {
        const uint32_t at = (uint32_t)(lane >> 1) * (uint32_t)hb;
        atomicOr(&b[at >> 2], cnt << (8u * (at & 3u)));
    }
    if (active) {
        const bool odd = lane & 1;
        uint32_t o = 0;   // bits of the lane placed so far
        // the low nb <= 32 bits of val (the others zero) as the lane's next bits
        auto put = [&](uint32_t val, uint32_t nb) {
            if (nb == 0) return;
            // odd lanes: the field's bits run backwards, so it sits reversed
            // at [end - o - nb, end - o)
            const uint32_t p = odd ? end - o - nb : start + o;
            const uint32_t f = odd ? __builtin_bitreverse32(val) >> (32u - nb) : val;
            const uint32_t sh = p & 31u;
            if (p + nb <= (uint32_t)kPackWords * 32u) {   // (a well-formed stream always fits)
                atomicOr(&b[p >> 5], f << sh);
                if (sh + nb > 32u) atomicOr(&b[(p >> 5) + 1], f >> (32u - sh));
            }
            o += nb;
        };
        put(st, (uint32_t)tans_pack::kStateBits);
        #pragma unroll
        for (int t = 0; t < kPackTiles; t++) {
            if (t >= nt) break;   // wave-uniform
            uint32_t total = 0;
            #pragma unroll
            for (int s = 0; s < F::kSegs; s++) total += (r[t].x >> (5 * s)) & 31u;
            put(r[t].y, total < 32u ? total : 32u);
            if (total > 32u) put(r[t].z, total < 64u ? total - 32u : 32u);
            if (total > 64u) {
                const uint32_t w = total < 96u ? total - 64u : 32u;
                put(ovf[(int64_t)t * K + k0 + lane] , w);
            }
        }
    }
    const int64_t base = offsets[g];
    const int64_t glen = offsets[g + 1] - base;
    for (int64_t i = lane; i < glen && i < kPackWords; i += kLanes) comp[base + i] = b[i];
}

}  // namespace

extern "C" {

int tans_gpu_encode_workspace(int64_t K, int64_t N, int32_t log2L, int64_t* workspace_bytes) {
    if (!workspace_bytes || K < 0 || N < 0 || N % 2)
        return fail(TANS_EINVAL, "gpu_encode: need K >= 0 and even N >= 0");
    if (log2L != TANS_PAIR_LOG2L && log2L != TANS_NIBBLE_LOG2L)
        return fail(TANS_EINVAL, "gpu_encode: log2L must be 12 (pair) or 11 (nibble)");
    *workspace_bytes = ws_layout(K, N, log2L).total;
    return TANS_OK;
}

}  // extern "C"

namespace {

// begin of every source and layout; packed: states == NULL (the workspace
// keeps them)
template <class Src>
int gpu_encode_begin(const Src& src, const void* data, int64_t K, int64_t N,
                     const uint32_t* enc_tab, const uint16_t* enc_next, int32_t log2L,
                     void* workspace, int64_t workspace_bytes, int64_t* offsets, uint16_t* states,
                     void* sm, int32_t* status, int64_t* result, void* stream, bool packed) {
    int64_t need = 0;
    int rc = tans_gpu_encode_workspace(K, N, log2L, &need);
    if (rc) return rc;
    if (packed && (log2L != TANS_PAIR_LOG2L || N > 2 * tans_pack::kMaxSteps))
        return fail(TANS_EINVAL, "gpu_encode_packed: needs log2L 12 and N <= 64");
    if (K == 0 || N == 0) {
        if (K == 0 && offsets) {   // offsets = {0}: the scan of no groups
            hipLaunchKernelGGL(enc_scan_kernel, dim3(1), dim3(kScanBlock), 0, (hipStream_t)stream,
                               nullptr, (int64_t)0, offsets, status, result);
            return hip_check(hipGetLastError(), "gpu_encode offsets");
        }
        return fail(TANS_EINVAL, "gpu_encode: N must be positive when K > 0");
    }
    if (!data || !enc_tab || !enc_next || !workspace || !offsets || (!states && !packed) || !sm ||
        (!status && !result))
        return fail(TANS_EINVAL, "gpu_encode: null pointer");
    if (workspace_bytes < need) return fail(TANS_EINVAL, "gpu_encode: workspace too small");
    const int sps = log2L == TANS_PAIR_LOG2L ? 2 : 1;
    const int64_t S = N / sps;
    const int64_t G = (K + kLanes - 1) / kLanes;
    // K within int32 keeps every grid within a launch's 32-bit work-item count
    if (K > INT32_MAX || S > (int64_t(1) << 24))
        return fail(TANS_EINVAL, "gpu_encode: tensor too large");
    const WsLayout l = ws_layout(K, N, log2L);
    char* ws = static_cast<char*>(workspace);
    uint32_t* rec = reinterpret_cast<uint32_t*>(ws + l.rec);
    uint32_t* ovf = reinterpret_cast<uint32_t*>(ws + l.ovf);
    uint32_t* glen = reinterpret_cast<uint32_t*>(ws + l.glen);
    uint16_t* plen = reinterpret_cast<uint16_t*>(ws + l.plen);
    uint16_t* st_out = packed ? reinterpret_cast<uint16_t*>(ws + l.pstate) : states;
    hipStream_t st = (hipStream_t)stream;
    auto walk = [&](auto kernel, int block = kEncBlock) {
        const int64_t per = block / kLanes;
        hipLaunchKernelGGL(kernel, dim3((unsigned)((G + per - 1) / per)), dim3((unsigned)block), 0,
                           st, src, K, N, enc_tab, enc_next,
                           (int)log2L, rec, ovf, st_out, glen, (uint32_t*)sm, plen);
    };
    bool done = false;
    if constexpr (std::is_same_v<Src, RowSrc>) {
        const int cus = tans_internal_cu_count();
        if (cus <= 0) return fail(TANS_EHIP, "gpu_encode: cannot query the device's CU count");
        const bool lines = tans_launch::whole_lines(G, N, cus);
        done = packed || lines;
        if (packed) walk(enc_walk_kernel<2, true, Src, false>);
        else if (lines && sps == 2) walk(enc_walk_kernel<2, false, Src, true>, kLinesBlock);
        else if (lines) walk(enc_walk_kernel<1, false, Src, true>, kLinesBlock);
    }
    if (!done) {
        if (sps == 2) walk(enc_walk_kernel<2, false, Src, false>);
        else walk(enc_walk_kernel<1, false, Src, false>);
    }
    if ((rc = hip_check(hipGetLastError(), "enc_walk_kernel launch"))) return rc;
    hipLaunchKernelGGL(enc_scan_kernel, dim3(1), dim3(kScanBlock), 0, st, glen, G, offsets,
                       status, result);
    return hip_check(hipGetLastError(), "enc_scan_kernel launch");
}

// begin of a tensor's rows
int gpu_encode_rows(const void* fp8, int64_t K, int64_t N, const uint32_t* enc_tab,
                    const uint16_t* enc_next, int32_t log2L, void* workspace,
                    int64_t workspace_bytes, int64_t* offsets, uint16_t* states, void* sm,
                    int32_t* status, int64_t* result, void* stream, bool packed) {
    if (reinterpret_cast<uintptr_t>(fp8) % 16)
        return fail(TANS_EINVAL, "gpu_encode: fp8 must be 16-byte aligned");
    return gpu_encode_begin(RowSrc{(const uint8_t*)fp8, K, N, nullptr, 0}, fp8, K, N, enc_tab,
                            enc_next, log2L, workspace, workspace_bytes, offsets, states, sm,
                            status, result, stream, packed);
}

int gpu_encode_finish(int64_t K, int64_t N, int32_t log2L, const void* workspace,
                      const int64_t* offsets, void* comp, int64_t comp_bytes, void* stream,
                      bool packed) {
    int64_t need = 0;
    int rc = tans_gpu_encode_workspace(K, N, log2L, &need);
    if (rc) return rc;
    if (packed && (log2L != TANS_PAIR_LOG2L || N > 2 * tans_pack::kMaxSteps))
        return fail(TANS_EINVAL, "gpu_encode_packed: needs log2L 12 and N <= 64");
    if (!workspace || !offsets || !comp) return fail(TANS_EINVAL, "gpu_encode: null pointer");
    if (comp_bytes < kTailWords * 4 || comp_bytes % 4)
        return fail(TANS_EINVAL, "gpu_encode: comp must hold the stream words and the 1 KiB tail");
    hipStream_t st = (hipStream_t)stream;
    const int64_t words_total = comp_bytes / 4 - kTailWords;
    uint32_t* c32 = static_cast<uint32_t*>(comp);
    if (K > 0 && N > 0) {
        const int64_t G = (K + kLanes - 1) / kLanes;
        const WsLayout l = ws_layout(K, N, log2L);
        const char* ws = static_cast<const char*>(workspace);
        const dim3 grid((unsigned)((G + kEncBlock / kLanes - 1) / (kEncBlock / kLanes)));
        const uint32_t* rec = reinterpret_cast<const uint32_t*>(ws + l.rec);
        const uint32_t* ovf = reinterpret_cast<const uint32_t*>(ws + l.ovf);
        // (the place kernels zero the tail words too)
        if (packed)
            hipLaunchKernelGGL(enc_place_packed_kernel, grid, dim3(kEncBlock), 0, st, rec, ovf,
                               reinterpret_cast<const uint16_t*>(ws + l.pstate),
                               reinterpret_cast<const uint16_t*>(ws + l.plen), K, N,
                               (uint32_t)(1u << log2L), offsets, c32, words_total);
        else if (log2L == TANS_NIBBLE_LOG2L)
            hipLaunchKernelGGL(enc_place_kernel<1>, grid, dim3(kEncBlock), 0, st, rec, ovf, K, N,
                               offsets, c32, words_total);
        else
            hipLaunchKernelGGL(enc_place_kernel<2>, grid, dim3(kEncBlock), 0, st, rec, ovf, K, N,
                               offsets, c32, words_total);
        return hip_check(hipGetLastError(), "enc_place_kernel launch");
    }
    hipLaunchKernelGGL(zero_words_kernel, dim3((unsigned)((kTailWords + kEncBlock - 1) / kEncBlock)),
                       dim3(kEncBlock), 0, st, c32 + words_total, kTailWords);
    return hip_check(hipGetLastError(), "gpu_encode tail");
}

}  // namespace

extern "C" {

int tans_gpu_encode_begin(const void* fp8, int64_t K, int64_t N, const uint32_t* enc_tab,
                          const uint16_t* enc_next, int32_t log2L, void* workspace,
                          int64_t workspace_bytes, int64_t* offsets, uint16_t* states, void* sm,
                          int32_t* status, void* stream) {
    return gpu_encode_rows(fp8, K, N, enc_tab, enc_next, log2L, workspace, workspace_bytes,
                            offsets, states, sm, status, nullptr, stream, false);
}

int tans_gpu_encode_lanes_begin(const void* fp8, int64_t K, int64_t N, int32_t packed,
                                const uint32_t* enc_tab, const uint16_t* enc_next, int32_t log2L,
                                void* workspace, int64_t workspace_bytes, int64_t* offsets,
                                uint16_t* states, void* sm, int64_t* result, void* stream) {
    if (!result) return fail(TANS_EINVAL, "gpu_encode_lanes: null result");
    return gpu_encode_rows(fp8, K, N, enc_tab, enc_next, log2L, workspace, workspace_bytes,
                           offsets, states, sm, nullptr, result, stream, packed != 0);
}

int tans_gpu_encode_matrix_begin(const void* w, int64_t R, int64_t C, int64_t S, int64_t Nc,
                                 int32_t pad, const uint32_t* enc_tab, const uint16_t* enc_next,
                                 int32_t log2L, void* workspace, int64_t workspace_bytes,
                                 int64_t* offsets, uint16_t* states, void* sm, int64_t* result,
                                 void* stream) {
    if (!result) return fail(TANS_EINVAL, "gpu_encode_matrix: null result");
    if (R <= 0 || C < 16 || S <= 0 || Nc <= 0 || Nc % 32 || Nc > 1024)
        return fail(TANS_EINVAL, "gpu_encode_matrix: need R > 0, C >= 16 and segments of at most "
                                 "1024 columns, a multiple of 32");
    if (S > INT32_MAX || S * Nc < C || (S - 1) * Nc >= C)
        return fail(TANS_EINVAL, "gpu_encode_matrix: S segments of Nc columns must cover C exactly");
    if (pad < 0 || pad > 255) return fail(TANS_EINVAL, "gpu_encode_matrix: pad must be a byte");
    // (R and S within int32 and K checked against it: no product overflows)
    if (R > INT32_MAX) return fail(TANS_EINVAL, "gpu_encode_matrix: matrix too large");
    const int64_t Rp = (R + kLanes - 1) / kLanes * kLanes;
    if (S > INT32_MAX / (4 * Rp)) return fail(TANS_EINVAL, "gpu_encode_matrix: matrix too large");
    const MatSrc src{(const uint8_t*)w, R, C, (int)(Rp / 16), (int)Nc,
                     (uint32_t)pad * 0x01010101u, nullptr, nullptr, 0, 0, false};
    return gpu_encode_begin(src, w, 4 * S * Rp, Nc / 4, enc_tab, enc_next, log2L, workspace,
                            workspace_bytes, offsets, states, sm, nullptr, result, stream, false);
}

int tans_gpu_encode_finish(int64_t K, int64_t N, int32_t log2L, const void* workspace,
                           const int64_t* offsets, void* comp, int64_t comp_bytes, void* stream) {
    return gpu_encode_finish(K, N, log2L, workspace, offsets, comp, comp_bytes, stream, false);
}

int tans_gpu_encode_packed_begin(const void* fp8, int64_t K, int64_t N, const uint32_t* enc_tab,
                                 const uint16_t* enc_next, int32_t log2L, void* workspace,
                                 int64_t workspace_bytes, int64_t* offsets, void* sm,
                                 int32_t* status, void* stream) {
    return gpu_encode_rows(fp8, K, N, enc_tab, enc_next, log2L, workspace, workspace_bytes,
                            offsets, nullptr, sm, status, nullptr, stream, true);
}

int tans_gpu_encode_packed_finish(int64_t K, int64_t N, int32_t log2L, const void* workspace,
                                  const int64_t* offsets, void* comp, int64_t comp_bytes,
                                  void* stream) {
    return gpu_encode_finish(K, N, log2L, workspace, offsets, comp, comp_bytes, stream, true);
}

}  // extern "C"
