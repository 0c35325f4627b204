// attn_prefill.hip -- prefill attention (two or more query tokens) on the
// gfx950 matrix cores, fp16 or int8 KV cache, any head_dim up to 256.
//
// Replaces flash_attention_prefill_batched_kernel (reference
// src/kernels/attention.cu:180-290): token t, head h sees positions
// [0, start + t] of KV head h / group; fp32 softmax, fp16 out.
//
// Query rows.  The rows of one KV head are numbered t * group + j (token t,
// j-th head of the group), whatever the group is; a workgroup takes a block
// of 128 of them and a chunk of the KV tiles (64 positions), wave w of each
// wave group 32 rows.  With G = 2 wave groups (8 waves, two per SIMD) group q
// takes the chunk's tiles q, q + 2, ... with its own LDS buffers and online
// softmax, and the groups merge through LDS.
//
// Per tile (lane l: query row l % 32, half h = l / 32):
//   S^T = K . Q^T   v_mfma_f32_32x32x16_f16, src0 = 32 positions x 16 dims of
//                   K (LDS), src1 = Q^T (registers); the lane ends up with
//                   positions 32 pt + 8 j + 4 h + i, i < 4, j < 4;
//   softmax         the row's maximum from the two lane halves (one row
//                   swap); the reference point m of the exponentials moves
//                   only when the maximum has grown by more than 2^kLazy, so
//                   O is rarely rescaled; row sums stay per lane to the end;
//   O^T += V^T P^T  src0 = 32 dims x 16 positions of V^T (two
//                   ds_read_tr16_b64 of the row-major V), src1 = P^T straight
//                   from the score registers: k = 8 h + e stands for position
//                   16 kk + 8 (e / 4) + 4 h + e % 4 in both operands.  P is
//                   split into fp16 hi + lo (two MFMAs): 22 bits of the fp32
//                   probabilities down to 2^-35 of the reference point.
// int8 caches: P holds the V scales, so m follows the maximum of score + log2
// |scale|; O and l are relative to it all the same.  Scales in P without that ran
// into fp16's ends: 2000 positions of head_dim 96, error of the split against 64
// bits at scales around 1e-3 / 1e-4 / 1e-5 2.0e-4 / 2.0e-3 / 2.1e-2, with it 6.5e-8
// each (an fp16 output's own rounding is 2.0e-4 / 2.2e-4 / 1.1e-3), and NaN from a
// scale of 4094.
// Bound: the matrix cores (48 MFMAs of 32 cycles a tile and wave at head_dim
// 128) and the VALU's exponentials beside them.  32 query rows a wave halve
// the LDS fragment bytes per MFMA against 16 rows (1 KB per 32 cycles and
// SIMD, the LDS rate), which bounded a 16-row kernel.
//
// Staging.  A tile is loaded into registers one tile ahead (16 bytes of fp16 or
// 8 of int8 a thread and chunk; int8 is widened, exactly, on its way) and
// written to the other LDS buffer between the softmax and the P.V products;
// one barrier a tile.  Chunk c (8 dims, 16 bytes) of K row p sits at
// k_pos(p, c) and of V row p at v_pos(p, c), so that 16 lanes of a K fragment
// read and 32 lanes of a transposed V read cover the 64 banks once.  Dims past
// head_dim (up to the instance's padded size) are zeros.  (Direct-to-LDS
// copies need no registers, but the compiler waits for all of them before a
// transposing LDS read.)
//
// Splits.  With few query rows (a short message after a long cached context,
// a draft being checked) the KV tiles are cut into chunks over the chip, each
// workgroup leaves (O, m, l) in the workspace in register order and
// prefill_combine_kernel adds the chunks in order; plan_prefill picks the
// chunk.
//
// Measured, 32 / 8 heads of 128, fp16 cache, other inputs each call, against the
// 16-row kernel of attn.hip (never split): 45 tokens after 8000 positions 125.5 ->
// 22.6 us, 128 after 16000 247 -> 61.5, 1000 from 0 31.4 -> 27.1, 2048 from 0 99.3 ->
// 60.8, 4096 from 0 337 -> 216 (636 TFLOP/s); int8 2048 from 0 141 -> 69.4; head_dim
// 80 and 256 against the VALU kernel, 512 tokens 115 -> 13.5 and 269 -> 39.7.
// Timing-only variants (replays of one input, which run up to a fifth longer) of an
// unsplit 8000-position walk (2.6 us per two tiles): without the tile loads
// 2.3, without the exponentials 2.5, without P.V 1.8, without the low half of
// P 2.2 us.  Not kept: half tiles of 32 positions with the next half's scores
// between this half's exponentials (8000 positions 163 -> 180 us), one wave
// group and two workgroups a CU (163 -> 225 us unsplit, 2048 tokens 68 -> 73),
// the second group one phase behind (148 us there, equal elsewhere, and the
// head_dim 256 instance spills: 512 after 4096 104 -> 122 us).
#include <math.h>

#include <algorithm>
#include <atomic>
#include <type_traits>

#include "launch.h"
#include "mfma_util.h"
#include "q4k_device.h"

namespace rxq4 {
namespace {

typedef short v4i16 __attribute__((ext_vector_type(4)));

constexpr int kTile = 64;    // positions per tile
constexpr int kBlock = 128;  // query rows per workgroup
constexpr int kMaxChunks = 64;  // KV chunks per block
// The reference point m of a row's exponentials moves when the row's maximum has
// outgrown it by 2^kLazy, and P holds 2^kShift times them, up to 2^(kLazy +
// kShift) = 2^15: fp16's range is used from its top (65504) and the low half of
// P ends at 2^-24 = 2^-35 of the reference point.
constexpr float kLazy = 4.0f;
constexpr float kShift = 11.0f;
// V scales below 2^kMinScale count as that where the reference point is chosen
// (what they weigh is 0 in an fp16 output) and those above 2^kMaxScale as that.
constexpr float kMinScale = -40.0f, kMaxScale = 127.0f;
// An int8 tile's floats in LDS: K scales, V scales, log2 |V scale|.
constexpr int kScl = 3 * kTile;

struct PrefillParams {
    uint16_t *out;
    const uint16_t *q;
    const void *k, *v;
    const float *ks, *vs;
    f32x4 *part;   // splits > 1: O pieces [kv][block][chunk][wave][HD / 8][64 lanes]
    float *stats;  // ... and [kv][block][chunk][wave][m, l][32 rows]
    int n_heads, n_kv, hd, group, n_tok, start;
    int n_blocks, n_chunks, chunk_tiles;
    float sl2;     // |scale| * log2(e), positive
    int negate;    // scale < 0: q enters negated
};

typedef const float __attribute__((address_space(1))) *GlobalFloat;
__device__ const float g_one = 1.0f;  // int8 caches without scales: read with stride 0

__device__ __forceinline__ f32x16 mfma32h(u32x4 a, u32x4 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a),
                                                  __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}

// Infinities and NaN among N x 8 fp16: whether there are any (times 0 they are
// NaN), and zeros in their place (a half with all exponent bits set carries into
// its top bit).
template <int N>
__device__ __forceinline__ bool not_finite16(const u32x4 *x) {
    f16x2 sum[4] = {};
#pragma unroll
    for (int j = 0; j < N; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t v = x[j][i];  // (a bit cast of the vector's element itself takes element 0)
            sum[i] = __builtin_elementwise_fma(__builtin_bit_cast(f16x2, v), f16x2{0, 0}, sum[i]);
        }
    const f16x2 all = (sum[0] + sum[1]) + (sum[2] + sum[3]);
    return !(all.x == 0) || !(all.y == 0);
}
template <int N>
__device__ __forceinline__ void zero_not_finite16(u32x4 *x) {
#pragma unroll
    for (int j = 0; j < N; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t all = (((x[j][i] & 0x7C007C00u) + 0x04000400u) >> 15) & 0x00010001u;
            x[j][i] &= ~(all * 0xFFFFu);
        }
}

// Token and head of query row row0 + r (r < 32), from the uniform division of
// row0: the quotient of rem0 + r < group + 32 by the group from a reciprocal
// ((x + 0.5) / group is at least 0.5 / group from an integer, far more than
// the reciprocal's error).
struct RowMap {
    int tok0, rem0, group;
    float rcp;
    __device__ void at(int r, int &tok, int &head) const {
        const int x = rem0 + r;
        const int q = (int)(((float)x + 0.5f) * rcp);
        tok = tok0 + q;
        head = x - q * group;
    }
};
__device__ __forceinline__ RowMap row_map(int row0, int group) {
    const int t = row0 / group;
    return RowMap{t, row0 - t * group, group, __builtin_amdgcn_rcpf((float)group)};
}

// Place of 16-byte chunk c of row p in the LDS row (HD fp16).
template <int HD>
__device__ __forceinline__ int k_pos(int p, int c) {
    if (HD == 64) return c ^ ((p >> 1) & 7);            // two rows cover the banks
    if (HD == 96) return (c & ~3) | ((c ^ (p >> 2)) & 3);  // rows p, p + 4, .. share a bank window
    return c ^ (p & 15);                                // a row (or half of it) covers them
}
template <int HD>
__device__ __forceinline__ int v_pos(int p, int c) {
    if (HD == 64) return c ^ (((p >> 1) & 1) << 2);
    if (HD == 96) return c;
    return c ^ ((p & 3) << 2);
}

// 4 int8 of w (xor 0x80 gives x + 128) as fp16: 0x6400 | byte = 1024 + byte
// exactly, and the subtraction is exact.
__device__ __forceinline__ u32x2 i8x4_to_f16(uint32_t w) {
    const uint32_t u = w ^ 0x80808080u;
    const half2_t off = as_half2(0x64806480u);  // 1152
    const half2_t a = as_half2(__builtin_amdgcn_perm(0x64646464u, u, 0x04010400u)) - off;
    const half2_t b = as_half2(__builtin_amdgcn_perm(0x64646464u, u, 0x04030402u)) - off;
    return u32x2{__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b)};
}

// Bytes of one K or V tile and of a wave group's LDS (two buffers of K, V).
template <int HD>
constexpr int tile_bytes() { return kTile * HD * 2; }
template <int HD, int G>
constexpr int prefill_lds() {
    return G * 4 * tile_bytes<HD>()      // K, V x 2 buffers
           + G * 2 * kScl * 4            // int8 scales
           + 2 * 256 * 4                 // (m, l) of the second group
           + G * 4 * 4;                  // a wave's flag: V not finite
}

template <int HD, bool I8, int G>
__global__ __launch_bounds__(256 * G) void attn_prefill_kernel(PrefillParams p) {
    constexpr int KS = HD / 16;             // k-steps of the scores
    constexpr int DT = HD / 32;             // 32-dim tiles of O
    constexpr int TB = tile_bytes<HD>();
    constexpr int CH = HD / 8;              // 16-byte chunks per row
    constexpr int NC = kTile * CH / 256;    // 8-dim chunks per thread and tile (K, V each)
    constexpr int esz = I8 ? 1 : 2;
    extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];

    const int gq = G == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
    const int tid = threadIdx.x & 255, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r32 = lane & 31, h = lane >> 5;
    uint8_t *const lds = smem + gq * 4 * TB;  // buffer b: K at 2 b TB, V at (2 b + 1) TB
    float *const scl = reinterpret_cast<float *>(smem + G * 4 * TB) + gq * 2 * kScl;
    float *const mgl = reinterpret_cast<float *>(smem + G * 4 * TB + G * 8 * kScl);
    int *const bad_v = reinterpret_cast<int *>(mgl + 512) + gq * 4;

    // Unit: longest blocks (the latest tokens) first.
    const int kvh = blockIdx.x % p.n_kv;
    const int v0 = blockIdx.x / p.n_kv;
    const int block = p.n_blocks - 1 - v0 % p.n_blocks;
    const int chunk = v0 / p.n_blocks;
    const int n_rows = p.n_tok * p.group;
    const int blk_last = min(n_rows, (block + 1) * kBlock) - 1;
    const int pos_end = p.start + blk_last / p.group + 1;  // positions the block sees
    const int t_beg = chunk * p.chunk_tiles;
    const int t_end = min((pos_end + kTile - 1) / kTile, t_beg + p.chunk_tiles);
    if (t_beg >= t_end) return;  // uniform

    // The lane's query row.
    const int row0 = block * kBlock + 32 * w;
    const bool live_wave = row0 < n_rows;
    const RowMap rm = row_map(min(row0, n_rows - 1), p.group);
    int tok, hj, tok_last, unused;
    rm.at(min(r32, max(0, n_rows - 1 - row0)), tok, hj);
    rm.at(min(31, max(0, n_rows - 1 - row0)), tok_last, unused);
    const int qpos = p.start + tok;  // last visible position
    const int wave_first = p.start + rm.tok0;
    const int wave_end = live_wave ? p.start + __builtin_amdgcn_readfirstlane(tok_last) + 1 : 0;
    const int64_t row_stride = (int64_t)p.n_kv * p.hd * esz;
    const uint8_t *kb = static_cast<const uint8_t *>(p.k) + (int64_t)kvh * p.hd * esz;
    const uint8_t *vb = static_cast<const uint8_t *>(p.v) + (int64_t)kvh * p.hd * esz;
    // (global pointers: a generic load would be waited for with the LDS reads)
    const GlobalFloat ksp = p.ks ? (GlobalFloat)(p.ks + kvh) : (GlobalFloat)&g_one;
    const GlobalFloat vsp = p.vs ? (GlobalFloat)(p.vs + kvh) : (GlobalFloat)&g_one;
    const int s_stride = p.ks ? p.n_kv : 0, v_stride = p.vs ? p.n_kv : 0;
    const int n_ch = p.hd >> 3;
    const int blk_first = p.start + block * kBlock / p.group;  // first query position of the block

    // Q^T fragments: dims 16 ks + 8 h .. + 7 of the row (zeros past hd).
    u32x4 qf[KS];
    {
        const uint16_t *qrow = p.q + ((int64_t)tok * p.n_heads + kvh * p.group + hj) * p.hd;
        const uint32_t flip = p.negate ? 0x80008000u : 0u;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            const int c = 2 * ks + h;
            u32x4 x = *reinterpret_cast<const u32x4 *>(qrow + 8 * min(c, n_ch - 1));
            x = u32x4{x.x ^ flip, x.y ^ flip, x.z ^ flip, x.w ^ flip};
            qf[ks] = c < n_ch ? x : u32x4{0u, 0u, 0u, 0u};
        }
    }

    // The thread's chunks of a tile: source offset within the tile's rows
    // (past the resource for dims past head_dim: zeros), LDS offsets.  Where a row
    // divides the 256 chunks, chunk j is kRows rows down and the places in a K row
    // repeat every kPerK chunks: only what differs is kept.
    constexpr bool kEven = 256 % CH == 0;
    constexpr int kRows = 256 / CH, kPer = kEven ? 1 : NC, kPerK = kEven && kRows % 16 ? 16 / kRows : kPer;
    static_assert(!kEven || kRows % 4 == 0, "the places in a V row repeat");
    int io[kPer], ik[kPerK], iv[kPer];
#pragma unroll
    for (int j = 0; j < kPerK; ++j) {
        const int id = tid + 256 * j, pr = id / CH, c = id % CH;
        ik[j] = pr * HD * 2 + 16 * k_pos<HD>(pr, c);
        if (j >= kPer) continue;
        io[j] = c < n_ch ? (int)(pr * row_stride) + 8 * esz * c : 0x7FFFFFF0;
        iv[j] = pr * HD * 2 + 16 * v_pos<HD>(pr, c);
    }
    const int io_step = tid % CH < n_ch ? kRows * (int)row_stride : 0;
    auto chunk_src = [&](int j) { return kEven ? io[0] + j * io_step : io[j % kPer]; };
    auto chunk_k = [&](int j) { return ik[j % kPerK] + (kEven ? j / kPerK * kPerK * kRows * HD * 2 : 0); };
    auto chunk_v = [&](int j) { return kEven ? iv[0] + j * kRows * HD * 2 : iv[j % kPer]; };
    // resources over a tile's visible rows (rows past them read zeros); the
    // base and bound are wave-uniform
    auto tile_rsrc = [&](const uint8_t *base, int p0) {
        const int bytes = __builtin_amdgcn_readfirstlane(
            (int)((min(pos_end - p0, kTile) - 1) * row_stride + p.hd * esz));
        const int64_t off = (int64_t)p0 * row_stride;
        const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)off);
        const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(off >> 32));
        return make_rsrc(base + (int64_t)(((uint64_t)hi << 32) | lo), bytes);
    };
    using Chunk = typename std::conditional<I8, u32x2, u32x4>::type;
    struct Raw {
        Chunk c[NC];
        float s;
    };
    auto load_raw = [&](const uint8_t *base, GlobalFloat scales, int stride, int t, Raw &R) {
        const __amdgpu_buffer_rsrc_t rs = tile_rsrc(base, t * kTile);
#pragma unroll
        for (int j = 0; j < NC; ++j) {
            if constexpr (I8) R.c[j] = buffer_load8(rs, chunk_src(j));
            else R.c[j] = buffer_load16(rs, chunk_src(j));
        }
        if (I8) R.s = scales[(int64_t)min(t * kTile + lane, pos_end - 1) * stride];  // (every wave)
    };
    auto widen = [](Chunk c) {
        if constexpr (I8) {
            const u32x2 a = i8x4_to_f16(c.x), b = i8x4_to_f16(c.y);
            return u32x4{a.x, a.y, b.x, b.y};
        } else {
            return c;
        }
    };
    auto store_raw = [&](const Raw &R, int off, auto place, int s_off) {
#pragma unroll
        for (int j = 0; j < NC; ++j) *reinterpret_cast<u32x4 *>(lds + off + place(j)) = widen(R.c[j]);
        if (I8 && tid < kTile) scl[s_off + tid] = R.s;
    };
    // log2 |V scale| of the tile's positions, clamped, and a bound of theirs that
    // seldom moves (a maximum over the lanes for every tile costs 3%).  None for
    // the first tile, where the row's maximum is taken exactly in any case.
    float most_log = kMaxScale;
    auto store_log = [&](float vs, int s_off, bool first) {
        if constexpr (I8) {
            const float lg = fminf(fmaxf(__builtin_amdgcn_logf(fabsf(vs)), kMinScale), kMaxScale);
            if (!first && (__builtin_amdgcn_ballot_w64(lg > most_log) != 0 || most_log >= kMaxScale))
                most_log = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(
                               int, butterfly_max<64>(lg) + 0.125f)));
            if (tid < kTile) scl[s_off + tid] = lg;
        }
    };

    // Positions that some row of the block does not see: a zero probability does
    // not stop an infinity or NaN there in the P.V products.  On the tiles that
    // hold such positions those V values (int8: V scales) are staged again as
    // zeros, and the rows that see them get them at the end.  (Looked over after
    // their LDS writes have gone out: 300 tokens after 700 at head_dim 96 15.5 ->
    // 15.7 us, 2048 from 0 at 128 60.4 -> 60.9; rows of a clean cache bit for bit.)
    if (lane == 0) bad_v[w] = 0;  // the wave's flag: some of its staging
    auto look_over = [&](Raw &R, int t, int off, int s_off) {
        if (t * kTile + kTile - 1 <= blk_first) return;  // uniform
        if constexpr (I8) {
            const bool bad = !(fabsf(R.s) < INFINITY);
            if (__builtin_amdgcn_ballot_w64(bad) == 0) return;
            if (bad && tid < kTile) scl[s_off + tid] = 0.0f;
        } else {
            if (__builtin_amdgcn_ballot_w64(not_finite16<NC>(R.c)) == 0) return;
            Raw Z = R;  // (copies: head_dim 80, 775 tokens, 20.2 us with the loaded registers changed in place, 19.5)
#pragma unroll
            for (int j = 0; j < NC; ++j) asm volatile("" : "+v"(Z.c[j]));
            zero_not_finite16<NC>(Z.c);
            store_raw(Z, off, chunk_v, s_off);
        }
        if (lane == 0) bad_v[w] = 1;
    };

    // Lane parts of the fragment addresses: K row 32 pt + r32, chunk
    // 2 ks + h; V row 16 kk + 8 x + 4 h + (r16 / 4), dims 32 dt + 16 (l / 16 % 2)
    // + 4 (r16 % 4) (the transposing read hands the lane dim 32 dt + r32).
    const int r16 = lane & 15;
    int ka[KS], va[DT];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) ka[ks] = r32 * HD * 2 + 16 * k_pos<HD>(r32, 2 * ks + h);
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
        const int vr = 4 * h + (r16 >> 2), d = 32 * dt + 16 * ((lane >> 4) & 1) + 4 * (r16 & 3);
        va[dt] = vr * HD * 2 + 16 * v_pos<HD>(vr, d >> 3) + 2 * (d & 7);
    }

    f32x16 o[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) o[dt] = f32x16{};
    float m = -INFINITY, l = 0.0f;  // l: this lane's positions only

    u32x4 ph[4], pl[4];  // P^T hi / lo operands per 16-position k step
    auto softmax = [&](int t, int b) {
        const int p0 = t * kTile;
        const uint8_t *kt = lds + b * 2 * TB;
        f32x16 s[2];
#pragma unroll
        for (int pt = 0; pt < 2; ++pt) {
            s[pt] = f32x16{};
#pragma unroll
            for (int ks = 0; ks < KS; ++ks)
                s[pt] = mfma32h(*reinterpret_cast<const u32x4 *>(kt + ka[ks] + pt * 64 * HD), qf[ks], s[pt]);
        }
        if constexpr (I8) {
            const float *sk = scl + b * kScl;
#pragma unroll
            for (int pt = 0; pt < 2; ++pt)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const f32x4 x = *reinterpret_cast<const f32x4 *>(sk + 32 * pt + 8 * j + 4 * h);
#pragma unroll
                    for (int i = 0; i < 4; ++i) s[pt][4 * j + i] *= x[i];
                }
        }
        if (p0 + kTile - 1 > wave_first) {  // uniform: the diagonal's tiles
#pragma unroll
            for (int pt = 0; pt < 2; ++pt)
#pragma unroll
                for (int i = 0; i < 16; ++i)
                    if (p0 + 32 * pt + 8 * (i >> 2) + 4 * h + (i & 3) > qpos) s[pt][i] = -INFINITY;
        }
        // the row's largest P in log2 units: the score, with V scales score +
        // log2 |scale|, at most the largest of each together
        float mx = -INFINITY;
#pragma unroll
        for (int pt = 0; pt < 2; ++pt)
#pragma unroll
            for (int i = 0; i < 16; ++i) mx = fmaxf(mx, s[pt][i]);
        mx = max_xor_rows<32>(mx) * p.sl2;
        if constexpr (I8) {
            const float *sg = scl + b * kScl + 2 * kTile;
            if (__builtin_amdgcn_ballot_w64(mx + most_log > m + kLazy) != 0) {  // m may have to move: exactly
                mx = -INFINITY;
#pragma unroll
                for (int pt = 0; pt < 2; ++pt)
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const f32x4 x = *reinterpret_cast<const f32x4 *>(sg + 32 * pt + 8 * j + 4 * h);
#pragma unroll
                        for (int i = 0; i < 4; ++i)
                            mx = fmaxf(mx, __builtin_fmaf(s[pt][4 * j + i], p.sl2, x[i]));
                    }
                mx = max_xor_rows<32>(mx);
            } else {
                mx = -INFINITY;
            }
        }
        // m moves when the row's maximum has outgrown it by 2^kLazy (always
        // at a row's first visible position): |P| <= 2^(kLazy + kShift), and O
        // and l stay relative to the same m
        if (__builtin_amdgcn_ballot_w64(mx > m + kLazy) != 0) {
            // (each row's by its own rule: no row depends on what others see)
            const float m_new = mx > m + kLazy ? mx : m;
            const float corr = m_new == -INFINITY ? 1.0f : __builtin_amdgcn_exp2f(m - m_new);
            m = m_new;
            l *= corr;
#pragma unroll
            for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                for (int i = 0; i < 16; ++i) o[dt][i] *= corr;
        }
        const float m_use = m == -INFINITY ? 0.0f : m - kShift;  // rows with nothing visible yet: e = 0
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) {
            f32x4 x0, x1;
            if constexpr (I8) {
                const float *sv = scl + b * kScl + kTile;
                x0 = *reinterpret_cast<const f32x4 *>(sv + 16 * kk + 4 * h);
                x1 = *reinterpret_cast<const f32x4 *>(sv + 16 * kk + 8 + 4 * h);
            }
#pragma unroll
            for (int e = 0; e < 8; e += 2) {
                const int i = 8 * (kk & 1) + e;  // register of k = e
                float e0 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[kk >> 1][i], p.sl2, -m_use));
                float e1 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[kk >> 1][i + 1], p.sl2, -m_use));
                l += e0;
                l += e1;
                if constexpr (I8) {
                    e0 *= e < 4 ? x0[e] : x1[e - 4];
                    e1 *= e < 4 ? x0[e + 1] : x1[e - 3];
                }
                const uint32_t hi = pack2<RXQ4_DTYPE_F16>(e0, e1);
                // lo = RNE_f16(e - f32(hi)): the difference is exact in fp32
                uint32_t lo;
                asm("v_fma_mixlo_f16 %0, %1, 1.0, -%2 op_sel_hi:[0,0,1]" : "=v"(lo) : "v"(e0), "v"(hi));
                asm("v_fma_mixhi_f16 %0, %1, 1.0, -%2 op_sel:[0,0,1] op_sel_hi:[0,0,1]"
                    : "+v"(lo) : "v"(e1), "v"(hi));
                ph[kk][e >> 1] = hi;
                pl[kk][e >> 1] = lo;
            }
        }
    };
    auto weigh = [&](int b) {
        const uint8_t *vt = lds + (b * 2 + 1) * TB;
#pragma unroll
        for (int kk = 0; kk < 4; ++kk)
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) {
                const uint8_t *vp = vt + va[dt] + kk * 32 * HD;
                const u32x2 v0 = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                                                               (__attribute__((address_space(3))) v4i16 *)vp));
                const u32x2 v1 = __builtin_bit_cast(
                    u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                               (__attribute__((address_space(3))) v4i16 *)(vp + 16 * HD)));
                const u32x4 a = u32x4{v0.x, v0.y, v1.x, v1.y};
                o[dt] = mfma32h(a, ph[kk], o[dt]);
                o[dt] = mfma32h(a, pl[kk], o[dt]);
            }
    };

    // Tiles t_beg + gq, + G, ...: tile j of the group is in buffer j & 1
    // during iteration j, and tile j + 1 is written to the other one, which
    // every wave has left at the barrier.  A tile past the wave's visible
    // positions changes nothing and is skipped.
    const int n_j = (t_end - t_beg - gq + G - 1) / G;  // this group's tiles
    const int n_it = (t_end - t_beg + G - 1) / G;      // every group's iterations
    const int t_first = t_beg + gq;
    Raw K, V;
    auto load_tile = [&](int t) {
        load_raw(kb, ksp, s_stride, t, K);
        load_raw(vb, vsp, v_stride, t, V);
    };
    auto store_tile = [&](int t, int b, bool first) {
        store_raw(K, b * 2 * TB, chunk_k, b * kScl);
        store_raw(V, (b * 2 + 1) * TB, chunk_v, b * kScl + kTile);
        store_log(V.s, b * kScl + 2 * kTile, first);
        look_over(V, t, (b * 2 + 1) * TB, b * kScl + kTile);
    };
    if (n_j > 0) {
        load_tile(t_first);
        store_tile(t_first, 0, true);
    }
    for (int j = 0; j < n_it; ++j) {
        wait_lgkmcnt0();
        lds_barrier();
        const int t = t_first + G * j;
        const bool next = j + 1 < n_j;
        const bool live = j < n_j && t * kTile < wave_end;  // uniform
        if (next) load_tile(t + G);
        if (live) softmax(t, j & 1);
        if (next) store_tile(t + G, (j + 1) & 1, false);
        if (live) weigh(j & 1);
    }
    wait_lgkmcnt0();
    lds_barrier();
    if (__builtin_amdgcn_readfirstlane(bad_v[0] | bad_v[1] | bad_v[2] | bad_v[3]) != 0) {
        for (int t = max(t_beg, (blk_first + 1) / kTile); t < t_end; ++t) {
            if ((t - t_beg) % G != gq) continue;
            for (int pos = t * kTile; pos < min(wave_end, t * kTile + kTile); ++pos) {
                const uint8_t *row = vb + pos * row_stride + 4 * esz * h;
                const float vs = I8 ? vsp[(int64_t)pos * v_stride] : 1.0f;
                if (pos > qpos || (I8 && fabsf(vs) < INFINITY)) continue;
                int n = n_ch;
                asm volatile("" : "+s"(n));  // (compared here, not kept as CH conditions)
#pragma unroll
                for (int c = 0; c < CH; ++c) {
                    if (c >= n) continue;  // uniform
                    const u32x2 x = I8 ? u32x2{*reinterpret_cast<const uint32_t *>(row + 8 * c), 0u}
                                       : *reinterpret_cast<const u32x2 *>(row + 16 * c);
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const float v = I8 ? vs * (float)(int8_t)(x.x >> (8 * i))
                                           : f16_bits_to_f32((i < 2 ? x.x : x.y) >> (16 * (i & 1)) & 0xFFFFu);
                        if (!(fabsf(v) < INFINITY)) o[c / 4][4 * (c % 4) + i] += v;
                    }
                }
            }
        }
    }

    // Merge: the second group hands (O, m, l) over through its own buffers.
    l = sum_xor_rows<32>(l);
    if (G == 2) {
        float *mb = reinterpret_cast<float *>(smem + 4 * TB);  // HD / 2 x 256 floats
        if (gq == 1) {
#pragma unroll
            for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                for (int i = 0; i < 16; ++i) mb[(16 * dt + i) * 256 + tid] = o[dt][i];
            mgl[tid] = m;
            mgl[256 + tid] = l;
        }
        wait_lgkmcnt0();
        lds_barrier();
        if (gq == 1) return;
        const float m1 = mgl[tid], l1 = mgl[256 + tid];
        const float mm = fmaxf(m, m1);
        const bool any = mm != -INFINITY;
        const float c0 = any ? __builtin_amdgcn_exp2f(m - mm) : 0.0f;
        const float c1 = any ? __builtin_amdgcn_exp2f(m1 - mm) : 0.0f;
        l = l * c0 + l1 * c1;
        m = mm;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int i = 0; i < 16; ++i) o[dt][i] = o[dt][i] * c0 + mb[(16 * dt + i) * 256 + tid] * c1;
    }
    if (!live_wave) return;
    if (p.n_chunks > 1) {
        const int64_t u = ((int64_t)(kvh * p.n_blocks + block) * p.n_chunks + chunk) * 4 + w;
        f32x4 *part = p.part + u * (CH * 64) + lane;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int j = 0; j < 4; ++j)
                part[(4 * dt + j) * 64] =
                    f32x4{o[dt][4 * j], o[dt][4 * j + 1], o[dt][4 * j + 2], o[dt][4 * j + 3]};
        if (h == 0) {
            p.stats[u * 64 + r32] = m;
            p.stats[u * 64 + 32 + r32] = l;
        }
        return;
    }
    // Output rows through the wave's own LDS rows: 16 bytes a lane, a row's
    // bytes together (straight from the registers: 8-byte pieces of 32 rows).
    const float inv = l > 0.0f ? 1.0f / l : 0.0f;
    constexpr int OP = 2 * HD + 16;  // LDS pitch of a staged row
    static_assert(4 * 32 * OP <= 4 * TB, "the staged rows fit the group's buffers");
    uint8_t *ow = lds + w * 32 * OP;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const uint32_t a = pack2<RXQ4_DTYPE_F16>(o[dt][4 * j] * inv, o[dt][4 * j + 1] * inv);
            const uint32_t c = pack2<RXQ4_DTYPE_F16>(o[dt][4 * j + 2] * inv, o[dt][4 * j + 3] * inv);
            *reinterpret_cast<u32x2 *>(ow + r32 * OP + 2 * (32 * dt + 8 * j + 4 * h)) = u32x2{a, c};
        }
    wait_lgkmcnt0();
#pragma unroll
    for (int i = 0; i < 32 * CH / 64; ++i) {
        const int id = lane + 64 * i, rr = id / CH, c = id % CH;
        const int orow = row0 + rr;
        if (orow < n_rows && c < n_ch) {
            int t, jj;
            rm.at(rr, t, jj);
            *reinterpret_cast<u32x4 *>(p.out + ((int64_t)t * p.n_heads + kvh * p.group + jj) * p.hd + 8 * c) =
                *reinterpret_cast<const u32x4 *>(ow + rr * OP + 16 * c);
        }
    }
}

// out = sum_c 2^(m_c - M) O_c / sum_c 2^(m_c - M) l_c over a block's chunks in
// order.  Workgroup: 32 query rows (a wave of the attention kernel) and four
// of the HD / 8 register pieces, one per wave, so every load is the coalesced
// mirror of a store.  The chunks' weights are formed once per workgroup: thread
// (k, r) takes the chunks k, k + 8, .. of row r; all sums have fixed orders.
template <int HD>
__global__ __launch_bounds__(256) void prefill_combine_kernel(PrefillParams p) {
    constexpr int CH = HD / 8, CG = CH / 4;
    __shared__ float wgt[kMaxChunks][32], red[2][8][32];
    const int tid = threadIdx.x, lane = tid & 63, r32 = lane & 31, h = lane >> 5;
    const int pg = blockIdx.x % CG, bw = blockIdx.x / CG, w = bw & 3, kb = bw >> 2;
    const int block = kb % p.n_blocks, kvh = kb / p.n_blocks;
    const int n_rows = p.n_tok * p.group;
    const int row0 = block * kBlock + 32 * w;
    if (row0 >= n_rows) return;
    const int blk_last = min(n_rows, (block + 1) * kBlock) - 1;
    const int tiles = (p.start + blk_last / p.group + kTile) / kTile;
    const int n_c = (tiles + p.chunk_tiles - 1) / p.chunk_tiles;
    const int64_t u0 = (int64_t)kb * p.n_chunks * 4 + w;
    // the first O pieces go out before the weights' round trip
    const f32x4 *src = p.part + (u0 * CH + 4 * pg + (tid >> 6)) * 64 + lane;
    constexpr int U = 8;
    f32x4 x[U];
#pragma unroll
    for (int i = 0; i < U; ++i) x[i] = src[(int64_t)min(i, n_c - 1) * (4 * CH * 64)];
    {
        const int r = tid & 31, k = tid >> 5;
        const float *st = p.stats + u0 * 64 + r;
        float mc[kMaxChunks / 8], lc[kMaxChunks / 8], mx = -INFINITY;
#pragma unroll
        for (int i = 0; i < kMaxChunks / 8; ++i) {
            const int c = min(k + 8 * i, n_c - 1);
            mc[i] = st[(int64_t)c * 256];
            lc[i] = st[(int64_t)c * 256 + 32];
        }
#pragma unroll
        for (int i = 0; i < kMaxChunks / 8; ++i) mx = fmaxf(mx, mc[i]);  // repeats change nothing
        red[0][k][r] = mx;
        __syncthreads();
        float M = red[0][0][r];
#pragma unroll
        for (int i = 1; i < 8; ++i) M = fmaxf(M, red[0][i][r]);
        float L = 0.0f;
#pragma unroll
        for (int i = 0; i < kMaxChunks / 8; ++i) {
            const int c = k + 8 * i;
            if (c < n_c) {
                const float e = M != -INFINITY ? __builtin_amdgcn_exp2f(mc[i] - M) : 0.0f;
                wgt[c][r] = e;
                L += e * lc[i];
            }
        }
        red[1][k][r] = L;
        __syncthreads();
    }
    float L = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; ++i) L += red[1][i][r32];
    f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int c0 = 0; c0 < n_c; c0 += U) {
        f32x4 nx[U];
#pragma unroll
        for (int i = 0; i < U; ++i) nx[i] = src[(int64_t)min(c0 + U + i, n_c - 1) * (4 * CH * 64)];
#pragma unroll
        for (int i = 0; i < U; ++i) {
            const float e = c0 + i < n_c ? wgt[c0 + i][r32] : 0.0f;
            if (c0 + i < n_c)
                acc = f32x4{acc[0] + e * x[i][0], acc[1] + e * x[i][1], acc[2] + e * x[i][2],
                            acc[3] + e * x[i][3]};
        }
#pragma unroll
        for (int i = 0; i < U; ++i) x[i] = nx[i];
    }
    const int d = 8 * (4 * pg + (tid >> 6)) + 4 * h;  // piece 4 dt + j: dims 32 dt + 8 j + 4 h
    if (row0 + r32 >= n_rows || d >= p.hd) return;
    const float inv = L > 0.0f ? 1.0f / L : 0.0f;
    int t, j;
    row_map(row0, p.group).at(r32, t, j);
    uint16_t *o = p.out + ((int64_t)t * p.n_heads + kvh * p.group + j) * p.hd + d;
    *reinterpret_cast<u32x2 *>(o) = u32x2{pack2<RXQ4_DTYPE_F16>(acc[0] * inv, acc[1] * inv),
                                          pack2<RXQ4_DTYPE_F16>(acc[2] * inv, acc[3] * inv)};
}

// Launch model, microseconds: a workgroup's fixed part and its tiles, the
// workgroups' rounds over the CUs and, for splits, the second launch and the
// partials' way through memory.  Two sets of constants.  kSplit picks the split; its
// workgroups are slower than those of a launch alone, which keeps launches of
// several rounds from being cut too finely (with the second set for both, int8 1050
// tokens, 32 / 8 heads of 64: 28.4 -> 39.2 us, 775 of 16 / 4 heads of 80 19.2 ->
// 22.8).  The other gives the plan's time, against the other kernels' in the
// dispatch, fitted to launches of 2 to 1500 tokens after 0 to 1500 positions: model
// and measured, 32 / 8 heads of 128, fp16, 200 tokens 11.3 / 10.9, 512 16.6 / 16.6,
// 400 after 400 23.2 / 23.0, 45 after 400 13.0 / 13.1 (4 chunks), 45 after 700 14.1 /
// 14.0 (6), 130 after 600 18.3 / 18.7 (3).
struct Cost {
    double fixed, tile, second, partials;  // partials: bytes a microsecond
};
Cost split_cost(int hd_pad) {
    if (hd_pad == 64) return {4.7, 0.93, 3.0, 3.5e6};
    if (hd_pad == 96) return {5.5, 1.15, 3.0, 3.5e6};
    if (hd_pad == 128) return {6.5, 1.3, 3.0, 3.5e6};
    return {6.0, 4.3, 3.0, 3.5e6};
}
Cost time_cost(int hd_pad, int kv_int8) {
    if (hd_pad == 64) return {kv_int8 ? 5.3 : 4.3, kv_int8 ? 1.2 : 0.93, 2.4, 2.6e6};
    if (hd_pad == 96) return {kv_int8 ? 5.6 : 4.8, kv_int8 ? 1.3 : 1.1, 2.4, 2.6e6};
    if (hd_pad == 128) return {kv_int8 ? 6.8 : 6.0, kv_int8 ? 1.55 : 1.32, 2.4, 2.6e6};
    return {kv_int8 ? 6.3 : 5.9, kv_int8 ? 4.5 : 4.3, 2.4, 2.6e6};
}
// `tiles` the longest workgroup's, `work` and `units` all workgroups' tiles and
// number, `bytes` of partials (0: no split).
double launch_us(const Cost &k, int tiles, double work, double units, double bytes, int cus) {
    double us = k.fixed + k.tile * tiles;
    if (units > cus) us = std::max(us, (k.tile * work + 0.5 * k.fixed * units) / cus) + 0.3 * us;
    return bytes > 0 ? us + k.second + bytes / k.partials : us;
}

// The cheapest chunk of KV tiles per workgroup (a multiple of the G wave
// groups) under the model.
PrefillPlan plan_prefill(int64_t rows, int group, int n_kv, int start, int n_tok, int hd_pad, int G,
                         int kv_int8, int cus, size_t room) {
    const int tiles = (start + n_tok + kTile - 1) / kTile;
    const int64_t blocks = (rows + kBlock - 1) / kBlock;
    const int64_t step = (blocks + 7) / 8;  // up to eight blocks stand for all
    const Cost pick = split_cost(hd_pad), time = time_cost(hd_pad, kv_int8);
    PrefillPlan best{tiles, 1, 0};
    double best_pick = 0;
    int last = 0;
    const int most = tuning().attn_split ? std::min(kMaxChunks, tuning().attn_split) : kMaxChunks;
    // 1, 2, 3, 4, 5, 6, 7, 8, 10, 12, .. splits, an eighth apart: a host call's worth
    for (int s = 1; s <= most && s <= tiles; s += std::max(1, s / 4)) {
        int ct = (tiles + s - 1) / s;
        ct = (ct + G - 1) / G * G;
        const int n_c = (tiles + ct - 1) / ct;
        if (n_c == last) continue;
        last = n_c;
        if (n_c > 1 && (size_t)(blocks * n_kv * n_c) * kBlock * (hd_pad + 2) * 4 > room) break;
        double work = 0, units = 0, seen = 0;  // block b ends at token ((b + 1) * kBlock - 1) / group
        for (int64_t b = 0; b < blocks; b += step, ++seen) {
            const int64_t last_row = std::min(rows, (b + 1) * kBlock) - 1;
            const int tb = (int)((start + last_row / group) / kTile + 1);
            work += tb;
            units += (tb + ct - 1) / ct;
        }
        work *= blocks / seen * n_kv;
        units *= blocks / seen * n_kv;
        const double chunk = (double)rows * (hd_pad + 2) * 8;  // a chunk of every block, per KV head
        const double us = launch_us(pick, std::min(ct, tiles), work, units, n_c > 1 ? chunk * n_kv * n_c : 0, cus);
        if (best_pick == 0 || us < best_pick) {
            best_pick = us;
            best = PrefillPlan{ct, n_c, launch_us(time, std::min(ct, tiles), work, units,
                                                  n_c > 1 ? chunk * units / blocks : 0, cus)};
        }
    }
    return best;
}

constexpr int kBigDim = 128;  // larger heads: one wave group, 512 registers a wave

template <int HD, bool I8>
hipError_t launch_prefill_t(PrefillParams &p, PrefillPlan plan, hipStream_t st) {
    constexpr int G = HD > kBigDim ? 1 : 2;
    const int64_t rows = (int64_t)p.n_tok * p.group;
    const int64_t blocks = (rows + kBlock - 1) / kBlock;
    const int64_t units0 = blocks * p.n_kv;
    if (plan.n_chunks > 1) {
        float *ws = nullptr;
        const int64_t slots = units0 * plan.n_chunks;
        const hipError_t e = Scratch{}.get(st, (size_t)slots * kBlock * (HD + 2) * 4, &ws);
        if (e != hipSuccess) {
            (void)hipGetLastError();  // no workspace: the unsplit plan needs none
            plan = PrefillPlan{(p.start + p.n_tok + kTile - 1) / kTile, 1, 0};
        } else {
            p.part = reinterpret_cast<f32x4 *>(ws);
            p.stats = ws + slots * kBlock * HD;
        }
    }
    if (units0 * plan.n_chunks > 0x7FFFFFFF) return hipErrorInvalidValue;
    p.n_blocks = (int)blocks;
    p.n_chunks = plan.n_chunks;
    p.chunk_tiles = plan.chunk_tiles;
    constexpr int lds = prefill_lds<HD, G>();
    // the dynamic LDS limit, raised once per device (devices 0..63)
    static std::atomic<uint64_t> raised{0};
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    const uint64_t bit = 1ull << (dev & 63);
    if (!(raised.load(std::memory_order_acquire) & bit)) {
        e = hipFuncSetAttribute(reinterpret_cast<const void *>(&attn_prefill_kernel<HD, I8, G>),
                                hipFuncAttributeMaxDynamicSharedMemorySize, lds);
        if (e != hipSuccess) return e;
        raised.fetch_or(bit, std::memory_order_acq_rel);
    }
    attn_prefill_kernel<HD, I8, G><<<(unsigned)(units0 * plan.n_chunks), 256 * G, lds, st>>>(p);
    if (plan.n_chunks > 1)
        prefill_combine_kernel<HD><<<(unsigned)(units0 * 4 * (HD / 32)), 256, 0, st>>>(p);
    return hipGetLastError();
}

template <bool I8>
hipError_t launch_prefill_i(PrefillParams &p, const PrefillPlan &plan, hipStream_t st) {
    if (p.hd <= 64) return launch_prefill_t<64, I8>(p, plan, st);
    if (p.hd <= 96) return launch_prefill_t<96, I8>(p, plan, st);
    if (p.hd <= 128) return launch_prefill_t<128, I8>(p, plan, st);
    return launch_prefill_t<256, I8>(p, plan, st);
}

}  // namespace

PrefillPlan plan_prefill_attention(int n_heads, int n_kv, int head_dim, int n_tok, int start, int kv_int8) {
    const int cus = device_info().cu_count > 0 ? device_info().cu_count : 256;
    const int group = n_heads / n_kv;
    const int pad = head_dim <= 64 ? 64 : head_dim <= 96 ? 96 : head_dim <= 128 ? 128 : 256;
    return plan_prefill((int64_t)n_tok * group, group, n_kv, start, n_tok, pad, pad > kBigDim ? 1 : 2,
                        kv_int8, cus, kWorkspaceBytes);
}

hipError_t launch_prefill_attention(uint16_t *out, const uint16_t *q, const void *k, const void *v,
                                    const float *ks, const float *vs, int n_heads, int n_kv,
                                    int head_dim, int n_tok, int start, float scale, int kv_int8,
                                    const PrefillPlan &plan, hipStream_t st) {
    PrefillParams p{};
    p.out = out;
    p.q = q;
    p.k = k;
    p.v = v;
    p.ks = ks;
    p.vs = vs;
    p.n_heads = n_heads;
    p.n_kv = n_kv;
    p.hd = head_dim;
    p.group = n_heads / n_kv;
    p.n_tok = n_tok;
    p.start = start;
    // a tiny positive scale for 0, so that masked scores stay -inf
    p.sl2 = std::max(fabsf(scale) * 1.4426950408889634f, 1e-30f);
    p.negate = scale < 0.0f;
    // row and tile offsets are 32-bit
    if ((int64_t)n_tok * p.group > 0x7FFFFF00 || (int64_t)n_kv * head_dim * 2 * kTile > 0x7FFFFF00 ||
        (int64_t)start + n_tok > 0x7FFFFF00)
        return hipErrorInvalidValue;
    return kv_int8 ? launch_prefill_i<true>(p, plan, st) : launch_prefill_i<false>(p, plan, st);
}

}  // namespace rxq4
