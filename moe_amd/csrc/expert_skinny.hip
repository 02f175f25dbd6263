// expert_skinny.hip — products of few tokens with row-major quantised weights
// (plain projections of few tokens: skinny_linear_pays; experts of few tokens)
// on gfx950 matrix cores.
//
// Such a product's time is its weight stream's, so the kernel is one
// continuous stream per wave, with the activations held in registers.
//
// A launch is one block of eight waves per CU.  The waves split K (chunks of
// CU 64-value units, one per wave; SETS = 8 / nkw sets of rows when K has
// fewer chunks than waves).  Work is counted in groups of 16 SETS result
// rows; the groups of all (token tile, K part) pairs, in that order, are
// dealt to the blocks in contiguous ranges.  A wave turns its chunk of the
// tile's activations into MFMA fragments once per pair it meets and then
// walks its groups: per step, the 16 row pieces of its chunk (CU units: 144 to
// 544 contiguous bytes, always whole 16-byte pieces) come by LDS DMA into the
// wave's own ring, D steps deep and running across groups and tiles, so the
// stream never drains.  Waits are exact vmcnt counts.  Every KS steps the
// waves' partial sums meet in LDS (two buffers, one barrier) and are summed in
// the order of the waves.
//
// V_MFMA_F32_16X16X32_F16, one 32-value block per step of K: A = 16 tokens'
// activation pieces, B = 16 weight rows' codes.  Lane (l & 15, g = l >> 4)
// decodes row l & 15's values {4 g .. 4 g + 3, 16 + 4 g .. + 3} of each block
// (the two runs one dword of nibbles holds) and has that row's scale at hand,
// which multiplies the block's sum into the step's.
//
// Precision: as expert_mfma.hip.  Activations are f16 hi + lo pieces of
// v 2^e (22 to 24 significant bits: lo is signed), e per (token, chunk) putting
// the chunk's largest finite |v| in [2^14, 2^15); codes are exact in f16; block
// sums, scales and accumulators are f32.  An infinity or a NaN is its own hi piece and
// has no part in e: it reaches the sums as it is, beside finite values that
// keep their scale.
//
// The last chunk of a row whose units are no multiple of CU starts early, so
// that it ends with the row, and leaves out the units it shares with the
// chunk before; the last group of a matrix likewise starts early and stores
// only its own rows.
//
// Measured on MI355X, plain projections (us, before: f32 GEMV up to 8 tokens,
// which streams the weights once per two tokens, then the LDS-ring MFMA
// kernel with K split over blocks and two more launches):
//   Q8_0 102400 x 2048   T=1 66.7 -> 43.6   T=4 165 -> 46.5   T=32 106 -> 60 (3.7 TB/s)
//   Q4_0 102400 x 2048   T=1 55.0 -> 34.0   T=4 149 -> 34.9   T=32 75.3 -> 52
//   Q8_0   3072 x 2048   T=4 20.7 ->  7.1   T=32 20.4 -> 11.8 (calls cost the host 7)
//   Q8_0  28672 x 4096   T=1 40.8 -> 33.9   T=32 69.0 -> 58.2
// Of the 43.6, 30 remain without the DMAs (decoding and MFMAs, ~60% of the
// vector issue slots) and 44 without the decoding: the two overlap, and what
// is left is the stream at 5.1 TB/s and ~6 us of start (launch, activations).
// Experts (untiled; before: integer-dot kernels, two tokens per weight load,
// then the LDS-ring MFMA tiles), us per layer: V2-Lite Q8_0 T=32 (3 tokens per
// expert) 241 -> 167, Qwen3 Q8_0 T=64 254 -> 161, Mixtral Q4_0 T=32 380 -> 231,
// Mixtral Q5_0 T=16 447 -> 274.  V2-Lite's gate/up streams 376 MB in 73 us
// (5.1 TB/s); its down rows (1408 wide: six chunks, so six of eight waves)
// 197 MB in 45 (4.4).  For Q4_0, half the bytes per code, decoding bounds it:
// 14 vector instructions per 32-value block and lane after taking two
// nibbles per mask-and-or (16 with byte permutes: Mixtral T=32 237 -> 231).
// Four-wave blocks, three to a CU, each with its own rows ran the same loop in
// 50: their starts and ends are not covered.  Activations read per chunk
// instead of kept cost 1.5 us per chunk and block.
#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "gmem.h"
#include "lds_dma.h"
#include "mfma_tiles.h"
#include "moe_internal.h"

namespace moe {
namespace {

using namespace lds;
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));

// Meet the other waves once this wave's LDS accesses are done; loads in
// flight stay in flight.
__device__ inline void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// One step's weights: 16 rows x one chunk.
template <int DT, int CU>
struct Step {
    static constexpr int unit = 2 * Fmt<DT>::bytes;      // 36, 44, 68
    static constexpr int row = CU * unit;                // bytes of a row's chunk
    static constexpr int pieces = row / 16;              // CU = 4: 9, 11, 17
    static constexpr int bytes = 16 * row;
    static constexpr int dmas = (16 * pieces + 63) / 64;
    static_assert(row % 16 == 0, "whole 16-byte pieces");
};

__device__ inline half2v bits_h2(uint32_t v) { return __builtin_bit_cast(half2v, v); }
__device__ inline half2v both(float v) { return half2v{(_Float16)v, (_Float16)v}; }
__device__ inline void put(half8 &b, int at, half2v v) { b[at] = v[0], b[at + 1] = v[1]; }
// The codes of one dword as f16, in the order the fragments use: values 0, 2,
// 1, 3 of the lane's first run, then of its second (kRun).  A code in the
// low mantissa bits under exponent 0x64 is 1024 + code exactly; one four bits
// higher is 1024 + 16 code, which a fused multiply-add by 1/16 brings down.
constexpr int kRun[4] = {0, 2, 1, 3};
// Q4_0: low nibbles are the first run, high nibbles the second.
// (c & mask) | 0x6400'6400 is one instruction only with the masks in scalar
// and the exponents in vector registers, which the compiler does not see by
// itself: it is handed them as values it cannot fold.
struct Magic {
    uint32_t m, l, h;
    __device__ Magic() {
        asm("v_mov_b32 %0, 0x64006400" : "=v"(m));
        asm("s_mov_b32 %0, 0x000f000f" : "=s"(l));
        asm("s_mov_b32 %0, 0x00f000f0" : "=s"(h));
    }
};
// NEG: the codes negated (see decode_unit).
template <bool NEG>
__device__ inline half2v minus(half2v v, float off) { return NEG ? both(off) - v : v - both(off); }
template <bool NEG>
__device__ inline void nibbles(uint32_t c, const Magic &k, half8 &b) {
    const uint32_t m = k.m, l = k.l, h = k.h, c8 = c >> 8;
    put(b, 0, minus<NEG>(bits_h2((c & l) | m), 1032.0f));
    put(b, 2, minus<NEG>(bits_h2((c8 & l) | m), 1032.0f));
    put(b, 4, minus<NEG>(bits_h2((c & h) | m) * both(0.0625f), 72.0f));
    put(b, 6, minus<NEG>(bits_h2((c8 & h) | m) * both(0.0625f), 72.0f));
}
// Four codes (bytes of c, without an offset bit) minus `off`.
template <bool NEG>
__device__ inline void codes4(uint32_t c, float off, half8 &b, int at) {
    put(b, at, minus<NEG>(bits_h2(perm(0x64646464u, c, 0x04020400u)), off));
    put(b, at + 2, minus<NEG>(bits_h2(perm(0x64646464u, c, 0x04030401u)), off));
}
// hb: fifth bits of the first run at 0 .. 3, of the second at 16 .. 19.
template <bool NEG>
__device__ inline void nibbles5(uint32_t c, uint32_t hb, half8 &b) {
    codes4<NEG>((c & 0x0f0f0f0fu) | spread4(hb & 15u), 1040.0f, b, 0);
    codes4<NEG>(((c >> 4) & 0x0f0f0f0fu) | spread4((hb >> 16) & 15u), 1040.0f, b, 4);
}
template <bool NEG>
__device__ inline void bytes4(uint32_t c, half8 &b, int at) {
    codes4<NEG>(c ^ 0x80808080u, 1152.0f, b, at);
}
// Unit at p of lane (row, g)'s row chunk: its two blocks' codes and scales.
// The second block has both negated (at no cost): scales are positive as the
// formats are packed, and the matrix cores' sums err to one side, which adds
// up over the blocks otherwise.  Error against 64 bits over N(0, 1)
// activations, Q8_0, K = 4096: 1.21e-7 -> 1.04e-7.
template <int DT>
__device__ inline void decode_unit(lds_p p, int g, const Magic &mk, half8 (&b)[2], float (&d)[2]) {
    const auto w = [&](int i) { return lds_u32(p + 4 * i); };
    const lds_p pg = p + 4 * g;
    const auto wg = [&](int i) { return lds_u32(pg + 4 * i); };
    const auto scale = [&](uint32_t v) { return __half2float(__ushort_as_half((unsigned short)v)); };
    if constexpr (DT == MOE_DT_Q4_0) {
        d[0] = scale(w(0) & 0xffffu), d[1] = -scale(w(4) >> 16);
        nibbles<false>(alignb(wg(1), wg(0), 2), mk, b[0]);
        nibbles<true>(wg(5), mk, b[1]);
    } else if constexpr (DT == MOE_DT_Q5_0) {
        const uint32_t w0 = w(0);
        d[0] = scale(w0 & 0xffffu), d[1] = -scale(w(5) >> 16);
        nibbles5<false>(alignb(wg(2), wg(1), 2), alignb(w(1), w0, 2) >> (4 * g), b[0]);
        nibbles5<true>(wg(7), w(6) >> (4 * g), b[1]);
    } else {
        d[0] = scale(w(0) & 0xffffu), d[1] = -scale(w(8) >> 16);
        bytes4<false>(alignb(wg(1), wg(0), 2), b[0], 0);
        bytes4<false>(alignb(wg(5), wg(4), 2), b[0], 4);
        bytes4<true>(wg(9), b[1], 0);
        bytes4<true>(wg(13), b[1], 4);
    }
}

// A wave's activations for one chunk and one 16-token tile: the A fragments
// of its blocks, and 2^-e of the tokens whose sums the lane holds (4 g + i).
template <int CU>
struct Acts {
    half8 hi[2 * CU], lo[2 * CU];
    float inv[4];
};
// row: the chunk's first value of this lane's token.  The first `skip` units
// belong to the chunk before and read as zero.
template <int CU>
__device__ inline void load_acts(const float *row, int lane, int skip, Acts<CU> &out) {
    const int g = lane >> 4;
    auto load = [&](int q, f32x4(&v)[16]) {
#pragma unroll
        for (int i = 0; i < 16; i++)
            v[i] = gload((const f32x4 *)(row + 256 * q + 32 * (i >> 1) + 16 * (i & 1) + 4 * g));
    };
    // The largest finite |v|: its bits without the sign, shifted up, order like
    // it, and adding one to the exponent wraps an infinity or a NaN to less
    // than any finite value (one instruction).
    constexpr uint32_t kOne = 1u << 24;
    uint32_t m = kOne;
#pragma unroll
    for (int q = 0; q < CU / 4; q++) {
        f32x4 v[16];
        load(q, v);
#pragma unroll
        for (int i = 0; i < 16; i++)
#pragma unroll
            for (int j = 0; j < 4; j++) m = max(m, (__float_as_uint(v[i][j]) << 1) + kOne);
    }
    m = max(m, (uint32_t)__shfl_xor((int)m, 16, 64));
    m = max(m, (uint32_t)__shfl_xor((int)m, 32, 64));
    // |v| in [2^(x - 127), 2^(x - 126)): scaled into [2^14, 2^15).
    const int x = (int)(m >> 24) - 1;
    const int e = min(141 - x, 126);
    const float sc = __uint_as_float((uint32_t)(e + 127) << 23);
#pragma unroll
    for (int q = 0; q < CU / 4; q++) {
        f32x4 v[16];
        load(q, v);
#pragma unroll
        for (int b = 0; b < 8; b++) {
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const float w = v[2 * b + i / 4][kRun[i % 4]];
                const _Float16 hi = (_Float16)(w * sc);
                out.hi[8 * q + b][i] = hi;
                // Beside an infinite or NaN hi piece any finite lo will do.
                out.lo[8 * q + b][i] = (_Float16)fmaxf(fmaf(w, sc, -(float)hi), -8192.0f);
            }
            // Block by block: the fragments take their values' registers.
            __builtin_amdgcn_sched_barrier(0);
        }
    }
#pragma unroll
    for (int u = 0; u < CU - 1; u++)
        if (u < skip) out.hi[2 * u] = out.hi[2 * u + 1] = out.lo[2 * u] = out.lo[2 * u + 1] = half8{};
#pragma unroll
    for (int i = 0; i < 4; i++)
        out.inv[i] = __uint_as_float((uint32_t)(127 - __shfl(e, 4 * g + i, 64)) << 23);
}

struct SkinnyArgs {
    // Experts: the layer's table and the dispatch's lists (tiles of 16
    // tokens); otherwise one matrix (up: gate w0 and up w1) over T tokens.
    const ExpertDev *experts;
    const int32_t *tiles, *ntiles, *counts, *offsets, *perm_tok;
    int shared_tiles;            // tiles at the end of the list that are not this launch's
    const uint8_t *w0, *w1;
    uint32_t stride;             // bytes between weight rows (one for all experts)
    int T;
    const float *x;              // token rows, cols wide (up: by token; down: permuted rows)
    float *y;                    // result rows, `rows` wide
    float *residual;             // += y, or null
    size_t ypart;                // elements between K parts of y
    int rows, cols;              // of a matrix
    int parts;                   // K parts
    int cu;                      // units of a chunk: 4 or 8
    int cus;                     // blocks at most
    int nkw;                     // waves across K
    int groups;                  // of one matrix (pair)
};

template <int DT, int CU, int NT, int KS>
constexpr int ring_steps() {
    constexpr int n = (159 * 1024 - 2 * 8 * KS * NT * 1024) / (8 * Step<DT, CU>::bytes);
    return n > 6 ? 6 : n;
}
template <int DT, int CU, int NT, int KS>
constexpr int skinny_lds() {
    return 8 * ring_steps<DT, CU, NT, KS>() * Step<DT, CU>::bytes + 2 * 8 * KS * NT * 1024;
}

// UP: gate and up rows in alternating steps, y = silu(gate) up.  NT: 16-token
// tiles of a token tile.  KS: steps between meetings (UP: even).
template <int DT, bool UP, int CU, int NT, int KS>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void skinny_kernel(const SkinnyArgs a) {
    using S = Step<DT, CU>;
    constexpr int D = ring_steps<DT, CU, NT, KS>();
    constexpr int M = UP ? 2 : 1;  // steps of a group
    static_assert(D >= 2 && D * S::dmas < 64 && KS % M == 0, "ring");
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int g = lane >> 4, l16 = lane & 15;
    const int kw = wave % a.nkw, set = wave / a.nkw, sets = 8 / a.nkw, lsets = 31 - __builtin_clz(sets);
    const int tiles = a.experts ? a.ntiles[0] - a.shared_tiles : (a.T + 16 * NT - 1) / (16 * NT);
    int g0, g1;
    {
        // Blocks of a whole number per pair where that leaves at most an
        // eighth of them idle (a block then meets one pair: turning a chunk
        // of activations into fragments costs a few microseconds), else even
        // shares of all groups.
        const int pairs = tiles * a.parts, b = blockIdx.x, per = pairs > 0 ? gridDim.x / pairs : 0;
        if (8 * per * pairs >= 7 * (int)gridDim.x && pairs > 0) {
            const int tp = b / per, i = b % per;
            if (tp >= pairs) return;
            g0 = tp * a.groups + (int)((long long)a.groups * i / per);
            g1 = tp * a.groups + (int)((long long)a.groups * (i + 1) / per);
        } else {
            const long long all = (long long)pairs * a.groups;
            g0 = (int)(all * b / gridDim.x), g1 = (int)(all * (b + 1) / gridDim.x);
        }
        if (g0 >= g1) return;
    }
    const int units = a.cols / 64, chunks = (units + CU - 1) / CU;
    const int last16 = a.rows - 16;

    // One (token tile, part): its weights from this wave's chunk on, tokens
    // and first result row.
    struct Pair {
        const uint8_t *w0, *w1;
        int n, out0, u0, skip, nk;  // nk: waves of the part that have a chunk
        bool on;
    };
    auto pair_of = [&](int tp) {
        Pair o;
        const int part = tp % a.parts, tile = tp / a.parts;
        const int c0 = chunks * part / a.parts, c1 = chunks * (part + 1) / a.parts;
        o.on = c0 + kw < c1;
        o.nk = min(a.nkw, c1 - c0);
        o.u0 = min(CU * (c0 + kw), units - CU);
        o.skip = CU * (c0 + kw) - o.u0;
        if (a.experts) {
            const int e = a.tiles[4 * tile], m0 = a.tiles[4 * tile + 1];
            const ExpertDev &ex = a.experts[e];
            o.w0 = UP ? ex.m[0].ptr : ex.m[2].ptr;
            o.w1 = UP ? ex.m[1].ptr : o.w0;
            o.n = min(16 * NT, a.counts[e] - m0), o.out0 = a.offsets[e] + m0;
        } else {
            o.w0 = a.w0, o.w1 = a.w1;
            o.out0 = tile * 16 * NT, o.n = min(16 * NT, a.T - o.out0);
        }
        const size_t at = (size_t)(16 * set) * a.stride + (size_t)o.u0 * S::unit;
        o.w0 = (const uint8_t *)uniform_ptr(o.w0 + at);
        o.w1 = (const uint8_t *)uniform_ptr(o.w1 + at);
        return o;
    };

    uint32_t off[S::dmas];
#pragma unroll
    for (int i = 0; i < S::dmas; i++) {
        const uint32_t p = 64 * i + lane;
        off[i] = p / S::pieces * a.stride + 16u * (p % S::pieces);
    }
    // The DMA side runs up to D steps ahead of the sums: its own pair, group
    // and offset.  Steps of pairs in which this wave has no chunk do not
    // exist for it (`sent` and `used` count the ones that do).
    const uint32_t lds0 = lds_addr(smem + wave * D * S::bytes);
    const uint32_t gstep = 16u * (uint32_t)sets * a.stride;
    int d_at = g0, d_gr = g0 % a.groups, d_tp = g0 / a.groups, d_half = 0, d_slot = 0;
    Pair dp = pair_of(d_tp);
    int sent = 0, used = 0;
    auto issue = [&]() {
        // Skip pairs without a chunk of ours.
        while (d_at < g1 && !dp.on) {
            d_at += a.groups - d_gr, d_gr = 0, d_tp++;
            if (d_at < g1) dp = pair_of(d_tp);
        }
        if (d_at >= g1) return;
        const int row = 16 * (d_gr * sets + set);
        // The matrix's last group starts early; sets past its end re-read it.
        const uint8_t *b = (UP && d_half ? dp.w1 : dp.w0) + (size_t)(uint32_t)d_gr * gstep;
        if (row > last16) b -= (size_t)(row - last16) * a.stride;
        const uint32_t dst = lds0 + (uint32_t)d_slot * S::bytes;
#pragma unroll
        for (int i = 0; i < S::dmas; i++)
            if (64 * i + 63 < 16 * S::pieces || 64 * i + lane < 16 * S::pieces) dma16(b, off[i], dst + 1024u * i);
        sent++;
        d_slot = d_slot + 1 == D ? 0 : d_slot + 1;
        if (UP && !d_half) {
            d_half = 1;
        } else {
            d_half = 0, d_at++;
            if (++d_gr == a.groups) {
                d_gr = 0, d_tp++;
                if (d_at < g1) dp = pair_of(d_tp);
            }
        }
    };
#pragma unroll 1
    for (int i = 0; i < D; i++) issue();

    const Magic magic;
    float *red0 = reinterpret_cast<float *>(smem + 8 * D * S::bytes);
    Acts<CU> act[NT];
    Pair cur = pair_of(g0 / a.groups);
    int tp = g0 / a.groups, gr = g0 % a.groups, slot = 0;
    bool fresh = true;
    for (int at = g0, buf = 0; at < g1; buf ^= 1) {
        const int ng = min(KS / M, min(g1 - at, a.groups - gr));
        if (fresh && cur.on) {
#pragma unroll
            for (int t = 0; t < NT; t++) {
                // Lanes without a token read the tile's first: their sums are
                // rows of the result that nothing stores.
                const int tok = cur.out0 + (16 * t + l16 < cur.n ? 16 * t + l16 : 0);
                const int src = UP && a.experts ? a.perm_tok[tok] : tok;
                load_acts<CU>(a.x + (size_t)src * a.cols + 64 * cur.u0, lane, cur.skip, act[t]);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        float *red = red0 + buf * (8 * KS * NT * 256);
        auto steps = [&](auto skip_c) {
            constexpr bool SK = decltype(skip_c)::value;
            float *rw = red + wave * (KS * NT * 256) + lane;
#pragma unroll 1
            for (int s = 0; s < M * ng; s++, rw += NT * 256) {
                f32x4 sum[NT];
#pragma unroll
                for (int t = 0; t < NT; t++) sum[t] = f32x4{0, 0, 0, 0};
                // This step's DMAs are the oldest: all but the newer ones.
                const int newer = sent - used - 1;
                if (newer >= D - 1) wait_vm<(D - 1) * S::dmas>();
                else if (D > 5 && newer == 4) wait_vm<4 * S::dmas>();
                else if (D > 4 && newer == 3) wait_vm<3 * S::dmas>();
                else if (D > 3 && newer == 2) wait_vm<2 * S::dmas>();
                else if (D > 2 && newer == 1) wait_vm<S::dmas>();
                else wait_vm<0>();
                const lds_p p = (lds_p)smem + (wave * D + slot) * S::bytes + l16 * S::row;
#pragma unroll
                for (int u = 0; u < CU; u++) {
                    half8 b[2];
                    float d[2];
                    decode_unit<DT>(p + u * S::unit, g, magic, b, d);
#pragma unroll
                    for (int k = 0; k < 2; k++) {
                        const float dk = SK && u < CU - 1 && u < cur.skip ? 0.0f : d[k];
#pragma unroll
                        for (int t = 0; t < NT; t++) {
                            // The small pieces' sum first: one rounding of the
                            // block's size, not two (error against 64 bits at
                            // K = 512, 9.0e-8 -> 8.2e-8; 2048, 9.9e-8 -> 9.1e-8).
                            f32x4 v = __builtin_amdgcn_mfma_f32_16x16x32_f16(act[t].lo[2 * u + k], b[k],
                                                                             f32x4{0, 0, 0, 0}, 0, 0, 0);
                            v = __builtin_amdgcn_mfma_f32_16x16x32_f16(act[t].hi[2 * u + k], b[k], v, 0, 0, 0);
#pragma unroll
                            for (int i = 0; i < 4; i++) sum[t][i] = fmaf(dk, v[i], sum[t][i]);
                        }
                    }
                }
                // The step's reads are done in every lane: refill its slot.
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                used++;
                slot = slot + 1 == D ? 0 : slot + 1;
                issue();
#pragma unroll
                for (int t = 0; t < NT; t++)
#pragma unroll
                    for (int i = 0; i < 4; i++) rw[t * 256 + 64 * i] = sum[t][i] * act[t].inv[i];
            }
        };
        if (cur.on) {
            if (cur.skip == 0)
                steps(std::false_type{});
            else
                steps(std::true_type{});
        }
        // One barrier per meeting: the next one uses the other buffer, and a
        // wave is past this one's sums before it reaches that barrier.
        lds_barrier();
        const int part = tp % a.parts;
        for (int q = wave; q < (ng * NT * 4) << lsets; q += 8) {
            const int i = q & 3, t = (q >> 2) % NT, st = (q >> 2) / NT & (sets - 1), s = (q >> 2) / NT >> lsets;
            auto total = [&](int step) {
                const float *r = red + ((st * a.nkw * KS + step) * NT + t) * 256 + 64 * i + lane;
                float v[8];
#pragma unroll
                for (int k = 0; k < 8; k++) v[k] = k < cur.nk ? r[k * KS * NT * 256] : 0.0f;
                return ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
            };
            float v = total(M * s);
            if constexpr (UP) {
                const float u = total(M * s + 1);
                v = (v / (1.0f + __expf(-v))) * u;
            }
            const int row = 16 * ((gr + s) * sets + st), r = min(row, last16) + l16;
            const int tk = 16 * t + 4 * g + i;
            if (r >= row && row < a.rows && tk < cur.n) {
                const size_t o = (size_t)(cur.out0 + tk) * a.rows + r;
                gstore(a.y + part * a.ypart + o, v);
                if (a.residual) a.residual[o] += v;
            }
        }
        at += ng, gr += ng;
        fresh = gr == a.groups;
        if (fresh) {
            gr = 0, tp++;
            if (at < g1) cur = pair_of(tp);
        }
    }
}

template <int DT, bool UP, int CU, int NT, int KS>
hipError_t launch_one(SkinnyArgs a, int tiles, hipStream_t s) {
    constexpr int lds = skinny_lds<DT, CU, NT, KS>();
    // The setting is per device, so every launch makes it.
    const hipError_t e = hipFuncSetAttribute((const void *)skinny_kernel<DT, UP, CU, NT, KS>,
                                             hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e != hipSuccess) return e;
    const int chunks = (a.cols / 64 + CU - 1) / CU, per = (chunks + a.parts - 1) / a.parts;
    if (per > 8) return hipErrorInvalidValue;
    a.nkw = 1;
    while (a.nkw < per) a.nkw *= 2;
    a.groups = (a.rows + 16 * (8 / a.nkw) - 1) / (16 * (8 / a.nkw));
    const long long all = (long long)a.groups * tiles * a.parts;
    hipLaunchKernelGGL((skinny_kernel<DT, UP, CU, NT, KS>), dim3((unsigned)std::min<long long>(all, a.cus)),
                       dim3(512), lds, s, a);
    return hipGetLastError();
}

// Units of a chunk and K parts for a width: four-unit chunks while eight of
// them cover K (shorter steps, half the registers), else eight-unit ones.
int chunk_units(int cols) { return cols <= 8 * 4 * 64 ? 4 : 8; }
int parts_for(int cols) {
    const int cu = chunk_units(cols);
    return (cols / 64 + 8 * cu - 1) / (8 * cu);
}

// tokens: of the one matrix; experts: minus the tokens of their tiles (a.T
// bounds the number of tiles).
template <int DT, bool UP>
hipError_t launch_dt(const SkinnyArgs &a, int tokens, hipStream_t s) {
    constexpr int M = UP ? 2 : 1;
    if (UP && a.parts != 1) return hipErrorInvalidValue;
    const int tiles = tokens > 0 ? (tokens + 15) / 16 : a.T;
    if (a.cu == 4) {
        if (tokens > 16 || tokens == -32)
            return launch_one<DT, UP, 4, 2, 2>(a, tokens > 0 ? (tokens + 31) / 32 : a.T, s);
        return launch_one<DT, UP, 4, 1, 4>(a, tiles, s);
    }
    // Q8_0 steps of eight units leave room for one meeting's sums only.
    if constexpr (DT == MOE_DT_Q8_0 && UP)
        return hipErrorInvalidValue;
    else
        return tokens == -32 ? hipErrorInvalidValue
                             : launch_one<DT, UP, 8, 1, DT == MOE_DT_Q8_0 ? 1 : (DT == MOE_DT_Q5_0 ? M : 2)>(a, tiles, s);
}
hipError_t launch_any(int dt, bool up, const SkinnyArgs &a, int tokens, hipStream_t s) {
    switch (dt) {
    case MOE_DT_Q4_0: return up ? launch_dt<MOE_DT_Q4_0, true>(a, tokens, s) : launch_dt<MOE_DT_Q4_0, false>(a, tokens, s);
    case MOE_DT_Q5_0: return up ? launch_dt<MOE_DT_Q5_0, true>(a, tokens, s) : launch_dt<MOE_DT_Q5_0, false>(a, tokens, s);
    default: return up ? launch_dt<MOE_DT_Q8_0, true>(a, tokens, s) : launch_dt<MOE_DT_Q8_0, false>(a, tokens, s);
    }
}

}  // namespace

bool skinny_ok(const MatDev &m) {
    return (m.dt == MOE_DT_Q4_0 || m.dt == MOE_DT_Q5_0 || m.dt == MOE_DT_Q8_0) && (uintptr_t)m.ptr % 4 == 0 &&
           m.stride % 4 == 0 && m.cols % 64 == 0 && m.cols >= 64 * chunk_units(m.cols) && m.rows >= 16;
}

bool skinny_layer_ok(const ExpertDev *experts, int n, int E) {
    // Every matrix takes the kernel; gate and up rows fit one K part; routed
    // experts share their row strides (launches pass one).
    for (int e = 0; e < n; e++) {
        const MatDev *m = experts[e].m;
        for (int i = 0; i < 3; i++)
            if (!skinny_ok(m[i])) return false;
        if (m[0].dt != m[1].dt || m[0].stride != m[1].stride || parts_for(m[0].cols) != 1 ||
            (m[0].dt == MOE_DT_Q8_0 && chunk_units(m[0].cols) != 4) || parts_for(m[2].cols) > kMaxKSplit)
            return false;
        if (e < E && (m[0].stride != experts[0].m[0].stride || m[2].stride != experts[0].m[2].stride)) return false;
    }
    return true;
}
// 32-token tiles where both widths leave registers for them (at most 2048)
// and experts often hold more than 16 tokens: Qwen3 Q8_0 T=256 (16 per
// expert) 239 -> 220 us per layer, V2-Lite T=192 (18) 290 -> 263, but Qwen3
// T=192 (12) 199 -> 215.
int skinny_tile(int H, int I, double tokens) {
    return tokens > 14.0 && chunk_units(H) == 4 && chunk_units(I) == 4 ? 32 : 16;
}
int skinny_parts(int I) { return parts_for(I); }
// The shared expert's down rows: four-unit chunks (and the 32-token tiles
// that go with them) while kMaxKSplit parts of them cover K.
int shared_units(int I_s) { return (I_s / 64 + 31) / 32 <= kMaxKSplit ? 4 : 8; }
int skinny_shared_parts(int I_s) {
    const int cu = shared_units(I_s);
    return (I_s / 64 + 8 * cu - 1) / (8 * cu);
}

hipError_t launch_skinny_experts(bool up, const MfmaArgs &m, int tile, const float *x, const ExpertDev &e0, hipStream_t s) {
    SkinnyArgs a{};
    a.experts = m.experts, a.tiles = m.tiles, a.ntiles = m.ntiles, a.counts = m.counts, a.offsets = m.offsets;
    a.perm_tok = m.perm_tok, a.shared_tiles = m.shared_tiles;
    const MatDev &w = up ? e0.m[0] : e0.m[2];
    a.stride = w.stride;
    a.T = m.max_tiles;
    a.x = up ? x : m.h, a.y = up ? m.h : m.y;
    a.ypart = up ? 0 : m.ypart;
    a.rows = w.rows, a.cols = w.cols, a.parts = up ? 1 : m.ksplit;
    a.cu = chunk_units(w.cols), a.cus = device_cus();
    return launch_any(w.dt, up, a, -tile, s);
}
hipError_t launch_skinny_shared(bool up, const MfmaArgs &m, const float *x, const ExpertDev &ex, bool beside,
                                hipStream_t s) {
    SkinnyArgs a{};
    const MatDev &w = up ? ex.m[0] : ex.m[2];
    a.w0 = w.ptr, a.w1 = up ? ex.m[1].ptr : w.ptr;
    a.stride = w.stride;
    a.T = m.T;
    a.x = up ? x : m.hs, a.y = up ? m.hs : m.ys;
    a.ypart = up ? 0 : m.yspart;
    a.rows = w.rows, a.cols = w.cols, a.parts = up ? 1 : skinny_shared_parts(w.cols);
    a.cu = up ? chunk_units(w.cols) : shared_units(w.cols);
    // Beside the routing it leaves CUs free: a block holds its CU's LDS, and
    // the dispatch kernel would wait for one to end.
    a.cus = beside ? device_cus() * 3 / 4 : device_cus();
    return launch_any(w.dt, up, a, m.T, s);
}

bool skinny_linear_ok(const MatDev &m) { return skinny_ok(m) && parts_for(m.cols) == 1; }

// Every 32 tokens (16 for rows wider than 2048) stream the weights again, so
// beyond one tile the launch pays while it stays short, counted in groups
// over all tiles.  Against the GEMV (up to 8 tokens) and the MFMA kernels, us:
// 16384 x 1408 Q8_0 T=64 (2048 groups) 22.2 / 27.3, T=128 (4096) 34.0 / 38.7
// but T=192 52 / 42; 32000 x 512 T=128 (2000) 29.5 / 32.8, T=192 (3000) 43 /
// 30; 4096 x 4096 T=64 (1024) 24.3 / 25.2, 8192 x 4096 T=64 (2048) 35 / 28;
// 102400 x 2048 T=64 95 / 114, T=96 145 / 139.  One or two tokens on few rows
// wider than 2048: the GEMV's start is shorter (1024 x 4096 T=1 8.8 / 7.6,
// 8192 x 4096 T=1 14.7 / 13.0, T=2 at 4096 rows 10.7 / 16.1).
bool skinny_linear_pays(const MatDev &m, int T) {
    const int cu = chunk_units(m.cols);
    if (T == 1 && cu == 8 && m.rows <= 8192) return false;
    if (T == 2 && cu == 8 && m.rows <= 1024) return false;
    if (T <= 32 || (cu == 4 && T <= 64)) return true;
    const int per = (m.cols / 64 + cu - 1) / cu;
    int nkw = 1;
    while (nkw < per) nkw *= 2;
    const long long groups = (m.rows + 16 * (8 / nkw) - 1) / (16 * (8 / nkw));
    return groups * (cu == 4 ? (T + 31) / 32 : (T + 15) / 16) <= (cu == 4 ? 2048 : 1024);
}

hipError_t launch_skinny_linear(const MatDev &w, const float *x, int T, float *y, float *residual, hipStream_t s) {
    if (!skinny_linear_ok(w) || T < 1) return hipErrorInvalidValue;
    SkinnyArgs a{};
    a.w0 = a.w1 = w.ptr, a.stride = w.stride;
    a.x = x, a.y = y, a.residual = residual, a.T = T;
    a.rows = w.rows, a.cols = w.cols, a.parts = 1;
    a.cu = chunk_units(w.cols), a.cus = device_cus();
    return launch_any(w.dt, false, a, T, s);
}

}  // namespace moe
