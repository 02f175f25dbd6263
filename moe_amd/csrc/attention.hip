// attention.hip — causal attention over the f32 caches (src/model.rs:790-831).
//
// Row r of q belongs to sequence seq[r] at position pos[r] and attends to
// that sequence's cache positions [lo, pos[r]].  seq and pos live on the
// device, so the host does not know whether consecutive rows are one prompt
// (a prefill, which should read keys and values once for many rows) or many
// sequences (a decode step): one kernel serves both.
//
// attention_tile_kernel: a block takes a group of consecutive rows and one
// key/value head, splits the group into runs of one sequence, and makes each
// run's (row, query head) pairs the 16 or 32 columns of its products on the
// f32 matrix cores.  Its waves split the cached positions, 16 at a time, and
// merge their softmax state at the end (through LDS), so nothing is shared
// between waves inside the loop and there is no barrier there:
//   S^T = K Q^T: the keys of 16 positions are the rows (A), loaded straight
//     from the cache, 16 bytes per lane; Q^T (B) sits in LDS in operand order;
//   P = exp(S - m): the product's result layout (lane = column, 4 positions
//     per lane) is the B layout of the next product, so the weights never move;
//   O^T += V^T P^T: the values of the same positions, 16 bytes per lane.
// The keys of the next 16 positions load while the weights and the second
// product run, the values while the first product runs.  The running
// maximum m moves only when a score exceeds it by more than 8 (weights then
// stay below e^8): the common step has no lane exchange and no rescale.
// Everything is f32: products by V_MFMA_F32_16X16X4_F32, accumulation in f32.
//
// A decode step has one row per run: most columns are empty, but 80 MFMAs
// (keys of 192, values of 128) per 20 KB of cache still leave the matrix
// pipe ~3x below what HBM delivers, so the kernel stays memory bound there.
//
// Measured on MI355X against one wavefront per (row, head) everywhere (key
// rows read lane by lane, a serial value loop): a decode step of 32 sequences
// of 600-1200 positions, 16 heads, keys of 192 and values of 128 (590 MB of
// cache) 439 -> 113 us (5.2 TB/s: HBM bound); a prompt of 1000 rows, 32 heads
// over 8, width 128 (8.2 GFLOP) 1408 -> 105 us (78 TFLOP/s of the ~151 the
// f32 matrix cores reach in a large product: the rest is the softmax between
// the two products).
//
// attention_kernel: one wavefront per (row, head), scores in LDS: head widths
// that are not a multiple of 4, values wider than 256, buffers off a 16-byte
// boundary, and head counts that are no multiple of the key/value heads.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "exact_math.h"
#include "gmem.h"
#include "moe_internal.h"

namespace moe {
int fail(int code, const char *fmt, ...);

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

// One wavefront per (row, head): scores of positions [lo, p] (one lane per
// position, the key read as a contiguous row), softmax with glibc's expf,
// then the weighted sum of values (one lane per output column, positions
// in order).
constexpr int kAttnMaxDim = 256;
__global__ __launch_bounds__(64) void attention_kernel(const float *__restrict__ q, int64_t q_stride, int heads,
                                                       int n_kv, int qd, int vd, float scale,
                                                       const float *__restrict__ kc, const float *__restrict__ vc,
                                                       int64_t ctx, const int32_t *__restrict__ seq,
                                                       const int32_t *__restrict__ pos, int window,
                                                       float *__restrict__ out, int64_t out_stride) {
    extern __shared__ float sc[];
    __shared__ float qs[kAttnMaxDim];
    const int r = blockIdx.x / heads, h = blockIdx.x % heads, lane = threadIdx.x;
    const int p = pos[r];
    const int lo = window > 0 ? max(0, p + 1 - window) : 0;
    const int n = p + 1 - lo;
    const int rep = heads / max(n_kv, 1);
    const int kvh = rep > 1 ? h / rep : min(h, n_kv - 1);
    const size_t kd = (size_t)n_kv * qd, vdim = (size_t)n_kv * vd;
    const float *qv = q + (size_t)r * q_stride + (size_t)h * qd;
    for (int i = lane; i < qd; i += 64) qs[i] = qv[i];
    __syncthreads();
    const float *kbase = kc + ((size_t)seq[r] * ctx) * kd + (size_t)kvh * qd;
    const float *vbase = vc + ((size_t)seq[r] * ctx) * vdim + (size_t)kvh * vd;
    float m = -INFINITY;
    for (int j = lane; j < n; j += 64) {
        const float *k = kbase + (size_t)(lo + j) * kd;
        float d = 0.0f;
        for (int i = 0; i < qd; i++) d = fmaf(qs[i], k[i], d);
        const float s = d * scale;
        sc[j] = s;
        m = fmaxf(m, s);
    }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
    float sum = 0.0f;
    for (int j = lane; j < n; j += 64) {
        const float e = expf_exact(sc[j] - m);
        sc[j] = e;
        sum += e;
    }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) sum += __shfl_xor(sum, o, 64);
    __syncthreads();
    float *o = out + (size_t)r * out_stride + (size_t)h * vd;
    for (int c = lane; c < vd; c += 64) {
        float acc = 0.0f;
        for (int j = 0; j < n; j++) {
            const float w = sc[j] / sum;
            acc += w * vbase[(size_t)(lo + j) * vdim + c];
        }
        o[c] = acc;
    }
}

struct AttnArgs {
    const float *q, *kc, *vc;
    const int32_t *seq, *pos;
    float *out;
    int64_t q_stride, out_stride, ctx;
    int rows, n_kv, rep, qd, vd, window;
    float scale;
    int tt;      // rows of a group
    int groups;  // groups of tt rows
    int rc;      // query heads of a block (of the rep that share its key/value head)
    int chunks;  // blocks that share the rep heads
    int split;   // blocks that share a group's runs
};

// exp(x) for x <= 8 or so, to about 1 ulp: 2^t by the hardware, the rounding
// of t = x log2(e) put back as a first-order factor.  -inf gives 0, NaN stays.
__device__ inline float exp_weight(float x) {
    x = x < -200.0f ? -200.0f : x;
    const float t = x * 1.44269504f;
    const float r = fmaf(x, 1.44269504f, -t) + x * 1.92596299e-8f;
    const float e = __builtin_amdgcn_exp2f(t);
    return fmaf(e, r * 0.693147181f, e);
}

// QC: 16-value steps of a key; EX: the key is exactly QC steps wide.  VB:
// 64-value blocks of a value row.  C: 16-column tiles.  W: waves.
template <int QC, bool EX, int VB, int C, int W>
__global__ __launch_bounds__(W * 64, 2) void attention_tile_kernel(const AttnArgs a) {
    constexpr int kQ = C * QC * 64, kMerge = (W / 2) * C * VB * 4 * 64;
    __shared__ f32x4 sm[kQ > kMerge ? kQ : kMerge];
    __shared__ float sm_m[W][C * 16], sm_l[W][C * 16];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, col = lane & 15, g = lane >> 4;
    // Blocks go to the XCDs in turn (block id mod 8).  Each XCD takes every
    // eighth (group, part of its runs) with all its key/value heads next to
    // each other: a cached row of all heads is contiguous, so together they
    // read whole rows, spread over all of the XCD's L2 channels, while one
    // head's pieces, a power of two apart, would sit in two of sixteen.
    int id = blockIdx.x >> 3;
    const int kv = id % a.n_kv;
    id /= a.n_kv;
    const int chunk = id % a.chunks;
    const int unit = id / a.chunks * 8 + (blockIdx.x & 7);
    if (unit >= a.groups * a.split) return;
    // A group's first part holds all of a prompt's work, its others leave at
    // once: the first parts come together, because the dispatcher deals blocks
    // to an XCD's shader engines in turn, and every second or fourth one doing
    // the work would leave the others idle.  (The parts of a group next to each
    // other and heads dealt over the XCDs -> this order: 32 heads over 8 of
    // width 128, a prompt of 2000 rows 603 -> 320 us, 8 x 64 rows past 1000 327
    // -> 109; 16 heads of 192/128, 4 x 1000 rows 475 -> 289.)  Later rows of a
    // prompt see more positions: the last groups go first.
    const int sub = unit / a.groups;
    const int r0 = (a.groups - 1 - unit % a.groups) * a.tt;
    const int nr = min(a.tt, a.rows - r0);
    const int h0 = kv * a.rep + chunk * a.rc, hn = min(a.rc, a.rep - chunk * a.rc);
    const int my_seq = gload(a.seq + r0 + min(lane, nr - 1)), my_pos = gload(a.pos + r0 + min(lane, nr - 1));
    const int before = __shfl_up(my_seq, 1, 64);
    unsigned long long starts = __ballot(lane < nr && (lane == 0 || my_seq != before));
    const size_t ks = (size_t)a.n_kv * a.qd, vs = (size_t)a.n_kv * a.vd;

    for (int run = 0; starts; run++) {
        const int first = __builtin_ctzll(starts);
        starts &= starts - 1;
        const int end = starts ? __builtin_ctzll(starts) : nr;
        if (run % a.split != sub) continue;
        const int ncol = (end - first) * hn;
        // The union of the run's position ranges, and each column's own.
        const bool mine = lane >= first && lane < end;
        int hi = mine ? my_pos : -1;
        int lo = mine ? (a.window > 0 ? max(0, my_pos + 1 - a.window) : 0) : 0x7fffffff;
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1) {
            hi = max(hi, __shfl_xor(hi, o, 64));
            lo = min(lo, __shfl_xor(lo, o, 64));
        }
        hi = __builtin_amdgcn_readfirstlane(hi);
        lo = __builtin_amdgcn_readfirstlane(lo);
        int cp[C], cl[C], ctok[C];
        bool cv[C];
#pragma unroll
        for (int c = 0; c < C; c++) {
            const int cc = c * 16 + col;
            cv[c] = cc < ncol;
            ctok[c] = first + (cv[c] ? cc / hn : 0);
            const int p = __shfl(my_pos, ctok[c], 64);
            cp[c] = p;
            cl[c] = a.window > 0 ? max(0, p + 1 - a.window) : 0;
        }
        __syncthreads();  // the previous run's reads of sm
        for (int i = threadIdx.x; i < kQ; i += W * 64) {
            const int l = i & 63, s = (i >> 6) % QC, cc = (i >> 6) / QC * 16 + (l & 15), d = 16 * s + 4 * (l >> 4);
            f32x4 v = {0.0f, 0.0f, 0.0f, 0.0f};
            if (cc < ncol && d < a.qd)
                v = gload((const f32x4 *)(a.q + (size_t)(r0 + first + cc / hn) * a.q_stride +
                                          (size_t)(h0 + cc % hn) * a.qd + d));
            sm[i] = v;
        }
        __syncthreads();
        const int sq = __builtin_amdgcn_readfirstlane(__shfl(my_seq, first, 64));
        const float *kb = a.kc + ((size_t)sq * a.ctx) * ks + (size_t)kv * a.qd;
        const float *vb = a.vc + ((size_t)sq * a.ctx) * vs + (size_t)kv * a.vd;
        const int ntiles = hi >= lo ? (hi - lo + 16) / 16 : 0;
        // Weights reach e^8 < 2^12 and there are at most 16 ntiles of them: so
        // scaled, a row's weights sum to less than 1, and its weighted sums stay
        // within the values' own range until they are divided.  A power of two
        // (exact), one multiplication per weight.
        const float unit = __uint_as_float((uint32_t)(127 - 12 - (36 - __clz(ntiles))) << 23);

        f32x4 o[C][VB][4];
        float m[C], l[C];
#pragma unroll
        for (int c = 0; c < C; c++) {
            m[c] = -INFINITY, l[c] = 0.0f;
#pragma unroll
            for (int t = 0; t < VB; t++)
#pragma unroll
                for (int j = 0; j < 4; j++) o[c][t][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        }
        if (wave < ntiles) {
            f32x4 k[QC];
            // Keys: lane (col, g) holds position col's values 16 s + 4 g ..
            // + 3.  Positions past the end re-read the last one (masked).
            auto load_k = [&](int tile) {
                const int p = min(lo + tile * 16 + col, hi);
                const float *row = kb + (size_t)p * ks;
#pragma unroll
                for (int s = 0; s < QC; s++) {
                    const int d = EX ? 16 * s + 4 * g : min(16 * s + 4 * g, a.qd - 4);
                    k[s] = gload((const f32x4 *)(row + d));
                }
            };
            load_k(wave);
            for (int tile = wave; tile < ntiles; tile += W) {
                const int base = lo + tile * 16;
                f32x4 v[4][VB];
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const float *row = vb + (size_t)min(base + 4 * g + i, hi) * vs;
#pragma unroll
                    for (int t = 0; t < VB; t++) v[i][t] = gload((const f32x4 *)(row + min(64 * t + 4 * col, a.vd - 4)));
                }
                // Two chains per column tile.
                f32x4 sa[C][2];
#pragma unroll
                for (int c = 0; c < C; c++) sa[c][0] = sa[c][1] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
                f32x4 qq[C];
#pragma unroll
                for (int c = 0; c < C; c++) qq[c] = sm[c * QC * 64 + lane];
#pragma unroll
                for (int s = 0; s < QC; s++) {
                    f32x4 kk = k[s], qn[C];
                    if (!EX && 16 * s + 4 * g >= a.qd) kk = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                    for (int c = 0; c < C; c++) qn[c] = sm[(c * QC + min(s + 1, QC - 1)) * 64 + lane];
#pragma unroll
                    for (int j = 0; j < 4; j++)
#pragma unroll
                        for (int c = 0; c < C; c++)
                            sa[c][j & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(kk[j], qq[c][j], sa[c][j & 1], 0, 0, 0);
#pragma unroll
                    for (int c = 0; c < C; c++) qq[c] = qn[c];
                    // One step of Q^T ahead, not all of them (registers).
                    __builtin_amdgcn_sched_barrier(0);
                }
                load_k(min(tile + W, ntiles - 1));
                // Scores; masked where a column does not see a position.
                float p[C][4];
                bool part = false;
#pragma unroll
                for (int c = 0; c < C; c++) part |= cv[c] && (base < cl[c] || base + 15 > cp[c]);
                part = __any(part);
#pragma unroll
                for (int c = 0; c < C; c++)
#pragma unroll
                    for (int i = 0; i < 4; i++) p[c][i] = (sa[c][0][i] + sa[c][1][i]) * a.scale;
                if (part) {
#pragma unroll
                    for (int c = 0; c < C; c++)
#pragma unroll
                        for (int i = 0; i < 4; i++) {
                            const int at = base + 4 * g + i;
                            if (at < cl[c] || at > cp[c]) p[c][i] = -INFINITY;
                        }
                }
                float top[C];
                bool move = false;
#pragma unroll
                for (int c = 0; c < C; c++) {
                    top[c] = fmaxf(fmaxf(p[c][0], p[c][1]), fmaxf(p[c][2], p[c][3]));
                    move |= top[c] > m[c] + 8.0f;
                }
                if (__any(move)) {
#pragma unroll
                    for (int c = 0; c < C; c++) {
                        float x = fmaxf(top[c], __shfl_xor(top[c], 16, 64));
                        x = fmaxf(x, __shfl_xor(x, 32, 64));
                        const float mn = fmaxf(m[c], x);
                        const float f = mn == -INFINITY ? 1.0f : exp_weight(m[c] - mn);
                        m[c] = mn;
                        l[c] *= f;
#pragma unroll
                        for (int t = 0; t < VB; t++)
#pragma unroll
                            for (int j = 0; j < 4; j++) o[c][t][j] *= f;
                    }
                }
#pragma unroll
                for (int c = 0; c < C; c++) {
                    const float ref = m[c] == -INFINITY ? 0.0f : m[c];
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        p[c][i] = exp_weight(p[c][i] - ref) * unit;
                        l[c] += p[c][i];
                    }
                }
                // A value no column may see weighs 0, and 0 times an infinity
                // or a NaN is a NaN: a partly masked step that holds such a
                // value goes row by row, unseen values read as 0.
                bool odd = false;
                if (part) {
                    float z = 0.0f;
#pragma unroll
                    for (int i = 0; i < 4; i++)
#pragma unroll
                        for (int t = 0; t < VB; t++)
#pragma unroll
                            for (int j = 0; j < 4; j++) z = fmaf(v[i][t][j], 0.0f, z);
                    odd = __any(!(z == 0.0f));
                }
                if (!odd) {
#pragma unroll
                    for (int i = 0; i < 4; i++)
#pragma unroll
                        for (int t = 0; t < VB; t++)
#pragma unroll
                            for (int j = 0; j < 4; j++)
#pragma unroll
                                for (int c = 0; c < C; c++)
                                    o[c][t][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[i][t][j], p[c][i], o[c][t][j], 0, 0,
                                                                                     0);
                } else {
#pragma unroll 1
                    for (int tok = first; tok < end; tok++) {
                        const int tp = __shfl(my_pos, tok, 64);
                        const int tl = a.window > 0 ? max(0, tp + 1 - a.window) : 0;
                        bool see[4];
#pragma unroll
                        for (int i = 0; i < 4; i++) see[i] = base + 4 * g + i >= tl && base + 4 * g + i <= tp;
#pragma unroll
                        for (int t = 0; t < VB; t++)
#pragma unroll
                            for (int j = 0; j < 4; j++) {
#pragma unroll
                                for (int c = 0; c < C; c++) {
                                    f32x4 x = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                                    for (int i = 0; i < 4; i++)
                                        x = __builtin_amdgcn_mfma_f32_16x16x4f32(see[i] ? v[i][t][j] : 0.0f, p[c][i], x, 0,
                                                                                 0, 0);
                                    if (ctok[c] == tok) o[c][t][j] += x;
                                }
                                __builtin_amdgcn_sched_barrier(0);
                            }
                    }
                }
            }
        }

        // Merge the waves: everyone to the block's maximum, then sums by halves.
#pragma unroll
        for (int c = 0; c < C; c++) {
            l[c] += __shfl_xor(l[c], 16, 64);
            l[c] += __shfl_xor(l[c], 32, 64);
            if (g == 0) sm_m[wave][c * 16 + col] = m[c], sm_l[wave][c * 16 + col] = l[c];
        }
        __syncthreads();
#pragma unroll
        for (int c = 0; c < C; c++) {
            float mm = -INFINITY, ll = 0.0f;
            for (int w = 0; w < W; w++) mm = fmaxf(mm, sm_m[w][c * 16 + col]);
            for (int w = 0; w < W; w++) {
                const float mw = sm_m[w][c * 16 + col];
                if (mw != -INFINITY) ll += sm_l[w][c * 16 + col] * exp_weight(mw - mm);
                else ll += sm_l[w][c * 16 + col];  // 0, or the NaN of NaN scores
            }
            const float f = m[c] == -INFINITY ? 1.0f : exp_weight(m[c] - mm);
            l[c] = ll;
#pragma unroll
            for (int t = 0; t < VB; t++)
#pragma unroll
                for (int j = 0; j < 4; j++) o[c][t][j] *= f;
        }
#pragma unroll
        for (int h = W / 2; h >= 1; h /= 2) {
            if (ntiles <= h) continue;  // the upper waves had no positions
            if (wave >= h && wave < 2 * h) {
#pragma unroll
                for (int c = 0; c < C; c++)
#pragma unroll
                    for (int t = 0; t < VB; t++)
#pragma unroll
                        for (int j = 0; j < 4; j++) sm[(((wave - h) * C + c) * VB * 4 + t * 4 + j) * 64 + lane] = o[c][t][j];
            }
            __syncthreads();
            if (wave < h) {
#pragma unroll
                for (int c = 0; c < C; c++)
#pragma unroll
                    for (int t = 0; t < VB; t++)
#pragma unroll
                        for (int j = 0; j < 4; j++) o[c][t][j] += sm[((wave * C + c) * VB * 4 + t * 4 + j) * 64 + lane];
            }
            __syncthreads();
        }
        if (wave != 0) continue;
#pragma unroll
        for (int c = 0; c < C; c++) {
            if (!cv[c]) continue;
            const int cc = c * 16 + col;
            float *dst = a.out + (size_t)(r0 + first + cc / hn) * a.out_stride + (size_t)(h0 + cc % hn) * a.vd;
            const float inv = 1.0f / l[c];
            const bool none = cp[c] < cl[c];
#pragma unroll
            for (int t = 0; t < VB; t++)
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const int d = 64 * t + 16 * g + 4 * i;
                    if (d >= a.vd) continue;
                    f32x4 x;
#pragma unroll
                    for (int j = 0; j < 4; j++) x[j] = none ? 0.0f : o[c][t][j][i] * inv;
                    // Few positions: the quotient correctly rounded (one step
                    // from the product with the reciprocal), which shows
                    // where there are one or two (error against 64 bits, width
                    // 24: 4.3e-8 -> 4.0e-8; the kernel for odd widths 4.1e-8).
                    // Beyond a tile the sums' roundings count.
                    if (ntiles == 1)
#pragma unroll
                        for (int j = 0; j < 4; j++) {
                            const float y = fmaf(fmaf(-x[j], l[c], o[c][t][j][i]), inv, x[j]);
                            x[j] = !none && fabsf(x[j]) < INFINITY ? y : x[j];
                        }
                    gstore((f32x4 *)(dst + d), x);
                }
        }
    }
}

bool aligned16(const void *p) { return (uintptr_t)p % 16 == 0; }

// What attention_tile_kernel takes: 16-byte loads of every row, query heads
// in whole groups per key/value head.
bool attention_tile_ok(const AttnArgs &a, int heads) {
    return a.qd % 4 == 0 && a.vd % 4 == 0 && a.vd <= 256 && heads % a.n_kv == 0 && a.q_stride % 4 == 0 &&
           a.out_stride % 4 == 0 && aligned16(a.q) && aligned16(a.kc) && aligned16(a.vc) && aligned16(a.out);
}

template <int QC, bool EX, int VB, int C, int W>
void launch_tile(AttnArgs a, hipStream_t s) {
    a.rc = std::min(a.rep, 16 * C);
    a.chunks = (a.rep + a.rc - 1) / a.rc;
    a.tt = 16 * C / a.rc;
    a.groups = (a.rows + a.tt - 1) / a.tt;
    // Runs of a group go to `split` blocks: enough that a decode step (every
    // row a run of its own) fills the chip, few where the groups already do,
    // since a prompt's groups are one run each and their other blocks leave
    // at once.
    const long long base = (long long)a.groups * a.chunks * a.n_kv;
    a.split = (int)std::max<long long>(1, std::min<long long>(a.tt, (2048 + base - 1) / base));
    const long long units = ((long long)a.groups * a.split + 7) / 8 * 8;
    hipLaunchKernelGGL((attention_tile_kernel<QC, EX, VB, C, W>), dim3((unsigned)(units * a.chunks * a.n_kv)),
                       dim3(W * 64), 0, s, a);
}

template <int QC, int VB>
void launch_width(const AttnArgs &a, hipStream_t s) {
    const bool ex = a.qd == QC * 16;
    // Two column tiles halve the cache traffic of a prefill once there is a
    // group of 32 columns for every CU; below that, 16 columns and more waves
    // over the positions of each.  16 -> 32 columns, 32 heads over 8 of width
    // 128: prompts of 250 and 500 rows 28.4 -> 22.1 and 62.1 -> 42.1 us, 16
    // sequences of 16 new rows 74.8 -> 57.0.  A decode step of many sequences
    // (one row per run, which the arguments here do not tell) pays for the empty
    // columns, 200 sequences 258 -> 312 us, which is why the line is not lower;
    // one of more than the line's pairs pays as well.
    const long long wide = ((long long)a.rows * a.rep + 31) / 32 * a.n_kv;
    if (QC < 16 && wide >= 256) {
        if (ex) launch_tile<QC, true, VB, QC < 16 ? 2 : 1, 4>(a, s);
        else launch_tile<QC, false, VB, QC < 16 ? 2 : 1, 4>(a, s);
    } else {
        constexpr int W = VB < 4 ? 8 : 4;
        if (ex) launch_tile<QC, true, VB, 1, W>(a, s);
        else launch_tile<QC, false, VB, 1, W>(a, s);
    }
}

}  // namespace
}  // namespace moe

using namespace moe;

extern "C" int moe_attention(const float *q, int64_t q_stride, int32_t rows, int32_t heads, int32_t n_kv, int32_t qd,
                             int32_t vd, float scale, const float *kcache, const float *vcache, int64_t ctx,
                             const int32_t *seq, const int32_t *pos, int32_t max_pos, int32_t window, float *out,
                             int64_t out_stride, void *stream) {
    if (!q || !kcache || !vcache || !seq || !pos || !out || rows < 0 || heads <= 0 || n_kv <= 0 || qd <= 0 ||
        vd <= 0 || qd > kAttnMaxDim || max_pos < 0 || max_pos >= ctx)
        return fail(MOE_EINVAL, "moe_attention: bad argument (qd %d, vd %d, max position %d, context %lld)", qd, vd,
                    max_pos, (long long)ctx);
    if (rows == 0) return MOE_OK;
    const int span = window > 0 ? std::min(window, max_pos + 1) : max_pos + 1;
    const size_t lds = (size_t)span * 4;
    if (lds > 64 * 1024) return fail(MOE_EUNSUP, "moe_attention: %d positions exceed the score buffer", span);
    hipStream_t s = (hipStream_t)stream;
    AttnArgs a{};
    a.q = q, a.kc = kcache, a.vc = vcache, a.seq = seq, a.pos = pos, a.out = out;
    a.q_stride = q_stride, a.out_stride = out_stride, a.ctx = ctx;
    a.rows = rows, a.n_kv = n_kv, a.rep = heads / n_kv, a.qd = qd, a.vd = vd, a.window = window;
    a.scale = scale;
    if (attention_tile_ok(a, heads)) {
        if (qd <= 64 && vd <= 64) launch_width<4, 1>(a, s);
        else if (qd <= 128 && vd <= 128) launch_width<8, 2>(a, s);
        else if (qd <= 192 && vd <= 128) launch_width<12, 2>(a, s);
        else launch_width<16, 4>(a, s);
    } else {
        // Past 32 KiB of scores the launch asks for the larger dynamic LDS limit
        // (on the current device, every time: the setting is per device).
        if (lds > 32 * 1024) {
            const hipError_t e = hipFuncSetAttribute((const void *)attention_kernel,
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, 64 * 1024);
            if (e != hipSuccess) return fail(MOE_EHIP, "moe_attention: LDS limit: %s", hipGetErrorString(e));
        }
        hipLaunchKernelGGL(attention_kernel, dim3((unsigned)rows * heads), dim3(64), lds, s, q, q_stride, heads, n_kv, qd,
                           vd, scale, kcache, vcache, ctx, seq, pos, window, out, out_stride);
    }
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? MOE_OK : fail(MOE_EHIP, "attention kernel: %s", hipGetErrorString(e));
}
