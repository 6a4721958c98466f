// Attention of the forward (qwen35_forward.rs:639-671) and its softmax
// (crates/unltd-tensor/src/kernels.rs:157-168), for one decode position or a
// prefill's rows of them. Caches are [n_ctx][n_head_kv][hd] f32; q head h
// reads kv head h / group (consecutive heads share a kv head).
//
// Bit contract: a score is the f64 pairwise sum (kernels.rs:21-42) of hd
// exact products rounded to f32, an output the f64 sum of soft[p] V[p] in
// position order rounded to f32. The products run on the f64 matrix cores
// (v_mfma_f64, same 64-bit products and sums as the vector units, 64 or 16
// products' operands converted once per lane instead of once per product),
// whose order of addition is another; each result carries a rigorous bound e
// on the distance between that sum S and the reference's, and where both ends
// of [S - e, S + e] round to the same f32 (rounding is monotonic) that is the
// reference's value. Elsewhere (about 1 in 10^4 to 10^5) the reference's
// order is replayed.
#include <algorithm>

#include "uq_device.h"
#include "uq_internal.h"

namespace uq {

namespace {

typedef double d4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));  // rows start at any float
typedef short s4 __attribute__((ext_vector_type(4)));

constexpr int kAttnMaxGroup = 8;

// r = lo. A NaN decides nothing, whether of S or of a bound whose parts left
// their range: its bits may equal themselves where the reference is finite.
__device__ __forceinline__ bool decided(double S, double e, float &r) {
    const float lo = (float)(S - e), hi = (float)(S + e);
    r = lo;
    return __float_as_uint(lo) == __float_as_uint(hi) && lo == lo;
}

// f64 sum over the lanes l, l ^ 16, l ^ 32, l ^ 48, in each of them.
__device__ __forceinline__ double quarter_sum(double v) {
    v += __shfl_xor(v, 16);
    return v + __shfl_xor(v, 32);
}

// ---- softmax --------------------------------------------------------------

// Pairwise tree (kernels.rs:27-42) of lv[0, len) in LDS, level by level:
// pairs (2i, 2i+1), an odd tail carried up. Every thread takes part;
// returns lv[0] to all (len <= 2 * kSmTPB * kTreeRegs).
constexpr int kSmTPB = 256;
constexpr int kTreeRegs = 16;
__device__ double lds_tree(double *lv, int len) {
    while (len > 1) {
        const int nl = (len + 1) / 2;
        double v[kTreeRegs];
        int c = 0;
        for (int p = threadIdx.x; p < nl; p += kSmTPB, c++) v[c] = 2 * p + 1 < len ? lv[2 * p] + lv[2 * p + 1] : lv[2 * p];
        __syncthreads();
        c = 0;
        for (int p = threadIdx.x; p < nl; p += kSmTPB, c++) lv[p] = v[c];
        __syncthreads();
        len = nl;
    }
    const double r = lv[0];
    __syncthreads();
    return r;
}

__device__ __forceinline__ float wave_max_f(float v) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) v = fmaxf(v, __shfl_xor(v, off));
    return v;
}

// Rows longer than kSmRowMax, one workgroup per row, in place allowed.
// The denominator is pairwise_sum_f64 over the row. For a chunk size C that
// is a power of two, level log2(C) of that tree holds the trees of the full
// C-chunks followed by the tree of the remainder (whose node is always the
// carried odd tail below that level), so the row sum is the pairwise tree
// over the chunk sums: each chunk is reduced in LDS, then the chunk sums.
constexpr int kSmChunk = 2 * kSmTPB * kTreeRegs;  // 8192
constexpr int kSmMaxChunks = 2048;
static_assert((kSmChunk & (kSmChunk - 1)) == 0, "chunk trees must be nodes of the row tree");
// Rows of token z = blockIdx.y (the attention of a prefill) are n + z dn
// long and start zst floats after token z - 1's.
__global__ __launch_bounds__(kSmTPB) void softmax_kernel(float *out, const float *x, int n, float scale, int dn,
                                                         size_t zst) {
    __shared__ double lv[kSmChunk / 2];
    __shared__ double cs[kSmMaxChunks];
    __shared__ float red[kSmTPB / 64];
    n += (int)blockIdx.y * dn;
    const size_t row0 = (size_t)blockIdx.y * zst + (size_t)blockIdx.x * n;
    const float *xr = x + row0;
    float *yr = out + row0;
    float m = -INFINITY;
    for (int i = threadIdx.x; i < n; i += kSmTPB) m = fmaxf(m, xr[i]);
    m = wave_max_f(m);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
    __syncthreads();
    for (int i = 0; i < kSmTPB / 64; i++) m = fmaxf(m, red[i]);
    auto ex = [&](int i) { return expf_cr(__fmul_rn(__fsub_rn(xr[i], m), scale)); };
    const int nch = (n + kSmChunk - 1) / kSmChunk;
    for (int c = 0; c < nch; c++) {
        const int base = c * kSmChunk, cl = min(kSmChunk, n - base);
        const int len = (cl + 1) / 2;  // level 1 straight from the exponentials
        for (int p = threadIdx.x; p < len; p += kSmTPB) {
            const int i = base + 2 * p;
            lv[p] = 2 * p + 1 < cl ? (double)ex(i) + (double)ex(i + 1) : (double)ex(i);
        }
        __syncthreads();
        const double t = lds_tree(lv, len);
        if (threadIdx.x == 0) cs[c] = t;
    }
    __syncthreads();
    const double sum = lds_tree(cs, nch);
    for (int i = threadIdx.x; i < n; i += kSmTPB) yr[i] = (float)((double)ex(i) / sum);
}

// Rows of at most 4 T J values, one workgroup of T per row, every value in
// registers from the one read to the one write and its exponential formed
// once (softmax_kernel forms it twice and reads the row three times). Thread
// t holds the quads t, t + T, ...: a quad's tree, then the wave's fixed tree
// over 64 adjacent quads (wave_sum_d) gives the trees of the row's 256-chunks,
// and every wave forms the tree over those. Missing elements are zeros: every
// term is an exponential (>= +0), so a zero added where the tree carries an
// odd tail up leaves the same value. The weight e / sum is e * (1 / sum)
// where that product's 2^-51 neighbourhood rounds to one f32, else the
// division: q = e * rn(1 / sum) lies within 2^-52 (relative) of the quotient,
// which the f64 division rounds by another 2^-53.
// Bound by the f64 exponential (about 40 f64 instructions a value): 16 rows of
// 24001 in 13.5 us against softmax_kernel's 77, 4080 rows of 3842 in 33 against 97.
// Rows up to 256 take a wave each: 5000 rows of 1, 4, 32 values in 4.8, 5.6, 5.6 us
// against 6.9, 8.0, 8.0 with four waves, three of them idle.
template <int T, int J>
__global__ __launch_bounds__(T) void softmax_row_kernel(float *out, const float *x, int n, float scale, int dn,
                                                        size_t zst) {
    constexpr int W = T / 64;
    static_assert(W * J <= 128, "a wave forms the tree over the chunks, two a lane");
    __shared__ float red[W];
    __shared__ double cs[128];
    n += (int)blockIdx.y * dn;
    const size_t row0 = (size_t)blockIdx.y * zst + (size_t)blockIdx.x * n;
    const float *xr = x + row0;
    float *yr = out + row0;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    float v[J][4];
    float m = -INFINITY;
#pragma unroll
    for (int j = 0; j < J; j++) {
        const int i = 4 * (tid + T * j);
        if (i + 4 <= n) {
            const f4u q = *(const f4u *)(xr + i);
#pragma unroll
            for (int k = 0; k < 4; k++) v[j][k] = q[k];
        } else {
#pragma unroll
            for (int k = 0; k < 4; k++) v[j][k] = i + k < n ? xr[i + k] : -INFINITY;
        }
    }
#pragma unroll
    for (int j = 0; j < J; j++)
#pragma unroll
        for (int k = 0; k < 4; k++) m = fmaxf(m, v[j][k]);
    m = wave_max_f(m);
    if (lane == 0) red[w] = m;
    for (int i = tid; i < 128; i += T) cs[i] = 0.0;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < W; i++) m = fmaxf(m, red[i]);
#pragma unroll
    for (int j = 0; j < J; j++) {
        const int i = 4 * (tid + T * j);
        if (256 * (w + W * j) >= n) break;  // wave-uniform: no element of the wave's chunk
#pragma unroll
        for (int k = 0; k < 4; k++) v[j][k] = i + k < n ? expf_cr(__fmul_rn(__fsub_rn(v[j][k], m), scale)) : 0.0f;
        const double t = wave_sum_d(((double)v[j][0] + (double)v[j][1]) + ((double)v[j][2] + (double)v[j][3]));
        if (lane == 0) cs[w + W * j] = t;
    }
    __syncthreads();
    const double sum = wave_sum_d(cs[2 * lane] + cs[2 * lane + 1]);
    const double inv = 1.0 / sum;
#pragma unroll
    for (int j = 0; j < J; j++) {
        const int i = 4 * (tid + T * j);
        if (256 * (w + W * j) >= n) break;
        float r[4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const double q = (double)v[j][k] * inv;
            if (!decided(q, q * 0x1p-51, r[k])) r[k] = (float)((double)v[j][k] / sum);
        }
        if (i + 4 <= n) {
            *(f4u *)(yr + i) = f4u{r[0], r[1], r[2], r[3]};
        } else {
#pragma unroll
            for (int k = 0; k < 4; k++)
                if (i + k < n) yr[i + k] = r[k];
        }
    }
}
constexpr int kSmRowMax = 4 * 1024 * 8;

hipError_t softmax_rows(float *out, const float *x, int n, int rows, float scale, int dn, int nz, size_t zst,
                        hipStream_t s) {
    const dim3 grid(rows, nz);
    const int hi = n + dn * (nz - 1);  // the longest row
#define UQ_SM(T, J) hipLaunchKernelGGL((softmax_row_kernel<T, J>), grid, dim3(T), 0, s, out, x, n, scale, dn, zst)
    if (hi <= 256)
        UQ_SM(64, 1);  // a wave a row
    else if (hi <= 1024)
        UQ_SM(256, 1);
    else if ((size_t)rows * nz >= 512 && hi <= 2048)
        UQ_SM(256, 2);
    else if ((size_t)rows * nz >= 512 && hi <= 4096)
        UQ_SM(256, 4);
    else if (hi <= 4096)
        UQ_SM(1024, 1);
    else if (hi <= 8192)
        UQ_SM(1024, 2);
    else if (hi <= 16384)
        UQ_SM(1024, 4);
    else if (hi <= kSmRowMax)
        UQ_SM(1024, 8);
    else
        hipLaunchKernelGGL(softmax_kernel, grid, dim3(kSmTPB), 0, s, out, x, n, scale, dn, zst);
#undef UQ_SM
    return hipGetLastError();
}

// ---- scores ---------------------------------------------------------------

// Pairwise sum (kernels.rs:21-42) of 64 * E values, lane l holding values
// [E*l, E*l + E). For a power-of-two count the tree adds adjacent nodes
// level by level: the lane-local tree, then the xor butterfly over lanes
// (both lanes of a pair form the same node: f64 addition is commutative).
template <int E>
__device__ double wave_pairwise(double (&t)[E]) {
#pragma unroll
    for (int w = E; w > 1; w /= 2)
#pragma unroll
        for (int j = 0; j < w / 2; j++) t[j] = t[2 * j] + t[2 * j + 1];
    double s = t[0];
#pragma unroll
    for (int off = 1; off < 64; off *= 2) s = s + __shfl_xor(s, off);
    return s;
}

// The reference's dot of two rows of HD, formed by the whole wave.
template <int HD>
__device__ float tree_dot(const float *__restrict__ a, const float *__restrict__ b) {
    constexpr int E = HD / 64;
    const int lane = threadIdx.x & 63;
    double d[E];
#pragma unroll
    for (int e = 0; e < E; e++) d[e] = (double)a[lane * E + e] * (double)b[lane * E + e];
    return (float)wave_pairwise<E>(d);
}

// Any order of adding the HD products, each add rounded by at most 2^-52,
// lies within HD 2^-52 A of the exact sum, the reference's tree within
// 9 * 2^-53 A, A = sum |q_i k_i| <= |q| |k| (Cauchy-Schwarz): the norms are
// one multiply-add per operand instead of one per product. (HD + 66) 2^-52
// leaves room for the roundings of the norms, of e and of S +- e.
template <int HD>
__device__ __forceinline__ double score_bound(double qn, double kn) {
    return (double)(HD + 66) * 0x1p-52 * (qn * kn);
}

// A norm from its square, at most 2^-10 above it. The root (v_sqrt_f64, 2^29
// units in the last place) has the range of f64, where squares of f32 neither
// underflow nor overflow. It is zero for a row of zeros: the score is then a
// zero with a bound of zero, of another sign than the reference's perhaps,
// which softmax drops (exp of either zero is 1).
__device__ __forceinline__ double norm_above(double sq) { return __builtin_amdgcn_sqrt(sq) * (1.0 + 0x1p-11); }

// Whether a score S that its bound left undecided needs a replay. Not so, and
// S itself the result r: a NaN or an infinity of these products, which is the
// reference's too, and a zero of a row of zeros.
__device__ __forceinline__ bool needs_replay(double S, double qn, double kn, float &r) {
    if (S - S == 0.0 && qn != 0.0 && kn != 0.0) return true;
    r = (float)S;
    return false;
}

// scores[h][p] for a few queries (a decode step, or the first rows of a
// short prefill), one wave per workgroup, no LDS. v_mfma_f64_4x4x4_4b: four
// blocks of 4 x 4 x 4, block b = heads 0..3 of the kv head (x 4 GB of them
// for groups above four) against positions 4 b .. 4 b + 3, so a tile of 16
// positions takes HD / 4 instructions (about 17 cycles each) and all products
// are wanted for a group of four. Operands: lane l holds element
// 16 c + 4 (l >> 4) + u of position l & 15 (K) and of head l & 3 (q), one
// 16-byte load per c feeding u = 0..3; result lane l: head l >> 4, position
// l & 15. A wave keeps its q in registers and strides over the tiles, the
// next tile's rows in flight (16 KB a wave) while this one is multiplied.
// Bound by reading K: 24001 positions x 4 x 256 (98 MB) in 25.7 us against
// 60 us for the vector-unit kernel it replaces.
// Query z = blockIdx.z (of a prefill) sees n_ctx + z positions; its q and
// scores are z q_st and z sc_st floats on.
template <int HD, int GB>
__global__ __launch_bounds__(64, 2) void attn_scores_kernel(float *__restrict__ scores, const float *__restrict__ q,
                                                         const float *__restrict__ kc, int n_ctx, int n_head_kv,
                                                         int group, size_t q_st, size_t sc_st) {
    constexpr int CH = HD < 256 ? HD : 256;  // dims per pass (registers)
    constexpr int NC = CH / 16, PASSES = HD / CH;
    n_ctx += (int)blockIdx.z;
    q += blockIdx.z * q_st;
    scores += blockIdx.z * sc_st;
    const int lane = threadIdx.x, kv = blockIdx.x, pos = lane & 15, kk = lane >> 4;
    const int ntile = (n_ctx + 15) / 16;
    if ((int)blockIdx.y >= ntile) return;
    const size_t kv_len = (size_t)n_head_kv * HD;
    const float *kb = kc + (size_t)kv * HD + 4 * kk;
    auto krow = [&](int t) { return kb + (size_t)min(16 * t + pos, n_ctx - 1) * kv_len; };
    // heads past the group repeat its last one (not stored)
    const float *qb[GB];
#pragma unroll
    for (int b = 0; b < GB; b++) qb[b] = q + ((size_t)kv * group + min(4 * b + (lane & 3), group - 1)) * HD + 4 * kk;
    f4 kx[NC], qx[GB][NC];
    auto load_k = [&](int t, int ps) {
        const float *r = krow(t) + ps * CH;
#pragma unroll
        for (int c = 0; c < NC; c++) kx[c] = *(const f4u *)(r + 16 * c);
    };
    auto load_q = [&](int ps) {
#pragma unroll
        for (int b = 0; b < GB; b++)
#pragma unroll
            for (int c = 0; c < NC; c++) qx[b][c] = *(const f4u *)(qb[b] + ps * CH + 16 * c);
    };
    load_k(blockIdx.y, 0);
    if constexpr (PASSES == 1) load_q(0);
    double qn[GB];  // |q| of head 4 b + (lane >> 4), the result's
    {
        double s[GB];
#pragma unroll
        for (int b = 0; b < GB; b++) {
            s[b] = 0.0;
#pragma unroll 1
            for (int ps = 0; ps < PASSES; ps++) {
                if constexpr (PASSES > 1) load_q(ps);
#pragma unroll
                for (int c = 0; c < NC; c++) {
#pragma unroll
                    for (int u = 0; u < 4; u++) s[b] = fma((double)qx[b][c][u], (double)qx[b][c][u], s[b]);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            qn[b] = __shfl(norm_above(quarter_sum(s[b])), kk);
        }
    }
    for (int t = blockIdx.y; t < ntile; t += gridDim.y) {
        double acc[GB], ks = 0.0;
#pragma unroll
        for (int b = 0; b < GB; b++) acc[b] = 0.0;
#pragma unroll 1
        for (int ps = 0; ps < PASSES; ps++) {
            if constexpr (PASSES > 1) load_q(ps);
            // q stays f32: the conversions below cost less than the registers of their results
#pragma unroll
            for (int b = 0; b < GB; b++)
#pragma unroll
                for (int c = 0; c < NC; c++) asm volatile("" : "+v"(qx[b][c]));
            // each 16-byte load of the next rows is issued as its registers fall free
            // (after the last tile: q again, which is in cache)
            const float *nr = ps + 1 < PASSES                 ? krow(t) + (ps + 1) * CH
                              : t + (int)gridDim.y < ntile ? krow(t + gridDim.y)
                                                              : qb[0];
#pragma unroll
            for (int c = 0; c < NC; c++) {
                const f4 cur = kx[c];
                kx[c] = *(const f4u *)(nr + 16 * c);
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    const double k = (double)cur[u];
                    ks = fma(k, k, ks);
#pragma unroll
                    for (int b = 0; b < GB; b++)
                        acc[b] = __builtin_amdgcn_mfma_f64_4x4x4f64((double)qx[b][c][u], k, acc[b], 0, 0, 0);
                }
                __builtin_amdgcn_sched_barrier(0);  // the loads stay spread over the steps
            }
        }
        const double kn = norm_above(quarter_sum(ks));
        const int p = 16 * t + pos;
#pragma unroll
        for (int b = 0; b < GB; b++) {
            const int g = 4 * b + kk;
            const bool in = g < group && p < n_ctx;
            float r;
            const bool ok = decided(acc[b], score_bound<HD>(qn[b], kn), r);
            unsigned long long mask = __ballot(in && !ok);
            if (mask) mask = __ballot(in && !ok && needs_replay(acc[b], qn[b], kn, r));
            while (mask) {
                const int l = __ffsll(mask) - 1;
                mask &= mask - 1;
                const float d = tree_dot<HD>(q + ((size_t)kv * group + 4 * b + (l >> 4)) * HD,
                                             kc + (size_t)(16 * t + (l & 15)) * kv_len + (size_t)kv * HD);
                if (lane == l) r = d;
            }
            if (in) scores[(size_t)(kv * group + g) * n_ctx + p] = r;
        }
    }
}

// scores of a prefill chunk, v_mfma_f64_16x16x4: a workgroup of four waves
// holds the K rows of 64 positions, 16 a wave, in registers, and goes
// over tiles of 16 (query, head) pairs of the kv head, each staged once into
// LDS as f64 in the operands' order (two tiles: the next one is written while
// this one is read, one barrier a tile). Lane l of a wave: position l & 15,
// elements 16 c + 4 (l >> 4) + u; a 16 x 16 tile takes HD / 4 instructions of
// 64 cycles against one 16-byte LDS read each for two of them: 255 queries x
// 16 heads over 3842 positions of 256, 16.0 GFLOP, take 181 us, the matrix
// cores busy 53% of it (58% for the next chunk's 4096 positions) and the vector
// units 16% (718 us for the lane-per-position vector kernel this replaces). f64 vector instructions do
// not overlap with f64 matrix ones here (4 to 7 cycles each, 16 more where the
// kinds alternate), so the loop holds none: K and q are converted outside.
// Query zz sees n_ctx + zz positions (causal): tiles of pairs that see none
// of the workgroup's positions are skipped. blockIdx.z splits the pair tiles.
template <int HD>
__global__ __launch_bounds__(256, 2) void attn_scores_tile_kernel(float *__restrict__ scores,
                                                                  const float *__restrict__ q,
                                                                  const float *__restrict__ kc, int n_ctx,
                                                                  int n_head_kv, int group, size_t q_st, size_t sc_st,
                                                                  int rows) {
    constexpr int NC = HD / 16;
    extern __shared__ __align__(16) double qs[];  // [2][NC][2][64][2]
    __shared__ __align__(16) double nrm[2][16][4];
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kv = blockIdx.y, p0 = blockIdx.x * 64, pairs = rows * group;
    const int ntile = (pairs + 15) / 16, per = (ntile + gridDim.z - 1) / gridDim.z;
    // the first pair that sees p0 and the workgroup's share of the tiles
    const int first = p0 < n_ctx ? 0 : (p0 - n_ctx + 1) * group / 16;
    const int t_lo = max((int)blockIdx.z * per, first), t_hi = min(ntile, ((int)blockIdx.z + 1) * per);
    if (t_lo >= t_hi) return;  // the whole workgroup
    const int n_last = n_ctx + rows - 1;
    const size_t kv_len = (size_t)n_head_kv * HD;
    const int pos = p0 + 16 * wv + (lane & 15), kk = lane >> 4;
    const float *kr = kc + (size_t)min(pos, n_last - 1) * kv_len + (size_t)kv * HD + 4 * kk;
    // staging: thread -> pair i of the tile, 16-byte group kk, c = wv, wv + 4, ...
    const int si = (lane >> 2) & 15, sk = lane & 3;
    constexpr int SI = NC / 4;
    static_assert(NC % 4 == 0, "the four waves stage alike");
    f4 st[SI];
    // pr / group, pr < 2^19: the remainder's error pr (group - 1) 2^-32 is below 1 / group
    const uint32_t rg = (uint32_t)((0x100000000ull + group - 1) / group);
    auto query = [&](int pr) { return group == 1 ? pr : (int)__umulhi((uint32_t)pr, rg); };
    auto stage_load = [&](int t) {
        const int pr = min(16 * t + si, pairs - 1), zz = query(pr);
        const float *r = q + (size_t)zz * q_st + ((size_t)kv * group + (pr - zz * group)) * HD + 4 * sk;
#pragma unroll
        for (int j = 0; j < SI; j++)
            st[j] = *(const f4u *)(r + 16 * (wv + 4 * j));
    };
    auto stage_store = [&](int b) {
        double *d = qs + (size_t)b * NC * 256 + 2 * (si + 16 * sk);
#pragma unroll
        for (int j = 0; j < SI; j++) {
            double2 *o = (double2 *)(d + (wv + 4 * j) * 256);
            o[0] = make_double2((double)st[j][0], (double)st[j][1]);
            o[64] = make_double2((double)st[j][2], (double)st[j][3]);
        }
        double qq = 0.0;  // the pair's |q|^2: this wave's part
#pragma unroll
        for (int j = 0; j < SI; j++)
#pragma unroll
            for (int u = 0; u < 4; u++) qq = fma((double)st[j][u], (double)st[j][u], qq);
        qq += dpp_d<0xB1>(qq);
        qq += dpp_d<0x4E>(qq);
        if (sk == 0) nrm[b][si][wv] = qq;
    };
    stage_load(t_lo);
    double kd[NC][4];
    double ks = 0.0;
#pragma unroll
    for (int c0 = 0; c0 < NC; c0 += 4) {
        f4 v[4];
#pragma unroll
        for (int c = 0; c < 4; c++) v[c] = *(const f4u *)(kr + 16 * (c0 + c));
#pragma unroll
        for (int c = 0; c < 4; c++)
#pragma unroll
            for (int u = 0; u < 4; u++) kd[c0 + c][u] = (double)v[c][u], ks = fma(kd[c0 + c][u], kd[c0 + c][u], ks);
    }
    const double kn = norm_above(quarter_sum(ks));
    stage_store(0);
    for (int t = t_lo; t < t_hi; t++) {
        const int b = (t - t_lo) & 1;
        __syncthreads();  // tile t is in buffer b; buffer b ^ 1 is no longer read
        if (t + 1 < t_hi) stage_load(t + 1);
        const double2 *d = (const double2 *)(qs + (size_t)b * NC * 256) + lane;
        d4 acc = {0.0, 0.0, 0.0, 0.0};
        double2 x = d[0], y = d[64];
#pragma unroll
        for (int c = 0; c < NC; c++) {
            const double2 nx = d[2 * min(c + 1, NC - 1) * 64], ny = d[(2 * min(c + 1, NC - 1) + 1) * 64];
            acc = __builtin_amdgcn_mfma_f64_16x16x4f64(x.x, kd[c][0], acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f64_16x16x4f64(x.y, kd[c][1], acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f64_16x16x4f64(y.x, kd[c][2], acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f64_16x16x4f64(y.y, kd[c][3], acc, 0, 0, 0);
            x = nx, y = ny;
            __builtin_amdgcn_sched_barrier(0);  // reads one step ahead, not all of them (registers)
        }
        double qn[4];  // |q| of pair kk + 4 r
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const double2 *o = (const double2 *)nrm[b][kk + 4 * r];
            qn[r] = norm_above((o[0].x + o[0].y) + (o[1].x + o[1].y));
        }
        if (t + 1 < t_hi) stage_store(b ^ 1);
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int pr = 16 * t + kk + 4 * r, zz = query(pr), g = pr - zz * group;
            const int nzc = n_ctx + zz;
            const bool in = pr < pairs && pos < nzc;
            float v;
            const bool ok = decided(acc[r], score_bound<HD>(qn[r], kn), v);
            unsigned long long mask = __ballot(in && !ok);
            if (mask) mask = __ballot(in && !ok && needs_replay(acc[r], qn[r], kn, v));
            while (mask) {
                const int l = __ffsll(mask) - 1;
                mask &= mask - 1;
                const int lp = 16 * t + (l >> 4) + 4 * r, lz = query(lp);
                const float dv = tree_dot<HD>(q + (size_t)lz * q_st + ((size_t)kv * group + (lp - lz * group)) * HD,
                                              kc + (size_t)(p0 + 16 * wv + (l & 15)) * kv_len + (size_t)kv * HD);
                if (lane == l) v = dv;
            }
            if (in) scores[(size_t)zz * sc_st + (size_t)(kv * group + g) * nzc + pos] = v;
        }
    }
}

// ---- values ---------------------------------------------------------------
// out[h][i] = (f32) of the f64 sum over p, in order, of t_p = soft[h][p]
// V[p][i] (every product exact in f64). Error of that order: each add rounds
// by at most u = 2^-53 of the partial sum it forms, |s_p| <= |P| + A_blk for
// the prefix P at the start of p's 16-block and the block's A_blk =
// sum |t|, so the reference lies within u (16 sum_blk |P| + 16 A) of the
// exact sum, A over all positions: with values of both signs that is tens of
// times tighter than the usual n u A, and so are the replays rarer. Prefixes
// are read off the running matrix-core accumulators. A segment of len
// positions that starts at prefix B adds len |B| to 16 PS, PS its own blocks'
// prefixes. This sum itself rounds by at most 2 u of its own partials: its
// adds per block go on top of the reference's 16 (per_block).
struct PvErr {
    double B = 0.0, E = 0.0;  // sum so far; error in units of u
    __device__ __forceinline__ void segment(double S, double PS, double A, int len, double per_block) {
        E += (double)(len + 4) * fabs(B) + per_block * (PS + A);
        B += S;
    }
    // 1 + 1/32: the roundings of PS, E and of S +- e, and by how much an A of rounded operands may be low
    // (attn_pv_tile_kernel: 2^-8 + 2^-12; four f32 |V| in attn_pv_kernel: less)
    __device__ __forceinline__ double bound() const { return (1.03125 * 0x1p-53) * (E + 8.0 * fabs(B)); }
};

// The reference's sum by a whole workgroup of T threads, all of which call it
// and get the result. The chain of n dependent adds is cut into runs of
// kRun positions, a thread each, on this ground: while a run's partial sums
// stay in one binade (spacing q), fl(x + m q + t) = fl(x + t) + m q for even m
// (ties to even see the parity of x / q only), so the run's effect on the
// exact incoming sum s is s + D[parity of s / q], with both D taken from two
// chains started at neighbouring doubles P and P + q near s. P is a parallel
// prefix sum; |s - P| <= dist bounds how far its chain may be from the real
// one, and a run is regular if its chain keeps that distance from the ends of
// the binade. Consecutive regular runs of one binade are combined by a scan
// (the pairs D compose; all exact: multiples of q below 2^53 q), then each
// wave in turn takes its chains of them in order, irregular runs by their
// adds, and passes the exact sum on. 24001 positions: 110 us against 235 for
// the adds one after another; 3071: 20 against 30. The loop over the chains is
// bound by its own instructions' fetch: placed anywhere, the kernel took 163 to
// 171 us for one and the same input, by what stood before it; from the start of
// a cache line, and with a select of the two D instead of a branch, 162.5.
constexpr int kRun = 16;
struct SeqLds {
    double tot[16], abs[16], dist[16], token;
};
__device__ __forceinline__ double lane_value(double v, int l) {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), l),
                            __builtin_amdgcn_readlane(__double2loint(v), l));
}
template <int T>
__device__ __forceinline__ double wg_replay(SeqLds &L, const float *__restrict__ sr, const float *__restrict__ vl,
                                         size_t kv_len, int n) {
    constexpr int W = T / 64;
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    double s = 0.0;
    for (int base = 0; base < n; base += T * kRun) {
        double t[kRun];
        {
            const int p0 = base + kRun * (int)threadIdx.x;
            float sv[kRun], vv[kRun];
#pragma unroll
            for (int k = 0; k < kRun; k++) vv[k] = vl[(size_t)min(p0 + k, n - 1) * kv_len];
            if (p0 + kRun <= n) {
#pragma unroll
                for (int k = 0; k < kRun; k += 4) {
                    const f4u x = *(const f4u *)(sr + p0 + k);
#pragma unroll
                    for (int e = 0; e < 4; e++) sv[k + e] = x[e];
                }
            } else {
#pragma unroll
                for (int k = 0; k < kRun; k++) sv[k] = sr[min(p0 + k, n - 1)];
            }
#pragma unroll
            for (int k = 0; k < kRun; k++) t[k] = p0 + k < n ? (double)sv[k] * (double)vv[k] : 0.0;  // s + 0 = s
        }
        double sum = 0.0, a = 0.0;
#pragma unroll
        for (int k = 0; k < kRun; k++) sum += t[k], a += fabs(t[k]);
        double inc = sum;  // inclusive over the lanes
#pragma unroll
        for (int off = 1; off < 64; off *= 2) {
            const double o = __shfl_up(inc, off);
            if (lane >= off) inc += o;
        }
        double P = __shfl_up(inc, 1);
        if (lane == 0) P = 0.0;
        const double wa = wave_sum_d(a);
        if (lane == 63) L.tot[w] = inc, L.abs[w] = wa;
        __syncthreads();
        double at = 0.0, before = s;
#pragma unroll
        for (int u = 0; u < W; u++) {
            at += L.abs[u];
            if (u < w) before += L.tot[u];
        }
        P += before;
        const double wd = wave_sum_d(kRun * (fabs(P) + a));
        if (lane == 0) L.dist[w] = wd;
        __syncthreads();
        // the sequential sum's error up to anywhere in the pass, and the scan's
        double dist = 0.0;
#pragma unroll
        for (int u = 0; u < W; u++) dist += L.dist[u];
        dist = 0x1p-53 * (1.0625 * dist + 64.0 * (at + fabs(s)));
        double r0 = P, r1 = __longlong_as_double(__double_as_longlong(P) + 1), mn = P, mx = P;
        const double q = fabs(r1 - P);
#pragma unroll
        for (int k = 0; k < kRun; k++) {
            r0 += t[k], r1 += t[k];
            mn = fmin(mn, r0), mx = fmax(mx, r0);
        }
        const double room = 1.0625 * dist + 4.0 * q;
        const int binade = __double2hiint(P) >> 20, ex = binade & 0x7FF;
        const bool regular = __double2hiint(mn - room) >> 20 == binade && __double2hiint(mx + room) >> 20 == binade &&
                             ex > 0 && ex < 0x7FF && r0 == r0;
        // by the parity of the incoming sum: the change and the parity after
        const bool odd = __double2loint(P) & 1;
        const double c0 = r0 - P, c1 = r1 - __longlong_as_double(__double_as_longlong(P) + 1);
        double d0 = odd ? c1 : c0, d1 = odd ? c0 : c1;
        const int p0 = __double2loint(r0) & 1, p1 = __double2loint(r1) & 1;
        int o = odd ? p1 | p0 << 1 : p0 | p1 << 1;  // bit j: parity after an incoming parity j
        // chains of consecutive regular runs of one binade compose (inclusive scan with the
        // chain's first lane as a barrier); lane l then holds its chain's change up to l
        const int key = regular ? binade : -1 - lane;  // an irregular run is a chain of its own
        const int up = __shfl_up(key, 1);
        bool head = lane == 0 || up != key;
        const unsigned long long heads = __ballot(head), regs = __ballot(regular);
#pragma unroll
        for (int off = 1; off < 64; off *= 2) {
            const double n0 = __shfl_up(d0, off), n1 = __shfl_up(d1, off);
            const int no = __shfl_up(o, off);
            const bool nh = __shfl_up((int)head, off);
            if (!head && lane >= off) {
                const double e0 = n0 + (no & 1 ? d1 : d0), e1 = n1 + (no & 2 ? d1 : d0);
                o = ((no & 1 ? o >> 1 : o) & 1) | ((no & 2 ? o >> 1 : o) & 1) << 1;
                d0 = e0, d1 = e1;
                head = nh;
            }
        }
        for (int u = 0; u < W; u++) {
            if (w == u) {
                unsigned long long ends = heads >> 1 | 1ull << 63;  // last lanes of the chains
                asm volatile(".p2align 6");  // the loop below from the start of a cache line
                while (ends) {
                    const int l = __ffsll(ends) - 1;
                    ends &= ends - 1;
                    if ((regs >> l) & 1) {
                        const bool odd_s = __builtin_amdgcn_readfirstlane(__double2loint(s)) & 1;
                        const double e0 = lane_value(d0, l), e1 = lane_value(d1, l);  // both: a select, no branch
                        s += odd_s ? e1 : e0;
                    } else {
                        double x = s;
#pragma unroll
                        for (int k = 0; k < kRun; k++) x += t[k];
                        s = lane_value(x, l);
                    }
                }
                if (lane == 0) L.token = s;
            }
            __syncthreads();
            s = L.token;
            if (base + (u + 1) * 64 * kRun >= n) break;  // no positions in the waves after this one
            __syncthreads();
        }
        __syncthreads();  // L is written again
    }
    return s;
}
// The same by the lane alone, its adds in order, where many outputs need it or
// the positions are few. Up to 1024 positions a workgroup takes 10 to 11 us an
// output, one after the other; the lanes 45 ns a position, all at once: 1 and 8
// outputs over 64 positions 11 and 80 us against 2 and 2, over 256 11 and 86
// against 10 and 10, one over 1024 10 against 43; 224 with 16 kv heads of 512, the
// rows not in cache, 10 against 13, hence 160. Few positions need it more
// often: a sum of a few values under weights of a few bits (1/2, 1/4) may end on
// a midpoint.
constexpr int kReplayMax = 8, kLaneReplay = 160;
__device__ double lane_replay(const float *__restrict__ sr, const float *__restrict__ vl, size_t kv_len, int n) {
    constexpr int RB = 16;
    double q = 0.0;
    for (int p0 = 0; p0 < n; p0 += RB) {
        float vb[RB], sb[RB];
#pragma unroll
        for (int u = 0; u < RB; u++) {
            const int p = min(p0 + u, n - 1);
            vb[u] = vl[(size_t)p * kv_len];
            sb[u] = sr[p];
        }
#pragma unroll
        for (int u = 0; u < RB; u++)
            if (p0 + u < n) q += (double)sb[u] * (double)vb[u];
        if (q != q) break;  // it stays one
    }
    return q;
}

// *(p + off bytes) for a pointer that is the same in every lane: the scalar
// register pair as the load's base and the lane's 32-bit offset, no 64-bit
// address arithmetic on the vector unit (the empty asm keeps the compiler from
// adding the lane's part to the base ahead of the loop).
using gptr = const __attribute__((address_space(1))) char *;
template <class V>
__device__ __forceinline__ V load_at(gptr &p, uint32_t off) {
    asm volatile("" : "+s"(p));
    return *(const __attribute__((address_space(1))) V *)(p + off);
}

struct PvStrides {
    size_t soft, out, gz, gated;
};

// Few queries: a workgroup of 16 waves per (16 columns, kv head, query), the
// waves each a contiguous segment of the positions, v_mfma_f64_4x4x4_4b. Lane
// l takes row l >> 2 of a 16-block: V's columns 4 (l & 3) .. + 3 (one 16-byte
// load) and the weight of head l & 3 (one dword). Instruction r = 0..3
// multiplies column 4 j + r of each row: block b = (l >> 2) & 3 of it sums the
// rows 4 k + b, so the four accumulators are independent and their blocks are
// added at the end; result lane l: head l >> 4, column 4 (l & 3) + r. A prefix
// is bounded by the sum over b of the blocks' |S|, A by one instruction per
// column and 64 positions: the largest of four weights times their sum of |V|.
// 16 columns and not 64 a workgroup: 64 workgroups at the 9B shape instead of
// 16, with nothing to exchange between them (a caller gives no workspace).
// 24001 positions of the 9B shape: 56 us without replays; 1738 on the vector
// units with 64 columns a workgroup. The 56 are spent on the 64 CUs that have a
// workgroup: there the matrix cores are busy 20% of the time and the vector
// units 23% (one after the other), and a wave waits for its loads 36% of its.
// Replays follow the values: 108 to 212 us over 14 inputs, 138 in the median;
// scores, softmax and values together 147 to 251, 182 in the mean. Lanes holding
// a column each (five loads, four times the weights' bytes, eight conversions and
// one chain of dependent instructions per 16 positions) took 74 without replays.
constexpr int kPvWaves = 16, kPvUnroll = 4;  // 16-blocks whose loads a wave keeps in flight
template <int G>
__global__ __launch_bounds__(64 * kPvWaves) void attn_pv_kernel(float *__restrict__ out, const float *__restrict__ soft,
                                                                const float *__restrict__ vc, int n_ctx, int n_head_kv,
                                                                int hd, const float *__restrict__ gz, int gzs,
                                                                float *__restrict__ gated, PvStrides zs) {
    constexpr int GB = (G + 3) / 4;
    __shared__ double part[kPvWaves][GB][3][64];
    __shared__ SeqLds seq;
    __shared__ int todo[kReplayMax], ntodo;
    if (threadIdx.x == 0) ntodo = 0;
    // pairs of column blocks (the halves of 128-byte lines) dealt to the XCDs in turn: an XCD's
    // blocks then lie in different parts of a cache row, that is in more channels of its L2
    // (24001 positions: 56 us without replays, 59 with contiguous ranges)
    const int ncol = hd / 16, total = ncol * n_head_kv;
    const int slot = (int)(blockIdx.x >> 3), wk = 2 * (8 * (slot >> 1) + (int)(blockIdx.x & 7)) + (slot & 1);
    if (wk >= total) return;  // the whole workgroup
    const int kv = __builtin_amdgcn_readfirstlane(wk / ncol), col0 = 16 * __builtin_amdgcn_readfirstlane(wk % ncol);
    n_ctx += (int)blockIdx.y;
    soft += blockIdx.y * zs.soft;
    out += blockIdx.y * zs.out;
    if (gated) {
        gz += blockIdx.y * zs.gz;
        gated += blockIdx.y * zs.gated;
    }
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), row = lane >> 2;
    const size_t kv_len = (size_t)n_head_kv * hd;
    // uniform bases and each lane's byte offset from them (a group's rows: at most 2^29 bytes)
    const float *vbase = vc + (size_t)kv * hd + col0, *sbase = soft + (size_t)kv * G * n_ctx;
    const uint32_t voff = 4 * (uint32_t)(row * (int)kv_len + 4 * (lane & 3));
    uint32_t soff[GB];
#pragma unroll
    for (int b = 0; b < GB; b++) soff[b] = 4 * (uint32_t)(min(4 * b + (lane & 3), G - 1) * n_ctx + row);
    const int nblk = (n_ctx + 15) / 16, per = (nblk + kPvWaves - 1) / kPvWaves;
    const int b_lo = min(w * per, nblk), b_hi = min(b_lo + per, nblk);
    const int b_full = min(b_hi, n_ctx / 16);  // blocks [b_lo, b_full) hold 16 positions
    double S[GB][4], PS[GB][4], A[GB][4];
    float smax[GB], vabs[4];
#pragma unroll
    for (int r = 0; r < 4; r++) {
        vabs[r] = 0.0f;
#pragma unroll
        for (int b = 0; b < GB; b++) S[b][r] = PS[b][r] = A[b][r] = 0.0, smax[b] = 0.0f;
    }
    auto block = [&](const float *sv, const f4 vv) {  // one 16-block
        double vd[4];
#pragma unroll
        for (int r = 0; r < 4; r++) vd[r] = (double)vv[r], vabs[r] += fabsf(vv[r]);
#pragma unroll
        for (int b = 0; b < GB; b++) {
            const double sd = (double)sv[b];
            smax[b] = fmaxf(smax[b], sv[b]);
#pragma unroll
            for (int r = 0; r < 4; r++) {
                PS[b][r] += fabs(S[b][r]);
                S[b][r] = __builtin_amdgcn_mfma_f64_4x4x4f64(sd, vd[r], S[b][r], 0, 0, 0);
            }
        }
    };
    auto flush = [&] {  // the blocks since the last flush into A
#pragma unroll
        for (int r = 0; r < 4; r++) {
#pragma unroll
            for (int b = 0; b < GB; b++)
                A[b][r] = __builtin_amdgcn_mfma_f64_4x4x4f64((double)smax[b], (double)vabs[r], A[b][r], 0, 0, 0);
            vabs[r] = 0.0f;
        }
#pragma unroll
        for (int b = 0; b < GB; b++) smax[b] = 0.0f;
    };
    float sx[kPvUnroll][GB];
    f4 vx[kPvUnroll];
    const size_t vblk = 64 * kv_len;  // bytes of a block's rows
    gptr vp = (gptr)(vbase + (size_t)16 * b_lo * kv_len), sp = (gptr)(sbase + 16 * b_lo);
    auto load = [&](int k) {  // the block at vp / sp into slot k; the pointers to the next block
        vx[k] = load_at<f4u>(vp, voff);
        vp += vblk;
#pragma unroll
        for (int b = 0; b < GB; b++) sx[k][b] = load_at<float>(sp, soff[b]);
        sp += 64;
    };
    int blk = b_lo;
    const int groups = max(b_full - b_lo, 0) / kPvUnroll;
    if (groups) {
#pragma unroll
        for (int k = 0; k < kPvUnroll; k++) {
            load(k);
            __builtin_amdgcn_sched_barrier(0);  // in this order: the loop waits by counting
        }
        for (int j = 0; j < groups; j++) {
            if (j + 1 == groups) vp -= kPvUnroll * vblk, sp -= 64 * kPvUnroll;  // the last group again
#pragma unroll
            for (int k = 0; k < kPvUnroll; k++) {
                block(sx[k], vx[k]);
                __builtin_amdgcn_sched_barrier(0);  // into the same registers: no copies to wait for
                load(k);
                __builtin_amdgcn_sched_barrier(0);
            }
            flush();
        }
        blk += groups * kPvUnroll;
    }
#pragma unroll
    for (int k = 0; k < kPvUnroll - 1; k++)
        if (blk + k < b_full) load(k);
#pragma unroll
    for (int k = 0; k < kPvUnroll - 1; k++)
        if (blk + k < b_full) block(sx[k], vx[k]);
    if (b_full < b_hi && b_lo < b_hi) {  // the ragged last block: absent positions as zeros
        const int p = 16 * b_full + row;
        const bool in = p < n_ctx;
        const int pc = min(p, n_ctx - 1);
        f4 v = *(const f4u *)(vbase + (size_t)pc * kv_len + 4 * (lane & 3));
        float sv[GB];
#pragma unroll
        for (int b = 0; b < GB; b++) {
            const float t = sbase[(size_t)min(4 * b + (lane & 3), G - 1) * n_ctx + pc];
            sv[b] = in ? t : 0.0f;
        }
        if (!in) v = f4{0.f, 0.f, 0.f, 0.f};
        block(sv, v);
    }
    flush();
    // the four blocks' sums, then lane l holds column 4 (l & 3) + (l >> 2 & 3) of head l >> 4
    const int c4 = (lane >> 2) & 3;
    auto blocks = [&](const double (&t)[4]) {
        double o = 0.0;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            double x = t[r] + dpp_d<0x124>(t[r]);  // row_ror:4
            x += dpp_d<0x128>(x);                  // row_ror:8
            o = r == c4 ? x : o;
        }
        return o;
    };
#pragma unroll
    for (int b = 0; b < GB; b++) {
        part[w][b][0][lane] = blocks(S[b]);
        part[w][b][1][lane] = blocks(PS[b]);
        part[w][b][2][lane] = blocks(A[b]);
    }
    __syncthreads();
    // waves 0 .. GB - 1 finish, wave b the heads 4 b ..
    const int g = 4 * w + (lane >> 4), i = col0 + 4 * (lane & 3) + c4;
    const bool fin = w < GB && g < G;
    float r = 0.0f;
    bool need = false;
    if (fin) {
        PvErr t;
#pragma unroll
        for (int u = 0; u < kPvWaves; u++)
            t.segment(part[u][w][0][lane], part[u][w][1][lane], part[u][w][2][lane], 16 * per, 16.0 + 12.0);
        if (!decided(t.B, t.bound(), r)) {
            need = t.B - t.B == 0.0;
            if (!need) r = (float)t.B;  // the sum's terms are the reference's: so is a NaN or an infinity of them
        }
    }
    if (need) {
        const int k = atomicAdd(&ntodo, 1);
        if (k < kReplayMax) todo[k] = threadIdx.x;
    }
    __syncthreads();
    const int nt = ntodo;
    if (nt > kReplayMax || n_ctx <= kLaneReplay * nt) {
        if (need) r = (float)lane_replay(soft + (size_t)(kv * G + g) * n_ctx, vc + (size_t)kv * hd + i, kv_len, n_ctx);
    } else {
        for (int k = 0; k < nt; k++) {
            const int id = todo[k];
            const double s = wg_replay<64 * kPvWaves>(seq, soft + (size_t)(kv * G + (id >> 4)) * n_ctx,
                                                      vbase + 4 * (id & 3) + ((id >> 2) & 3), kv_len, n_ctx);
            if ((int)threadIdx.x == id) r = (float)s;
        }
    }
    if (!fin) return;
    out[(size_t)(kv * G + g) * hd + i] = r;
    // the gated output (qwen35_forward.rs:677-684, as mul_act_kernel)
    if (gated) gated[(size_t)(kv * G + g) * hd + i] = __fmul_rn(r, sigmoid1(gz[(size_t)(kv * G + g) * gzs + i]));
}

// Four values to bf16, to nearest (relative error 2^-9; v_cvt_pk_bf16_f32).
__device__ __forceinline__ s4 bf16_4(float a, float b, float c, float d) {
    typedef float v2 __attribute__((ext_vector_type(2)));
    typedef __bf16 b2 __attribute__((ext_vector_type(2)));
    const b2 lo = __builtin_convertvector((v2{a, b}), b2), hi = __builtin_convertvector((v2{c, d}), b2);
    const uint2 o = make_uint2(__builtin_bit_cast(uint32_t, lo), __builtin_bit_cast(uint32_t, hi));
    return __builtin_bit_cast(s4, o);
}

// A prefill chunk: a workgroup takes 64 (query, head) pairs of a kv head and
// 64 columns; of its eight waves, wave (k, a, c) holds pairs 32 a .. and
// columns 32 c .. as 2 x 2 tiles of v_mfma_f64_16x16x4 (64 cycles) over half
// k of the positions. Lane l: soft of pair l & 15, V of column l & 15, both
// at positions 4 (l >> 4) + u of a 16-block, straight from memory (each
// 16-block: 16 matrix instructions per wave against 2 + 8 loads, the next
// block's in flight). A is bounded from above with one bf16 instruction per
// tile and block, the operands rounded to nearest: the sum is low by at most
// 2^-8 of itself, and the f32 additions by 2^-12, which the 2^-5 in
// PvErr::bound covers. 255 queries x 16 heads over 3842 positions take 195 to
// 206 us, the matrix cores busy 52% of it and the vector units 23% (their f64
// instructions do not overlap); a chunk over 4096 takes 223 to 237, 48% and
// 21%: the workgroups that replay an output end last.
// Workgroups of one pair tile (its four column blocks at hd 256) are adjacent
// on one XCD, so the weights are read from its L2.
constexpr int kPvTileWaves = 8;
struct PvTile {
    d4 S;  // pairs (lane >> 4) + 4 r, column lane & 15
    double PS[4], A[4];
};
__global__ __launch_bounds__(64 * kPvTileWaves, 2) void attn_pv_tile_kernel(
    float *__restrict__ out, const float *__restrict__ soft, const float *__restrict__ vc, int n_ctx, int n_head_kv,
    int hd, int group, int rows, const float *__restrict__ gz, int gzs, float *__restrict__ gated, PvStrides zs) {
    // S and PS + A of the tiles the partner finishes, one column tile's half at a time
    __shared__ double xch[2][kPvTileWaves][4][64];
    __shared__ SeqLds seq;
    __shared__ int todo[kReplayMax], ntodo;
    if (threadIdx.x == 0) ntodo = 0;
    const int pairs = rows * group, npt = (pairs + 63) / 64, ncol = hd / 64;
    // XCD x = blockIdx.x & 7 takes a contiguous range of (kv, pair tile, column block)
    const int total = npt * ncol * n_head_kv, perx = (total + 7) / 8;
    const int slot = (int)(blockIdx.x >> 3), wk = (int)(blockIdx.x & 7) * perx + slot;
    if (slot >= perx || wk >= total) return;
    // (readfirstlane: divisions run on the vector unit)
    const int cb = __builtin_amdgcn_readfirstlane(wk % ncol), kv = __builtin_amdgcn_readfirstlane(wk / (ncol * npt)),
              pt = __builtin_amdgcn_readfirstlane((wk / ncol) % npt);
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int kh = wv >> 2, pa = (wv >> 1) & 1, ca = wv & 1, x = lane & 15, kk = lane >> 4;
    const int pr0 = 64 * pt + 32 * pa, col0 = 64 * cb + 32 * ca;
    const size_t kv_len = (size_t)n_head_kv * hd;
    // uniform bases and each lane's byte offset from them (a chunk's weights: at most 2^26 bytes)
    const int z_lo = __builtin_amdgcn_readfirstlane(64 * pt / group),
              z_hi = __builtin_amdgcn_readfirstlane((min(64 * pt + 64, pairs) - 1) / group);
    const float *vbase = vc + (size_t)kv * hd + col0, *sbase = soft + (size_t)z_lo * zs.soft;
    const uint32_t voff = 4 * (uint32_t)(4 * kk * (int)kv_len + x);
    const float *vb = vbase + x;
    const float *sr[2];
    uint32_t soff[2];
    int nz[2];
#pragma unroll
    for (int a = 0; a < 2; a++) {
        const int pr = min(pr0 + 16 * a + x, pairs - 1), zz = pr / group;
        nz[a] = n_ctx + zz;
        const size_t row = (size_t)(zz - z_lo) * zs.soft + (size_t)(kv * group + (pr - zz * group)) * nz[a];
        sr[a] = sbase + row;
        soff[a] = 4 * (uint32_t)(row + 4 * kk);
    }
    // the workgroup's positions: blocks every pair sees in full, then masked ones
    const int nblk = (n_ctx + z_hi + 15) / 16, nfull = (n_ctx + z_lo) / 16;
    const int half = (nblk + 1) / 2, b_lo = kh ? half : 0, b_hi = kh ? nblk : half, b_full = min(b_hi, nfull);
    PvTile T[2][2];
    f4 Af[2][2];
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
        for (int c = 0; c < 2; c++) {
#pragma unroll
            for (int r = 0; r < 4; r++) T[a][c].S[r] = T[a][c].PS[r] = T[a][c].A[r] = 0.0;
            Af[a][c] = f4{0.f, 0.f, 0.f, 0.f};
        }
    auto flush = [&] {  // the f32 sums of A into f64 (at most 64 blocks: within 2^-12)
#pragma unroll
        for (int a = 0; a < 2; a++)
#pragma unroll
            for (int c = 0; c < 2; c++) {
#pragma unroll
                for (int r = 0; r < 4; r++) T[a][c].A[r] += (double)Af[a][c][r];
                Af[a][c] = f4{0.f, 0.f, 0.f, 0.f};
            }
    };
    float sv[2][4], vv[2][4];
    uint32_t vany[2] = {0, 0};  // or of the bits of the lane's V values: is the column all zeros
    const uint32_t vrow = 4 * (uint32_t)kv_len;  // bytes
    // a block's rows as buffer loads (any 32-bit offset): the block in the base, the row in the scalar offset, no
    // address arithmetic on the vector unit (its cycles and the f64 matrix instructions' add up)
    auto load = [&](int blk) {
        const auto vr = __builtin_amdgcn_make_buffer_rsrc((void *)(vbase + (size_t)16 * blk * kv_len), 0, -1, 0x00020000);
        const auto sb = __builtin_amdgcn_make_buffer_rsrc((void *)(sbase + 16 * blk), 0, -1, 0x00020000);
#pragma unroll
        for (int a = 0; a < 2; a++) {
            const uint4 t = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(sb, soff[a], 0, 0));
            sv[a][0] = __uint_as_float(t.x), sv[a][1] = __uint_as_float(t.y);
            sv[a][2] = __uint_as_float(t.z), sv[a][3] = __uint_as_float(t.w);
        }
#pragma unroll
        for (int u = 0; u < 4; u++)
#pragma unroll
            for (int c = 0; c < 2; c++)
                vv[c][u] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(vr, voff + 64 * c, u * vrow, 0));
    };
    auto load_masked = [&](int blk) {  // positions a pair does not see as zero weights
        const int p = 16 * blk + 4 * kk;
#pragma unroll
        for (int u = 0; u < 4; u++) {
#pragma unroll
            for (int a = 0; a < 2; a++) {
                const float t = sr[a][min(p + u, nz[a] - 1)];
                sv[a][u] = p + u < nz[a] ? t : 0.0f;
            }
            const int pc = min(p + u, n_ctx + z_hi - 1);
#pragma unroll
            for (int c = 0; c < 2; c++) {
                const float t = vb[(size_t)pc * kv_len + 16 * c];
                vv[c][u] = p + u == pc ? t : 0.0f;
            }
        }
    };
    auto prefixes = [&] {  // every 32 positions
#pragma unroll
        for (int a = 0; a < 2; a++)
#pragma unroll
            for (int c = 0; c < 2; c++)
#pragma unroll
                for (int r = 0; r < 4; r++) T[a][c].PS[r] += fabs(T[a][c].S[r]);
        __builtin_amdgcn_sched_barrier(0);  // before S changes in place
    };
    auto block = [&](int next) {  // sv, vv; block next (< b_full) is loaded over them
        s4 sb[2], vbf[2];
        double sd[2][4], vd[2][4];
#pragma unroll
        for (int a = 0; a < 2; a++) {
            // weights at least the smallest normal value: none lost beside a large |V|
            float m[4];
#pragma unroll
            for (int u = 0; u < 4; u++) {
                m[u] = __uint_as_float(max(__float_as_uint(sv[a][u]), 0x00800000u));  // never negative
                sd[a][u] = (double)sv[a][u], vd[a][u] = (double)vv[a][u];
            }
            sb[a] = bf16_4(m[0], m[1], m[2], m[3]);
            vbf[a] = bf16_4(fabsf(vv[a][0]), fabsf(vv[a][1]), fabsf(vv[a][2]), fabsf(vv[a][3]));
            vany[a] = vany[a] | __float_as_uint(vv[a][0]) | __float_as_uint(vv[a][1]);
            vany[a] = vany[a] | __float_as_uint(vv[a][2]) | __float_as_uint(vv[a][3]);
        }
        __builtin_amdgcn_sched_barrier(0);  // the vector work, the loads, then the matrix instructions together
        if (next < b_full) load(next);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int a = 0; a < 2; a++)
#pragma unroll
            for (int c = 0; c < 2; c++)
                Af[a][c] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(sb[a], vbf[c], Af[a][c], 0, 0, 0);
#pragma unroll
        for (int u = 0; u < 4; u++)
#pragma unroll
            for (int a = 0; a < 2; a++)
#pragma unroll
                for (int c = 0; c < 2; c++)
                    T[a][c].S = __builtin_amdgcn_mfma_f64_16x16x4f64(sd[a][u], vd[c][u], T[a][c].S, 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
    };
    int blk = b_lo;
    if (blk < b_full) load(blk);
    for (; blk < b_full; blk++) {
        if (((blk - b_lo) & 1) == 0) prefixes();
        block(blk + 1);
        if ((blk & 63) == 63) flush();
    }
    for (; blk < b_hi; blk++) {
        load_masked(blk);
        if (((blk - b_lo) & 1) == 0) prefixes();
        block(b_full);
        if ((blk & 63) == 63) flush();
    }
    flush();
    // bf16 products lost below the f32 range; none in a column of zeros, whose bound stays zero
    // (a bound above a sum of zero is never decided: every output of the column would be replayed)
    const double tiny = (double)nblk * 0x1p-121;
#pragma unroll
    for (int c = 0; c < 2; c++) {
        vany[c] |= __shfl_xor(vany[c], 16);
        vany[c] |= __shfl_xor(vany[c], 32);
        if (vany[c] << 1)
#pragma unroll
            for (int a = 0; a < 2; a++)
#pragma unroll
                for (int r = 0; r < 4; r++) T[a][c].A[r] += tiny;
    }
    // wave (k, a, c) finishes its column tile k, its partner (k ^ 1, a, c) the other
    float res[2][4];
    unsigned need = 0;
#pragma unroll
    for (int a = 0; a < 2; a++) {
        const PvTile &give = kh ? T[a][0] : T[a][1], &m = kh ? T[a][1] : T[a][0];
        if (a) __syncthreads();
#pragma unroll
        for (int r = 0; r < 4; r++) xch[0][wv][r][lane] = give.S[r], xch[1][wv][r][lane] = give.PS[r] + give.A[r];
        __syncthreads();
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const double oS = xch[0][wv ^ 4][r][lane], oX = xch[1][wv ^ 4][r][lane], mX = m.PS[r] + m.A[r];
            PvErr t;
            t.segment(kh ? oS : m.S[r], kh ? oX : mX, 0.0, 16 * half, 32.0 + 64.0);
            t.segment(kh ? m.S[r] : oS, kh ? mX : oX, 0.0, 16 * half, 32.0 + 64.0);
            const int pr = pr0 + 16 * a + kk + 4 * r;
            // a NaN too: positions this pair may not see took part, as zero weights, and 0 x infinity is one;
            // an infinite sum is of the pair's own terms
            if (!decided(t.B, t.bound(), res[a][r]) && pr < pairs) {
                if (fabs(t.B) == INFINITY) {
                    res[a][r] = (float)t.B;
                } else {
                    need |= 1u << (4 * a + r);
                    const int k = atomicAdd(&ntodo, 1);
                    if (k < kReplayMax) todo[k] = (int)threadIdx.x * 8 + 4 * a + r;
                }
            }
        }
    }
    __syncthreads();
    const int i = col0 + 16 * kh + x, nt = ntodo;
    // a lane takes its outputs one after the other: their number does not count here
    const bool lanes = nt > kReplayMax || n_ctx + z_hi <= kLaneReplay;
    auto srow = [&](int pr) {
        const int zz = pr / group;
        return soft + (size_t)zz * zs.soft + (size_t)(kv * group + (pr - zz * group)) * (n_ctx + zz);
    };
    if (!lanes) {
        for (int k = 0; k < nt; k++) {
            const int id = todo[k] >> 3, ar = todo[k] & 7, il = id & 63, iw = id >> 6;
            const int pr = 64 * pt + 32 * ((iw >> 1) & 1) + 16 * (ar >> 2) + (il >> 4) + 4 * (ar & 3);
            const int col = 64 * cb + 32 * (iw & 1) + 16 * (iw >> 2) + (il & 15);
            const double s = wg_replay<64 * kPvTileWaves>(seq, srow(pr), vc + (size_t)kv * hd + col, kv_len,
                                                          n_ctx + pr / group);
#pragma unroll
            for (int j = 0; j < 8; j++)
                if ((int)threadIdx.x == id && j == ar) res[j >> 2][j & 3] = (float)s;
        }
    }
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int pr = pr0 + 16 * a + kk + 4 * r;
            if (pr >= pairs) continue;
            const int zz = pr / group;
            float v = res[a][r];
            if (lanes && ((need >> (4 * a + r)) & 1))
                v = (float)lane_replay(srow(pr), vc + (size_t)kv * hd + i, kv_len, n_ctx + zz);
            const size_t o = (size_t)(kv * group + (pr - zz * group));
            out[(size_t)zz * zs.out + o * hd + i] = v;
            if (gated)
                gated[(size_t)zz * zs.gated + o * hd + i] = __fmul_rn(v, sigmoid1(gz[(size_t)zz * zs.gz + o * gzs + i]));
        }
}

}  // namespace

int softmax_max_len() { return kSmChunk * kSmMaxChunks; }

hipError_t launch_softmax(float *out, const float *x, int n, int rows, float scale, hipStream_t s) {
    if (rows == 0 || n == 0) return hipSuccess;
    if (n > softmax_max_len()) return hipErrorInvalidValue;
    return softmax_rows(out, x, n, rows, scale, 0, 1, 0, s);
}

bool attn_shape_ok(int hd, int group) {
    return (hd == 64 || hd == 128 || hd == 256 || hd == 512) && group >= 1 && group <= kAttnMaxGroup;
}

// Which kernels take a few queries, from a sweep of 2 .. 128 of them over 16,
// 500 and 3500 positions of the 9B shape (layer times).
// Scores: a query of its own reads K once more, a pair tile has a fixed cost
// (8 queries: 104 against 108 us at 16 positions, 110 / 113 at 500, 139 / 125
// at 3500).
inline bool scores_per_query(int rows, int n) { return rows == 1 || (size_t)rows * n <= 8192; }
// Values: the tile kernel's time hardly depends on how many of its 64-pair
// tiles there are until they fill the chip (about 5 us + 42 ns a position);
// the other's workgroups (16 columns of a kv head and query) take about
// 1.2 us + 2.5 ns a position, 256 of them at a time. Times cross at 18 queries
// at 16 positions, 40 at 500, 64 at 3500.
inline bool values_per_query(int rows, int n, int n_head_kv, int hd) {
    const double groups = (double)rows * n_head_kv * (hd / 16);
    return rows == 1 || groups / 256.0 * (480.0 + n) < 2000.0 + 17.0 * n;
}

hipError_t launch_attn_rows(float *out, size_t out_st, float *soft, size_t soft_st, const float *q, size_t q_st,
                            const float *kc, const float *vc, int n_ctx, int rows, int n_head_kv, int hd, int group,
                            float kq_scale, hipStream_t s, const float *gz, int gzs, size_t gz_st, float *gated,
                            size_t gated_st) {
    if (n_ctx <= 0 || n_head_kv <= 0 || rows <= 0) return hipSuccess;
    const int n_last = n_ctx + rows - 1;
    if (!attn_shape_ok(hd, group) || n_last > softmax_max_len() || rows > 65535) return hipErrorInvalidValue;
    if (hd <= 256 && !scores_per_query(rows, n_last)) {
        // pair tiles split until about eight workgroups per CU, four tiles each at least
        const int base = (n_last + 63) / 64 * n_head_kv, ntile = (rows * group + 15) / 16;
        const int split = std::max(1, std::min((2048 + base - 1) / base, ntile / 4));
        const dim3 g((n_last + 63) / 64, n_head_kv, split);
        const size_t lds = (size_t)2 * (hd / 16) * 256 * 8;
        hipError_t e = hipSuccess;
#define UQ_ST(HD)                                                                                                      \
    if ((e = allow_lds((const void *)attn_scores_tile_kernel<HD>, lds)) != hipSuccess) return e;                       \
    hipLaunchKernelGGL(attn_scores_tile_kernel<HD>, g, dim3(256), lds, s, soft, q, kc, n_ctx, n_head_kv, group, q_st,  \
                       soft_st, rows)
        if (hd == 64) {
            UQ_ST(64);
        } else if (hd == 128) {
            UQ_ST(128);
        } else {
            UQ_ST(256);
        }
#undef UQ_ST
    } else {
        // about eight waves per CU, an even number of tiles for each
        const int ntile = (n_last + 15) / 16, per = std::max(1, ntile * n_head_kv * rows / 2048);
        const dim3 g(n_head_kv, (ntile + per - 1) / per, rows);  // a tile's kv heads, whole cache rows, side by side
#define UQ_SC(HD)                                                                                                     \
    do {                                                                                                              \
        if (group <= 4)                                                                                               \
            hipLaunchKernelGGL((attn_scores_kernel<HD, 1>), g, dim3(64), 0, s, soft, q, kc, n_ctx, n_head_kv, group,   \
                               q_st, soft_st);                                                                        \
        else                                                                                                          \
            hipLaunchKernelGGL((attn_scores_kernel<HD, 2>), g, dim3(64), 0, s, soft, q, kc, n_ctx, n_head_kv, group,   \
                               q_st, soft_st);                                                                        \
    } while (0)
        switch (hd) {
            case 64: UQ_SC(64); break;
            case 128: UQ_SC(128); break;
            case 256: UQ_SC(256); break;
            default: UQ_SC(512); break;
        }
#undef UQ_SC
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    if ((e = softmax_rows(soft, soft, n_ctx, n_head_kv * group, kq_scale, 1, rows, soft_st, s)) != hipSuccess) return e;
    const PvStrides pst{soft_st, out_st, gz_st, gated_st};
    if (!values_per_query(rows, n_last, n_head_kv, hd)) {
        const int total = (rows * group + 63) / 64 * (hd / 64) * n_head_kv;
        hipLaunchKernelGGL(attn_pv_tile_kernel, dim3((total + 7) / 8 * 8), dim3(64 * kPvTileWaves), 0, s, out, soft, vc,
                           n_ctx, n_head_kv, hd, group, rows, gz, gzs, gated, pst);
        return hipGetLastError();
    }
    const dim3 gp((hd / 16 * n_head_kv + 15) / 16 * 16, rows);
#define UQ_PV(G) hipLaunchKernelGGL(attn_pv_kernel<G>, gp, dim3(64 * kPvWaves), 0, s, out, soft, vc, n_ctx, n_head_kv, \
                                    hd, gz, gzs, gated, pst)
    switch (group) {
        case 1: UQ_PV(1); break;
        case 2: UQ_PV(2); break;
        case 3: UQ_PV(3); break;
        case 4: UQ_PV(4); break;
        case 5: UQ_PV(5); break;
        case 6: UQ_PV(6); break;
        case 7: UQ_PV(7); break;
        default: UQ_PV(8); break;
    }
#undef UQ_PV
    return hipGetLastError();
}

hipError_t launch_attn_decode(float *out, float *soft, const float *q, const float *kc, const float *vc, int n_ctx,
                              int n_head_kv, int hd, int group, float kq_scale, hipStream_t s, const float *gz,
                              int gzs, float *gated) {
    return launch_attn_rows(out, 0, soft, 0, q, 0, kc, vc, n_ctx, 1, n_head_kv, hd, group, kq_scale, s, gz, gzs, 0,
                            gated, 0);
}

}  // namespace uq
