// gt_backward.hip -- gradients of the all-pairs distance vector.
//
// gputools has no backward; these kernels differentiate the forward formulas
// of inst/cuda/distance.cu (euclidean :40-78, minkowski :453-493).  For the
// packed distance vector D and an upstream gradient G = dL/dD (packed, R
// 'dist' order):
//   dL/dx_ic = sum_{j != i} G_ij * dd_ij/dx_ic,
//   euclidean   dd_ij/dx_ic = (x_ic - x_jc) / d_ij
//   minkowski   dd_ij/dx_ic = sign(t) |t|^(p-1) / d_ij^(p-1),  t = x_ic - x_jc
// and a pair with d_ij == 0 contributes 0 (subgradient).
//
// Row-owner sweep: a workgroup owns 64 rows i and one block of up to 128
// features, and visits a share of the 64-row blocks j.  Per (i, j) tile it
// recomputes d_ij exactly (FP32 differences, two-level summation over LDS
// chunks of up to 32 features; D is never stored), forms
// w_ij = G_ij / d_ij^(p-1) in LDS, then accumulates dX_i over its features.
// The 64 x 64 block of packed G is loaded coalesced (lanes along the
// contiguous index of R's 'dist' order, which is i below the diagonal and j
// above it) and staged through LDS.
// When there are few row blocks, the j blocks are split over JS workgroups
// per row block, which write partial dX into a workspace; a second kernel
// adds the JS partials in a fixed order.  No atomics: deterministic.
//
// Euclidean gradients of up to 128 features run on the matrix cores instead
// (gradient_kernel below): the distances in the split-precision Gram form of
// gt_gram.hip, with near pairs recomputed from differences, and the
// accumulation sum_j w_ij x_j as a product of split operands.
//
// The same sweep computes the metric-MDS stress S = sum_{i<j} (d_ij - delta_ij)^2
// of an embedding Y and its gradient (G_ij = 2 (d_ij - delta_ij)); S is summed
// in FP64 from per-workgroup partials (the only FP64 on the device).
#include "gt_common.h"
#include "gt_internal.h"
#include "gt_mfma.h"

namespace gt {
namespace {

constexpr int BI = 64;          // owned rows per workgroup
constexpr int BJ = 64;          // rows per visited block
constexpr int BTH = 256;        // threads
constexpr int DKC = 32;         // features per distance chunk
constexpr int DLD = BI + 4;     // LDS row length of the k-major distance chunks
constexpr int KBMAX = 128;      // largest feature block per workgroup
constexpr int WLD = BI + 4;     // LDS row length of the G / weight tile (float4 rows)

enum { MODE_GRAD = 0, MODE_MDS = 1 };
enum { BW_EUCLID = 0, BW_MINK3 = 1, BW_MINKP = 2 };

struct BwArgs {
    const float *x;
    int64_t n, k, ldx;
    const float *g;        // MODE_GRAD: packed dL/dD; MODE_MDS: packed delta
    float *dx;
    int64_t lddx;
    float *dxp;            // JS > 1: JS partial dX slices, n x k each
    double *partials;      // MODE_MDS: one per (row block, j split) workgroup
    float p, pm1;          // p and p - 1
    // row blocks that gradient_kernel left (1 = left): only those run; null:
    // every block runs
    const uint8_t *left;
};

template <int OP>
__device__ __forceinline__ float dterm(float t)
{
    // contribution of one feature difference to the distance accumulator
    if (OP == BW_EUCLID) return t * t;
    const float a = fabsf(t);
    if (OP == BW_MINK3) return a * a * a;
    return 0.0f;  // BW_MINKP handled by the caller (needs p)
}

// KB: features per workgroup (4, 32 or 128, chosen from k on the host).
// blockIdx.z = js of JS = gridDim.z: this workgroup visits j blocks
// js, js + JS, ...; with JS > 1 it writes partial dX to args.dxp.
template <int OP, int MODE, int KB>
__global__ __launch_bounds__(BTH) void backward_kernel(BwArgs args)
{
    constexpr int XLD = KB + 4;   // LDS row length of the x_J feature block (float4 rows)
    constexpr int DK = KB < DKC ? KB : DKC;   // features per distance chunk
    __shared__ float xi_s[DK][DLD];
    __shared__ float xj_s[DK][DLD];
    __shared__ float w_s[BI][WLD];            // G, then the weights
    __shared__ float xb_s[BJ][XLD];
    __shared__ double red_s[BTH / 64];

    const int tid = threadIdx.x;
    const int64_t n = args.n, k = args.k, ldx = args.ldx;
    const int64_t i0 = (int64_t)blockIdx.x * BI;
    if (MODE == MODE_GRAD && args.left && args.left[blockIdx.x] == 0) return;
    const int64_t f0 = (int64_t)blockIdx.y * KB;
    const int64_t fcount = (k - f0) < KB ? (k - f0) : KB;

    // distance phase mapping: 4 x 4 pairs per thread
    const int ty = tid >> 4, tx = tid & 15;
    // accumulation phase mapping (a register-blocked W x_J product): rows
    // rg * RPT + r, features fg * FPT + m of the feature block
    constexpr int RPT = KB >= 32 ? 4 : 1;            // rows per thread
    constexpr int FPT = KB * BI / (BTH * RPT);       // features per thread: 8, 2, 1
    constexpr int FGROUPS = KB / FPT;
    const int rg = tid / FGROUPS, fg = tid % FGROUPS;
    float xi_r[RPT][FPT], acc[RPT][FPT], rowsum[RPT];
#pragma unroll
    for (int r = 0; r < RPT; ++r) {
        rowsum[r] = 0.0f;
        const int64_t gi = i0 + rg * RPT + r;
#pragma unroll
        for (int m = 0; m < FPT; ++m) {
            const int c = fg * FPT + m;
            // euclidean needs x_i only at the end (dX_i = x_i sum_j w_ij - sum_j w_ij x_j)
            xi_r[r][m] = (OP != BW_EUCLID && gi < n && c < fcount) ? args.x[gi * ldx + f0 + c] : 0.0f;
            acc[r][m] = 0.0f;
        }
    }
    double stress = 0.0;

    // the 64 x 64 block of G is element e = tid + 256 q; below the diagonal
    // (i > j) the packed index runs along i, above it along j
    const int js = blockIdx.z, JS = gridDim.z;
    // G of tile j0 into registers: loaded one tile ahead, so its latency
    // overlaps the previous tile's work
    float gq[(BI * BJ) / BTH];
    auto gfetch = [&](int64_t jt) {
        const bool up = jt > i0;
#pragma unroll
        for (int q = 0; q < (BI * BJ) / BTH; ++q) {
            const int e = tid + BTH * q;
            const int li = up ? (e >> 6) : (e & 63), lj = up ? (e & 63) : (e >> 6);
            const int64_t i = i0 + li, j = jt + lj;
            float g = 0.0f;
            if (i < n && j < n && i != j) {
                const int64_t hi = i > j ? i : j, lo = i > j ? j : i;
                g = args.g[packed_base(n, lo) + hi];
            }
            gq[q] = g;
        }
    };
    if ((int64_t)js * BJ < n) gfetch((int64_t)js * BJ);
    for (int64_t j0 = (int64_t)js * BJ; j0 < n; j0 += (int64_t)JS * BJ) {
        const bool upper = j0 > i0;   // every i < j in this tile
        // ---- d_ij for the 64 x 64 tile, exact FP32 differences ------------
        float dsum[4][4];
#pragma unroll
        for (int a = 0; a < 4; ++a)
#pragma unroll
            for (int b = 0; b < 4; ++b) dsum[a][b] = 0.0f;
        for (int64_t kb = 0; kb < k; kb += DK) {
            __syncthreads();
#pragma unroll
            for (int q = 0; q < (BI * DK) / BTH; ++q) {
                const int e = tid + BTH * q;
                const int row = e / DK, kc = e % DK;
                const int64_t kk = kb + kc;
                const int64_t ri = i0 + row, rj = j0 + row;
                // with one chunk (k <= DK) the owned rows' chunk is the same
                // for every tile: staged on the first only
                if (k > DK || j0 == (int64_t)js * BJ)
                    xi_s[kc][row] = (ri < n && kk < k) ? args.x[ri * ldx + kk] : 0.0f;
                xj_s[kc][row] = (rj < n && kk < k) ? args.x[rj * ldx + kk] : 0.0f;
            }
            __syncthreads();
            float part[4][4];
#pragma unroll
            for (int a = 0; a < 4; ++a)
#pragma unroll
                for (int b = 0; b < 4; ++b) part[a][b] = 0.0f;
#pragma unroll 4
            for (int kc = 0; kc < DK; ++kc) {
                const float4 vi = *reinterpret_cast<const float4 *>(&xi_s[kc][ty * 4]);
                const float4 vj = *reinterpret_cast<const float4 *>(&xj_s[kc][tx * 4]);
                const float ai[4] = {vi.x, vi.y, vi.z, vi.w};
                const float aj[4] = {vj.x, vj.y, vj.z, vj.w};
#pragma unroll
                for (int a = 0; a < 4; ++a)
#pragma unroll
                    for (int b = 0; b < 4; ++b) {
                        const float t = ai[a] - aj[b];
                        if (OP == BW_MINKP)
                            part[a][b] += exp2f(args.p * log2f(fabsf(t)));
                        else
                            part[a][b] += dterm<OP>(t);
                    }
            }
#pragma unroll
            for (int a = 0; a < 4; ++a)
#pragma unroll
                for (int b = 0; b < 4; ++b) dsum[a][b] += part[a][b];
        }
        // ---- G to LDS (the previous tile's weights were read before the
        // distance phase's barriers), then w_ij = G_ij / d_ij^(p-1) ---------
#pragma unroll
        for (int q = 0; q < (BI * BJ) / BTH; ++q) {
            const int e = tid + BTH * q;
            const int li = upper ? (e >> 6) : (e & 63), lj = upper ? (e & 63) : (e >> 6);
            w_s[li][lj] = gq[q];
        }
        if (j0 + (int64_t)JS * BJ < n) gfetch(j0 + (int64_t)JS * BJ);
        __syncthreads();
        float w_r[4][4];
#pragma unroll
        for (int a = 0; a < 4; ++a)
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                const int li = ty * 4 + a, lj = tx * 4 + b;
                const int64_t i = i0 + li, j = j0 + lj;
                float w = 0.0f;
                if (i < n && j < n && i != j) {
                    const float s = dsum[a][b];
                    const float d = (OP == BW_EUCLID) ? sqrtf(s)
                                    : (OP == BW_MINK3) ? cbrtf(s)
                                                       : powf(s, 1.0f / args.p);
                    const float gv = w_s[li][lj];
                    if (d > 0.0f) {
                        float gij;
                        if (MODE == MODE_MDS) {
                            const float r = d - gv;     // gv = delta_ij
                            stress += (double)r * (double)r;
                            gij = 2.0f * r;
                        } else {
                            gij = gv;
                        }
                        // d^(p-1): p = 2 -> d, p = 3 -> d^2
                        const float dp = (OP == BW_EUCLID) ? d
                                         : (OP == BW_MINK3) ? d * d
                                                            : powf(d, args.pm1);
                        w = gij / dp;
                    } else if (MODE == MODE_MDS) {
                        const float r = -gv;            // d == 0
                        stress += (double)r * (double)r;
                    }
                }
                w_r[a][b] = w;
            }
        // every G value is read: store the weights transposed, w_s[j][i]
        __syncthreads();
#pragma unroll
        for (int a = 0; a < 4; ++a)
#pragma unroll
            for (int b = 0; b < 4; ++b) w_s[tx * 4 + b][ty * 4 + a] = w_r[a][b];
        // ---- x_J feature block ----------------------------------------------
        for (int e = tid; e < BJ * KB; e += BTH) {
            const int row = e / KB, c = e % KB;
            const int64_t rj = j0 + row;
            xb_s[row][c] = (rj < n && c < fcount) ? args.x[rj * ldx + f0 + c] : 0.0f;
        }
        __syncthreads();
        // ---- dX_i += sum_j w_ij phi(x_i - x_j) ------------------------------
        const int jmax = (n - j0) < BJ ? (int)(n - j0) : BJ;
        for (int lj = 0; lj < jmax; ++lj) {
            float w[RPT], xj[FPT];
            if (RPT == 4) {
                const float4 v = *reinterpret_cast<const float4 *>(&w_s[lj][rg * 4]);
                w[0] = v.x;
                w[1] = v.y;
                w[2 % RPT] = v.z;
                w[3 % RPT] = v.w;
            } else {
                w[0] = w_s[lj][rg];
            }
            if (FPT % 4 == 0) {
#pragma unroll
                for (int m = 0; m < FPT; m += 4) {
                    const float4 v = *reinterpret_cast<const float4 *>(&xb_s[lj][fg * FPT + m]);
                    xj[m] = v.x;
                    xj[(m + 1) % FPT] = v.y;
                    xj[(m + 2) % FPT] = v.z;
                    xj[(m + 3) % FPT] = v.w;
                }
            } else if (FPT == 2) {
                const float2 v = *reinterpret_cast<const float2 *>(&xb_s[lj][fg * 2]);
                xj[0] = v.x;
                xj[1 % FPT] = v.y;
            } else {
                xj[0] = xb_s[lj][fg];
            }
#pragma unroll
            for (int r = 0; r < RPT; ++r) {
                if (OP == BW_EUCLID) {
                    rowsum[r] += w[r];
#pragma unroll
                    for (int m = 0; m < FPT; ++m) acc[r][m] = fmaf(-w[r], xj[m], acc[r][m]);
                } else {
#pragma unroll
                    for (int m = 0; m < FPT; ++m) {
                        const float t = xi_r[r][m] - xj[m];
                        const float a = fabsf(t);
                        // sign(t) |t|^(p-1); 0 at t == 0 (p >= 1)
                        const float ph = (OP == BW_MINK3) ? a * t
                                         : (a > 0.0f ? copysignf(exp2f(args.pm1 * log2f(a)), t) : 0.0f);
                        acc[r][m] = fmaf(w[r], ph, acc[r][m]);
                    }
                }
            }
        }
    }

    if (args.dx) {
#pragma unroll
        for (int r = 0; r < RPT; ++r) {
            const int64_t gi = i0 + rg * RPT + r;
            if (gi >= n) continue;
            // JS > 1: partial sums to slice js of the workspace (row stride k)
            float *const out = JS > 1 ? args.dxp + (int64_t)js * n * k + gi * k
                                      : args.dx + gi * args.lddx;
#pragma unroll
            for (int m = 0; m < FPT; ++m) {
                const int c = fg * FPT + m;
                if (c < fcount) {
                    const float v = (OP == BW_EUCLID)
                                        ? fmaf(args.x[gi * ldx + f0 + c], rowsum[r], acc[r][m])
                                        : acc[r][m];
                    out[f0 + c] = v;
                }
            }
        }
    }

    if (MODE == MODE_MDS && blockIdx.y == 0) {
        // each unordered pair was seen by both of its row owners: S = sum / 2
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) stress += __shfl_xor(stress, d, 64);
        __syncthreads();
        if ((tid & 63) == 0) red_s[tid >> 6] = stress;
        __syncthreads();
        if (tid == 0) {
            double s = 0.0;
            for (int w = 0; w < BTH / 64; ++w) s += red_s[w];
            args.partials[(int64_t)js * gridDim.x + blockIdx.x] = 0.5 * s;
        }
    }
}

// ---------------------------------------------------------------------------
// Euclidean gradient on the matrix cores
// ---------------------------------------------------------------------------
// dX_i = x_i sum_j w_ij - sum_j w_ij x_j with w_ij = G_ij / d_ij, on the centred
// rows (both terms move alike).  A wave owns 32 rows i and visits blocks of 32
// rows j.  The Gram block is computed with j along the accumulator's rows and i
// along its columns, so element r of lane l is pair (i = l % 32, j = 8 (r / 4) +
// 4 (l / 32) + r % 4): as it stands, registers 8 s .. 8 s + 7 of the weights are
// the A operand of the second product for sixteen j, whose B operand (x_j, one
// feature per lane) a pre-pass lays out in the same order of j.  Weights never
// leave the registers.
constexpr int GW = 8;                  // waves per workgroup, 32 rows i each
constexpr int GROWS = GW * 32;
constexpr int GTL = 36;                // row of a wave's transposed block of G
constexpr int GOWN = 512 + 1024;       // floats of a wave's region: G, or near pairs and distances
static_assert(32 * GTL <= GOWN, "transpose region");
constexpr float GRAD_W_MIN = 0x1p-100f;
constexpr int GRAD_NEAR_MAX = 256;     // near pairs of a 32 x 32 block, on average
constexpr int GRAD_SAMPLES = 512;      // blocks of 32 x 32 pairs; a thread of gradient_kernel each
static_assert(GRAD_SAMPLES == GW * 64, "samples");

__device__ __forceinline__ uint16_t *gradient_samples(uint8_t *left)
{
    return reinterpret_cast<uint16_t *>(left) - GRAD_SAMPLES;
}

typedef float f32x4u_t __attribute__((ext_vector_type(4), aligned(4)));   // rows start anywhere

// This lane's rank among the set bits of m.
__device__ __forceinline__ int rank_in(unsigned long long m)
{
    return (int)__builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
}

// norms read through the scalar cache: uniform addresses, not written by the kernel
typedef const __attribute__((address_space(4))) float uniform_float_t;

struct GradArgs {
    const float *x;                    // FP32 rows (exact pairs)
    int64_t n, k, ldx;
    const unsigned short *terms;       // operand blocks of the centred rows (gt_mfma.h)
    const unsigned short *tterms;      // the same values, features along the rows
    const float *norms;                // squared norms of the centred rows
    const float *center;
    const float *g;                    // packed dL/dD
    float *dx;
    int64_t lddx;
    float *dxp;                        // gridDim.y > 1: partial dX slices
    // per BI rows: 1 = left to backward_kernel; before them the near pairs of the
    // blocks that gradient_sample visits
    uint8_t *left;
    int64_t jblocks;                   // blocks of 32 rows j, per workgroup
    float tau;
};

// Near pairs of sample s, a block of 32 x 32 pairs, from the first terms alone: the
// rows i of the samples are spread over all rows, and so are the rows j of the
// even ones; those of the odd ones are the rows i, which shows near points that
// lie in order (the eight waves of a workgroup meet such a block one after the
// other, each while the others wait).
__device__ __forceinline__ void gradient_sample(const GradArgs &args, int s, int nch)
{
    typedef Split<SPLIT_BF16> S;
    const int lane = threadIdx.x & 63, h = lane >> 5;
    const int64_t n = args.n, nblk = operand_rows(n) / 32;
    const int64_t ib = s * nblk / GRAD_SAMPLES;
    const int64_t jb = s & 1 ? ib : (ib + 1 + s * (int64_t)617 % nblk) % nblk;
    const unsigned short *const a = args.terms + jb * nch * 3 * OPERAND_VALUES + lane * 8;
    const unsigned short *const b = args.terms + ib * nch * 3 * OPERAND_VALUES + lane * 8;
    const int64_t i = ib * 32 + (lane & 31);
    const float ni = args.norms[i < n ? i : n - 1];
    float nj[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int64_t j = jb * 32 + 8 * (r >> 2) + 4 * h + (r & 3);
        nj[r] = args.norms[j < n ? j : n - 1];
    }
    f32x16_t w;
#pragma unroll
    for (int r = 0; r < 16; ++r) w[r] = 0.0f;
#pragma unroll 8
    for (int c = 0; c < nch; ++c)
        w = S::mfma(*reinterpret_cast<const bf16x8_t *>(a + c * 3 * OPERAND_VALUES),
                    *reinterpret_cast<const bf16x8_t *>(b + c * 3 * OPERAND_VALUES), w);
    int near = 0;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int64_t j = jb * 32 + 8 * (r >> 2) + 4 * h + (r & 3);
        const float ss = ni + nj[r], d2 = fmaf(-2.0f, w[r], ss);
        const bool ok = d2 >= fmaf(args.tau, ss, GRAM_SQRT_MIN) && d2 < 0x1p127f;
        near += __popcll(__builtin_amdgcn_ballot_w64(i < n && j < n && i != j && !ok));
    }
    if (lane == 0) gradient_samples(args.left)[s] = (uint16_t)near;
}

// B operands of the second product: block jb (32 rows j), feature block cb (32
// features), step s (sixteen j: 16 s + 8 p + 4 h + e, p < 2, e < 4), term t at
// (((jb * ncb + cb) * 2 + s) * 3 + t) * OPERAND_VALUES, lane 32 h + c.  Also
// clears `left`, and the first workgroups count the samples.
__global__ __launch_bounds__(256) void gradient_terms_kernel(GradArgs args, int64_t ncb,
                                                             unsigned short *__restrict__ tterms)
{
    constexpr int SAMPLERS = GRAD_SAMPLES / 4;   // workgroups
    if (blockIdx.x < SAMPLERS) {
        gradient_sample(args, (int)blockIdx.x * 4 + (threadIdx.x >> 6), (int)ncb * 2);
        return;
    }
    const int lane = threadIdx.x & 63, h = lane >> 5;
    const int64_t n = args.n, k = args.k, ldx = args.ldx;
    const int64_t wg = (int64_t)blockIdx.x - SAMPLERS, wgs = (int64_t)gridDim.x - SAMPLERS;
    const float *const __restrict__ x = args.x, *const __restrict__ center = args.center;
    const int64_t nleft = (n + BI - 1) / BI;
    for (int64_t t = wg * 256 + threadIdx.x; t < nleft; t += wgs * 256) args.left[t] = 0;
    const int64_t blocks = operand_rows(n) / 32 * ncb * 2;
    for (int64_t blk = wg * 4 + (threadIdx.x >> 6); blk < blocks; blk += wgs * 4) {
        const int64_t s = blk & 1, cb = (blk >> 1) % ncb, jb = (blk >> 1) / ncb;
        const int64_t c = cb * 32 + (lane & 31);
        unsigned short t[8][3];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int64_t j = jb * 32 + s * 16 + (e >> 2) * 8 + h * 4 + (e & 3);
            const float v = (j < n && c < k) ? x[j * ldx + c] - center[c] : 0.0f;
            Split<SPLIT_BF16>::split(v, t[e]);
        }
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            uint4 w;
            w.x = t[0][q] | ((unsigned)t[1][q] << 16);
            w.y = t[2][q] | ((unsigned)t[3][q] << 16);
            w.z = t[4][q] | ((unsigned)t[5][q] << 16);
            w.w = t[6][q] | ((unsigned)t[7][q] << 16);
            *reinterpret_cast<uint4 *>(tterms + (blk * 3 + q) * OPERAND_VALUES + lane * 8) = w;
        }
    }
}

// NC: chunks of 16 features (2, 4, 6 or 8).  A workgroup owns 256 rows i (blockIdx.x)
// and a range of row blocks j (blockIdx.y); each block's two operand forms
// stream through a two-stage LDS ring, G through registers.
// Bound: the matrix cores and the VALU about alike (per 32 x 32 block and wave
// 96 products, 3072 cycles, and about 500 VALU instructions, 2000 cycles, the
// weights and their split).  Two waves a SIMD, from registers that hold the
// wave's rows of the Gram product and its share of dX.  16384 x 128: 5.2 ms for
// the sweep (two distances and an fma per feature and ordered pair on the
// VALU), 1.1 ms here; the relative error of dX against FP64 8.2e-7 -> 4.0e-7.
// A pair with d^2 < tau (||x_i||^2 + ||x_j||^2), or a d^2 that is not a normal
// number, is recomputed from FP32 differences.  Rows with a weight that is not
// finite or too small for three BF16 terms, or (in the blocks that one wave has
// seen) more near pairs than GRAD_NEAR_MAX, are left to backward_kernel, and so are
// all rows where the samples show many near pairs: more than 144 of 1024 (80 up
// to 32 features, where the sweep is faster).  In ms, here and in the sweep, with
// 64 and 128 of 1024 near: 16384 x 128 2.51, 3.42 and 5.19; 3000 x 48 0.122,
// 0.141 and 0.175; 16384 x 32 1.29, 1.63 and 1.73; 6000 x 32 0.28, 0.42 and 0.26.
// Left without samples, by each wave once it had seen too many, a row was found
// after other waves had done their work on it: 12000 x 128 with one dominant
// direction 5.15 ms, in 8 clusters that lie in order 4.20, with the samples 3.24
// and 3.22, the sweep 3.20.  Of the samples on the diagonal more than a quarter may
// not hold more than 400 near pairs: in groups of 12 and 32 rows that lie in order
// 3000 x 64 took 0.178 and 0.41 ms here, 0.175 in the sweep.
template <int NC>
__global__ __launch_bounds__(GW * 64, 2) void gradient_kernel(GradArgs args)
{
    typedef Split<SPLIT_BF16> S;
    constexpr int NCB = NC / 2;                       // blocks of 32 features
    constexpr int HALF = NC * 3 * OPERAND_BYTES;      // one block j in one form
    // [two stages of both operand forms][a region per wave].  One array: with
    // two, the compiler waits for the direct loads in flight before every LDS
    // read.
    __shared__ __attribute__((aligned(1024))) unsigned char smem[2 * 2 * HALF + GW * GOWN * 4];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    float *const own = reinterpret_cast<float *>(smem + 2 * 2 * HALF) + wave * GOWN;
    const int h = lane >> 5, col = lane & 31;
    const int64_t n = args.n, k = args.k;
    const int64_t i0 = (int64_t)blockIdx.x * GROWS + wave * 32;
    const int64_t nblk = operand_rows(n) / 32;
    const int64_t jb0 = (int64_t)blockIdx.y * args.jblocks;
    const int64_t jb1 = jb0 + args.jblocks < nblk ? jb0 + args.jblocks : nblk;
    {
        // many near pairs, or groups of near points in order: all rows are left
        const int v = gradient_samples(args.left)[tid];
        const int ordered = __syncthreads_count((tid & 1) && v > 400);
        int sum = tid & 1 ? 0 : v;
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) sum += __shfl_xor(sum, d, 64);
        int *const part = reinterpret_cast<int *>(smem);
        if (lane == 0) part[wave] = sum;
        __syncthreads();
        sum = 0;
        for (int w = 0; w < GW; ++w) sum += part[w];
        __syncthreads();   // the region is free again
        if (sum > (NC == 2 ? 80 : 144) * (GRAD_SAMPLES / 2) || ordered > GRAD_SAMPLES / 8) {
            if (blockIdx.y == 0 && tid < GROWS / BI && (int64_t)blockIdx.x * GROWS + tid * BI < n)
                args.left[(int64_t)blockIdx.x * (GROWS / BI) + tid] = 1;
            return;
        }
    }
    bool idle = i0 >= n;                              // only helps to load
    const int64_t i = i0 + col;
    const int64_t ic = i < n ? i : n - 1;

    typedef __attribute__((address_space(3))) void lds_void_t;
    typedef const __attribute__((address_space(1))) void gbl_void_t;
    auto issue = [&](int64_t jb) {
        unsigned char *const st = smem + (jb & 1) * 2 * HALF;
        const unsigned short *const a = args.terms + jb * NC * 3 * OPERAND_VALUES + lane * 8;
        const unsigned short *const b = args.tterms + jb * NC * 3 * OPERAND_VALUES + lane * 8;
        for (int u = wave; u < NC * 3; u += GW) {
            __builtin_amdgcn_global_load_lds((gbl_void_t *)(a + u * OPERAND_VALUES),
                                             (lds_void_t *)(st + u * OPERAND_BYTES), 16, 0, 0);
            __builtin_amdgcn_global_load_lds((gbl_void_t *)(b + u * OPERAND_VALUES),
                                             (lds_void_t *)(st + HALF + u * OPERAND_BYTES), 16, 0, 0);
        }
    };
    // G of block j0: below the diagonal (i > j) the packed index runs along i,
    // the lanes; above it along j, so the lanes take j and the block is
    // transposed through LDS when it is used
    float gq[16] = {};
    auto gfetch = [&](int64_t jb) {
        const int64_t j0 = jb * 32;
        if (j0 < i0) {
            const float *const base = args.g + packed_base(n, j0) + ic;
            const unsigned cw = (unsigned)(n - 1 - j0);
            // row j0 + d + 4 h starts d cw - d (d + 1) / 2 + h (4 cw - 4 d - 10) on
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const unsigned d = 8 * (r >> 2) + (r & 3);
                gq[r] = base[d * cw - d * (d + 1) / 2 + (h ? 4 * cw - 4 * d - 10 : 0u)];
            }
        } else if (j0 > i0) {
            const int64_t j = j0 + col < n ? j0 + col : n - 1;
            const float *const base = args.g + packed_base(n, i0) + j;
            unsigned cw = (unsigned)(n - 1 - i0);
            // the sixteen offsets do not change with jb: computed here each
            // time, or they would be kept in registers that are not there
            asm volatile("" : "+s"(cw));
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const unsigned d = 2 * r;
                gq[r] = base[d * cw - d * (d + 1) / 2 + (h ? cw - d - 1 : 0u)];
            }
        } else {
            int h4 = 4 * h;
            asm volatile("" : "+v"(h4));
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int64_t j = j0 + 8 * (r >> 2) + (r & 3) + h4;
                const int64_t hi = i > j ? i : j, lo = i > j ? j : i;
                gq[r] = (hi < n && lo != hi) ? args.g[packed_base(n, lo) + hi] : 0.0f;
            }
        }
    };

    bf16x8_t xi[NC][3];
    f32x16_t dacc[NCB];
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int t = 0; t < 3; ++t)
            xi[c][t] = *reinterpret_cast<const bf16x8_t *>(
                args.terms + (((idle ? nblk - 1 : i0 / 32) * NC + c) * 3 + t) * OPERAND_VALUES + lane * 8);
#pragma unroll
    for (int cb = 0; cb < NCB; ++cb)
#pragma unroll
        for (int r = 0; r < 16; ++r) dacc[cb][r] = 0.0f;
    const float ni = args.norms[ic];
    float rowsum = 0.0f;
    bool bad = false;
    int seen = 0, seen_near = 0;                      // blocks, near pairs in them

    if (jb0 < jb1) {
        issue(jb0);
        if (!idle) gfetch(jb0);
    }
    for (int64_t jb = jb0; jb < jb1; ++jb) {
        const int64_t j0 = jb * 32;
        // this block's operands (and G) have landed, in every wave, and every
        // wave is done with the stage that the next issue overwrites
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        // (a use of G here, or the compiler would wait for the next block's
        // loads at its first use below)
#pragma unroll
        for (int r = 0; r < 16; ++r) asm volatile("" : "+v"(gq[r]));
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (jb + 1 < jb1) issue(jb + 1);
        if (idle) continue;
        const unsigned char *const st = smem + (jb & 1) * 2 * HALF + lane * 16;
        // ---- Gram block ------------------------------------------------------
        // The smaller products of all chunks first: an addition rounds at the size
        // of the sum, and so only the last NC do at its full size.  (By chunks, all
        // 6 NC did: with three dominant directions and gradients at near pairs alone,
        // 4000 x 128, the largest relative error of a row of dX 5.3e-7 and 3.5e-7
        // here, 2.4e-7 in the sweep; 16384 x 128 1.04 and 1.06 ms.)
        f32x16_t w;
#pragma unroll
        for (int r = 0; r < 16; ++r) w[r] = 0.0f;
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            bf16x8_t a[3];
#pragma unroll
            for (int t = 0; t < 3; ++t)
                a[t] = *reinterpret_cast<const bf16x8_t *>(st + (c * 3 + t) * OPERAND_BYTES);
            w = S::mfma(a[1], xi[c][1], w);
            w = S::mfma(a[2], xi[c][0], w);
            w = S::mfma(a[0], xi[c][2], w);
            w = S::mfma(a[1], xi[c][0], w);
            w = S::mfma(a[0], xi[c][1], w);
            // keeps the later chunks' operands out of the registers
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            w = S::mfma(*reinterpret_cast<const bf16x8_t *>(st + c * 3 * OPERAND_BYTES), xi[c][0], w);
            __builtin_amdgcn_sched_barrier(0);
        }
        // ---- weights -----------------------------------------------------------
        if (j0 > i0) {
            // G back with lanes along i (a wave's own region; LDS is in order)
            float *const tr = own;
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int r = 0; r < 16; ++r) tr[(2 * r + h) * GTL + col] = gq[r];
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const float4 v = *reinterpret_cast<const float4 *>(tr + col * GTL + 8 * q + 4 * h);
                gq[4 * q] = v.x;
                gq[4 * q + 1] = v.y;
                gq[4 * q + 2] = v.z;
                gq[4 * q + 3] = v.w;
            }
        }
        const bool edge = j0 == i0 || j0 + 32 > n || i0 + 32 > n;
        unsigned flags = 0;
        float part = 0.0f;
        // (past the last row these read what follows the norms: no pair uses it)
        uniform_float_t *const nj = (uniform_float_t *)(args.norms + j0);
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int lj = 8 * (r >> 2) + 4 * h + (r & 3);
            const int64_t j = j0 + lj;
            const float ss = ni + (h ? nj[8 * (r >> 2) + 4 + (r & 3)] : nj[8 * (r >> 2) + (r & 3)]);
            const float d2 = fmaf(-2.0f, w[r], ss);
            bool ok = d2 >= fmaf(args.tau, ss, GRAM_SQRT_MIN) && d2 < 0x1p127f;
            // 1 / sqrt(d^2): the hardware estimate and one Newton step
            float y = __builtin_amdgcn_rsqf(d2);
            y = fmaf(0.5f * y, fmaf(-d2 * y, y, 1.0f), y);
            float v = gq[r] * y;
            if (edge) {
                const bool pair = i < n && j < n && i != j;
                ok = ok || !pair;
                v = pair ? v : 0.0f;
            }
            w[r] = ok ? v : 0.0f;
            flags |= ok ? 0u : 1u << r;
        }
        if (__builtin_amdgcn_ballot_w64(flags != 0u)) {
            // Near pairs from differences: their list goes to LDS (the wave's
            // own region), four lanes take a pair, sixteen pairs at a time,
            // and the distances come back through LDS.
            unsigned short *const list = reinterpret_cast<unsigned short *>(own);
            float *const res = own + 512;
            int near = 0;
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const bool f = (flags >> r) & 1u;
                const unsigned long long m = __builtin_amdgcn_ballot_w64(f);
                if (f) list[near + rank_in(m)] = (unsigned short)(lane | (r << 6));
                near += __popcll(m);
            }
            __builtin_amdgcn_wave_barrier();
            seen_near += near;
            if (seen_near > (seen < 1 ? 2 : seen + 1) * GRAD_NEAR_MAX) {
                // points in a few clusters: differences throughout are cheaper
                bad = idle = true;
                continue;
            }
#pragma unroll 1
            for (int e0 = 0; e0 < near; e0 += 16) {
                const int e = e0 + (lane >> 2);
                const int ent = list[e < near ? e : near - 1];
                const int src = ent & 63, q = ent >> 6;
                const float *const pi = args.x + (i0 + (src & 31)) * args.ldx;
                const float *const pj = args.x + (j0 + 8 * (q >> 2) + 4 * (src >> 5) + (q & 3)) * args.ldx;
                float s = 0.0f;
#pragma unroll 2
                for (int f = (lane & 3) * 4; f < (int)k; f += 16) {
                    if (f + 4 <= (int)k) {
                        const f32x4u_t d = *reinterpret_cast<const f32x4u_t *>(pi + f) -
                                           *reinterpret_cast<const f32x4u_t *>(pj + f);
                        s = fmaf(d[0], d[0], s);
                        s = fmaf(d[1], d[1], s);
                        s = fmaf(d[2], d[2], s);
                        s = fmaf(d[3], d[3], s);
                    } else {
                        for (int u = f; u < (int)k; ++u) {
                            const float d = pi[u] - pj[u];
                            s = fmaf(d, d, s);
                        }
                    }
                }
                s += __shfl_xor(s, 1, 64);
                s += __shfl_xor(s, 2, 64);
                if ((lane & 3) == 0 && e < near) res[e] = sqrtf(s);
            }
            __builtin_amdgcn_wave_barrier();
            near = 0;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const bool f = (flags >> r) & 1u;
                const unsigned long long m = __builtin_amdgcn_ballot_w64(f);
                if (f) {
                    const float dist = res[near + rank_in(m)];
                    w[r] = dist > 0.0f ? gq[r] / dist : 0.0f;
                }
                near += __popcll(m);
            }
            __builtin_amdgcn_wave_barrier();
        }
        ++seen;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const float a = fabsf(w[r]);
            bad = bad || !(a < INFINITY) || (a < GRAD_W_MIN && a != 0.0f);
            part += w[r];
        }
        rowsum += part;
        if (jb + 1 < jb1) gfetch(jb + 1);
        // ---- dX += W x_J ---------------------------------------------------------
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            bf16x8_t a[3];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                unsigned short t[3];
                S::split(w[8 * s + e], t);
#pragma unroll
                for (int q = 0; q < 3; ++q) a[q][e] = __builtin_bit_cast(__bf16, t[q]);
            }
#pragma unroll
            for (int cb = 0; cb < NCB; ++cb) {
                bf16x8_t b[3];
#pragma unroll
                for (int t = 0; t < 3; ++t)
                    b[t] = *reinterpret_cast<const bf16x8_t *>(st + HALF + ((cb * 2 + s) * 3 + t) * OPERAND_BYTES);
                dacc[cb] = S::mfma(a[1], b[1], dacc[cb]);
                dacc[cb] = S::mfma(a[2], b[0], dacc[cb]);
                dacc[cb] = S::mfma(a[0], b[2], dacc[cb]);
                dacc[cb] = S::mfma(a[1], b[0], dacc[cb]);
                dacc[cb] = S::mfma(a[0], b[1], dacc[cb]);
                dacc[cb] = S::mfma(a[0], b[0], dacc[cb]);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    }
    if (__builtin_amdgcn_ballot_w64(bad) != 0 && lane == 0) args.left[i0 / BI] = 1;
    if (idle) return;

    rowsum += __shfl_xor(rowsum, 32, 64);
    const bool slices = gridDim.y > 1;
    float *const out = slices ? args.dxp + (int64_t)blockIdx.y * n * k : args.dx;
    const int64_t ldo = slices ? k : args.lddx;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int li = 8 * (r >> 2) + 4 * h + (r & 3);
        const float rs = __shfl(rowsum, li, 64);
        const int64_t row = i0 + li;
        if (row >= n) continue;
#pragma unroll
        for (int cb = 0; cb < NCB; ++cb) {
            const int64_t c = cb * 32 + col;
            if (c < k) out[row * ldo + c] = fmaf(args.x[row * args.ldx + c] - args.center[c], rs, -dacc[cb][r]);
        }
    }
}

// ---------------------------------------------------------------------------
// MDS of few features
// ---------------------------------------------------------------------------
// Up to 8 features a pair is a handful of instructions and four bytes of
// delta, so each pair is visited once and serves both of its rows.  A workgroup
// owns 256 rows i and 4 jw columns j < i, a wave jw of the columns; a lane holds
// four rows i (lanes along i, as the packed columns run) and walks the columns,
// whose rows are uniform (scalar loads).  The sums of row i stay in its lane;
// those of row j are added over the lane's four rows, then over the wave by
// data-parallel adds.  Each term is w (y_i - y_j): sums of w and of w y_j apart
// cancel where points are close.  Both sides go to partial slices, which
// mds_finish_kernel adds in a fixed order: deterministic, no atomics.  The
// slices are about n / 128 for each row: beyond MDS_SLICE_BYTES the row blocks are
// taken some at a time, each pass adding to dY.
// Bound: VALU issue (about 45 instructions per pair with 2 features, two of them
// FP64; delta alone would take 0.11 ms).  16384 x 2: 0.67 ms for the sweep, which
// visits each pair from both rows and pads 2 features to 4, 0.18 ms here; the
// relative error of dY against FP64 9.0e-7 -> 5.2e-8.
constexpr int MI = 256;                            // rows of a workgroup
constexpr int MR = MI / 64;                        // rows per lane
constexpr int MSUM = 8;                            // threads per row in mds_finish_kernel

struct MdsArgs {
    const float *y;
    int64_t n, q, ldy;
    const float *delta;
    int jw;                    // columns per wave: 16, 32 or 64
    int64_t c0, c1;            // this pass's row blocks
    int t0;                    // tiles before them
    // [slice][feature][row]: rows i of the pass (irows of them) by column block,
    // rows j by row block of the pass; the pointers are those of row 0 and block 0
    float *ipart, *jpart;
    int irows;
    double *partials;          // stress, one per workgroup (of this pass)
};

// Sum over the wave, in lane 63.
__device__ __forceinline__ float wave_total(float v)
{
#define GT_DPP_ADD(ctrl, rows) \
    v += __uint_as_float((unsigned)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(v), ctrl, rows, 0xf, false))
    GT_DPP_ADD(0x111, 0xf);   // row_shr:1
    GT_DPP_ADD(0x112, 0xf);   // row_shr:2
    GT_DPP_ADD(0x114, 0xf);   // row_shr:4
    GT_DPP_ADD(0x118, 0xf);   // row_shr:8
    GT_DPP_ADD(0x142, 0xa);   // row_bcast:15
    GT_DPP_ADD(0x143, 0xc);   // row_bcast:31
#undef GT_DPP_ADD
    return v;
}

extern "C" __device__ int gt_mds_writelane(int value, int lane, int old) __asm("llvm.amdgcn.writelane.i32");

// One column j against the lane's rows.  EDGE: rows at or before j, or past
// the end, do not count.
template <int Q, bool GRAD, bool EDGE>
__device__ __forceinline__ void mds_column(const float (&xi)[MR][Q], const float (&xj)[Q], const float (&dl)[MR],
                                           int64_t i0, int64_t j, int64_t n, int lane, double &stress,
                                           float (&wi)[MR][Q], float (&wj)[Q])
{
#pragma unroll
    for (int c = 0; c < Q; ++c) wj[c] = 0.0f;
#pragma unroll
    for (int r = 0; r < MR; ++r) {
        float t[Q], d2 = 0.0f;
#pragma unroll
        for (int c = 0; c < Q; ++c) {
            t[c] = xi[r][c] - xj[c];
            d2 = fmaf(t[c], t[c], d2);
        }
        // d = sqrt(d2) and inv = 1 / d: the hardware estimate of the inverse
        // root, one correction of the root
        float inv = __builtin_amdgcn_rsqf(d2);
        float d = d2 * inv;
        d = fmaf(0.5f * inv, fmaf(-d, d, d2), d);
        bool apart = true;
        if (!(d2 >= 0x1p-100f && d2 <= 0x1p120f)) {   // 0, tiny, huge, not a number
            d = sqrtf(d2);
            inv = 1.0f / d;
            apart = d > 0.0f;
        }
        float res = apart ? d - dl[r] : -dl[r];
        if (EDGE) {
            const int64_t i = i0 + r * 64 + lane;
            const bool pair = i > j && i < n;
            res = pair ? res : 0.0f;
            apart = apart && pair;
        }
        stress = fma((double)res, (double)res, stress);
        if (GRAD) {
            const float w = apart ? 2.0f * res * inv : 0.0f;
#pragma unroll
            for (int c = 0; c < Q; ++c) {
                wi[r][c] = fmaf(w, t[c], wi[r][c]);
                wj[c] = fmaf(-w, t[c], wj[c]);
            }
        }
    }
}

template <int Q, bool GRAD>
__global__ __launch_bounds__(256) void mds_small_kernel(MdsArgs args)
{
    __shared__ float red[3][MI][Q];
    __shared__ double red_s[4];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int64_t n = args.n;
    // row block ci has f (ci + 1) column blocks, f = 256 / (4 jw)
    const int64_t t = args.t0 + blockIdx.x;
    const int f = 64 / args.jw;
    int ci, cm;
    tri_tile(t / f, ci, cm);
    const int64_t cj = (int64_t)cm * f + t % f;
    const int64_t i0 = (int64_t)ci * MI;
    const int64_t j0 = (cj * 4 + wave) * args.jw;
    int64_t j1 = j0 + args.jw < n ? j0 + args.jw : n;

    float xi[MR][Q], wi[MR][Q];
#pragma unroll
    for (int r = 0; r < MR; ++r) {
        const int64_t i = i0 + r * 64 + lane;
#pragma unroll
        for (int c = 0; c < Q; ++c) xi[r][c] = (i < n && c < args.q) ? args.y[i * args.ldy + c] : 0.0f;
#pragma unroll
        for (int c = 0; c < Q; ++c) wi[r][c] = 0.0f;
    }
    double stress = 0.0;
    const bool edge = j1 > i0 || i0 + MI > n;
    auto load = [&](int64_t j, float (&xj)[Q], float (&dl)[MR]) {
        uniform_float_t *const yj = (uniform_float_t *)(args.y + j * args.ldy);
#pragma unroll
        for (int c = 0; c < Q; ++c) xj[c] = c < args.q ? yj[c] : 0.0f;
        const float *const col = args.delta + packed_base(n, j) + i0;
#pragma unroll
        for (int r = 0; r < MR; ++r) {
            const int li = r * 64 + lane;
            dl[r] = (!edge || (i0 + li > j && i0 + li < n)) ? col[li] : 0.0f;
        }
    };
    if (j0 < j1) {
        const int64_t jc = j0;
        const int count = (int)(j1 - j0);
        float out[Q];   // lane l: the sums of row jc + l
#pragma unroll
        for (int c = 0; c < Q; ++c) out[c] = 0.0f;
        for (int l = 0; l < count; l += 4) {
            float xj[4][Q], dl[4][MR];
#pragma unroll
            for (int u = 0; u < 4; ++u)
                load(l + u < count ? jc + l + u : jc + count - 1, xj[u], dl[u]);
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                if (l + u >= count) break;
                float wj[Q];
                if (edge)
                    mds_column<Q, GRAD, true>(xi, xj[u], dl[u], i0, jc + l + u, n, lane, stress, wi, wj);
                else
                    mds_column<Q, GRAD, false>(xi, xj[u], dl[u], i0, jc + l + u, n, lane, stress, wi, wj);
                if (GRAD) {
#pragma unroll
                    for (int c = 0; c < Q; ++c) {
                        const int total = __builtin_amdgcn_readlane((int)__float_as_uint(wave_total(wj[c])), 63);
                        out[c] = __uint_as_float((unsigned)gt_mds_writelane(total, l + u, (int)__float_as_uint(out[c])));
                    }
                }
            }
        }
        if (GRAD && lane < count) {
#pragma unroll
            for (int c = 0; c < Q; ++c)
                if (c < args.q) args.jpart[(ci * args.q + c) * n + jc + lane] = out[c];
        }
    }
    // the four waves' sums of the rows i, in order
    if (GRAD) {
        if (wave > 0)
#pragma unroll
            for (int r = 0; r < MR; ++r)
#pragma unroll
                for (int c = 0; c < Q; ++c) red[wave - 1][r * 64 + lane][c] = wi[r][c];
        __syncthreads();
        if (wave == 0)
#pragma unroll
            for (int r = 0; r < MR; ++r) {
                const int64_t i = i0 + r * 64 + lane;
#pragma unroll
                for (int c = 0; c < Q; ++c) {
                    float v = wi[r][c];
                    for (int w = 0; w < 3; ++w) v += red[w][r * 64 + lane][c];
                    if (i < n && c < args.q) args.ipart[(cj * args.q + c) * args.irows + i] = v;
                }
            }
    }
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) stress += __shfl_xor(stress, d, 64);
    if (lane == 0) red_s[wave] = stress;
    __syncthreads();
    if (tid == 0) args.partials[blockIdx.x] = ((red_s[0] + red_s[1]) + red_s[2]) + red_s[3];
}

// dY_r from the slices of row r in this pass: its column blocks as a row i, then
// the row blocks from its own on as a row j; rows of earlier passes only as a
// row j, added to what they have.  MSUM threads a row; the last workgroup adds
// the stress partials (stress null: not the last pass).
__global__ __launch_bounds__(256) void mds_finish_kernel(MdsArgs args, float *__restrict__ dy, int64_t lddy,
                                                         int64_t count, double *__restrict__ stress)
{
    if (blockIdx.x == gridDim.x - 1) {
        if (stress == nullptr) return;
        __shared__ double s_[256];
        double s = 0.0;
        const double *const all = args.partials - args.t0;
        for (int64_t e = threadIdx.x; e < count; e += 256) s += all[e];
        s_[threadIdx.x] = s;
        __syncthreads();
        for (int d = 128; d >= 1; d >>= 1) {
            if ((int)threadIdx.x < d) s_[threadIdx.x] += s_[threadIdx.x + d];
            __syncthreads();
        }
        if (threadIdx.x == 0) *stress = s_[0];
        return;
    }
    constexpr int ROWS = 256 / MSUM;
    __shared__ float red[MSUM][ROWS];
    const int lr = threadIdx.x % ROWS, part = threadIdx.x / ROWS;
    const int64_t n = args.n, row = (int64_t)blockIdx.x * ROWS + lr, ci = row / MI;
    const bool earlier = ci < args.c0;
    const int64_t first = earlier ? args.c0 : ci;
    const int64_t islices = earlier ? 0 : 64 / args.jw * (ci + 1), slices = islices + args.c1 - first;
    const bool in = row < n && ci < args.c1;
    for (int64_t c = 0; c < args.q; ++c) {
        float v = 0.0f;
        if (in)
#pragma unroll 4
            for (int64_t e = part; e < slices; e += MSUM)
                v += e < islices ? args.ipart[(e * args.q + c) * args.irows + row]
                                 : args.jpart[((first + e - islices) * args.q + c) * n + row];
        __syncthreads();
        red[part][lr] = v;
        __syncthreads();
        float total = red[0][lr];
#pragma unroll
        for (int e = 1; e < MSUM; ++e) total += red[e][lr];
        if (part == 0 && in) dy[row * lddy + c] = earlier ? dy[row * lddy + c] + total : total;
    }
}

// Sum of the per-workgroup FP64 partials, fixed order (deterministic).
__global__ __launch_bounds__(256) void reduce_partials_kernel(const double *partials, int64_t count,
                                                              double *out)
{
    __shared__ double s_[256];
    double s = 0.0;
    for (int64_t e = threadIdx.x; e < count; e += 256) s += partials[e];
    s_[threadIdx.x] = s;
    __syncthreads();
    for (int d = 128; d >= 1; d >>= 1) {
        if ((int)threadIdx.x < d) s_[threadIdx.x] += s_[threadIdx.x + d];
        __syncthreads();
    }
    if (threadIdx.x == 0) *out = s_[0];
}

// dx = sum over the JS partial slices, in slice order (left_count slices for
// the rows of the BI-row blocks marked in left).
__global__ __launch_bounds__(256) void sum_partial_dx_kernel(const float *__restrict__ dxp, int64_t n,
                                                             int64_t k, int js_count,
                                                             const uint8_t *__restrict__ left, int left_count,
                                                             float *__restrict__ dx, int64_t lddx)
{
    const int64_t total = n * k;
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < total;
         e += (int64_t)gridDim.x * blockDim.x) {
        float s = dxp[e];
        const int count = left && left[e / k / BI] ? left_count : js_count;
        for (int q = 1; q < count; ++q) s += dxp[(int64_t)q * total + e];
        dx[(e / k) * lddx + e % k] = s;
    }
}

// Workspace of gradient_kernel: the Gram pre-passes' (gt_gram.hip), the second
// operand form, the flags and the partial slices.
struct GradPlan {
    int64_t kp, ncb, slices, jblocks;
    int sweep_slices;      // of the rows that are left
    size_t off_tterms, off_left, off_slices, bytes;
};

int j_splits(int64_t n, int64_t k);

size_t align256(size_t v) { return (v + 255) / 256 * 256; }

// Whether the matrix-core gradient takes the call.  Its operands of a block of
// rows fit the registers up to 128 features; below 16 most pairs are near by
// its rule (5 features, 4000 points: 206 us, and 115 for the sweep); with few
// points the pre-passes cost more than they save (times in us, sweep and here:
// 1000 x 96 50 and 55, 2000 x 96 88 and 70; 2000 x 32 41 and 58, 4000 x 32 122
// and 77; at 3000 x 32 95 and 74, but 130 where all rows are left).  A sweep that
// needs no workspace can be captured; it stays.
bool gradient_applies(int op, int64_t n, int64_t k)
{
    return op == OP_EUCLID && k <= 128 && ((k > 32 && n >= 1500) || (k >= 16 && n >= 4000)) &&
           j_splits(n, k) > 1;
}

GradPlan gradient_plan(int64_t n, int64_t k)
{
    GradPlan g;
    g.kp = (k + 31) / 32 * 32;
    g.ncb = g.kp / 32;
    const int64_t rows = (n + GROWS - 1) / GROWS, nblk = operand_rows(n) / 32;
    // about 1024 workgroups in all, at most 16 slices, at least two blocks each
    int64_t js = (1024 + rows - 1) / rows;
    if (js > 16) js = 16;
    if (js > (nblk + 1) / 2) js = (nblk + 1) / 2;
    g.jblocks = (nblk + js - 1) / js;
    g.slices = (nblk + g.jblocks - 1) / g.jblocks;
    g.sweep_slices = j_splits(n, k) < g.slices ? j_splits(n, k) : (int)g.slices;
    size_t p = align256(gram_workspace_bytes(n, k, 1));
    g.off_tterms = p;
    p += (size_t)operand_rows(n) * (size_t)g.kp * 3 * sizeof(unsigned short);
    p += GRAD_SAMPLES * sizeof(uint16_t);
    g.off_left = p;
    p += align256((size_t)nblk);
    g.off_slices = p;
    if (g.slices > 1) p += (size_t)g.slices * (size_t)n * (size_t)k * sizeof(float);
    g.bytes = p;
    return g;
}

int feature_block(int64_t k) { return k <= 4 ? 4 : (k <= 32 ? 32 : KBMAX); }

// j splits: about 2048 workgroups in all, at most 16 splits and no more than
// the number of j blocks.
int j_splits(int64_t n, int64_t k)
{
    const int64_t gx = (n + BI - 1) / BI, gy = (k + feature_block(k) - 1) / feature_block(k);
    int64_t js = (2048 + gx * gy - 1) / (gx * gy);
    if (js > 16) js = 16;
    if (js > gx) js = gx;
    return (int)(js < 1 ? 1 : js);
}

hipError_t launch_sum(const float *dxp, int64_t n, int64_t k, int slices, const uint8_t *left, int left_slices,
                      float *dx, int64_t lddx, hipStream_t stream)
{
    int64_t blocks = (n * k + 255) / 256;
    if (blocks > 65536) blocks = 65536;
    hipLaunchKernelGGL(sum_partial_dx_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, dxp, n, k, slices,
                       left, left_slices, dx, lddx);
    return hipGetLastError();
}

template <int MODE, int KB>
hipError_t launch_kb(int op, BwArgs &args, int js, hipStream_t stream)
{
    dim3 grid((unsigned)((args.n + BI - 1) / BI), (unsigned)((args.k + KB - 1) / KB), (unsigned)js);
    if (op == BW_EUCLID)
        hipLaunchKernelGGL((backward_kernel<BW_EUCLID, MODE, KB>), grid, dim3(BTH), 0, stream, args);
    else if (op == BW_MINK3)
        hipLaunchKernelGGL((backward_kernel<BW_MINK3, MODE, KB>), grid, dim3(BTH), 0, stream, args);
    else
        hipLaunchKernelGGL((backward_kernel<BW_MINKP, MODE, KB>), grid, dim3(BTH), 0, stream, args);
    return hipGetLastError();
}

template <int MODE>
hipError_t launch_sweep(int op, BwArgs &args, int js, hipStream_t stream)
{
    if (args.k <= 4) return launch_kb<MODE, 4>(op, args, js, stream);
    if (args.k <= 32) return launch_kb<MODE, 32>(op, args, js, stream);
    return launch_kb<MODE, KBMAX>(op, args, js, stream);
}

template <int MODE>
hipError_t launch_mode(int op, BwArgs &args, hipStream_t stream)
{
    const int js = j_splits(args.n, args.k);
    const hipError_t e = launch_sweep<MODE>(op, args, js, stream);
    if (e != hipSuccess || js == 1 || args.dx == nullptr) return e;
    return launch_sum(args.dxp, args.n, args.k, js, nullptr, 0, args.dx, args.lddx, stream);
}

// The matrix-core gradient: pre-passes, products, the sweep over the rows that
// were left, sum of the slices.
hipError_t launch_gradient(BwArgs &args, void *workspace, hipStream_t stream)
{
    const GradPlan g = gradient_plan(args.n, args.k);
    char *ws = static_cast<char *>(workspace);
    GramPrep prep;
    hipError_t e = gram_prepare(1, args.x, args.n, args.k, args.ldx, workspace, prep, stream);
    if (e != hipSuccess) return e;
    GradArgs ga;
    ga.x = args.x;
    ga.n = args.n;
    ga.k = args.k;
    ga.ldx = args.ldx;
    ga.terms = prep.terms;
    ga.tterms = reinterpret_cast<unsigned short *>(ws + g.off_tterms);
    ga.norms = prep.norms;
    ga.center = prep.center;
    ga.g = args.g;
    ga.dx = args.dx;
    ga.lddx = args.lddx;
    ga.dxp = reinterpret_cast<float *>(ws + g.off_slices);
    ga.left = reinterpret_cast<uint8_t *>(ws + g.off_left);
    ga.jblocks = g.jblocks;
    // pairs this near lose more in the Gram form than differences do
    ga.tau = fmaxf(gram_tau(1, args.k), 0.25f);
    int64_t blocks = (operand_rows(args.n) / 32 * g.ncb * 2 + 3) / 4;
    if (blocks > 65536) blocks = 65536;
    hipLaunchKernelGGL(gradient_terms_kernel, dim3((unsigned)(GRAD_SAMPLES / 4 + blocks)), dim3(256), 0, stream, ga,
                       g.ncb, const_cast<unsigned short *>(ga.tterms));
    if ((e = hipGetLastError()) != hipSuccess) return e;
    const dim3 grid((unsigned)((args.n + GROWS - 1) / GROWS), (unsigned)g.slices);
    switch (g.ncb) {
    case 1: hipLaunchKernelGGL(gradient_kernel<2>, grid, dim3(GW * 64), 0, stream, ga); break;
    case 2: hipLaunchKernelGGL(gradient_kernel<4>, grid, dim3(GW * 64), 0, stream, ga); break;
    case 3: hipLaunchKernelGGL(gradient_kernel<6>, grid, dim3(GW * 64), 0, stream, ga); break;
    default: hipLaunchKernelGGL(gradient_kernel<8>, grid, dim3(GW * 64), 0, stream, ga); break;
    }
    if ((e = hipGetLastError()) != hipSuccess) return e;
    // the rows that were left, over their slices
    args.left = ga.left;
    args.dxp = ga.dxp;
    e = launch_sweep<MODE_GRAD>(BW_EUCLID, args, g.sweep_slices, stream);
    if (e != hipSuccess || g.slices == 1) return e;
    // (sweep_slices > 1 here: gradient_applies)
    return launch_sum(ga.dxp, args.n, args.k, (int)g.slices, ga.left, g.sweep_slices, args.dx, args.lddx,
                      stream);
}

}  // namespace

namespace {

// Columns per wave of mds_small_kernel: few for few points, where there would be
// too few waves and each one's chain of loads would show (2000 x 2: 111 us with
// 128 columns a wave, 31 with 16; 16384 x 2: 229 with 128, 182 with 64).
int mds_jw(int64_t n) { return n <= 2500 ? 16 : n <= 6000 ? 32 : 64; }

// Its workgroups: row block ci has 64 / jw (ci + 1) column blocks.
int64_t mds_tiles(int64_t n)
{
    const int64_t ni = (n + MI - 1) / MI;
    return 64 / mds_jw(n) * (ni * (ni + 1) / 2);
}

// Few features: each pair once (mds_small_kernel).  Times in us, sweep and here:
// 16384 x 8 1738 and 502, 4000 x 6 125 and 70, 2000 x 6 42 and 41, 2000 x 8 42
// and 50; with 16 features its sums no longer fit the registers (4000: 128 and
// 329).
bool mds_small_applies(int64_t n, int64_t q) { return n >= 2 && (q <= 6 || (q <= 8 && n >= 3000)); }

// Slices of the rows as i (column blocks) and as j (row blocks).
int64_t mds_islices(int64_t n) { return 64 / mds_jw(n) * ((n + MI - 1) / MI); }

// Row blocks of a pass: all of them while the slices fit MDS_SLICE_BYTES (up to
// 32768 x 8), else what fits, at least one (65536 x 8: 6.59 ms with 1.07 GB in one
// pass, 7.30 with 128 MB, 6.84 with 256).
constexpr size_t MDS_SLICE_BYTES = (size_t)256 << 20;
size_t mds_slice_bytes(int64_t n, int64_t q, int64_t blocks)
{
    const int64_t ni = (n + MI - 1) / MI, irows = blocks == ni ? n : blocks * MI;
    return (size_t)(mds_islices(n) * irows + blocks * n) * (size_t)q * sizeof(float);
}
int64_t mds_pass_blocks(int64_t n, int64_t q)
{
    const int64_t ni = (n + MI - 1) / MI;
    if (mds_slice_bytes(n, q, ni) <= MDS_SLICE_BYTES) return ni;
    const int64_t blocks = (int64_t)(MDS_SLICE_BYTES / mds_slice_bytes(n, q, 1));
    return blocks < 1 ? 1 : blocks;
}

template <int Q>
void launch_mds_small(const MdsArgs &args, bool grad, hipStream_t stream)
{
    const dim3 grid((unsigned)(64 / args.jw * (args.c1 * (args.c1 + 1) / 2) - args.t0));
    if (grad)
        hipLaunchKernelGGL((mds_small_kernel<Q, true>), grid, dim3(256), 0, stream, args);
    else
        hipLaunchKernelGGL((mds_small_kernel<Q, false>), grid, dim3(256), 0, stream, args);
}

}  // namespace

int64_t mds_partials_count(int64_t n, int64_t q, bool lean)
{
    if (!lean && mds_small_applies(n, q)) return mds_tiles(n);
    return (n + BI - 1) / BI * j_splits(n, q);
}

static size_t sweep_workspace_bytes(int64_t n, int64_t k)
{
    if (n < 2 || k < 1) return 0;
    const int js = j_splits(n, k);
    return js > 1 ? (size_t)js * (size_t)n * (size_t)k * sizeof(float) : 0;
}

size_t mds_workspace_bytes(int64_t n, int64_t q, bool lean)
{
    if (!lean && mds_small_applies(n, q)) return mds_slice_bytes(n, q, mds_pass_blocks(n, q));
    return sweep_workspace_bytes(n, q);
}

size_t backward_workspace_bytes(int op, int64_t n, int64_t k, bool lean)
{
    if (n < 2 || k < 1) return 0;
    if (!lean && gradient_applies(op, n, k)) return gradient_plan(n, k).bytes;
    return sweep_workspace_bytes(n, k);
}

hipError_t launch_backward(int op, const float *x, int64_t n, int64_t k, int64_t ldx, float p,
                           const float *g_packed, float *dx, int64_t lddx, float *workspace,
                           bool lean, hipStream_t stream)
{
    if (n <= 0 || k <= 0) return hipSuccess;
    BwArgs args;
    args.x = x;
    args.n = n;
    args.k = k;
    args.ldx = ldx;
    args.g = g_packed;
    args.dx = dx;
    args.lddx = lddx;
    args.dxp = workspace;
    args.partials = nullptr;
    args.p = p;
    args.pm1 = p - 1.0f;
    args.left = nullptr;
    if (!lean && gradient_applies(op, n, k)) return launch_gradient(args, workspace, stream);
    const int bop = (op == OP_EUCLID) ? BW_EUCLID : (op == OP_MINK3) ? BW_MINK3 : BW_MINKP;
    return launch_mode<MODE_GRAD>(bop, args, stream);
}

hipError_t launch_mds(const float *y, int64_t n, int64_t q, int64_t ldy, const float *delta,
                      float *dy, int64_t lddy, double *stress, double *partials, float *workspace,
                      bool lean, hipStream_t stream)
{
    if (!lean && mds_small_applies(n, q)) {
        MdsArgs ma;
        ma.y = y;
        ma.n = n;
        ma.q = q;
        ma.ldy = ldy;
        ma.delta = delta;
        ma.jw = mds_jw(n);
        const int64_t ni = (n + MI - 1) / MI, blocks = dy ? mds_pass_blocks(n, q) : ni;
        for (int64_t c0 = 0; c0 < ni; c0 += blocks) {
            ma.c0 = c0;
            ma.c1 = c0 + blocks < ni ? c0 + blocks : ni;
            const int64_t end = ma.c1 * MI < n ? ma.c1 * MI : n;
            ma.irows = (int)(end - c0 * MI);
            ma.t0 = (int)(64 / ma.jw * (c0 * (c0 + 1) / 2));
            ma.partials = partials + ma.t0;
            ma.ipart = dy ? workspace - c0 * MI : nullptr;
            ma.jpart = dy ? workspace + mds_islices(n) * ma.irows * q - c0 * q * n : nullptr;
            switch (q) {
            case 1: launch_mds_small<1>(ma, dy != nullptr, stream); break;
            case 2: launch_mds_small<2>(ma, dy != nullptr, stream); break;
            case 3: launch_mds_small<3>(ma, dy != nullptr, stream); break;
            case 4: launch_mds_small<4>(ma, dy != nullptr, stream); break;
            case 5: case 6: launch_mds_small<6>(ma, dy != nullptr, stream); break;
            default: launch_mds_small<8>(ma, dy != nullptr, stream); break;
            }
            hipError_t e = hipGetLastError();
            if (e != hipSuccess) return e;
            const unsigned rows = dy ? (unsigned)((end + 256 / MSUM - 1) / (256 / MSUM)) : 0u;
            hipLaunchKernelGGL(mds_finish_kernel, dim3(rows + 1), dim3(256), 0, stream, ma, dy, lddy,
                               mds_tiles(n), ma.c1 == ni ? stress : nullptr);
            if ((e = hipGetLastError()) != hipSuccess) return e;
        }
        return hipSuccess;
    }
    BwArgs args;
    args.x = y;
    args.n = n;
    args.k = q;
    args.ldx = ldy;
    args.g = delta;
    args.dx = dy;
    args.lddx = lddy;
    args.dxp = workspace;
    args.partials = partials;
    args.p = 2.0f;
    args.pm1 = 1.0f;
    args.left = nullptr;
    hipError_t e = launch_mode<MODE_MDS>(BW_EUCLID, args, stream);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(reduce_partials_kernel, dim3(1), dim3(256), 0, stream, partials,
                       mds_partials_count(n, q, lean), stress);
    return hipGetLastError();
}

}  // namespace gt
