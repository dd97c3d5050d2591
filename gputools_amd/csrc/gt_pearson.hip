// gt_pearson.hip -- Pearson correlation of gpuCor(method = "pearson") on gfx950.
//
// Replaces pmcc (src/correlation.cpp:66-160) and its kernels
// (inst/cuda/correlation.cu:7-290).  gputools launches three kernels over an
// na x nb grid of 16-thread blocks, one block per pair, each re-reading both
// variables from global memory (means, then standard deviations, then the sum
// of standard-score products), and computes the t-scores on the host
// (correlation.cpp:51-64).
//
// use = "everything": every pair uses every sample, so means and standard
// deviations belong to the variables, not to the pairs.  A pre-pass
// standardises each variable once,
//     z = (v - mean) / sqrt(sum (v - mean)^2),
// and the correlation of a pair is the dot product z_x . z_y, which equals
// the reference's sum of standard-score products / (n - 1).  The dot products
// of a 256 x 256 tile of pairs run on the matrix cores with split-precision
// operands (gt_mfma.h), or in FP32 on the VALU (the plain distance tile with a
// dot-product term).
//
// use = "pairwise.complete.obs": a pair uses the samples where both values
// are present, so means and deviations are per pair.  The six sums a pair needs
// (count, two sums, three second moments of shifted values) are products of
// values, squares and presence masks: the matrix cores form them from split
// operands that a pre-pass lays out once (pmcc_moments_kernel).  Pairs whose
// moments cancel, or whose data is not finite, and calls without a workspace
// take a VALU tile kernel (pmcc_pairwise_kernel), which keeps the reference's
// two passes per pair where it must: counts and sums give the pair's means,
// then the centred second moments give the correlation
//     sum d_x d_y / (sqrt(sum d_x^2) sqrt(sum d_y^2)).
//
// Every path writes pairs, corr and hostSignif's t-score in one epilogue.
// With a == b (gpuCor(x)) only the tiles on and below the diagonal are
// computed and each value is stored at (x, y) and (y, x), so the result is
// exactly symmetric, as the reference's is.
#include "gt_common.h"
#include "gt_internal.h"
#include "gt_mfma.h"

#include <math.h>

namespace gt {
namespace {

// t-score of a correlation over npairs samples, operation by operation as
// hostSignif (src/correlation.cpp:51-64, CAP) or gpuSignif
// (inst/cuda/correlation.cu:292-310, no cap) compute it in FP32: IEEE
// division and square root, cor^2 rounded before the subtraction.
template <bool CAP>
__device__ __forceinline__ float t_score(float npairs, float cor)
{
    if (CAP && cor >= 0.999f) return 10000.0f;
    float c2 = cor * cor;
    asm volatile("" : "+v"(c2));
    return cor * sqrtf((npairs - 2.0f) / (1.0f - c2));
}

__device__ __forceinline__ float wave_sum(float v)
{
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) v += __shfl_xor(v, d, 64);
    return v;
}

__device__ __forceinline__ float wave_max(float v)
{
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) v = fmaxf(v, __shfl_xor(v, d, 64));
    return v;
}

// ---------------------------------------------------------------------------
// Pre-pass of use = "everything"
// ---------------------------------------------------------------------------
// z = (v - mean) / sqrt(sum (v - mean)^2), the mean and the sum over all dim
// samples (NaN in, NaN out; a constant variable gives 0 / 0 = NaN, as the
// reference's zero standard deviation does), and max |v - mean| for the FP16
// scale.  One wave per variable; the sums' order is the same in every form.
struct RowStats {
    float mean, root, mx;
};
__device__ __forceinline__ RowStats row_stats(const float *xr, int64_t dim)
{
    const int lane = threadIdx.x & 63;
    RowStats st;
    float s = 0.0f;
#pragma unroll 8
    for (int64_t c = lane; c < dim; c += 64) s += xr[c];
    st.mean = wave_sum(s) / (float)dim;
    float q = 0.0f, mx = 0.0f;
#pragma unroll 8
    for (int64_t c = lane; c < dim; c += 64) {
        const float d = xr[c] - st.mean;
        q = fmaf(d, d, q);
        mx = fmaxf(mx, fabsf(d));
    }
    st.root = sqrtf(wave_sum(q));
    st.mx = wave_max(mx);
    return st;
}

// z (n x dim) for the FP32 form
__global__ __launch_bounds__(256) void pmcc_zscore_kernel(const float *__restrict__ x, int64_t n,
                                                          int64_t dim, int64_t ldx, float *__restrict__ z)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (int64_t row = (int64_t)blockIdx.x * 4 + wave; row < n; row += (int64_t)gridDim.x * 4) {
        const float *xr = x + row * ldx;
        const RowStats st = row_stats(xr, dim);
        for (int64_t c = lane; c < dim; c += 64) z[row * dim + c] = (xr[c] - st.mean) / st.root;
    }
}

// The split forms: the terms of z in operand blocks (gt_mfma.h), samples
// dim..kp-1 zero.  FP16 scales z by a power of two that brings max |z| into
// [2^14, 2^15) and records the inverse.  `split` workgroups per block of 32
// variables: each finds the statistics, a wave per variable, and writes its
// share of the chunks, a wave per chunk, so that a store is a whole 1 KB
// block (few variables would otherwise leave CUs idle).  Rows past n fill
// their block with the last row; they only feed pairs that are never stored.
// Bound: memory (a read, then one from the caches, and six bytes out per
// value).  8192 x 1024, BF16: 25 us; a wave that wrote its own variable's
// 16-byte pieces of the blocks took 51.
constexpr int PTHREADS = 1024;
template <int PREP>
__global__ __launch_bounds__(PTHREADS) void pmcc_prep_kernel(const float *__restrict__ x, int64_t n,
                                                             int64_t dim, int64_t ldx, int64_t kp, int split,
                                                             bool vec,
                                                             unsigned short *__restrict__ terms,
                                                             float *__restrict__ iscale)
{
    constexpr int NT = Split<PREP>::NT;
    __shared__ float row_mean[32], row_root[32], row_scale[32];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 31, h = lane >> 5;
    const int64_t part = blockIdx.x % split, blocks = operand_rows(n) / 32;
    for (int64_t rb = blockIdx.x / split; rb < blocks; rb += gridDim.x / split) {
        __syncthreads();   // the last block's statistics are read
        for (int q = wave; q < 32; q += PTHREADS / 64) {
            const int64_t row = rb * 32 + q;
            const RowStats st = row_stats(x + (row < n ? row : n - 1) * ldx, dim);
            float sc = 1.0f;
            if (PREP == SPLIT_FP16) {
                const float m = st.mx / st.root;   // max |z|
                int e = 0;
                if (m > 0.0f && m < INFINITY) {
                    e = ilogbf(m);
                    e = e < -100 ? -100 : (e > 100 ? 100 : e);
                }
                sc = ldexpf(1.0f, 14 - e);
                if (lane == 0 && part == 0 && row < n) iscale[row] = ldexpf(1.0f, e - 14);
            }
            if (lane == 0) {
                row_mean[q] = st.mean;
                row_root[q] = st.root;
                row_scale[q] = sc;
            }
        }
        __syncthreads();
        const int64_t row = rb * 32 + r, nch = kp / OPERAND_K;
        const float *xr = x + (row < n ? row : n - 1) * ldx;
        const float mean = row_mean[r], root = row_root[r], sc = row_scale[r];
        for (int64_t ch = part * (PTHREADS / 64) + wave; ch < nch; ch += (int64_t)split * (PTHREADS / 64)) {
            const int64_t c0 = ch * OPERAND_K + h * 8;
            float v[8];
            if (vec && c0 + 8 <= dim) {
                const float4 a = *reinterpret_cast<const float4 *>(xr + c0);
                const float4 b = *reinterpret_cast<const float4 *>(xr + c0 + 4);
                v[0] = a.x, v[1] = a.y, v[2] = a.z, v[3] = a.w;
                v[4] = b.x, v[5] = b.y, v[6] = b.z, v[7] = b.w;
            } else {
#pragma unroll
                for (int c = 0; c < 8; ++c) v[c] = c0 + c < dim ? xr[c0 + c] : 0.0f;
            }
            unsigned short t[8][NT];
#pragma unroll
            for (int c = 0; c < 8; ++c)
                Split<PREP>::split(c0 + c < dim ? ((v[c] - mean) / root) * sc : 0.0f, t[c]);
            unsigned short *const out = terms + (rb * nch + ch) * NT * OPERAND_VALUES + lane * 8;
#pragma unroll
            for (int q = 0; q < NT; ++q) {
                uint4 w;
                w.x = t[0][q] | ((unsigned)t[1][q] << 16);
                w.y = t[2][q] | ((unsigned)t[3][q] << 16);
                w.z = t[4][q] | ((unsigned)t[5][q] << 16);
                w.w = t[6][q] | ((unsigned)t[7][q] << 16);
                *reinterpret_cast<uint4 *>(out + q * OPERAND_VALUES) = w;
            }
        }
    }
}

// ---------------------------------------------------------------------------
// MFMA tile of use = "everything": corr(x, y) = z_x . z_y.
// ---------------------------------------------------------------------------
constexpr int MBM = 256;        // side of a square of pairs (variables), two workgroups'
constexpr int MBK = 16;         // samples per main-loop chunk (one MFMA k-step)
constexpr int MKPAD = 32;       // split terms are zero-padded to a multiple of this
constexpr int MTHREADS = 512;   // 8 waves of 64 x 64 pairs
constexpr int MSUPER = 2;       // super-tile side in tiles (L2 locality)
constexpr int MBLOCKS = MBM / 2 * 3 / 32;   // operand blocks of one term, one chunk
constexpr int MNSTAGE = 2;

struct PmccTileArgs {
    const unsigned short *ta, *tb;   // split terms, in operand blocks (gt_mfma.h)
    int64_t na, nb, kp;
    const float *isa, *isb;          // FP16: inverse power-of-two scales
    float *corr, *ts, *pairs;
    int64_t ldo;
    float fpairs;                    // samples per pair (dim)
    int64_t super_b;                 // super-tiles along y (rectangular schedule)
    int64_t tiles_a, tiles_b;
    int64_t id_offset, ids_this;
};

// SYM: a == b; tiles with J <= I, values mirrored to (y, x).  VEC: ldo and the
// output pointers allow 16-byte mirrored stores.
// Two workgroups share a CU, so one's stores and waits lie under the other's
// products, and the last round of tiles is shorter: one workgroup of 16 waves
// on a 256 x 256 tile with a three-stage ring ran 8192 variables x 1024 samples
// (BF16, self) in 572 us, two of 8 waves on 256 x 128 with two stages in 491.
// Bound: the matrix cores (six products, 0.41 TFLOP: 361 us at the 1.14
// PFLOP/s of a large BF16 product) and 0.8 GB of results (117 us) beneath.
// Unaligned rows, 4001 x 201: 153 us with 4-byte mirrored stores, 111 as rows.
template <int SPLIT, bool SYM, bool VEC>
__global__ __launch_bounds__(MTHREADS, 4) void pmcc_tile_kernel(PmccTileArgs args)
{
    typedef typename Split<SPLIT>::vec vec;
    constexpr int NT = Split<SPLIT>::NT;
    // half a square: 256 x by 128 y where both (x, y) and (y, x) are stored; else
    // 128 x by 256 y, whose rows of results are longer (5671 x 3400 variables x 27
    // samples, FP16: 68 us with whole squares, 5% more with 128 y, 60 so)
    constexpr int TX = SYM ? MBM : MBM / 2, TY = SYM ? MBM / 2 : MBM, WAVES_Y = TY / 64;
    constexpr int STAGE = MBLOCKS * NT * OPERAND_BYTES;
    // after the main loop the stages hold each wave's transpose region for
    // the mirrored stores: 64 rows of MTRL floats
    constexpr int MTRL = 36;
    constexpr int TRBYTES = (MTHREADS / 64) * 64 * MTRL * 4;
    constexpr int SBYTES = MNSTAGE * STAGE > TRBYTES ? MNSTAGE * STAGE : TRBYTES;
    __shared__ __attribute__((aligned(1024))) unsigned char smem[SBYTES + (TX + TY) * 4];
    float *iA = reinterpret_cast<float *>(smem + SBYTES);
    float *iB = iA + TX;

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wr = wave / WAVES_Y, wc = wave % WAVES_Y;   // x rows wr*64.., y rows wc*64..

    // Super-tiled schedule: super-tile st covers MSUPER x MSUPER tiles; tiles
    // past the edge (or above the diagonal when SYM) exit at once.
    const int64_t gid = args.id_offset + xcd_remap(blockIdx.x, args.ids_this);
    const int64_t id = gid / 2;
    const int64_t st = id / (MSUPER * MSUPER);
    const int w = (int)(id % (MSUPER * MSUPER));
    int64_t SI, SJ;
    if (SYM) {
        int si, sj;
        tri_tile(st, si, sj);
        SI = si;
        SJ = sj;
    } else {
        SI = st / args.super_b;
        SJ = st % args.super_b;
    }
    const int64_t I = SI * MSUPER + w / MSUPER;
    const int64_t J = SJ * MSUPER + w % MSUPER;
    if (I >= args.tiles_a || J >= args.tiles_b || (SYM && J > I)) return;
    const int64_t x0 = I * MBM + (SYM ? 0 : (gid & 1) * TX), y0 = J * MBM + (SYM ? (gid & 1) * TY : 0);
    const int64_t na = args.na, nb = args.nb, kp = args.kp;
    if (x0 >= na || y0 >= nb) return;

    if (SPLIT == SPLIT_FP16) {
        if (tid < TX) {
            const int64_t r = x0 + tid;
            iA[tid] = r < na ? args.isa[r] : 1.0f;
        } else if (tid < TX + TY) {
            const int64_t r = y0 + (tid - TX);
            iB[tid - TX] = r < nb ? args.isb[r] : 1.0f;
        }
    }

    // ---- main loop: direct global -> LDS loads, MNSTAGE-deep, MFMA products
    // LDS chunk image: side x, then side y, 12 blocks of 32 rows together (8 + 4
    // where SYM, else 4 + 8), each NT terms of 1 KB as they lie in memory
    // (gt_mfma.h).  These pieces go to the 8 waves round robin, one per
    // instruction: global_load_lds writes lane l's 16 B at the wave's LDS base +
    // 16 l, and a lane's operand read is its own 16 B, free of bank conflicts.
    // Blocks past the last one repeat it: they only feed pairs that are never
    // stored.
    // (Row-major terms moved 32 bytes of 32 rows per instruction: 8192 x 1024
    // self, BF16, 643 -> 613 us.)
    typedef __attribute__((address_space(3))) void lds_void_t;
    typedef const __attribute__((address_space(1))) void gbl_void_t;
    constexpr int PIECES = MBLOCKS * NT, PMAX = (PIECES + 7) / 8;
    const unsigned short *gsrc[PMAX];
#pragma unroll
    for (int q = 0; q < PMAX; ++q) {
        const int p = min(wave + 8 * q, PIECES - 1), blk = p / NT;
        const int lside = blk >= TX / 32;
        const int64_t last = operand_rows(lside ? nb : na) / 32 - 1;
        const int64_t rb = lside ? y0 / 32 + blk - TX / 32 : x0 / 32 + blk;
        gsrc[q] = (lside ? args.tb : args.ta) +
                  ((rb < last ? rb : last) * (kp / OPERAND_K) * NT + p % NT) * OPERAND_VALUES + lane * 8;
    }
    auto issue = [&](int chunk) {
        const int g = chunk % MNSTAGE;
#pragma unroll
        for (int q = 0; q < PMAX; ++q)
            if (wave + 8 * q < PIECES)
                __builtin_amdgcn_global_load_lds(
                    (gbl_void_t *)(gsrc[q] + (int64_t)chunk * NT * OPERAND_VALUES),
                    (lds_void_t *)(smem + g * STAGE + (wave + 8 * q) * OPERAND_BYTES), 16, 0, 0);
    };
    const int roff = lane * 16;

    f32x16_t acc[2][2];
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[a][b][r] = 0.0f;

    const int nchunks = (int)(kp / MBK);
#pragma unroll
    for (int c = 0; c < MNSTAGE - 1; ++c)
        if (c < nchunks) issue(c);
    for (int c = 0; c < nchunks; ++c) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        // every wave's part of chunk c is in LDS and every wave finished chunk
        // c-1, whose stage the next issue overwrites
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (c + MNSTAGE - 1 < nchunks) issue(c + MNSTAGE - 1);
        const unsigned char *sg = smem + (c % MNSTAGE) * STAGE + roff;
        vec av[NT][2];
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int a = 0; a < 2; ++a)
                av[t][a] = *reinterpret_cast<const vec *>(sg + ((wr * 2 + a) * NT + t) * OPERAND_BYTES);
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            vec bv[NT];
#pragma unroll
            for (int t = 0; t < NT; ++t)
                bv[t] = *reinterpret_cast<const vec *>(sg + ((TX / 32 + wc * 2 + b) * NT + t) * OPERAND_BYTES);
#pragma unroll
            for (int a = 0; a < 2; ++a) {
                acc[a][b] = Split<SPLIT>::mfma(av[0][a], bv[0], acc[a][b]);
                acc[a][b] = Split<SPLIT>::mfma(av[0][a], bv[1], acc[a][b]);
                acc[a][b] = Split<SPLIT>::mfma(av[1][a], bv[0], acc[a][b]);
                if (NT == 3) {
                    acc[a][b] = Split<SPLIT>::mfma(av[0][a], bv[NT - 1], acc[a][b]);
                    acc[a][b] = Split<SPLIT>::mfma(av[NT - 1][a], bv[0], acc[a][b]);
                    acc[a][b] = Split<SPLIT>::mfma(av[1][a], bv[1], acc[a][b]);
                }
            }
        }
    }
    if (SPLIT == SPLIT_FP16) __syncthreads();   // iA / iB visible (written before the loop)

    // ---- epilogue: corr, t-score, pairs ------------------------------------
    // 32x32 accumulator layout: element r of lane l is x row 8(r/4) + 4(l/32)
    // + r%4 and y column l%32, so lanes 0..31 store 32 consecutive y of one x.
    const int ly0 = wc * 64 + (lane & 31);
    const float fp = args.fpairs;
    const int64_t ldo = args.ldo;
    float sb[2];
#pragma unroll
    for (int b = 0; b < 2; ++b) sb[b] = (SPLIT == SPLIT_FP16) ? iB[ly0 + b * 32] : 1.0f;
    // SYM: off-diagonal tiles store (x, y) and (y, x); diagonal tiles store
    // x >= y and mirror x > y, so the two halves are the same values
    const bool diag = SYM && (I == J);
    // off-diagonal tiles mirror through LDS: each wave writes its 64 x 32
    // block (one output, one a) transposed into its own region, then stores it
    // back as rows of 32 consecutive x (128 B per row), instead of 16-byte (or,
    // unaligned, 4-byte) pieces of 32 rows
    const bool fastm = SYM && !diag;
    const bool whole = x0 + TX <= na && y0 + TY <= nb;
    float *const tr = reinterpret_cast<float *>(smem) + wave * 64 * MTRL;
    // lane's four x (8 rq + 4 (lane >> 5) ..) of row (lane & 31) + 32 b
    auto tr_put = [&](int rq, int b, const float (&v)[4]) {
        *reinterpret_cast<float4 *>(tr + ((lane & 31) + 32 * b) * MTRL + 8 * rq + 4 * (lane >> 5)) =
            make_float4(v[0], v[1], v[2], v[3]);
    };
    // the wave's transposed 64 x 32 block out as rows of 32 x
    auto tr_store = [&](float *out, int a) {
        if (!VEC || !whole) {
#pragma unroll 4
            for (int it = 0; it < 32; ++it) {
                const int ly = 2 * it + (lane >> 5), lx = lane & 31;
                const int64_t y = y0 + wc * 64 + ly, x = x0 + wr * 64 + a * 32 + lx;
                if (x < na && y < nb) out[y * ldo + x] = tr[ly * MTRL + lx];
            }
            return;
        }
#pragma unroll
        for (int it = 0; it < 8; ++it) {
            const int ly = 8 * it + (lane >> 3), lx = (lane & 7) * 4;
            const float4 v = *reinterpret_cast<const float4 *>(tr + ly * MTRL + lx);
            *reinterpret_cast<float4 *>(out + (y0 + wc * 64 + ly) * ldo + x0 + wr * 64 + a * 32 + lx) = v;
        }
    };
#pragma unroll
    for (int a = 0; a < 2; ++a) {
        if (fastm) __syncthreads();   // the region's earlier reads (or the main loop's) are done
        float tva[4][2][4];
#pragma unroll
        for (int rq = 0; rq < 4; ++rq) {
            // the four x rows of this lane: lx0 .. lx0 + 3
            const int lx0 = wr * 64 + a * 32 + 8 * rq + 4 * (lane >> 5);
            float cv[2][4];
            float (&tv)[2][4] = tva[rq];
#pragma unroll
            for (int r4 = 0; r4 < 4; ++r4) {
                const int64_t x = x0 + lx0 + r4;
                const float sj = (SPLIT == SPLIT_FP16) ? iA[lx0 + r4] : 1.0f;
#pragma unroll
                for (int b = 0; b < 2; ++b) {
                    float g = acc[a][b][rq * 4 + r4];
                    // undo the scales one at a time (their product can overflow)
                    if (SPLIT == SPLIT_FP16) g = (g * sj) * sb[b];
                    cv[b][r4] = g;
                    tv[b][r4] = t_score<true>(fp, g);
                    const int64_t y = y0 + ly0 + b * 32;
                    if (x < na && y < nb && (!diag || x >= y)) {
                        const int64_t o = x * ldo + y;
                        args.corr[o] = g;
                        args.ts[o] = tv[b][r4];
                        args.pairs[o] = fp;
                    }
                }
            }
            if (fastm) {
#pragma unroll
                for (int b = 0; b < 2; ++b) tr_put(rq, b, cv[b]);
            } else if (SYM) {
                // the diagonal tile: (y, x) for the four x of this lane
#pragma unroll
                for (int b = 0; b < 2; ++b) {
                    const int64_t y = y0 + ly0 + b * 32;
                    const int64_t x = x0 + lx0;
                    if (y >= nb) continue;
                    const int64_t o = y * ldo + x;
#pragma unroll
                    for (int r4 = 0; r4 < 4; ++r4) {
                        if (x + r4 >= na || x + r4 <= y) continue;
                        args.corr[o + r4] = cv[b][r4];
                        args.ts[o + r4] = tv[b][r4];
                        args.pairs[o + r4] = fp;
                    }
                }
            }
        }
        if (fastm) {
            __syncthreads();
            tr_store(args.corr, a);
            __syncthreads();
#pragma unroll
            for (int rq = 0; rq < 4; ++rq)
#pragma unroll
                for (int b = 0; b < 2; ++b) tr_put(rq, b, tva[rq][b]);
            __syncthreads();
            tr_store(args.ts, a);
        }
    }
    if (fastm) {
        // pairs is one value: the wave's mirrored 64 x 64 block as rows
        if (!VEC || !whole) {
#pragma unroll 4
            for (int ly = 0; ly < 64; ++ly) {
                const int64_t y = y0 + wc * 64 + ly, x = x0 + wr * 64 + lane;
                if (x < na && y < nb) args.pairs[y * ldo + x] = fp;
            }
            return;
        }
#pragma unroll
        for (int it = 0; it < 16; ++it) {
            const int ly = 4 * it + (lane >> 4), lx = (lane & 15) * 4;
            *reinterpret_cast<float4 *>(args.pairs + (y0 + wc * 64 + ly) * ldo + x0 + wr * 64 + lx) =
                make_float4(fp, fp, fp, fp);
        }
    }
}

// ---------------------------------------------------------------------------
// VALU tile of use = "pairwise.complete.obs": two passes per pair.
// ---------------------------------------------------------------------------
constexpr int WBM = 64;        // variables per tile side
constexpr int WBK = 32;        // samples per LDS chunk
constexpr int WTHREADS = 256;  // 16 x 16 lanes, 4 x 4 pairs each
constexpr int WLD = WBM + 4;   // LDS row length (16-byte aligned rows)
// second moments whose squares neither overflowed nor lost bits that count (a
// sum of up to 2^24 of them)
constexpr float MOMENT_MIN = 0x1p-100f, MOMENT_MAX = 0x1p120f;

struct PairwiseArgs {
    const float *a;
    int64_t na, lda;
    const float *b;
    int64_t nb, ldb;
    int64_t dim;
    float *corr, *ts, *pairs;
    int64_t ldo;
    int64_t tiles_b;
    int64_t tile_offset, tiles_this;
    bool vec;   // ldo and the output pointers allow 16-byte stores
    // LEFT: the tiles to run (one byte per tile, 1 = left), and each variable's
    // power of two (pmcc_moments_prep_kernel)
    const uint8_t *left;
    const float *scale_a, *scale_b;
};

// A sample of a pair counts when both values are present (not NaN): counts
// and sums (gpuMeans, correlation.cu:7-51) give the pair's means, then the
// centred moments over the same samples (gpuSD and gpuPMCC,
// correlation.cu:53-150).  Masked samples are selected away, never multiplied
// by zero, so an Inf beside a missing value does not leak into the sums.
// Each chunk's sums are accumulated separately and then added to the totals.
// LEFT: only the tiles that pmcc_moments_kernel left, with two passes over the
// values as they are.  A variable's power of two fits its largest value, which a
// pair need not contain (one 1e30 beside ordinary values, missing in the
// partner, would scale the pair's squares to nothing).  The passes run again
// with it only where a variable of the tile is far from 1 in scale and a pair's
// squares over- or underflowed; such pairs take the scaled moments if those are
// in range.
template <bool SYM, bool LEFT>
__global__ __launch_bounds__(WTHREADS) void pmcc_pairwise_kernel(PairwiseArgs args)
{
    __shared__ float lds[2][WBK][WLD];   // [0] x side, [1] y side; sample-major
    const int tid = threadIdx.x;
    const int tx = tid & 15, ty = tid >> 4;   // y = 4 tx + j, x = 4 ty + i
    const int64_t t = args.tile_offset + xcd_remap(blockIdx.x, args.tiles_this);
    if (LEFT && args.left[t] == 0) return;
    int64_t I, J;
    if (SYM) {
        int ti, tj;
        tri_tile(t, ti, tj);
        I = ti;
        J = tj;
    } else {
        I = t / args.tiles_b;
        J = t % args.tiles_b;
    }
    const int64_t x0 = I * WBM, y0 = J * WBM;
    const int64_t dim = args.dim;

    // staging: variable tid >> 2, samples 8 (tid & 3) .. + 7 of the chunk;
    // samples past dim and variables past the end read as missing
    const int sv = tid >> 2, sk = (tid & 3) * 8;
    const bool va_ok = x0 + sv < args.na, vb_ok = y0 + sv < args.nb;
    const float *pa = args.a + (va_ok ? (x0 + sv) * args.lda : 0);
    const float *pb = args.b + (vb_ok ? (y0 + sv) * args.ldb : 0);
    const float qnan = __builtin_nanf("");
    float fa = 1.0f, fb = 1.0f;   // LEFT: factors of this lane's variables
    unsigned settled = 0;         // LEFT: the pairs whose moments were in range without factors
    float ra[8], rb[8];
    auto gload = [&](int64_t kb) {
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const int64_t kk = kb + sk + q;
            ra[q] = (va_ok && kk < dim) ? (LEFT ? pa[kk] * fa : pa[kk]) : qnan;
            rb[q] = (vb_ok && kk < dim) ? (LEFT ? pb[kk] * fb : pb[kk]) : qnan;
        }
    };
    auto stage = [&]() {
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            lds[0][sk + q][sv] = ra[q];
            lds[1][sk + q][sv] = rb[q];
        }
    };

    float cnt[4][4], qa[4][4], qb[4][4], qab[4][4];

    // ---- one pass ---------------------------------------------------------
    // Each variable is shifted by c, the mean of its present values in the
    // first chunk, and the pair's count and its five shifted sums come from
    // one pass: n = sum m_a m_b, Sa = sum a' m_b, Sb = sum m_a b',
    // Saa = sum a'^2 m_b, Sbb = sum m_a b'^2, Sab = sum a' b' (a' = a - c where
    // present, else 0).  The centred moments are then Saa - Sa^2 / n, ... .
    // Where that subtraction cancels (Caa <= Saa / 16: a subset mean far from
    // c, a constant subset, fewer than two samples) or a sum is not finite
    // (Inf in the data), the tile runs the two passes below instead.
    if constexpr (!LEFT) {
        __shared__ float lds1[3][2][WBK][WLD];   // a', a'^2, presence; [side]
        gload(0);
        float csum[2] = {0.0f, 0.0f}, ccnt[2] = {0.0f, 0.0f};
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            if (fabsf(ra[q]) < INFINITY) {
                csum[0] += ra[q];
                ccnt[0] += 1.0f;
            }
            if (fabsf(rb[q]) < INFINITY) {
                csum[1] += rb[q];
                ccnt[1] += 1.0f;
            }
        }
        // the four lanes of a variable are consecutive lanes of one wave
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            csum[h] += __shfl_xor(csum[h], 1, 64);
            ccnt[h] += __shfl_xor(ccnt[h], 1, 64);
            csum[h] += __shfl_xor(csum[h], 2, 64);
            ccnt[h] += __shfl_xor(ccnt[h], 2, 64);
        }
        const float ca = ccnt[0] > 0.0f ? csum[0] / ccnt[0] : 0.0f;
        const float cb = ccnt[1] > 0.0f ? csum[1] / ccnt[1] : 0.0f;

        float sa[4][4], sb[4][4], saa[4][4], sbb[4][4], sab[4][4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j)
                cnt[i][j] = sa[i][j] = sb[i][j] = saa[i][j] = sbb[i][j] = sab[i][j] = 0.0f;
        for (int64_t kb = 0; kb < dim; kb += WBK) {
            __syncthreads();
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                const bool pa_ = ra[q] == ra[q], pb_ = rb[q] == rb[q];
                const float da = pa_ ? ra[q] - ca : 0.0f, db = pb_ ? rb[q] - cb : 0.0f;
                lds1[0][0][sk + q][sv] = da;
                lds1[1][0][sk + q][sv] = da * da;
                lds1[2][0][sk + q][sv] = pa_ ? 1.0f : 0.0f;
                lds1[0][1][sk + q][sv] = db;
                lds1[1][1][sk + q][sv] = db * db;
                lds1[2][1][sk + q][sv] = pb_ ? 1.0f : 0.0f;
            }
            __syncthreads();
            if (kb + WBK < dim) gload(kb + WBK);
            // the second-moment sums are two-level (chunk partials, then
            // totals); Sa and Sb, small sums of shifted values that only
            // enter as Sa^2 / n, accumulate directly
            float p_aa[4][4], p_bb[4][4], p_ab[4][4];
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) p_aa[i][j] = p_bb[i][j] = p_ab[i][j] = 0.0f;
#pragma unroll 2
            for (int kc = 0; kc < WBK; ++kc) {
                const float4 av4 = *reinterpret_cast<const float4 *>(&lds1[0][0][kc][ty * 4]);
                const float4 aq4 = *reinterpret_cast<const float4 *>(&lds1[1][0][kc][ty * 4]);
                const float4 am4 = *reinterpret_cast<const float4 *>(&lds1[2][0][kc][ty * 4]);
                const float4 bv4 = *reinterpret_cast<const float4 *>(&lds1[0][1][kc][tx * 4]);
                const float4 bq4 = *reinterpret_cast<const float4 *>(&lds1[1][1][kc][tx * 4]);
                const float4 bm4 = *reinterpret_cast<const float4 *>(&lds1[2][1][kc][tx * 4]);
                const float av[4] = {av4.x, av4.y, av4.z, av4.w}, aq[4] = {aq4.x, aq4.y, aq4.z, aq4.w};
                const float am[4] = {am4.x, am4.y, am4.z, am4.w};
                const float bv[4] = {bv4.x, bv4.y, bv4.z, bv4.w}, bq[4] = {bq4.x, bq4.y, bq4.z, bq4.w};
                const float bm[4] = {bm4.x, bm4.y, bm4.z, bm4.w};
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        cnt[i][j] = fmaf(am[i], bm[j], cnt[i][j]);   // exact: small integers
                        sa[i][j] = fmaf(av[i], bm[j], sa[i][j]);
                        sb[i][j] = fmaf(am[i], bv[j], sb[i][j]);
                        p_aa[i][j] = fmaf(aq[i], bm[j], p_aa[i][j]);
                        p_bb[i][j] = fmaf(am[i], bq[j], p_bb[i][j]);
                        p_ab[i][j] = fmaf(av[i], bv[j], p_ab[i][j]);
                    }
            }
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    saa[i][j] += p_aa[i][j];
                    sbb[i][j] += p_bb[i][j];
                    sab[i][j] += p_ab[i][j];
                }
        }
        bool ill = false;
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float n = cnt[i][j];
                // Sa Sb / n with the product first, so (x, y) and (y, x) round alike
                qa[i][j] = saa[i][j] - sa[i][j] * sa[i][j] / n;
                qb[i][j] = sbb[i][j] - sb[i][j] * sb[i][j] / n;
                qab[i][j] = sab[i][j] - sa[i][j] * sb[i][j] / n;
                const bool inside = x0 + ty * 4 + i < args.na && y0 + tx * 4 + j < args.nb;
                ill = ill || (inside && !(qa[i][j] > saa[i][j] * 0.0625f && qb[i][j] > sbb[i][j] * 0.0625f));
            }
        if (__syncthreads_or(ill) == 0) goto finish;
    }

    // ---- two passes (tiles the one pass does not settle) -------------------
#pragma unroll 1
    for (int attempt = 0; attempt < (LEFT ? 2 : 1); ++attempt) {
        float s1[4][4], s2[4][4];
    #pragma unroll
        for (int i = 0; i < 4; ++i)
    #pragma unroll
            for (int j = 0; j < 4; ++j) cnt[i][j] = s1[i][j] = s2[i][j] = 0.0f;

        // pass 1: count, sum x, sum y over the pair's samples.  A chunk without
        // Inf uses products with 0/1 masks (x * 0 = 0 for finite x): one fma per
        // sum instead of a select and an add, with the same sums bit for bit; a
        // chunk with an Inf selects.
        gload(0);
        for (int64_t kb = 0; kb < dim; kb += WBK) {
            __syncthreads();
            stage();
            bool inf_here = false;
    #pragma unroll
            for (int q = 0; q < 8; ++q) inf_here = inf_here || __builtin_isinf(ra[q]) || __builtin_isinf(rb[q]);
            const bool any_inf = __syncthreads_or(inf_here) != 0;
            if (kb + WBK < dim) gload(kb + WBK);
            float p1[4][4], p2[4][4];
    #pragma unroll
            for (int i = 0; i < 4; ++i)
    #pragma unroll
                for (int j = 0; j < 4; ++j) p1[i][j] = p2[i][j] = 0.0f;
            if (!any_inf) {
    #pragma unroll 4
                for (int kc = 0; kc < WBK; ++kc) {
                    const float4 a4 = *reinterpret_cast<const float4 *>(&lds[0][kc][ty * 4]);
                    const float4 b4 = *reinterpret_cast<const float4 *>(&lds[1][kc][tx * 4]);
                    const float av[4] = {a4.x, a4.y, a4.z, a4.w};
                    const float bv[4] = {b4.x, b4.y, b4.z, b4.w};
                    float am[4], a0[4], bm[4], b0[4];
    #pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        am[i] = av[i] == av[i] ? 1.0f : 0.0f;
                        a0[i] = av[i] == av[i] ? av[i] : 0.0f;
                        bm[i] = bv[i] == bv[i] ? 1.0f : 0.0f;
                        b0[i] = bv[i] == bv[i] ? bv[i] : 0.0f;
                    }
    #pragma unroll
                    for (int i = 0; i < 4; ++i)
    #pragma unroll
                        for (int j = 0; j < 4; ++j) {
                            cnt[i][j] = fmaf(am[i], bm[j], cnt[i][j]);
                            p1[i][j] = fmaf(a0[i], bm[j], p1[i][j]);
                            p2[i][j] = fmaf(b0[j], am[i], p2[i][j]);
                        }
                }
            } else {
    #pragma unroll 4
                for (int kc = 0; kc < WBK; ++kc) {
                    const float4 a4 = *reinterpret_cast<const float4 *>(&lds[0][kc][ty * 4]);
                    const float4 b4 = *reinterpret_cast<const float4 *>(&lds[1][kc][tx * 4]);
                    const float av[4] = {a4.x, a4.y, a4.z, a4.w};
                    const float bv[4] = {b4.x, b4.y, b4.z, b4.w};
    #pragma unroll
                    for (int i = 0; i < 4; ++i)
    #pragma unroll
                        for (int j = 0; j < 4; ++j) {
                            const bool m = (av[i] == av[i]) && (bv[j] == bv[j]);
                            cnt[i][j] += m ? 1.0f : 0.0f;
                            p1[i][j] += m ? av[i] : 0.0f;
                            p2[i][j] += m ? bv[j] : 0.0f;
                        }
                }
            }
    #pragma unroll
            for (int i = 0; i < 4; ++i)
    #pragma unroll
                for (int j = 0; j < 4; ++j) {
                    s1[i][j] += p1[i][j];
                    s2[i][j] += p2[i][j];
                }
        }
        // the pair's means (0 / 0 = NaN for a pair without samples: its result
        // is set below)
    #pragma unroll
        for (int i = 0; i < 4; ++i)
    #pragma unroll
            for (int j = 0; j < 4; ++j) {
                s1[i][j] = s1[i][j] / cnt[i][j];
                s2[i][j] = s2[i][j] / cnt[i][j];
            }

        // pass 2: sum dx^2, sum dy^2, sum dx dy
    #pragma unroll
        for (int i = 0; i < 4; ++i)
    #pragma unroll
            for (int j = 0; j < 4; ++j) qa[i][j] = qb[i][j] = qab[i][j] = 0.0f;
        gload(0);
        for (int64_t kb = 0; kb < dim; kb += WBK) {
            __syncthreads();
            stage();
            __syncthreads();
            if (kb + WBK < dim) gload(kb + WBK);
            float pa2[4][4], pb2[4][4], pab[4][4];
    #pragma unroll
            for (int i = 0; i < 4; ++i)
    #pragma unroll
                for (int j = 0; j < 4; ++j) pa2[i][j] = pb2[i][j] = pab[i][j] = 0.0f;
    #pragma unroll 2
            for (int kc = 0; kc < WBK; ++kc) {
                const float4 a4 = *reinterpret_cast<const float4 *>(&lds[0][kc][ty * 4]);
                const float4 b4 = *reinterpret_cast<const float4 *>(&lds[1][kc][tx * 4]);
                const float av[4] = {a4.x, a4.y, a4.z, a4.w};
                const float bv[4] = {b4.x, b4.y, b4.z, b4.w};
    #pragma unroll
                for (int i = 0; i < 4; ++i)
    #pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const bool m = (av[i] == av[i]) && (bv[j] == bv[j]);
                        const float d = m ? av[i] - s1[i][j] : 0.0f;
                        const float e = m ? bv[j] - s2[i][j] : 0.0f;
                        pa2[i][j] = fmaf(d, d, pa2[i][j]);
                        pb2[i][j] = fmaf(e, e, pb2[i][j]);
                        pab[i][j] = fmaf(d, e, pab[i][j]);
                    }
            }
    #pragma unroll
            for (int i = 0; i < 4; ++i)
    #pragma unroll
                for (int j = 0; j < 4; ++j) {
                    qa[i][j] += pa2[i][j];
                    qb[i][j] += pb2[i][j];
                    qab[i][j] += pab[i][j];
                }
        }
        if constexpr (LEFT) {
            // the first attempt's correlations, if there is a second
            __shared__ float kept[16][WTHREADS];
            unsigned in_range = 0;
            bool again = false;
    #pragma unroll
            for (int i = 0; i < 4; ++i)
    #pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const bool ok = qa[i][j] >= MOMENT_MIN && qa[i][j] <= MOMENT_MAX &&
                                    qb[i][j] >= MOMENT_MIN && qb[i][j] <= MOMENT_MAX;   // (not for NaN)
                    in_range |= ok ? 1u << (i * 4 + j) : 0u;
                    const bool inside = x0 + ty * 4 + i < args.na && y0 + tx * 4 + j < args.nb;
                    again = again || (inside && !ok);
                }
            if (attempt > 0) {
    #pragma unroll
                for (int i = 0; i < 4; ++i)
    #pragma unroll
                    for (int j = 0; j < 4; ++j)
                        if (((in_range & ~settled) >> (i * 4 + j) & 1u) == 0) {
                            qab[i][j] = kept[i * 4 + j][tid];
                            qa[i][j] = qb[i][j] = 1.0f;
                        }
                break;
            }
            settled = in_range;
            fa = va_ok ? args.scale_a[x0 + sv] : 1.0f;
            fb = vb_ok ? args.scale_b[y0 + sv] : 1.0f;
            // (with every largest value within 2^+-40, no sum overflows, and
            // factors would not bring back what underflows)
            const bool far = !(fa >= 0x1p-40f && fa <= 0x1p40f && fb >= 0x1p-40f && fb <= 0x1p40f);
            if (__syncthreads_or(far) == 0 || __syncthreads_or(again) == 0) break;
    #pragma unroll
            for (int i = 0; i < 4; ++i)
    #pragma unroll
                for (int j = 0; j < 4; ++j)
                    kept[i * 4 + j][tid] = qab[i][j] / (sqrtf(qa[i][j]) * sqrtf(qb[i][j]));
        }
    }

finish:
    // epilogue: no samples gives the reference's 0 / (0 - 1) = -0
    const bool mirror = SYM && (I != J);
    float rv[4][4], tv[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float c = cnt[i][j];
            rv[i][j] = (c == 0.0f) ? -0.0f : qab[i][j] / (sqrtf(qa[i][j]) * sqrtf(qb[i][j]));
            tv[i][j] = t_score<true>(c, rv[i][j]);
        }
    // a lane's 4 x 4 pairs are four consecutive y per x (and four
    // consecutive x per y): 16-byte stores where the rows allow them
    const bool vec = args.vec && x0 + WBM <= args.na && y0 + WBM <= args.nb;
    if (vec) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int64_t o = (x0 + ty * 4 + i) * args.ldo + y0 + tx * 4;
            *reinterpret_cast<float4 *>(args.corr + o) = make_float4(rv[i][0], rv[i][1], rv[i][2], rv[i][3]);
            *reinterpret_cast<float4 *>(args.ts + o) = make_float4(tv[i][0], tv[i][1], tv[i][2], tv[i][3]);
            *reinterpret_cast<float4 *>(args.pairs + o) =
                make_float4(cnt[i][0], cnt[i][1], cnt[i][2], cnt[i][3]);
        }
        if (mirror) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int64_t o = (y0 + tx * 4 + j) * args.ldo + x0 + ty * 4;
                *reinterpret_cast<float4 *>(args.corr + o) = make_float4(rv[0][j], rv[1][j], rv[2][j], rv[3][j]);
                *reinterpret_cast<float4 *>(args.ts + o) = make_float4(tv[0][j], tv[1][j], tv[2][j], tv[3][j]);
                *reinterpret_cast<float4 *>(args.pairs + o) =
                    make_float4(cnt[0][j], cnt[1][j], cnt[2][j], cnt[3][j]);
            }
        }
        return;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int64_t x = x0 + ty * 4 + i;
        if (x >= args.na) continue;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int64_t y = y0 + tx * 4 + j;
            if (y >= args.nb) continue;
            const int64_t o = x * args.ldo + y;
            args.corr[o] = rv[i][j];
            args.ts[o] = tv[i][j];
            args.pairs[o] = cnt[i][j];
            if (mirror) {
                const int64_t om = y * args.ldo + x;
                args.corr[om] = rv[i][j];
                args.ts[om] = tv[i][j];
                args.pairs[om] = cnt[i][j];
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Matrix-core form of use = "pairwise.complete.obs"
// ---------------------------------------------------------------------------
// Per variable and sample seven BF16 values, in operand blocks (gt_mfma.h, NT =
// 7): the shifted and scaled value a' in three terms, its FP32 square q in three
// terms (both splits are exact), the presence mask m.  Missing samples, samples
// past dim and rows past the last variable are zero in all seven.  The shift c
// is the mean of the present values among the first 32 samples; the scale is
// the power of two that brings max |v - c| to [1, 2), so that the terms stay
// clear of the denormal range.  A pair need not contain that largest value:
// where its own squares are below MOMENTS_FLOOR on average, their terms run into
// the denormal range, and the pair is left to the two passes.
constexpr int QT = 7;
constexpr float MOMENTS_FLOOR = 0x1p-90f;
enum { Q_VALUE = 0, Q_SQUARE = 3, Q_MASK = 6 };
constexpr int QTHREADS = 1024;

// `split` workgroups per block of 32 variables: each finds the shift and the
// scale from all samples and writes its share of the chunks (few variables
// would otherwise leave CUs idle).  Lane 32 h + r of a wave reads samples 8 h
// .. + 7 of 16 of variable r.  Also clears `left`.
__global__ __launch_bounds__(QTHREADS) void pmcc_moments_prep_kernel(const float *__restrict__ x, int64_t n,
                                                                     int64_t dim, int64_t ldx, int64_t nch,
                                                                     int split,
                                                                     unsigned short *__restrict__ terms,
                                                                     float *__restrict__ scales,
                                                                     uint8_t *__restrict__ left, int64_t nleft)
{
    __shared__ float row_shift[32], row_scale[32];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 31, h = lane >> 5;
    for (int64_t t = (int64_t)blockIdx.x * QTHREADS + threadIdx.x; t < nleft;
         t += (int64_t)gridDim.x * QTHREADS)
        left[t] = 0;
    const int64_t rb = blockIdx.x / split, part = blockIdx.x % split;
    // shift and scale, a wave per variable
    for (int q = wave; q < 32; q += QTHREADS / 64) {
        const int64_t row = rb * 32 + q;
        float shift = 0.0f, m = 0.0f;
        if (row < n) {
            const float *xr = x + row * ldx;
            const float first = lane < 32 && lane < dim ? xr[lane] : __builtin_nanf("");
            const bool present = fabsf(first) < INFINITY;
            const float s = wave_sum(present ? first : 0.0f), c = wave_sum(present ? 1.0f : 0.0f);
            shift = c > 0.0f ? s / c : 0.0f;
#pragma unroll 4
            for (int64_t k = lane; k < dim; k += 64) {
                const float d = fabsf(xr[k] - shift);
                if (d < INFINITY) m = fmaxf(m, d);
            }
            m = wave_max(m);
        }
        if (lane == 0) {
            int e = m > 0.0f ? ilogbf(m) : 0;
            e = e < -120 ? -120 : (e > 120 ? 120 : e);
            row_shift[q] = shift;
            row_scale[q] = ldexpf(1.0f, -e);
            if (part == 0 && row < n) scales[row] = row_scale[q];
        }
    }
    __syncthreads();
    const int64_t row = rb * 32 + r;
    const bool in = row < n;
    const float *xr = x + (in ? row : 0) * ldx;
    const float shift = row_shift[r], scale = row_scale[r];
    float v[8];
    auto load = [&](int64_t ch) {
        const int64_t k0 = ch * OPERAND_K + h * 8;
#pragma unroll
        for (int k = 0; k < 8; ++k) v[k] = (in && k0 + k < dim) ? xr[k0 + k] : __builtin_nanf("");
    };
    for (int64_t ch = part * (QTHREADS / 64) + wave; ch < nch; ch += (int64_t)split * (QTHREADS / 64)) {
        load(ch);
        unsigned short t[8][QT];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const bool present = v[k] == v[k];
            const float d = present ? (v[k] - shift) * scale : 0.0f;
            Split<SPLIT_BF16>::split(d, t[k] + Q_VALUE);
            Split<SPLIT_BF16>::split(d * d, t[k] + Q_SQUARE);
            t[k][Q_MASK] = present ? 0x3f80 : 0;   // BF16 1.0
        }
        unsigned short *const out = terms + (rb * nch + ch) * QT * OPERAND_VALUES + lane * 8;
#pragma unroll
        for (int q = 0; q < QT; ++q) {
            uint4 w;
            w.x = t[0][q] | ((unsigned)t[1][q] << 16);
            w.y = t[2][q] | ((unsigned)t[3][q] << 16);
            w.z = t[4][q] | ((unsigned)t[5][q] << 16);
            w.w = t[6][q] | ((unsigned)t[7][q] << 16);
            *reinterpret_cast<uint4 *>(out + q * OPERAND_VALUES) = w;
        }
    }
}

constexpr double MOMENTS_MAX_BYTES = 1073741824.0;

constexpr int QBM = WBM;                 // variables per tile side
constexpr int QWAVES = 4;                // 2 (x) x 2 (y), 32 x 32 pairs each
constexpr int QSTAGE = 2 * QBM / 32 * QT * OPERAND_BYTES;   // one chunk of 16 samples (28 KB)
constexpr int QNSTAGE = 2;
constexpr int QTRL = 33;                 // row of a wave's transposed 32 x 32 block

struct MomentsArgs {
    const unsigned short *ta, *tb;   // operand blocks of pmcc_moments_prep_kernel
    int64_t na, nb;
    int nch, fold;                   // chunks, chunks per partial second moment
    float *corr, *ts, *pairs;
    int64_t ldo;
    uint8_t *left;                   // per WBM x WBM tile: a pair here is left to two passes
    int64_t tiles_b;                 // tiles along y (rectangular schedule)
    int64_t id_offset, ids_this;
};

// A 64 x 64 tile of pairs; the operand blocks stream through a two-stage LDS
// ring (direct loads).  A wave
// holds 32 x 32 pairs: n = m m', Sa = a m', Sb = m b', Saa = q m', Sbb = m q'
// and Sab = a b' take 1, 3, 3, 3, 3 and 6 products of 16 samples, all with
// FP32 accumulation.  The second moments are two-level sums: `fold` chunks in
// the accumulator, then added to a total, which keeps their error at that of
// the VALU form's two levels.  With two levels and six sums a 32 x 32 block
// takes 144 registers, which is what sets the tile.
// Two workgroups share a CU, so one's waits lie under the other's products.
// Bound: the matrix cores (19 products, 0.9 PFLOP/s of a measured 1.1 for a
// large BF16 product).  4001 variables x 777 samples, self case: 1.14 ms on
// the VALU (6 fused products per pair and sample), 0.28 ms here; 128 x 64
// tiles of 8 waves, one workgroup per CU, took 0.34 ms (five rounds of tiles,
// the last nearly empty).
// SYM: a == b; tiles on and below the diagonal, each pair stored twice.
template <bool SYM>
__global__ __launch_bounds__(QWAVES * 64, 2) void pmcc_moments_kernel(MomentsArgs args)
{
    typedef Split<SPLIT_BF16> S;
    __shared__ __attribute__((aligned(1024))) unsigned char smem[QNSTAGE * QSTAGE];
    static_assert(QWAVES * 32 * QTRL * 4 <= (int)sizeof(smem), "transpose regions");
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wx = wave >> 1, wy = wave & 1;
    const int64_t t = args.id_offset + xcd_remap(blockIdx.x, args.ids_this);
    int64_t I, J;
    if (SYM) {
        int ti, tj;
        tri_tile(t, ti, tj);
        I = ti;
        J = tj;
    } else {
        I = t / args.tiles_b;
        J = t % args.tiles_b;
    }
    const int64_t x0 = I * QBM + wx * 32, y0 = J * QBM + wy * 32;   // this wave's pairs
    const int64_t na = args.na, nb = args.nb;
    const int nch = args.nch;

    typedef __attribute__((address_space(3))) void lds_void_t;
    typedef const __attribute__((address_space(1))) void gbl_void_t;
    // wave w moves block w: side x in waves 0 and 1, side y in 2 and 3
    const unsigned short *src;
    {
        const bool sb = wave >= 2;
        const int64_t last = operand_rows(sb ? nb : na) / 32 - 1;
        int64_t rb = (sb ? J : I) * (QBM / 32) + (wave & 1);
        if (rb > last) rb = last;   // only feeds pairs that are not stored
        src = (sb ? args.tb : args.ta) + rb * nch * QT * OPERAND_VALUES + lane * 8;
    }
    auto issue = [&](int c) {
        unsigned char *const st = smem + (c % QNSTAGE) * QSTAGE + wave * QT * OPERAND_BYTES;
#pragma unroll
        for (int q = 0; q < QT; ++q)
            __builtin_amdgcn_global_load_lds((gbl_void_t *)(src + ((int64_t)c * QT + q) * OPERAND_VALUES),
                                             (lds_void_t *)(st + q * OPERAND_BYTES), 16, 0, 0);
    };
    // blocks above the diagonal or past the end only help to load
    const bool idle = x0 >= na || y0 >= nb || (SYM && y0 > x0);

    f32x16_t cn, sa, sb, paa, pbb, pab, saa, sbb, sab;
#pragma unroll
    for (int r = 0; r < 16; ++r)
        cn[r] = sa[r] = sb[r] = paa[r] = pbb[r] = pab[r] = saa[r] = sbb[r] = sab[r] = 0.0f;

#pragma unroll
    for (int c = 0; c < QNSTAGE - 1; ++c)
        if (c < nch) issue(c);
    int folded = 0;
    for (int c = 0; c < nch; ++c) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        // every wave's part of chunk c is in LDS, and every wave is done with
        // chunk c - 1, whose stage the next issue overwrites
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (c + QNSTAGE - 1 < nch) issue(c + QNSTAGE - 1);
        if (idle) continue;
        const unsigned char *const st = smem + (c % QNSTAGE) * QSTAGE + lane * 16;
        bf16x8_t av[QT], bv[QT];
#pragma unroll
        for (int q = 0; q < QT; ++q) {
            av[q] = *reinterpret_cast<const bf16x8_t *>(st + (wx * QT + q) * OPERAND_BYTES);
            bv[q] = *reinterpret_cast<const bf16x8_t *>(st + ((QBM / 32 + wy) * QT + q) * OPERAND_BYTES);
        }
        cn = S::mfma(av[Q_MASK], bv[Q_MASK], cn);
#pragma unroll
        for (int q = 2; q >= 0; --q) {
            sa = S::mfma(av[Q_VALUE + q], bv[Q_MASK], sa);
            sb = S::mfma(av[Q_MASK], bv[Q_VALUE + q], sb);
            paa = S::mfma(av[Q_SQUARE + q], bv[Q_MASK], paa);
            pbb = S::mfma(av[Q_MASK], bv[Q_SQUARE + q], pbb);
            // the products of three terms down to 2^-16: 1 1, 0 2, 2 0, 0 1, 1 0, 0 0
            if (q == 2) {
                pab = S::mfma(av[Q_VALUE + 1], bv[Q_VALUE + 1], pab);
                pab = S::mfma(av[Q_VALUE], bv[Q_VALUE + 2], pab);
            } else if (q == 1) {
                pab = S::mfma(av[Q_VALUE + 2], bv[Q_VALUE], pab);
                pab = S::mfma(av[Q_VALUE], bv[Q_VALUE + 1], pab);
            } else {
                pab = S::mfma(av[Q_VALUE + 1], bv[Q_VALUE], pab);
                pab = S::mfma(av[Q_VALUE], bv[Q_VALUE], pab);
            }
        }
        if (++folded == args.fold || c + 1 == nch) {
            folded = 0;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                saa[r] += paa[r];
                sbb[r] += pbb[r];
                sab[r] += pab[r];
                paa[r] = pbb[r] = pab[r] = 0.0f;
            }
        }
    }
    // the stages become the transpose regions
    __syncthreads();
    if (idle) return;

    // 32 x 32 accumulator layout: element r of lane l is x row 8 (r / 4) +
    // 4 (l / 32) + r % 4 and y column l % 32
    const bool diag = SYM && x0 == y0;
    const int64_t y = y0 + (lane & 31);
    bool ill = false;
    float rv[16], tv[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int64_t x = x0 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
        const float n = cn[r];
        // Sa Sb / n with the product first, so (x, y) and (y, x) round alike
        const float qa = saa[r] - sa[r] * sa[r] / n;
        const float qb = sbb[r] - sb[r] * sb[r] / n;
        const float qab = sab[r] - sa[r] * sb[r] / n;
        const bool inside = x < na && y < nb && (!diag || x >= y);
        ill = ill || (inside && !(qa > saa[r] * 0.0625f && qb > sbb[r] * 0.0625f &&
                                  fminf(saa[r], sbb[r]) >= n * MOMENTS_FLOOR));
        rv[r] = qab / (sqrtf(qa) * sqrtf(qb));
        tv[r] = t_score<true>(n, rv[r]);
        if (inside) {
            const int64_t o = x * args.ldo + y;
            args.corr[o] = rv[r];
            args.ts[o] = tv[r];
            args.pairs[o] = n;
        }
    }
    if (__builtin_amdgcn_ballot_w64(ill) != 0 && lane == 0) args.left[t] = 1;
    if (!SYM) return;
    // the mirrored block, transposed through this wave's own LDS region, as
    // rows of 32 consecutive x
    float *const tr = reinterpret_cast<float *>(smem) + wave * 32 * QTRL;
    auto mirror = [&](const float (&v)[16], float *out) {
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int r = 0; r < 16; ++r)
            tr[(lane & 31) * QTRL + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3)] = v[r];
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int it = 0; it < 16; ++it) {
            const int ly = 2 * it + (lane >> 5), lx = lane & 31;
            if (y0 + ly < nb && x0 + lx < na && (!diag || lx > ly))
                out[(y0 + ly) * args.ldo + x0 + lx] = tr[ly * QTRL + lx];
        }
    };
    float nv[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) nv[r] = cn[r];
    mirror(rv, args.corr);
    mirror(tv, args.ts);
    mirror(nv, args.pairs);
}

// ---------------------------------------------------------------------------
// Elementwise kernels
// ---------------------------------------------------------------------------

// t-scores and counts beside a correlation matrix the FP32 dot-product tiles
// wrote (use = "everything": every pair has fpairs samples).
__global__ void pmcc_finish_kernel(const float *__restrict__ corr, float *__restrict__ ts,
                                   float *__restrict__ pairs, int64_t na, int64_t nb, int64_t ldo,
                                   float fpairs)
{
    const int64_t total = na * nb;
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < total;
         e += (int64_t)gridDim.x * blockDim.x) {
        const int64_t o = (e / nb) * ldo + e % nb;
        ts[o] = t_score<true>(fpairs, corr[o]);
        pairs[o] = fpairs;
    }
}

// dim == 0: no samples, corr = 0 / (0 - 1) = -0 for every pair.
__global__ void pmcc_empty_kernel(float *__restrict__ corr, float *__restrict__ ts,
                                  float *__restrict__ pairs, int64_t na, int64_t nb, int64_t ldo)
{
    const int64_t total = na * nb;
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < total;
         e += (int64_t)gridDim.x * blockDim.x) {
        const int64_t o = (e / nb) * ldo + e % nb;
        corr[o] = -0.0f;
        ts[o] = t_score<true>(0.0f, -0.0f);
        pairs[o] = 0.0f;
    }
}

// gpuSignif (inst/cuda/correlation.cu:292-310): t-scores without the cap.
__global__ void ttest_kernel(const float *__restrict__ pairs, const float *__restrict__ corr,
                             float *__restrict__ ts, int64_t n)
{
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < n;
         e += (int64_t)gridDim.x * blockDim.x)
        ts[e] = t_score<false>(pairs[e], corr[e]);
}

unsigned grid_for(int64_t total, int threads)
{
    int64_t blocks = (total + threads - 1) / threads;
    if (blocks > 65536) blocks = 65536;
    if (blocks < 1) blocks = 1;
    return (unsigned)blocks;
}

size_t align256(size_t v) { return (v + 255) / 256 * 256; }

int64_t padded_dim(int64_t dim) { return (dim + MKPAD - 1) / MKPAD * MKPAD; }

int prep_terms(int precision) { return precision == 1 ? 3 : 2; }

// Workspace layout of use = "everything": the standardised variables of a,
// then (unless same) of b.  FP32: z rows; split forms: terms, then inverse
// scales.
struct PmccWs {
    unsigned short *ta = nullptr, *tb = nullptr;
    float *isa = nullptr, *isb = nullptr, *za = nullptr, *zb = nullptr;
};

size_t side_bytes(int precision, int64_t rows, int64_t dim)
{
    if (precision == 0) return align256((size_t)rows * (size_t)dim * sizeof(float));
    return align256((size_t)prep_terms(precision) * (size_t)operand_rows(rows) *
                    (size_t)padded_dim(dim) * sizeof(unsigned short)) +
           align256((size_t)rows * sizeof(float));
}

// The form that computes a call of use = "everything": the split terms are laid
// out for variables in multiples of 32, so a few long variables would take up to
// 32 times their bytes (2 x 10^8 samples 19 GB, BF16).  Where the rounding adds
// half of them again and more than 256 MB (one tile of few variables then), the
// FP32 form does the work, in 4 bytes a value: its products and sums are no less
// exact (see the sums of gt_plain.hip), and such a call takes about as long (20
// variables x 100000: 3.7 ms, BF16 5.9, FP16 3.4).
int everything_form(int precision, int64_t na, int64_t nb, bool same, int64_t dim)
{
    if (precision == 0) return 0;
    const double value = 2.0 * prep_terms(precision) * (double)padded_dim(dim);
    const double rows = (double)na + (same ? 0.0 : (double)nb);
    const double rounded = (double)operand_rows(na) + (same ? 0.0 : (double)operand_rows(nb));
    return rounded >= 1.5 * rows && (rounded - rows) * value > 268435456.0 ? 0 : precision;
}

PmccWs carve(int precision, int64_t na, int64_t nb, bool same, int64_t dim, void *ws)
{
    PmccWs w;
    char *p = static_cast<char *>(ws);
    auto side = [&](int64_t rows, unsigned short *&t, float *&is, float *&z) {
        if (precision == 0) {
            z = reinterpret_cast<float *>(p);
        } else {
            t = reinterpret_cast<unsigned short *>(p);
            is = reinterpret_cast<float *>(
                p + align256((size_t)prep_terms(precision) * (size_t)operand_rows(rows) *
                             (size_t)padded_dim(dim) * sizeof(unsigned short)));
        }
        p += side_bytes(precision, rows, dim);
    };
    side(na, w.ta, w.isa, w.za);
    if (same) {
        w.tb = w.ta;
        w.isb = w.isa;
        w.zb = w.za;
    } else {
        side(nb, w.tb, w.isb, w.zb);
    }
    return w;
}

hipError_t launch_prep(int precision, const float *x, int64_t n, int64_t dim, int64_t ldx,
                       unsigned short *terms, float *iscale, float *z, hipStream_t stream)
{
    if (precision == 0) {
        int64_t blocks = (n + 3) / 4;
        if (blocks > 65536) blocks = 65536;
        hipLaunchKernelGGL(pmcc_zscore_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, x, n, dim, ldx, z);
        return hipGetLastError();
    }
    // workgroups per block of 32 variables: to fill the CUs, while each has a
    // chunk per wave
    const int64_t kp = padded_dim(dim), blocks = operand_rows(n) / 32;
    int64_t split = 256 / (blocks > 0 ? blocks : 1), most = kp / OPERAND_K / (PTHREADS / 64);
    if (split > most) split = most;
    if (split < 1) split = 1;
    const bool vec = ldx % 4 == 0 && (reinterpret_cast<uintptr_t>(x) & 15) == 0;
    const dim3 grid((unsigned)((blocks < 65536 ? blocks : 65536) * split));
    if (precision == 1)
        hipLaunchKernelGGL(pmcc_prep_kernel<SPLIT_BF16>, grid, dim3(PTHREADS), 0, stream, x, n, dim, ldx, kp,
                           (int)split, vec, terms, iscale);
    else
        hipLaunchKernelGGL(pmcc_prep_kernel<SPLIT_FP16>, grid, dim3(PTHREADS), 0, stream, x, n, dim, ldx, kp,
                           (int)split, vec, terms, iscale);
    return hipGetLastError();
}

template <int SPLIT, bool SYM, bool VEC>
hipError_t launch_tile(PmccTileArgs &args, int64_t ids, hipStream_t stream)
{
    const int64_t max_ids = int64_t(1) << 23;
    for (int64_t off = 0; off < ids; off += max_ids) {
        args.id_offset = off;
        args.ids_this = (ids - off) < max_ids ? (ids - off) : max_ids;
        hipLaunchKernelGGL((pmcc_tile_kernel<SPLIT, SYM, VEC>), dim3((unsigned)args.ids_this),
                           dim3(MTHREADS), 0, stream, args);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

template <int SPLIT>
hipError_t launch_tile_split(bool same, bool vec, PmccTileArgs &args, int64_t ids,
                             hipStream_t stream)
{
    if (same)
        return vec ? launch_tile<SPLIT, true, true>(args, ids, stream)
                   : launch_tile<SPLIT, true, false>(args, ids, stream);
    return launch_tile<SPLIT, false, false>(args, ids, stream);
}

// Workspace of the matrix-core form of use = "pairwise.complete.obs": the
// operand blocks of a, then (unless same) of b, the scales, the tile flags.  bytes is
// 0 where the VALU form is taken: few samples, where three launches cost
// more than the sums (500 x 300 variables, times in us, VALU and here: 28 and
// 37 at 48 samples, 44 and 30 at 100), unless the pairs are many (3000
// variables x 20 samples: 70 and 50), and above a gigabyte of operands.
struct MomentsPlan {
    int64_t nch, tiles64;
    size_t off_b, off_scale, off_left, bytes;
};

MomentsPlan moments_plan(int64_t na, int64_t nb, bool same, int64_t dim)
{
    MomentsPlan m;
    m.nch = (dim + OPERAND_K - 1) / OPERAND_K;
    const int64_t ta = (na + WBM - 1) / WBM, tb = (nb + WBM - 1) / WBM;
    m.tiles64 = same ? ta * (ta + 1) / 2 : ta * tb;
    const double row = 2.0 * QT * OPERAND_K * (double)m.nch;
    const double all = row * ((double)operand_rows(na) + (same ? 0.0 : (double)operand_rows(nb)));
    if (!(dim >= 80 || (dim >= 16 && m.tiles64 >= 1000)) || all > MOMENTS_MAX_BYTES) {
        m.bytes = 0;
        return m;
    }
    m.off_b = (size_t)operand_rows(na) * (size_t)m.nch * OPERAND_K * QT * sizeof(unsigned short);
    m.off_scale = m.off_b + (same ? 0 : (size_t)operand_rows(nb) * (size_t)m.nch * OPERAND_K * QT *
                                            sizeof(unsigned short));
    m.off_left = m.off_scale + align256(((size_t)na + (same ? 0 : (size_t)nb)) * sizeof(float));
    m.bytes = m.off_left + align256((size_t)m.tiles64);
    return m;
}

hipError_t launch_moments_prep(const float *x, int64_t n, int64_t dim, int64_t ldx, int64_t nch,
                               unsigned short *terms, float *scales, uint8_t *left, int64_t nleft,
                               hipStream_t stream)
{
    const int64_t blocks = operand_rows(n) / 32;
    int64_t split = (512 + blocks - 1) / blocks;
    const int64_t rounds = (nch + QTHREADS / 64 - 1) / (QTHREADS / 64);   // chunks per wave
    if (split > rounds) split = rounds;
    hipLaunchKernelGGL(pmcc_moments_prep_kernel, dim3((unsigned)(blocks * split)), dim3(QTHREADS), 0, stream,
                       x, n, dim, ldx, nch, (int)split, terms, scales, left, nleft);
    return hipGetLastError();
}

template <bool SYM>
hipError_t launch_moments(const MomentsPlan &m, MomentsArgs &args, hipStream_t stream)
{
    args.tiles_b = (args.nb + QBM - 1) / QBM;
    const int64_t ids = m.tiles64;
    const int64_t max_ids = int64_t(1) << 22;
    for (int64_t off = 0; off < ids; off += max_ids) {
        args.id_offset = off;
        args.ids_this = (ids - off) < max_ids ? (ids - off) : max_ids;
        hipLaunchKernelGGL(pmcc_moments_kernel<SYM>, dim3((unsigned)args.ids_this), dim3(QWAVES * 64), 0,
                           stream, args);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace

size_t pmcc_workspace_bytes(int use, int precision, int64_t na, int64_t nb, bool same,
                            int64_t dim)
{
    if (dim <= 0 || na <= 0 || nb <= 0) return 0;
    if (use == 1) return moments_plan(na, nb, same, dim).bytes;
    precision = everything_form(precision, na, nb, same, dim);
    return side_bytes(precision, na, dim) + (same ? 0 : side_bytes(precision, nb, dim));
}

hipError_t launch_pmcc(int use, int precision, const float *a, int64_t na, int64_t lda,
                       const float *b, int64_t nb, int64_t ldb, bool same, int64_t dim,
                       float *pairs, float *corr, float *ts, int64_t ldo, void *workspace,
                       hipStream_t stream)
{
    if (na <= 0 || nb <= 0) return hipSuccess;
    if (dim == 0) {
        hipLaunchKernelGGL(pmcc_empty_kernel, dim3(grid_for(na * nb, 256)), dim3(256), 0, stream,
                           corr, ts, pairs, na, nb, ldo);
        return hipGetLastError();
    }
    if (use == 1) {
        PairwiseArgs args;
        args.a = a;
        args.na = na;
        args.lda = lda;
        args.b = b;
        args.nb = nb;
        args.ldb = ldb;
        args.dim = dim;
        args.corr = corr;
        args.ts = ts;
        args.pairs = pairs;
        args.ldo = ldo;
        args.vec = (ldo % 4 == 0) && ((reinterpret_cast<uintptr_t>(corr) | reinterpret_cast<uintptr_t>(ts) |
                                       reinterpret_cast<uintptr_t>(pairs)) & 15u) == 0;
        const int64_t ta = (na + WBM - 1) / WBM, tb = (nb + WBM - 1) / WBM;
        args.tiles_b = tb;
        args.left = nullptr;
        args.scale_a = args.scale_b = nullptr;
        const MomentsPlan m = moments_plan(na, nb, same, dim);
        if (m.bytes > 0 && workspace != nullptr) {
            char *ws = static_cast<char *>(workspace);
            MomentsArgs ma;
            unsigned short *terms_a = reinterpret_cast<unsigned short *>(ws);
            unsigned short *terms_b = same ? terms_a : reinterpret_cast<unsigned short *>(ws + m.off_b);
            float *scale_a = reinterpret_cast<float *>(ws + m.off_scale);
            float *scale_b = same ? scale_a : scale_a + na;
            ma.left = reinterpret_cast<uint8_t *>(ws + m.off_left);
            hipError_t e = launch_moments_prep(a, na, dim, lda, m.nch, terms_a, scale_a, ma.left,
                                               m.tiles64, stream);
            if (e == hipSuccess && !same)
                e = launch_moments_prep(b, nb, dim, ldb, m.nch, terms_b, scale_b, ma.left, 0, stream);
            if (e != hipSuccess) return e;
            ma.ta = terms_a;
            ma.tb = terms_b;
            ma.na = na;
            ma.nb = nb;
            ma.nch = (int)m.nch;
            // about sqrt(chunks) chunks per partial sum, so that both levels
            // add about as many
            ma.fold = 1;
            while ((int64_t)(ma.fold + 1) * (ma.fold + 1) <= m.nch) ++ma.fold;
            ma.corr = corr;
            ma.ts = ts;
            ma.pairs = pairs;
            ma.ldo = ldo;
            e = same ? launch_moments<true>(m, ma, stream) : launch_moments<false>(m, ma, stream);
            if (e != hipSuccess) return e;
            args.left = ma.left;   // the tiles left to two passes
            args.scale_a = scale_a;
            args.scale_b = scale_b;
        }
        const int64_t total = same ? ta * (ta + 1) / 2 : ta * tb;
        const int64_t max_tiles = int64_t(1) << 23;
        for (int64_t off = 0; off < total; off += max_tiles) {
            args.tile_offset = off;
            args.tiles_this = (total - off) < max_tiles ? (total - off) : max_tiles;
            const dim3 grid((unsigned)args.tiles_this), block(WTHREADS);
            if (args.left) {
                if (same)
                    hipLaunchKernelGGL((pmcc_pairwise_kernel<true, true>), grid, block, 0, stream, args);
                else
                    hipLaunchKernelGGL((pmcc_pairwise_kernel<false, true>), grid, block, 0, stream, args);
            } else {
                if (same)
                    hipLaunchKernelGGL((pmcc_pairwise_kernel<true, false>), grid, block, 0, stream, args);
                else
                    hipLaunchKernelGGL((pmcc_pairwise_kernel<false, false>), grid, block, 0, stream, args);
            }
            hipError_t e = hipGetLastError();
            if (e != hipSuccess) return e;
        }
        return hipSuccess;
    }

    precision = everything_form(precision, na, nb, same, dim);
    PmccWs w = carve(precision, na, nb, same, dim, workspace);
    hipError_t e = launch_prep(precision, a, na, dim, lda, w.ta, w.isa, w.za, stream);
    if (e != hipSuccess) return e;
    if (!same) {
        e = launch_prep(precision, b, nb, dim, ldb, w.tb, w.isb, w.zb, stream);
        if (e != hipSuccess) return e;
    }
    const float fpairs = (float)dim;
    if (precision == 0) {
        // corr[x * ldo + y] = z_x . z_y: the plain cross tile with x on its
        // row side and y on its column side; with a == b the symmetric
        // layout computes the lower tiles and mirrors them
        if (same)
            e = launch_plain(OP_DOT, OUT_FULL, w.za, na, dim, w.za, na, dim, dim, 2.0f, corr, ldo,
                             stream);
        else
            e = launch_plain(OP_DOT, OUT_CROSS, w.zb, nb, dim, w.za, na, dim, dim, 2.0f, corr, ldo,
                             stream);
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL(pmcc_finish_kernel, dim3(grid_for(na * nb, 256)), dim3(256), 0, stream,
                           corr, ts, pairs, na, nb, ldo, fpairs);
        return hipGetLastError();
    }
    PmccTileArgs args;
    args.ta = w.ta;
    args.tb = w.tb;
    args.na = na;
    args.nb = nb;
    args.kp = padded_dim(dim);
    args.isa = w.isa;
    args.isb = w.isb;
    args.corr = corr;
    args.ts = ts;
    args.pairs = pairs;
    args.ldo = ldo;
    args.fpairs = fpairs;
    args.tiles_a = (na + MBM - 1) / MBM;
    args.tiles_b = (nb + MBM - 1) / MBM;
    const int64_t sa = (args.tiles_a + MSUPER - 1) / MSUPER;
    const int64_t sbt = (args.tiles_b + MSUPER - 1) / MSUPER;
    args.super_b = sbt;
    const int64_t ids = (same ? sa * (sa + 1) / 2 : sa * sbt) * MSUPER * MSUPER * 2;
    const bool vec = (ldo % 4 == 0) && ((reinterpret_cast<uintptr_t>(corr) |
                                         reinterpret_cast<uintptr_t>(ts) |
                                         reinterpret_cast<uintptr_t>(pairs)) & 15u) == 0;
    return precision == 1 ? launch_tile_split<SPLIT_BF16>(same, vec, args, ids, stream)
                          : launch_tile_split<SPLIT_FP16>(same, vec, args, ids, stream);
}

hipError_t launch_ttest(const float *pairs, const float *corr, float *ts, int64_t n,
                        hipStream_t stream)
{
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(ttest_kernel, dim3(grid_for(n, 256)), dim3(256), 0, stream, pairs, corr,
                       ts, n);
    return hipGetLastError();
}

}  // namespace gt
