// gt_gram.hip -- split-precision MFMA Gram form of the euclidean distance.
//
// d(x_i, x_j)^2 = ||x_i||^2 + ||x_j||^2 - 2 x_i.x_j.  The dot products of a
// 256 x 256 square of pairs (or half of one) run on the gfx950 matrix cores
// (v_mfma_f32_32x32x16_{bf16,f16}) with FP32 accumulation.  A pre-pass splits
// every FP32 input value once into 16-bit terms (stored in the workspace), and
// the tile kernel accumulates the products whose error terms matter:
//   BF16 (8-bit significand): three terms x = h + m + l, exact (x - h and
//     x - h - m are exact in FP32 and the last remainder has at most 8
//     significant bits); six products hh' + hm' + mh' + hl' + lh' + mm'; the
//     dropped ml' + lm' + ll' are below 2^-23 |x_c y_c| per feature.
//   FP16 (11-bit significand): two terms x = h + l (+ r, |r| <= 2^-22|x|),
//     three products hh' + hl' + lh'; dropped terms below 3 * 2^-22 |x_c y_c|.
//     Rows are first scaled by a power of two so that max |x| lies in
//     [2^14, 2^15) (keeps l out of the subnormal range and h below the FP16
//     maximum); the scale is undone exactly on the dot product.
// (A two-term BF16 split leaves ~3 * 2^-16 |x_c y_c| per feature, which no
// cancellation threshold can bring under 1e-5 for small k.)
//
// The Gram form loses relative accuracy when d^2 is small against
// ||x||^2 + ||y||^2 (cancellation).  Every pair with
//   d^2 < tau (||x||^2 + ||y||^2)
// is flagged in the epilogue and recomputed in the same workgroup from exact
// FP32 differences, sum (x_c - y_c)^2, with the FP32 rows re-streamed through
// LDS in 32-feature chunks (two-level summation).  Flagged pairs are processed
// through an LDS list of 1024 entries per pass, as many passes as needed, so
// any number of near-coincident pairs is handled.  tau is derived on the host
// from k (gram_tau) so that the Gram-form error stays below 1.6e-5 d^2.
//
// The reference computes this distance with exact differences only
// (inst/cuda/distance.cu:40-78); this path produces the same distance within
// the stated tolerance (max relative error <= 1e-5 against FP64).
#include "gt_common.h"
#include "gt_internal.h"
#include "gt_mfma.h"

namespace gt {
namespace {

constexpr int GBM = 256;        // side of a square of pairs (points)
constexpr int GBK = 16;         // features per main-loop chunk (one MFMA k-step)
constexpr int KPAD = 32;        // the split terms are zero-padded to a multiple of this
constexpr int GSUPER = 4;       // super-tile side in tiles (L2 locality)
constexpr int FBK = 32;         // features per fix-up chunk
constexpr int FLD = FBK + 4;    // fix-up LDS row length (floats, 16 B aligned rows)
constexpr int FCAP = 1024;      // flagged pairs per fix-up pass
// Gram-form values are finished with the hardware square root (v_sqrt_f32)
// plus one residual correction (sqrt_rn), which rounds correctly for normal
// inputs; d^2 below 2^-100 goes to the exact pass instead.
constexpr int LIST_BYTES = FCAP * 4;

// A workgroup's tile: GAM rows j (side A) x 256 rows i (side B) on NW waves,
// NW / 4 along A x 4 along B, 64 x 64 pairs each as 2 x 2 blocks of 32 x 32
// accumulators (128 VGPRs per lane).  NW = 16: a whole square, one workgroup per
// CU.  NW = 8: half a square, two workgroups per CU.
constexpr int WC = 4;   // B-row groups
constexpr int NB = 2;   // 32-row accumulator blocks along B per wave
template <int NW>
struct Tile {
    static constexpr int THREADS = NW * 64;
    static constexpr int GAM = NW * 16;
    static constexpr int PARTS = GBM / GAM;                                // workgroups per square
    static constexpr int ABLOCKS = GAM / 32, BLOCKS = (GAM + GBM) / 32;    // operand blocks: A, both
    static constexpr int FUNITS = (GAM + GBM) * FBK / 4 / THREADS;         // fix-up float4 units per thread
    static constexpr int FPER = FCAP / THREADS;                            // fix-up list entries per thread
    static constexpr int FIX_BYTES = (GAM + GBM) * FLD * 4;                // fix-up staging, both sides
    static constexpr int SIDE_BYTES = 2 * (GAM + GBM) * 4 + 16 * 4;        // norms, inverse scales, scan
};

// LDS: [split terms | (aliased) fix-up staging + pair list] [side data]
template <int NT, int NW>
struct TileLds : Tile<NW> {
    typedef Tile<NW> T;
    static constexpr int PIECES = T::BLOCKS * NT;        // 1 KB each, per chunk
    static constexpr int GPW = (PIECES + NW - 1) / NW;   // per wave
    // main-loop ring depth: what two workgroups per CU leave room for (two
    // stages with one: 15.67 vs 15.55 ms on the 65536 x 512 mixture, BF16)
    static constexpr int NSTAGE = NW == 8 && NT == 3 ? 2 : 3;
    static constexpr int STAGE = PIECES * OPERAND_BYTES;
    static constexpr int MAIN = NSTAGE * STAGE;
    static constexpr int FIX = T::FIX_BYTES + LIST_BYTES;
    static constexpr int REGION = MAIN > FIX ? MAIN : FIX;
    static constexpr int SIDE = REGION;
    static constexpr int BYTES = REGION + T::SIDE_BYTES;
    static_assert(NSTAGE == 2 || PIECES % NW == 0, "the same number of loads in flight in every wave");
};

struct GramArgs {
    const float *x;        // FP32 points (exact passes)
    int64_t n, k, ldx;
    const unsigned short *terms;  // split terms, in operand blocks (gt_mfma.h)
    int64_t kp;            // k padded to KPAD
    const float *norms;    // ||x_i - c||^2 (FP32)
    const float *iscale;   // FP16 path: inverse power-of-two row scale
    float *out;
    int64_t ldd;
    int64_t T;             // tiles per side
    int64_t id_offset, ids_this;
    float tau;
};

// Exclusive scan of one int per thread over a workgroup of NW waves.
template <int NW>
__device__ __forceinline__ int block_exclusive_scan(int v, int *tmp, int &total)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int incl = v;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int t = __shfl_up(incl, d, 64);
        if (lane >= d) incl += t;
    }
    if (lane == 63) tmp[wave] = incl;
    __syncthreads();
    int before = 0;
    total = 0;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
        const int c = tmp[w];
        if (w < wave) before += c;
        total += c;
    }
    __syncthreads();
    return before + incl - v;
}

// Wait until at most N vector memory operations of this wave are outstanding.
template <int N>
__device__ __forceinline__ void wait_vmcnt()
{
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

typedef __attribute__((address_space(3))) void lds_void_t;
typedef const __attribute__((address_space(1))) void gbl_void_t;

// Main-loop LDS image of one chunk: side A (rows j), then side B (rows i),
// blocks of 32 rows, each NT terms of 1 KB as they lie in memory.
// global_load_lds writes lane l's 16 B at the wave's LDS base + 16 l, so each
// wave instruction moves one term of one block, eight whole lines; a lane's
// operand read is its own 16 B, free of bank conflicts.  These pieces go to the
// waves round robin.  Blocks past the last one repeat it: they only feed pairs
// that are never stored.
// (Row-major terms moved 32 bytes of 32 rows per instruction, each line in four
// parts: 65536 x 512 mixture, BF16, 15.77 -> 14.94 ms; 9001 x 130, FP16, 122 ->
// 114 us, both with one workgroup per CU.)
template <int NT, int NW>
__device__ __forceinline__ void chunk_sources(const GramArgs &args, int64_t i0, int64_t j0,
                                              int wave, int lane,
                                              const unsigned short *(&gsrc)[TileLds<NT, NW>::GPW])
{
    const int64_t last = operand_rows(args.n) / 32 - 1, nch = args.kp / OPERAND_K;
#pragma unroll
    for (int q = 0; q < TileLds<NT, NW>::GPW; ++q) {
        const int p = min(wave + q * NW, TileLds<NT, NW>::PIECES - 1), g = p / NT;
        constexpr int ABLOCKS = Tile<NW>::ABLOCKS;
        const int64_t rb = g < ABLOCKS ? j0 / 32 + g : i0 / 32 + g - ABLOCKS;
        gsrc[q] = args.terms + ((rb < last ? rb : last) * nch * NT + p % NT) * OPERAND_VALUES + lane * 8;
    }
}

template <int NT, int NW>
__device__ __forceinline__ void issue_chunk(const unsigned short *const (&gsrc)[TileLds<NT, NW>::GPW],
                                            unsigned char *stage, int wave, int chunk)
{
    const int64_t off = (int64_t)chunk * NT * OPERAND_VALUES;
#pragma unroll
    for (int q = 0; q < TileLds<NT, NW>::GPW; ++q)
        if (wave + q * NW < TileLds<NT, NW>::PIECES)
            __builtin_amdgcn_global_load_lds((gbl_void_t *)(gsrc[q] + off),
                                             (lds_void_t *)(stage + (wave + q * NW) * OPERAND_BYTES), 16, 0,
                                             0);
}

// One chunk of MFMA products for this wave's pairs (acc[a][b]: A rows
// wr*64 + a*32.., B rows wc*NB*32 + b*32..); sg = stage + the lane's operand
// offset.
template <int SPLIT, int NW>
__device__ __forceinline__ void mfma_chunk(f32x16_t (&acc)[2][NB], const unsigned char *sg, int wr,
                                           int wc)
{
    typedef typename Split<SPLIT>::vec vec;
    constexpr int NT = Split<SPLIT>::NT;
    vec av[NT][2];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int a = 0; a < 2; ++a)
            av[t][a] = *reinterpret_cast<const vec *>(sg + ((wr * 2 + a) * NT + t) * OPERAND_BYTES);
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        vec bv[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t)
            bv[t] = *reinterpret_cast<const vec *>(sg + ((Tile<NW>::ABLOCKS + wc * NB + b) * NT + t) * OPERAND_BYTES);
        // hh' first, then the cross terms in decreasing magnitude
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

// Norms (and FP16 inverse row scales) of the tile's rows into LDS.
template <int SPLIT, int NW>
__device__ __forceinline__ void load_side(const GramArgs &args, int64_t i0, int64_t j0, float *nA,
                                          float *nB, float *iA, float *iB)
{
    constexpr int GAM = Tile<NW>::GAM;
    for (int t = threadIdx.x; t < GAM + GBM; t += Tile<NW>::THREADS) {
        if (t < GAM) {
            const int64_t r = j0 + t;
            nA[t] = r < args.n ? args.norms[r] : 0.0f;
            if (SPLIT == SPLIT_FP16) iA[t] = r < args.n ? args.iscale[r] : 1.0f;
        } else {
            const int64_t r = i0 + (t - GAM);
            nB[t - GAM] = r < args.n ? args.norms[r] : 0.0f;
            if (SPLIT == SPLIT_FP16) iB[t - GAM] = r < args.n ? args.iscale[r] : 1.0f;
        }
    }
}

// Epilogue of one tile: d^2 = ||x||^2 + ||y||^2 - 2g for this wave's pairs;
// every valid pair that is not flagged (d^2 >= tau (||x||^2 + ||y||^2)) is
// stored.  Flag bits: index (a * NB + b) * 16 + r marks accumulator element
// r of block (a, b), in fm[index / 64].  32x32 accumulator layout: element r
// of lane l is row 8(r/4) + 4(l/32) + r%4 (A side, j) and column l%32 (B
// side, i); lanes 0..31 hold 32 consecutive i of one j, so packed stores are
// contiguous runs.
template <int SPLIT, int LAYOUT>
__device__ __forceinline__ void gram_epilogue(const f32x16_t (&acc)[2][NB], const GramArgs &args,
                                              int64_t i0, int64_t j0, bool interior, int wr,
                                              int wc, int lane, const float *nA, const float *nB,
                                              const float *iA, const float *iB,
                                              unsigned long long (&fm)[NB / 2])
{
    const int64_t n = args.n;
    const int li0 = wc * NB * 32 + (lane & 31);
    float ni[NB], sb[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        ni[b] = nB[li0 + b * 32];
        sb[b] = (SPLIT == SPLIT_FP16) ? iB[li0 + b * 32] : 1.0f;
    }
#pragma unroll
    for (int q = 0; q < NB / 2; ++q) fm[q] = 0ull;
    const float tau = args.tau;
    if (interior) {
        // every pair valid, i > j: stored branch-free.  Rows jw + d (d < 64)
        // of this wave: element offsets from the start of row jw fit in 32
        // bits (the host limits n to below 2^24), and the row-dependent part
        // of each offset is wave-uniform
        const int64_t jw = j0 + wr * 64;
        float *const outw =
            args.out + ((LAYOUT == OUT_PACKED) ? packed_base(n, jw) : jw * args.ldd) + i0;
        const unsigned cw = (LAYOUT == OUT_PACKED) ? (unsigned)(n - 1 - jw) : (unsigned)args.ldd;
        const bool hi = (lane >> 5) != 0;
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const unsigned dc = a * 32 + 8 * (r >> 2) + (r & 3);
                const unsigned base_u = (LAYOUT == OUT_PACKED) ? dc * cw - dc * (dc + 1) / 2 : dc * cw;
                const unsigned step_u = (LAYOUT == OUT_PACKED) ? 4 * cw - 4 * dc - 10 : 4 * cw;
                const unsigned ro = base_u + (hi ? step_u : 0u) + (unsigned)li0;
                const int lj = wr * 64 + (int)dc + (hi ? 4 : 0);
                const float nj = nA[lj];
                const float sj = (SPLIT == SPLIT_FP16) ? iA[lj] : 1.0f;
#pragma unroll
                for (int b = 0; b < NB; ++b) {
                    float g = acc[a][b][r];
                    if (SPLIT == SPLIT_FP16) g = (g * sj) * sb[b];
                    const float ss = nj + ni[b];
                    const float d2 = fmaf(-2.0f, g, ss);
                    const bool ok = d2 >= fmaf(tau, ss, GRAM_SQRT_MIN);
                    const int bit = (a * NB + b) * 16 + r;
                    fm[bit >> 6] |= ok ? 0ull : (1ull << (bit & 63));
                    const float v = sqrt_rn(d2);
                    outw[ro + (unsigned)(b * 32)] = v;
                    if (LAYOUT == OUT_FULL) args.out[(i0 + li0 + b * 32) * args.ldd + jw + lj - wr * 64] = v;
                }
            }
    } else {
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int lj = wr * 64 + a * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
                const int64_t j = j0 + lj;
                const float nj = nA[lj];
                const float sj = (SPLIT == SPLIT_FP16) ? iA[lj] : 1.0f;
                float *rowp = args.out + ((LAYOUT == OUT_PACKED) ? packed_base(n, j) : j * args.ldd) +
                              i0 + li0;
#pragma unroll
                for (int b = 0; b < NB; ++b) {
                    float g = acc[a][b][r];
                    // undo the row scales one at a time (their product can overflow)
                    if (SPLIT == SPLIT_FP16) g = (g * sj) * sb[b];
                    const float ss = nj + ni[b];
                    const float d2 = fmaf(-2.0f, g, ss);
                    const bool flag = !(d2 >= fmaxf(tau * ss, GRAM_SQRT_MIN));
                    const int li = li0 + b * 32;
                    const bool valid = i0 + li < n && i0 + li > j;
                    if (valid) {
                        if (!flag) {
                            const float v = sqrt_rn(fmaxf(d2, 0.0f));
                            rowp[b * 32] = v;
                            if (LAYOUT == OUT_FULL) args.out[(i0 + li) * args.ldd + j] = v;
                        } else {
                            const int bit = (a * NB + b) * 16 + r;
                            fm[bit >> 6] |= 1ull << (bit & 63);
                        }
                    }
                    if (LAYOUT == OUT_FULL && i0 + li == j && j < n) rowp[b * 32] = 0.0f;
                }
            }
    }
}

// Tile position of flag index `bit` of this lane: (A row << 16) | B row.
__device__ __forceinline__ unsigned flag_entry(int bit, int wr, int li0, int lane)
{
    const int a = bit / (NB * 16), b = (bit / 16) % NB, r = bit & 15;
    const int lj = wr * 64 + a * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
    return ((unsigned)lj << 16) | (unsigned)(li0 + b * 32);
}

// Exact distance of a flagged pair (entry as flag_entry) of tile (i0, j0).
template <int LAYOUT>
__device__ __forceinline__ void store_exact(const GramArgs &args, int64_t i0, int64_t j0,
                                            unsigned ent, float sum)
{
    const int64_t j = j0 + (ent >> 16), i = i0 + (ent & 0xffffu);
    const float v = sqrtf(sum);
    if (LAYOUT == OUT_PACKED) {
        args.out[packed_base(args.n, j) + i] = v;
    } else {
        args.out[j * args.ldd + i] = v;
        args.out[i * args.ldd + j] = v;
    }
}

// Exact FP32 recompute of the tile's flagged pairs: the FP32 rows of both
// sides are re-streamed through LDS in 32-feature chunks (two-level sums);
// the pairs go through an LDS list of FCAP entries per pass.  myoff: this
// lane's rank among the flagged pairs; total: their number.  The caller has
// let the epilogue's stores land.
template <int LAYOUT, bool VEC4, int NW>
__device__ __forceinline__ void gram_fixup(const GramArgs &args, unsigned char *smem, int64_t i0,
                                           int64_t j0,
                                           const unsigned long long (&fm)[NB / 2],
                                           int myoff, int total, int wr, int li0, int lane)
{
    typedef Tile<NW> T;
    constexpr int THREADS = T::THREADS, GAM = T::GAM, FUNITS = T::FUNITS, FPER = T::FPER;
    const int tid = threadIdx.x;
    float *fS = reinterpret_cast<float *>(smem);
    unsigned int *list = reinterpret_cast<unsigned int *>(smem + T::FIX_BYTES);
    const int64_t n = args.n, k = args.k, ldx = args.ldx;
    // Staging unit e = tid + THREADS q (q < FUNITS): tile row e >> 3 (A side
    // rows first, then B side), features (e & 7) * 4..+3 of a chunk; the
    // unit's column is (tid & 7) * 4 for every q.  The accumulators are dead
    // here, so their registers hold a ring of FRING chunks in flight (the
    // pass is bound by load latency, not bandwidth).
    constexpr int FRING = NW == 16 ? 2 : 1;   // (two workgroups hide the latency too)
    int frow[FUNITS];
#pragma unroll
    for (int q = 0; q < FUNITS; ++q) {
        const int row = (tid + THREADS * q) >> 3;
        const int64_t g = row < GAM ? j0 + row : i0 + (row - GAM);
        frow[q] = (int)(g < n ? g : n - 1);
    }
    const float *const fx = args.x + (tid & 7) * 4;
    const int nf = (int)((k + FBK - 1) / FBK);
    float4 fr0[FUNITS], fr1[FUNITS];
#define GT_FLOAD(buf, chunk)                                                               \
    do {                                                                                   \
        const int64_t fb_ = (int64_t)(chunk) * FBK;                                        \
        const int64_t kk = fb_ + (tid & 7) * 4;                                            \
        _Pragma("unroll") for (int q = 0; q < FUNITS; ++q) {                               \
            const float *src_ = fx + (int64_t)frow[q] * ldx + fb_;                         \
            if (VEC4) {                                                                    \
                buf[q] = kk < k ? *reinterpret_cast<const float4 *>(src_)                  \
                                : make_float4(0.f, 0.f, 0.f, 0.f);                         \
            } else {                                                                       \
                float v_[4];                                                               \
                _Pragma("unroll") for (int c_ = 0; c_ < 4; ++c_) v_[c_] =                  \
                    (kk + c_ < k) ? src_[c_] : 0.0f;                                       \
                buf[q] = make_float4(v_[0], v_[1], v_[2], v_[3]);                          \
            }                                                                              \
        }                                                                                  \
    } while (0)
    // one chunk: registers -> LDS, refill the registers FRING chunks ahead,
    // then accumulate this thread's flagged pairs over the chunk
#define GT_FSTEP(buf, chunk)                                                               \
    do {                                                                                   \
        __syncthreads();                                                                   \
        _Pragma("unroll") for (int q = 0; q < FUNITS; ++q) {                               \
            const int e = tid + THREADS * q;                                               \
            *reinterpret_cast<float4 *>(fS + (e >> 3) * FLD + (e & 7) * 4) = buf[q];       \
        }                                                                                  \
        __syncthreads();                                                                   \
        if ((chunk) + FRING < nf) GT_FLOAD(buf, (chunk) + FRING);                          \
        _Pragma("unroll") for (int c = 0; c < FPER; ++c) {                                 \
            if (tid + THREADS * c < cnt) {                                                 \
                const float4 *ra = reinterpret_cast<const float4 *>(fS + (ent[c] >> 16) * FLD); \
                const float4 *rb =                                                         \
                    reinterpret_cast<const float4 *>(fS + (GAM + (ent[c] & 0xffffu)) * FLD); \
                float part = 0.0f;                                                         \
                _Pragma("unroll") for (int q = 0; q < FBK / 4; ++q) {                      \
                    const float4 u = ra[q], v = rb[q];                                     \
                    float t = u.x - v.x;                                                   \
                    part = fmaf(t, t, part);                                               \
                    t = u.y - v.y;                                                         \
                    part = fmaf(t, t, part);                                               \
                    t = u.z - v.z;                                                         \
                    part = fmaf(t, t, part);                                               \
                    t = u.w - v.w;                                                         \
                    part = fmaf(t, t, part);                                               \
                }                                                                          \
                sum[c] += part;                                                            \
            }                                                                              \
        }                                                                                  \
    } while (0)
    for (int base = 0; base < total; base += FCAP) {
        {
            int rank = myoff;
#pragma unroll
            for (int qw = 0; qw < NB / 2; ++qw) {
                unsigned long long m = fm[qw];
                while (m) {
                    const int bit = __builtin_ctzll(m);
                    m &= m - 1;
                    if (rank >= base && rank < base + FCAP)
                        list[rank - base] = flag_entry(qw * 64 + bit, wr, li0, lane);
                    ++rank;
                }
            }
        }
        const int cnt = (total - base) < FCAP ? (total - base) : FCAP;
        float sum[FPER];
        unsigned ent[FPER];
#pragma unroll
        for (int c = 0; c < FPER; ++c) sum[c] = 0.0f;
        GT_FLOAD(fr0, 0);
        if (FRING == 2 && nf > 1) GT_FLOAD(fr1, 1);
        __syncthreads();
#pragma unroll
        for (int c = 0; c < FPER; ++c) {
            const int e = tid + THREADS * c;
            ent[c] = e < cnt ? list[e] : 0u;
        }
        for (int ch = 0; ch < nf; ch += FRING) {
            GT_FSTEP(fr0, ch);
            if (FRING == 2 && ch + 1 < nf) GT_FSTEP(fr1, ch + 1);
        }
#pragma unroll
        for (int c = 0; c < FPER; ++c)
            if (tid + THREADS * c < cnt) store_exact<LAYOUT>(args, i0, j0, ent[c], sum[c]);
        __syncthreads();
    }
#undef GT_FSTEP
#undef GT_FLOAD
}

// One workgroup per tile: main loop, epilogue, then the exact pass of the
// flagged pairs.  Bound: the matrix cores' power for long rows (65536 x 512
// mixture, BF16: 13.2 TFLOP of products, 11.6 ms at the 1.14 PFLOP/s of a large
// BF16 product, and 3.3 ms of exact pass: 14.9 ms), the stores for short ones.
template <int SPLIT, int LAYOUT, bool VEC4, int NW>
__global__ __launch_bounds__(NW * 64, 4) void gram_tile_kernel(GramArgs args)
{
    constexpr int NT = Split<SPLIT>::NT;
    typedef TileLds<NT, NW> L;
    constexpr int GPW = L::GPW, GAM = L::GAM;
    __shared__ __attribute__((aligned(1024))) unsigned char smem[L::BYTES];
    float *nA = reinterpret_cast<float *>(smem + L::SIDE);
    float *nB = nA + GAM, *iA = nB + GBM, *iB = iA + GAM;
    int *scan_tmp = reinterpret_cast<int *>(iB + GBM);

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wr = wave / WC, wc = wave % WC;

    // Super-tiled lower-triangular schedule: super-tile s covers GSUPER x
    // GSUPER tiles; tiles above the diagonal or past the edge exit at once.
    const int64_t gid = args.id_offset + xcd_remap(blockIdx.x, args.ids_this);
    const int64_t id = gid / L::PARTS;
    const int64_t st = id / (GSUPER * GSUPER);
    const int w = (int)(id % (GSUPER * GSUPER));
    int SI, SJ;
    tri_tile(st, SI, SJ);
    const int64_t I = (int64_t)SI * GSUPER + w / GSUPER;
    const int64_t J = (int64_t)SJ * GSUPER + w % GSUPER;
    if (I >= args.T || J > I) return;
    const int64_t i0 = I * GBM, j0 = J * GBM + gid % L::PARTS * GAM;
    if (j0 >= args.n) return;
    load_side<SPLIT, NW>(args, i0, j0, nA, nB, iA, iB);

    const unsigned short *gsrc[GPW];
    chunk_sources<NT, NW>(args, i0, j0, wave, lane, gsrc);
    const int roff = lane * 16;
    f32x16_t acc[2][NB];
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[a][b][r] = 0.0f;

    const int nchunks = (int)(args.kp / GBK);
    // NSTAGE stages: chunks c + 1 .. c + NSTAGE - 1 in flight while c is
    // computed
    constexpr int NS = L::NSTAGE;
#pragma unroll
    for (int c = 0; c < NS - 1; ++c)
        if (c < nchunks) issue_chunk<NT, NW>(gsrc, smem + c * L::STAGE, wave, c);
    for (int c = 0; c < nchunks; ++c) {
        // chunk c landed when at most the next chunk's loads of this wave
        // are outstanding (vector memory loads complete in order)
        if (NS == 3 && c + 1 < nchunks)
            wait_vmcnt<GPW>();
        else
            wait_vmcnt<0>();
        // every wave's part of chunk c is in LDS, and every wave finished
        // chunk c-1, whose stage the next issue overwrites.  A bare s_barrier:
        // __syncthreads() would also drain the later chunks' loads.
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (c + NS - 1 < nchunks)
            issue_chunk<NT, NW>(gsrc, smem + ((c + NS - 1) % NS) * L::STAGE, wave, c + NS - 1);
        mfma_chunk<SPLIT, NW>(acc, smem + (c % NS) * L::STAGE + roff, wr, wc);
    }
    // the fix-up below reuses the stage memory
    __syncthreads();

    const bool interior = (I > J) && (i0 + GBM <= args.n);
    unsigned long long fm[NB / 2];
    gram_epilogue<SPLIT, LAYOUT>(acc, args, i0, j0, interior, wr, wc, lane, nA, nB, iA, iB, fm);
    int cnt = 0;
#pragma unroll
    for (int q = 0; q < NB / 2; ++q) cnt += __popcll(fm[q]);
    int total;
    const int myoff = block_exclusive_scan<NW>(cnt, scan_tmp, total);
    if (total == 0) return;
    // the epilogue's stores of flagged pairs land before the exact values
    wait_vmcnt<0>();
    __syncthreads();
    gram_fixup<LAYOUT, VEC4, NW>(args, smem, i0, j0, fm, myoff, total, wr,
                                 wc * NB * 32 + (lane & 31), lane);
}

// Column centre c_j of the Gram form.  Euclidean distances do not change
// when every point is moved by the same vector, but the Gram form's error
// scales with ||x||^2 + ||y||^2: centring the columns makes that as small as
// the data's spread allows (U[0,1) data: 4x; N(0,1) + 100: 10^4 x).  c_j is
// the column mean rounded to a power-of-two grid no coarser than 1/64 of the
// column's range, so that x - c_j is often exact (integer columns keep
// integer centres); a constant column takes its value; a column holding a
// NaN or an infinity is not moved.
constexpr int CS_ROWS = 256;    // rows per partial-statistics block
constexpr int PREP_THREADS = 1024, PREP_WAVES = PREP_THREADS / 64;

// 64 columns per workgroup, a wave per 16 rows, their sums combined in wave
// order.  Bound: latency; 9001 x 130 12 us with a thread per column and all 256
// rows, 5.0 us here.
__global__ __launch_bounds__(PREP_THREADS) void colstats_partial_kernel(const float *__restrict__ x,
                                                                        int64_t n, int64_t k, int64_t ldx,
                                                                        float *__restrict__ psum,
                                                                        float *__restrict__ pmin,
                                                                        float *__restrict__ pmax)
{
    constexpr int ROWS = CS_ROWS / PREP_WAVES;
    __shared__ float red[3][PREP_WAVES][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t r0 = (int64_t)blockIdx.x * CS_ROWS + wave * ROWS;
    for (int64_t cb = (int64_t)blockIdx.y * 64; cb < k; cb += (int64_t)gridDim.y * 64) {
        const int64_t c = cb + lane;
        float sum = 0.0f, mn = __builtin_inff(), mx = -__builtin_inff();
        if (c < k) {
            float v[ROWS];
#pragma unroll
            for (int q = 0; q < ROWS; ++q) v[q] = r0 + q < n ? x[(r0 + q) * ldx + c] : 0.0f;
#pragma unroll
            for (int q = 0; q < ROWS; ++q) {
                if (r0 + q >= n) break;
                sum += v[q];              // a NaN or an infinity makes the sum non-finite
                mn = fminf(mn, v[q]);
                mx = fmaxf(mx, v[q]);
            }
        }
        red[0][wave][lane] = sum;
        red[1][wave][lane] = mn;
        red[2][wave][lane] = mx;
        __syncthreads();
        if (wave == 0 && c < k) {
            for (int w = 1; w < PREP_WAVES; ++w) {
                sum += red[0][w][lane];
                mn = fminf(mn, red[1][w][lane]);
                mx = fmaxf(mx, red[2][w][lane]);
            }
            psum[blockIdx.x * k + c] = sum;
            pmin[blockIdx.x * k + c] = mn;
            pmax[blockIdx.x * k + c] = mx;
        }
        __syncthreads();
    }
}

// Column statistics from the partials: 16 columns per workgroup, 16
// threads per column, each over every 16th partial block; the 16 partial
// results are combined in a fixed order.
constexpr int CS_COLS = 16, CS_SLICES = 16;

__global__ __launch_bounds__(256) void colstats_finish_kernel(const float *__restrict__ psum,
                                                              const float *__restrict__ pmin,
                                                              const float *__restrict__ pmax,
                                                              int64_t blocks, int64_t n, int64_t k,
                                                              float *__restrict__ center)
{
    __shared__ float red[3][CS_SLICES][CS_COLS];
    const int cl = threadIdx.x % CS_COLS, sl = threadIdx.x / CS_COLS;
    for (int64_t cb = (int64_t)blockIdx.x * CS_COLS; cb < k; cb += (int64_t)gridDim.x * CS_COLS) {
        const int64_t c = cb + cl;
        float sum = 0.0f, mn = __builtin_inff(), mx = -__builtin_inff();
        if (c < k) {
            for (int64_t b = sl; b < blocks; b += CS_SLICES) {
                sum += psum[b * k + c];
                mn = fminf(mn, pmin[b * k + c]);
                mx = fmaxf(mx, pmax[b * k + c]);
            }
        }
        red[0][sl][cl] = sum;
        red[1][sl][cl] = mn;
        red[2][sl][cl] = mx;
        __syncthreads();
        if (sl == 0 && c < k) {
            sum = 0.0f;
            for (int q = 0; q < CS_SLICES; ++q) {
                sum += red[0][q][cl];
                mn = fminf(mn, red[1][q][cl]);
                mx = fmaxf(mx, red[2][q][cl]);
            }
            float cc = 0.0f;
            const float range = mx - mn;
            if (isfinite(sum) && isfinite(range)) {
                if (range == 0.0f) {
                    cc = mn;
                } else {
                    const float mean = sum / (float)n;
                    const float g = ldexpf(1.0f, ilogbf(range) - 6);   // <= range / 64
                    const float q = mean / g;
                    cc = (fabsf(q) < 0x1p24f) ? rintf(q) * g : mean;
                }
            }
            center[c] = cc;
        }
        __syncthreads();
    }
}

// ||v||^2 of one centred row by one wave, and max |v|.  The squares are summed
// with compensation (each product split exactly by an fma, each addition's
// rounding error recovered by TwoSum), so the norm is within about 2u of exact
// whatever k.
__device__ __forceinline__ void centred_norm(const float *xr, const float *center, int64_t k, float &norm,
                                             float &m)
{
#pragma clang fp contract(off)
    const int lane = threadIdx.x & 63;
    float s = 0.0f, comp = 0.0f;
    m = 0.0f;
#pragma unroll 4
    for (int64_t c = lane; c < k; c += 64) {
        const float v = xr[c] - center[c];
        const float p = v * v;
        const float pe = fmaf(v, v, -p);          // v * v = p + pe exactly
        const float t = s + p;
        const float bp = t - s;
        comp += ((s - (t - bp)) + (p - bp)) + pe;  // s + p = t + (TwoSum error)
        s = t;
        m = fmaxf(m, fabsf(v));
    }
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) {
        const float so = __shfl_xor(s, d, 64), co = __shfl_xor(comp, d, 64);
        const float t = s + so;
        const float bp = t - s;
        comp = (comp + co) + ((s - (t - bp)) + (so - bp));
        s = t;
        m = fmaxf(m, __shfl_xor(m, d, 64));
    }
    norm = s + comp;
}

// Row norms ||x_i - c||^2, for FP16 the power-of-two row scales and their
// inverses, and every centred value x - c split once into operand blocks
// (gt_mfma.h; features k..kp-1 and rows past n are zero).  `split` workgroups
// per block of 32 rows: a wave per row for the norms, then a wave per chunk of
// 16 features, one 1 KB block per term.  One launch and one read of the rows
// from memory; a kernel for the norms and one for the terms took 5.1 + 8.5 us
// at 9001 x 130, this one 13.5, and its
// launch comes once.
template <int SPLIT, bool VEC4>
__global__ __launch_bounds__(PREP_THREADS) void row_prep_kernel(const float *__restrict__ x, int64_t n,
                                                                int64_t k, int64_t ldx, int64_t kp, int split,
                                                                const float *__restrict__ center,
                                                                float *__restrict__ norms,
                                                                float *__restrict__ scales,
                                                                float *__restrict__ iscales,
                                                                unsigned short *__restrict__ terms)
{
    constexpr int NT = Split<SPLIT>::NT;
    __shared__ float row_scale[32];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t part = blockIdx.x % split, blocks = operand_rows(n) / 32, nch = kp / OPERAND_K;
    for (int64_t rb = blockIdx.x / split; rb < blocks; rb += gridDim.x / split) {
        __syncthreads();   // the last block's scales are read
        for (int q = wave; q < 32 && (SPLIT == SPLIT_FP16 || part == 0); q += PREP_WAVES) {
            const int64_t row = rb * 32 + q;
            if (row >= n) break;
            float norm, m;
            centred_norm(x + row * ldx, center, k, norm, m);
            if (lane != 0) continue;
            if (part == 0) norms[row] = norm;
            if (SPLIT == SPLIT_FP16) {
                // power of two that brings max|x - c| into [2^14, 2^15)
                int e = 0;
                if (m > 0.0f) {
                    e = ilogbf(m);
                    if (e < -100) e = -100;
                    if (e > 100) e = 100;
                }
                row_scale[q] = ldexpf(1.0f, 14 - e);
                if (part == 0) {
                    scales[row] = row_scale[q];
                    iscales[row] = ldexpf(1.0f, e - 14);
                }
            }
        }
        __syncthreads();
        const int64_t row = rb * 32 + (lane & 31), r = row < n ? row : n - 1;
        const float sc = SPLIT == SPLIT_FP16 && row < n ? row_scale[lane & 31] : 1.0f;
        for (int64_t ch = part * PREP_WAVES + wave; ch < nch; ch += (int64_t)split * PREP_WAVES) {
            const int64_t c0 = ch * OPERAND_K + (lane >> 5) * 8;
            float v[8];
            if (VEC4 && c0 + 8 <= k) {
                const float4 a = *reinterpret_cast<const float4 *>(x + r * ldx + c0);
                const float4 b = *reinterpret_cast<const float4 *>(x + r * ldx + c0 + 4);
                const float4 ca = *reinterpret_cast<const float4 *>(center + c0);
                const float4 cb = *reinterpret_cast<const float4 *>(center + c0 + 4);
                v[0] = a.x - ca.x; v[1] = a.y - ca.y; v[2] = a.z - ca.z; v[3] = a.w - ca.w;
                v[4] = b.x - cb.x; v[5] = b.y - cb.y; v[6] = b.z - cb.z; v[7] = b.w - cb.w;
            } else {
#pragma unroll
                for (int c = 0; c < 8; ++c) v[c] = (c0 + c < k) ? x[r * ldx + c0 + c] - center[c0 + c] : 0.0f;
            }
            unsigned short t[8][NT];
#pragma unroll
            for (int c = 0; c < 8; ++c) {
                if (SPLIT == SPLIT_FP16) v[c] *= sc;
                Split<SPLIT>::split(v[c], t[c]);
            }
#pragma unroll
            for (int q = 0; q < NT; ++q) {
                uint4 w;
                w.x = t[0][q] | ((unsigned)t[1][q] << 16);
                w.y = t[2][q] | ((unsigned)t[3][q] << 16);
                w.z = t[4][q] | ((unsigned)t[5][q] << 16);
                w.w = t[6][q] | ((unsigned)t[7][q] << 16);
                if (row >= n) w = make_uint4(0, 0, 0, 0);
                *reinterpret_cast<uint4 *>(terms + ((rb * nch + ch) * NT + q) * OPERAND_VALUES + lane * 8) = w;
            }
        }
    }
}

template <int SPLIT, int LAYOUT, bool VEC4, int NW>
hipError_t launch_tiles(GramArgs &args, hipStream_t stream)
{
    const int64_t S = (args.T + GSUPER - 1) / GSUPER;
    const int64_t ids = S * (S + 1) / 2 * GSUPER * GSUPER * Tile<NW>::PARTS;
    const int64_t max_ids = int64_t(1) << 23;
    for (int64_t off = 0; off < ids; off += max_ids) {
        args.id_offset = off;
        args.ids_this = (ids - off) < max_ids ? (ids - off) : max_ids;
        hipLaunchKernelGGL((gram_tile_kernel<SPLIT, LAYOUT, VEC4, NW>), dim3((unsigned)args.ids_this),
                           dim3(Tile<NW>::THREADS), 0, stream, args);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

// Half squares while every half has a CU to itself (3000 points x 256 features
// 74 -> 58 us in BF16, x 1024 162 -> 110), and for short rows, where a tile's
// stores take as long as its products and the second workgroup fills them
// (30000 x 64: 740 -> 716 us BF16, 649 -> 625 FP16; 9001 x 130 FP16 114 -> 109).
// Else whole squares, which read fewer operands per pair (30000 x 1024 BF16
// 4.73 ms whole, 5.16 halves).
bool half_squares(const GramArgs &args, int terms)
{
    return args.T * (args.T + 1) <= 256 || args.kp * terms <= 512;
}

template <int SPLIT, int LAYOUT, bool VEC4>
hipError_t launch_waves(GramArgs &args, hipStream_t stream)
{
    return half_squares(args, Split<SPLIT>::NT) ? launch_tiles<SPLIT, LAYOUT, VEC4, 8>(args, stream)
                                                : launch_tiles<SPLIT, LAYOUT, VEC4, 16>(args, stream);
}

template <int SPLIT>
hipError_t launch_layout(int layout, bool vec4, GramArgs &args, hipStream_t stream)
{
    if (layout == OUT_PACKED)
        return vec4 ? launch_waves<SPLIT, OUT_PACKED, true>(args, stream)
                    : launch_waves<SPLIT, OUT_PACKED, false>(args, stream);
    return vec4 ? launch_waves<SPLIT, OUT_FULL, true>(args, stream)
                : launch_waves<SPLIT, OUT_FULL, false>(args, stream);
}

template <int SPLIT>
hipError_t launch_rows(bool vec4, const float *x, int64_t n, int64_t k, int64_t ldx, const GramPrep &prep,
                       hipStream_t stream)
{
    // workgroups per block of 32 rows: to fill the CUs, while each has a chunk
    // per wave
    const int64_t blocks = operand_rows(n) / 32;
    int64_t split = 512 / (blocks > 0 ? blocks : 1), most = prep.kp / OPERAND_K / PREP_WAVES;
    if (split > most) split = most;
    if (split < 1) split = 1;
    const dim3 grid((unsigned)((blocks < 65536 ? blocks : 65536) * split));
    if (vec4)
        hipLaunchKernelGGL((row_prep_kernel<SPLIT, true>), grid, dim3(PREP_THREADS), 0, stream, x, n, k, ldx,
                           prep.kp, (int)split, prep.center, prep.norms, prep.scales, prep.iscales, prep.terms);
    else
        hipLaunchKernelGGL((row_prep_kernel<SPLIT, false>), grid, dim3(PREP_THREADS), 0, stream, x, n, k, ldx,
                           prep.kp, (int)split, prep.center, prep.norms, prep.scales, prep.iscales, prep.terms);
    return hipGetLastError();
}

bool rows_vec4(const float *x, int64_t k, int64_t ldx)
{
    return (k % 4 == 0) && (ldx % 4 == 0) && ((reinterpret_cast<uintptr_t>(x) & 15u) == 0);
}

size_t align256(size_t v) { return (v + 255) / 256 * 256; }

int64_t padded_k(int64_t k) { return (k + KPAD - 1) / KPAD * KPAD; }

int split_terms(int precision) { return precision == 1 ? 3 : 2; }

}  // namespace

int64_t colstats_blocks(int64_t n) { return (n + CS_ROWS - 1) / CS_ROWS; }

// Workspace: split terms (NT x rows x kp 16-bit values, rows = n rounded up to
// 32), then norms, scales and
// inverse scales (n floats each), the column centres (k floats) and the
// partial column statistics (3 x ceil(n / 256) x k floats).
static size_t terms_bytes(int64_t rows, int64_t k, int precision)
{
    return align256((size_t)split_terms(precision) * (size_t)rows * (size_t)padded_k(k) *
                    sizeof(unsigned short));
}

// Above this tau nearly every pair would be recomputed: the request is
// computed by the FP32 difference kernel instead (from 8305 features on in BF16,
// 15457 in FP16), which needs no workspace.
constexpr float GRAM_TAU_MAX = 0.9f;

static int64_t terms_rows(int64_t n, int64_t k, int precision)
{
    return gram_tau(precision, k) > GRAM_TAU_MAX ? n : operand_rows(n);
}

// Bytes of gram_workspace_bytes that come from rounding the rows up to 32: at
// most GRAM_ROW_SLACK.
size_t gram_rounding_bytes(int64_t n, int64_t k, int precision)
{
    return terms_bytes(terms_rows(n, k, precision), k, precision) - terms_bytes(n, k, precision);
}

size_t gram_workspace_bytes(int64_t n, int64_t k, int precision)
{
    return terms_bytes(terms_rows(n, k, precision), k, precision) + 3 * align256((size_t)n * sizeof(float)) + align256((size_t)k * sizeof(float)) +
           3 * align256((size_t)colstats_blocks(n) * (size_t)k * sizeof(float));
}

// Cancellation threshold: pairs with d^2 < tau (||x||^2 + ||y||^2) (norms
// of the centred rows) are recomputed from exact differences of the original
// rows.  The Gram-form error of d^2, in units of ||x||^2 + ||y||^2
// (u = 2^-24):
//   split    BF16 three terms: 4u; FP16 two terms: 12u (= 3 * 2^-22)
//            (|dg| <= c sum|x_c y_c| <= c (||x||^2+||y||^2)/2 and |d(d^2)| = 2|dg|)
//   accumulation of the MFMA partial sums, one FP32 rounding per product
//            instruction: statistical bound 4 sqrt(#adds) u
//   norms    4u for the two compensated row norms together
//   final    3u for ||x||^2 + ||y||^2 - 2g
// Relative to d^2 of a pair that is not flagged (d^2 >= tau (...)), that is
// at most E / tau.  Centring moves each difference x_c - y_c by at most
// u (|x~_c| + |y~_c|), so d^2 by at most 2u d (||x~|| + ||y~||) <=
// 2u sqrt(2 / tau) d^2 <= 8u d^2 for tau >= 1/8.  tau is chosen so that
// E / tau + 8u = 1.6e-5, the allowed relative error of d^2 (8e-6 on d).
float gram_tau(int precision, int64_t k)
{
    const double u = 1.0 / 16777216.0;
    const bool bf16 = (precision == 1);
    const double split = bf16 ? 4.0 * u : 12.0 * u;
    const double nadds = (bf16 ? 6.0 : 3.0) * (double)((k + 15) / 16);
    const double accum = 4.0 * sqrt(nadds) * u;
    const double total = split + accum + 4.0 * u + 3.0 * u;
    const double tau = total / (1.6e-5 - 8.0 * u);
    return (float)(tau > 0.125 ? tau : 0.125);
}

// The pre-passes: column centres, row norms (FP16: row scales) and the split
// terms, all in the workspace (gram_workspace_bytes).
hipError_t gram_prepare(int precision, const float *x, int64_t n, int64_t k, int64_t ldx, void *workspace,
                        GramPrep &prep, hipStream_t stream)
{
    prep.kp = padded_k(k);
    char *ws = static_cast<char *>(workspace);
    prep.terms = reinterpret_cast<unsigned short *>(ws);
    ws += align256((size_t)split_terms(precision) * (size_t)operand_rows(n) * (size_t)prep.kp *
                   sizeof(unsigned short));
    prep.norms = reinterpret_cast<float *>(ws);
    ws += align256((size_t)n * sizeof(float));
    prep.scales = reinterpret_cast<float *>(ws);
    ws += align256((size_t)n * sizeof(float));
    prep.iscales = reinterpret_cast<float *>(ws);
    ws += align256((size_t)n * sizeof(float));
    prep.center = reinterpret_cast<float *>(ws);
    ws += align256((size_t)k * sizeof(float));
    const int64_t csb = colstats_blocks(n);
    const size_t pbytes = align256((size_t)csb * (size_t)k * sizeof(float));
    float *psum = reinterpret_cast<float *>(ws);
    float *pmin = reinterpret_cast<float *>(ws + pbytes);
    float *pmax = reinterpret_cast<float *>(ws + 2 * pbytes);
    const bool fp16 = (precision == 2);
    {
        const int64_t cb = (k + 63) / 64;
        hipLaunchKernelGGL(colstats_partial_kernel, dim3((unsigned)csb, (unsigned)(cb < 1024 ? cb : 1024)),
                           dim3(PREP_THREADS), 0, stream, x, n, k, ldx, psum, pmin, pmax);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        const int64_t fb = (k + CS_COLS - 1) / CS_COLS;
        hipLaunchKernelGGL(colstats_finish_kernel, dim3((unsigned)(fb < 65536 ? fb : 65536)), dim3(256),
                           0, stream, psum, pmin, pmax, csb, n, k, prep.center);
        e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    const bool vec4 = rows_vec4(x, k, ldx);
    return fp16 ? launch_rows<SPLIT_FP16>(vec4, x, n, k, ldx, prep, stream)
                : launch_rows<SPLIT_BF16>(vec4, x, n, k, ldx, prep, stream);
}

hipError_t launch_gram(int precision, int layout, const float *x, int64_t n, int64_t k,
                       int64_t ldx, float *out, int64_t ldd, void *workspace, hipStream_t stream)
{
    if (n < 2 && layout == OUT_PACKED) return hipSuccess;
    const float tau = gram_tau(precision, k);
    if (tau > GRAM_TAU_MAX)
        return launch_plain(OP_EUCLID, layout, x, n, ldx, x, n, ldx, k, 2.0f, out, ldd, stream);
    GramPrep prep;
    hipError_t e = gram_prepare(precision, x, n, k, ldx, workspace, prep, stream);
    if (e != hipSuccess) return e;
    const bool fp16 = (precision == 2);
    GramArgs args;
    args.x = x;
    args.n = n;
    args.k = k;
    args.ldx = ldx;
    args.terms = prep.terms;
    args.kp = prep.kp;
    args.norms = prep.norms;
    args.iscale = prep.iscales;
    args.out = out;
    args.ldd = ldd;
    args.T = (n + GBM - 1) / GBM;
    args.tau = tau;
    const bool vec4 = rows_vec4(x, k, ldx);
    return fp16 ? launch_layout<SPLIT_FP16>(layout, vec4, args, stream)
                : launch_layout<SPLIT_BF16>(layout, vec4, args, stream);
}

}  // namespace gt
