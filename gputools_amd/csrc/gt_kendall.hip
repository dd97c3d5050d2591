// gt_kendall.hip -- Kendall's tau of gpuCor(method = "kendall") on gfx950.
//
// Replaces masterKendall (src/kendall.cpp:13-55) and gpuKendall
// (inst/cuda/kendall.cu:4-47).  For variables x (of A) and y (of B) over n
// samples, gputools counts the sample pairs i < j that are concordant, where
//   (x_j > x_i and y_j > y_i) or (x_j < x_i and y_j < y_i)
//   or (x_j == x_i and y_j == y_i)                        (kendall.cu:18-22)
// (any comparison with NaN is false), and returns
//   (concordant - discordant) / (n (n - 1) / 2),  discordant = that - concordant
// with the final steps in FP32 and the quotient in FP64 (kendall.cu:40-45).
// It runs one 256-thread block per pair of variables, each re-comparing the
// raw values of both variables n^2/2 times.
//
// Here the comparisons are made once per variable, and the counting is a
// contraction on the matrix cores.  A planes pass writes each sample pair of a
// variable as bits: P (x_j > x_i) always, N (x_j < x_i) and E (x_j == x_i)
// only where a tie or a non-finite value makes them more than ~P and 0.
// Where every sample pair of two variables is exactly one of P and N, the
// number of agreeing pairs is (bits + sum s s') / 2 with s = +1 or -1: the
// count pass expands the bits to FP4 values (E2M1: the sign is the bit, the
// magnitude 1) in registers and sums the products with
// v_mfma_f32_32x32x64_f8f6f4, exactly, as FP32 sums of integers below 2^24.
// Elsewhere it sums the 0/1 products of the three planes, also in FP4.
// The reference accumulates the count in FP32 (kendall.cu:14, 23, 28-38):
// below 2^24 concordant pairs (always when n <= 5793) that sum is exact and
// the results are identical; above it the reference's sum can round, and this
// build keeps the exact count.
#include "gt_common.h"
#include "gt_internal.h"

namespace gt {
namespace {

// ---------------------------------------------------------------------------
// Layout of the sample pairs
// ---------------------------------------------------------------------------
// Sample pairs (i, j) are cut into tiles of 64 rows i by 32 columns j: tile
// (rb, jw) holds i = 64 rb + r and j = 32 jw + u, for every rb and every jw
// from 2 rb on (j > i).  A tile is 64 words per variable, word r = row r, bit
// u = column u.  The bits of the tile that are no sample pair (j <= i, or past
// the end) have P = E = 0 and N = 1 for every variable, so they count as
// agreeing everywhere and the finish pass subtracts their number.
//
// Variables are taken in blocks of 32 and words in groups of 8, the operand of
// four matrix products: group g of block vb is 1 KB, 16 bytes for each of 64
// lanes, lane 32 h + v holding words 8 q + 4 h .. + 3 of variable 32 vb + v.
// The count pass moves groups as they are from memory to LDS to registers.
constexpr int KVB = 32;      // variables per block
constexpr int KGW = 8;       // words per group
constexpr int KTG = 8;       // groups per tile of sample pairs (64 words)
constexpr int KGWORDS = KVB * KGW;   // words of one group (256, 1 KB)

// Tiles before row block rb (jwn = ceil(n / 32) column words).
__host__ __device__ __forceinline__ int64_t tiles_before(int64_t rb, int64_t jwn)
{
    return rb * jwn - rb * (rb - 1);
}

__host__ __device__ __forceinline__ int64_t column_words(int64_t n) { return (n + 31) / 32; }

__host__ __device__ __forceinline__ int64_t pair_tiles(int64_t n)
{
    return tiles_before((n - 1 + 63) / 64, column_words(n));
}

// ---------------------------------------------------------------------------
// Planes pass
// ---------------------------------------------------------------------------
struct PlanesSide {
    const float *x;
    int64_t nvar, ldx;
    uint32_t *planes;    // plane p (0 = P, 1 = N, 2 = E), block vb, group g at
                         // ((p * nvb + vb) * ngroups + g) * KGWORDS
    uint8_t *flags;      // flags[g * fstride + vb]: the group's N and E words are stored
    int64_t nvb, fstride;
};

struct PlanesArgs {
    PlanesSide a, b;     // b.nvb = 0: the self case
    int64_t n, ngroups;
    int64_t tile_begin, ntiles;   // this segment's tiles of sample pairs
    int64_t runs;
    int64_t run;         // tiles per workgroup
    // the counts, cleared here before the first count pass adds to them (by
    // stores, not a memset node, so that a captured graph replays correctly)
    unsigned long long *count;
    int64_t ncount;
};

constexpr int KRUN = 4;      // tiles per workgroup

// x read through the scalar cache: uniform addresses, not written by the kernel
typedef const __attribute__((address_space(4))) float uniform_float_t;

// One workgroup per (variable block, run of tiles); a wave takes 8 variables,
// a lane one row i.  The bit of (i, j) is the sign of x_i - x_j, shifted into
// the lane's word by v_alignbit_b32: a subtract and a shift per 64 sample
// pairs, plus half a v_min3_u32 that notices a zero difference.  x_i has its
// zero made +0, so that equal values always give the difference +0.  x_j is
// uniform and comes through scalar loads.  This took 1024 variables x 2048
// samples from 0.52 ms (a ballot per 64 pairs, moved between lanes) to
// 0.23 ms.  Bound: VALU issue (1.2e8 wave instructions, 108 per word of 64
// lanes: 80 in the column loop, the rest masks, tests and the LDS transpose).
// A word with a zero difference or a non-finite value is redone (from the columns
// in the lanes: few variables with ties took 76 us of scalar loads, 15 so) with the
// three comparisons; if it holds a tie (or a NaN may be about), its group is
// flagged and the N and E words of the whole group are stored.
__global__ __launch_bounds__(256) void kendall_planes_kernel(PlanesArgs args)
{
    // a tile's P words, padded so that the 16 four-word pieces of a wave's
    // store fall in different banks
    constexpr int HS = 132, QS = 264;
    __shared__ __attribute__((aligned(16))) uint32_t buf[2][KTG * QS];
    __shared__ unsigned special[3];   // per tile: groups whose N and E words are needed
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    for (int64_t e = (int64_t)blockIdx.x * 256 + tid; e < args.ncount; e += (int64_t)gridDim.x * 256)
        args.count[e] = 0ull;
    const int64_t n = args.n, jwn = column_words(n);
    int64_t vb = blockIdx.x / args.runs;
    const int64_t run = blockIdx.x % args.runs;
    const bool second = vb >= args.a.nvb;
    if (second) vb -= args.a.nvb;
    const int64_t nvb = second ? args.b.nvb : args.a.nvb, nvar = second ? args.b.nvar : args.a.nvar;
    const int64_t ldx = second ? args.b.ldx : args.a.ldx, fstride = second ? args.b.fstride : args.a.fstride;
    uint8_t *const flags = second ? args.b.flags : args.a.flags;
    const int64_t tb = run * args.run;
    const int nt = (int)(args.ntiles - tb < args.run ? args.ntiles - tb : args.run);
    const int64_t t0 = args.tile_begin + tb;
    // row block of tile t0: the last rb with tiles_before(rb) <= t0
    int64_t rb;
    {
        const double b = (double)(jwn + 1);
        rb = (int64_t)((b - sqrt(fmax(b * b - 4.0 * (double)t0, 0.0))) * 0.5);
        while (rb > 0 && tiles_before(rb, jwn) > t0) --rb;
        while (tiles_before(rb + 1, jwn) <= t0) ++rb;
    }
    int64_t jw = 2 * rb + (t0 - tiles_before(rb, jwn));
    const int64_t v0 = vb * KVB + wave * 8;
    const float *const x = second ? args.b.x : args.a.x;
    const int64_t pstride = nvb * args.ngroups * KGWORDS;
    uint32_t *const pv = (second ? args.b.planes : args.a.planes) + vb * args.ngroups * KGWORDS;
    const int slot = (lane >> 3) * QS + ((lane >> 2) & 1) * HS + (lane & 3);

    float xi[8];
    auto load_rows = [&]() {
        int64_t i = rb * 64 + lane;
        if (i > n - 1) i = n - 1;
#pragma unroll
        for (int vv = 0; vv < 8; ++vv) {
            const int64_t v = v0 + vv < nvar ? v0 + vv : nvar - 1;
            xi[vv] = x[v * ldx + i] + 0.0f;
        }
    };
    // the three comparisons of up to 32 columns, column u in bit u, which lane u
    // holds (scalar loads here would be waited for one after the other), eight at
    // a time: few samples have one tile of few columns
    auto exact = [&](float a, float xl, int cols, uint32_t &gt, uint32_t &lt, uint32_t &eq) {
        gt = lt = eq = 0u;
#pragma unroll 1
        for (int u0 = (cols - 1) & ~7; u0 >= 0; u0 -= 8)
#pragma unroll
            for (int u = u0 + 7; u >= u0; --u) {
                const float b = __uint_as_float((unsigned)__builtin_amdgcn_readlane((int)__float_as_uint(xl), u));
                gt = (gt << 1) | (b > a ? 1u : 0u);
                lt = (lt << 1) | (b < a ? 1u : 0u);
                eq = (eq << 1) | (b == a ? 1u : 0u);
            }
    };
    load_rows();
    if (tid == 0) special[0] = 0u;
    __syncthreads();
    for (int k = 0; k < nt; ++k) {
        if (tid == 0) special[(k + 1) % 3] = 0u;   // last read two tiles ago
        const int64_t j0 = jw * 32;
        const int cols = n - j0 < 32 ? (int)(n - j0) : 32;
        // bits of the columns i < j < n
        const int lo = (int)(rb * 64 - j0) + lane + 1;   // -n .. 64
        uint32_t valid = cols >= 32 ? 0xffffffffu : (1u << cols) - 1u;
        if (lo > 0) valid &= lo >= 32 ? 0u : 0xffffffffu << lo;
        unsigned sp = 0, compared = 0;   // compared: the variables with ltw and eqw
        uint32_t ltw[8], eqw[8];         // x_j < x_i and x_j == x_i
        uint32_t *const pb = buf[k & 1] + slot + wave * 8 * 4;
#pragma unroll
        for (int vv = 0; vv < 8; ++vv) {
            const int64_t v = v0 + vv < nvar ? v0 + vv : nvar - 1;
            const float *xv = x + v * ldx + j0;
            uniform_float_t *xj = (uniform_float_t *)xv;
            const float xl = xv[(lane & 31) < cols ? lane & 31 : cols - 1];
            uint32_t w = 0u, m = 0xffffffffu;
            if (cols == 32) {
#pragma unroll
                for (int u = 31; u >= 0; --u) {
                    const uint32_t d = __float_as_uint(xi[vv] - xj[u]);
                    w = __builtin_amdgcn_alignbit(w, d, 31);
                    m = d < m ? d : m;
                }
            }
            const bool odd = !(fabsf(xi[vv]) < INFINITY) || !(fabsf(xl) < INFINITY);
            const unsigned long long oddw = __builtin_amdgcn_ballot_w64(odd);
            // (a tile of fewer columns, the only one of few samples, is compared at
            // once: 300 variables x 7 samples 15.8 us with the differences first,
            // which took each x_i - x_i for a tie, 8.1 so)
            if (cols < 32 || (__builtin_amdgcn_ballot_w64(m == 0u) | oddw)) {
                uint32_t lt, eq;
                exact(xi[vv], xl, cols, w, lt, eq);
                ltw[vv] = lt;
                eqw[vv] = eq;
                compared |= 1u << vv;
                const unsigned long long tied = __builtin_amdgcn_ballot_w64((eq & valid) != 0u);
                if (oddw) {
                    sp = 0xffu;
                } else {
#pragma unroll
                    for (int q = 0; q < KTG; ++q)
                        if ((tied >> (8 * q)) & 0xffull) sp |= 1u << q;
                }
            }
            pb[vv * 4] = w & valid;
        }
        if (sp != 0u && lane == 0) atomicOr(&special[k % 3], sp);
        __syncthreads();
        const int64_t g = (tb + k) * KTG;
        uint32_t *const pt = pv + g * KGWORDS;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int unit = tid + 256 * h, q = unit >> 6, l = unit & 63;
            *reinterpret_cast<uint4 *>(pt + unit * 4) =
                *reinterpret_cast<const uint4 *>(buf[k & 1] + q * QS + (l >> 5) * HS + (l & 31) * 4);
        }
        const unsigned mask = special[k % 3];
        if (tid < KTG) flags[(g + tid) * fstride + vb] = (uint8_t)((mask >> tid) & 1u);
        if (mask != 0u) {
            const int q = lane >> 3;
            uint32_t *const po = pt + q * KGWORDS + ((lane >> 2) & 1) * 128 + (lane & 3);
#pragma unroll
            for (int vv = 0; vv < 8; ++vv) {
                // not compared: no tie and nothing odd, so N = ~P and E = 0
                const bool c = (compared >> vv) & 1u;
                const uint32_t lt = c ? (ltw[vv] & valid) | ~valid : ~pb[vv * 4];
                const uint32_t eq = c ? eqw[vv] & valid : 0u;
                if ((mask >> q) & 1u) {
                    po[pstride + (wave * 8 + vv) * 4] = lt;
                    po[2 * pstride + (wave * 8 + vv) * 4] = eq;
                }
            }
        }
        if (++jw == jwn && k + 1 < nt) {
            ++rb;
            jw = 2 * rb;
            load_rows();
        }
    }
}

// ---------------------------------------------------------------------------
// Count pass
// ---------------------------------------------------------------------------
constexpr int KBX = 256, KBY = 128;      // variables per tile side
constexpr int KTX = KBX / KVB, KTY = KBY / KVB;   // blocks per tile side
constexpr int KTHREADS = 256;            // 4 waves, 2 (x) x 2 (y), 128 x 64 pairs each
constexpr int KSTAGE = (KTX + KTY) * KGWORDS * 4;   // bytes of one group of both sides (12 KB)
constexpr int KNSTAGE = 4;
// FP32 sums of +-2 per bit stay exact below 2^24: 32768 groups of 256 bits
constexpr int64_t KMAXGROUPS = 32000;

typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef int i32x8_t __attribute__((ext_vector_type(8)));
typedef float kf32x16_t __attribute__((ext_vector_type(16)));

struct KendallArgs {
    const uint32_t *pa, *pb;   // planes of A and B (PlanesArgs)
    const uint8_t *fa, *fb;
    int64_t nvb_a, nvb_b, fs_a, fs_b, ngroups;
    int64_t na, nb;
    unsigned long long *count; // na x nb (row stride ldc), pair (x, y) at x * ldc + y
    int64_t ldc;
    int64_t tiles_b, ntiles;
    int64_t split_g;           // groups per workgroup
    int64_t id_offset, ids_this;
};

// 32 bits -> 32 FP4 values: nibble t of dword s is bit 4 t + s of w, placed at
// mask's bit of the nibble, over the other bits of one.  Signs: mask 8, one 2
// (+1 where the bit is clear, -1 where it is set).  0 / 1: w rotated right by
// 2, mask 2; 0 / 2: w rotated right by 1, mask 4; one 0.
__device__ __forceinline__ i32x8_t expand(uint32_t w, uint32_t mask, uint32_t one)
{
    i32x8_t r = {};
#pragma unroll
    for (int s = 0; s < 4; ++s)
        r[s] = (int)(((s < 3 ? __builtin_rotateleft32(w, 3 - s) : w) & mask) | one);
    return r;
}

// Four blocks of side A and two of side B, 16 bytes a lane, loaded and waited
// for here: as ordinary loads in the loop they would make the compiler wait
// for every load in flight, the ring's among them, in groups that do not take
// this path (634 against 612 us for the whole pass).
__device__ __forceinline__ void load_six(const uint32_t *a, const int64_t (&sa)[4], const uint32_t *b,
                                         const int64_t (&sb)[2], u32x4_t (&w)[6])
{
    const uint32_t *a0 = a + sa[0], *a1 = a + sa[1], *a2 = a + sa[2], *a3 = a + sa[3];
    const uint32_t *b0 = b + sb[0], *b1 = b + sb[1];
    asm volatile("global_load_dwordx4 %0, %6, off\n\t"
                 "global_load_dwordx4 %1, %7, off\n\t"
                 "global_load_dwordx4 %2, %8, off\n\t"
                 "global_load_dwordx4 %3, %9, off\n\t"
                 "global_load_dwordx4 %4, %10, off\n\t"
                 "global_load_dwordx4 %5, %11, off\n\t"
                 "s_waitcnt vmcnt(0)"
                 : "=&v"(w[0]), "=&v"(w[1]), "=&v"(w[2]), "=&v"(w[3]), "=&v"(w[4]), "=&v"(w[5])
                 : "v"(a0), "v"(a1), "v"(a2), "v"(a3), "v"(b0), "v"(b1)
                 : "memory");
}

__device__ __forceinline__ kf32x16_t mfma_fp4(i32x8_t a, i32x8_t b, kf32x16_t c)
{
    // format 4 = E2M1 on both sides, block scales 2^0
    return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a, b, c, 4, 4, 0, 127, 0, 127);
}

// A 256 x 128 tile of pairs of variables over a range of groups.  Both sides'
// groups stream from memory through a four-stage LDS ring (direct loads); a
// wave expands its 4 + 2 blocks in registers, 7 VALU instructions per operand
// of two (A) or four (B) products, which leaves the matrix cores the longer
// side (256 against 168 cycles per 64 sample pairs and wave).  The popcount
// form this replaces spent 2 VALU operations per 32 sample pairs and pair.
// 1024 variables x 2048 samples, self case: 3.18 -> 0.61 ms, 4.6 PFLOP/s.
// Bound: the matrix cores at the clock they hold on such data; a register-only
// loop of the same products and expansions takes 0.51 - 0.61 ms (constant
// operands would run at 7.5 PFLOP/s, 0.38 ms).  256 x 256 tiles of 8 waves, one
// workgroup per CU, took 0.72 ms.
// SYM: pa == pb; tiles with J <= I only, and only x >= y is stored.
template <bool SYM>
__global__ __launch_bounds__(KTHREADS, 2) void kendall_count_kernel(KendallArgs args)
{
    __shared__ __attribute__((aligned(1024))) unsigned char smem[KNSTAGE * KSTAGE];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wx = wave >> 1, wy = wave & 1;
    const int64_t id = args.id_offset + xcd_remap(blockIdx.x, args.ids_this);
    const int64_t split = id / args.ntiles, t = id % args.ntiles;
    int64_t I, J;
    if (SYM) {
        // tile row I has 2 (I + 1) tiles
        I = (int64_t)((sqrt(4.0 * (double)t + 1.0) - 1.0) * 0.5);
        while ((I + 1) * (I + 2) <= t) ++I;
        while (I * (I + 1) > t) --I;
        J = t - I * (I + 1);
    } else {
        I = t / args.tiles_b;
        J = t % args.tiles_b;
    }
    const int64_t x0 = I * KBX, y0 = J * KBY;
    const int64_t g0 = split * args.split_g;
    int64_t g1 = g0 + args.split_g;
    if (g1 > args.ngroups) g1 = args.ngroups;
    if (g0 >= g1) return;
    const int ng = (int)(g1 - g0);
    // a wave with no pair, or none x >= y, only helps to load
    const bool idle = x0 + wx * 128 >= args.na || y0 + wy * 64 >= args.nb ||
                      (SYM && y0 + wy * 64 > x0 + wx * 128 + 127);

    // wave w loads blocks 3 w .. 3 w + 2 of the 8 + 4; blocks past a side's last
    // one repeat it (they only feed pairs that are not stored)
    typedef __attribute__((address_space(3))) void lds_void_t;
    typedef const __attribute__((address_space(1))) void gbl_void_t;
    const uint32_t *src[3];
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        const int blk = wave * 3 + q;
        const bool sb = blk >= KTX;
        const int64_t nvb = sb ? args.nvb_b : args.nvb_a;
        int64_t v = sb ? J * KTY + blk - KTX : I * KTX + blk;
        if (v >= nvb) v = nvb - 1;
        src[q] = (sb ? args.pb : args.pa) + (v * args.ngroups + g0) * KGWORDS + lane * 4;
    }
    auto issue = [&](int c) {
        unsigned char *const st = smem + (c % KNSTAGE) * KSTAGE + wave * 3 * (KGWORDS * 4);
#pragma unroll
        for (int q = 0; q < 3; ++q)
            __builtin_amdgcn_global_load_lds((gbl_void_t *)(src[q] + (int64_t)c * KGWORDS),
                                             (lds_void_t *)(st + q * KGWORDS * 4), 16, 0, 0);
    };
    // which of the next 64 groups hold N and E words for a block of this wave
    const int64_t la = args.nvb_a - (I * KTX + wx * 4), lb = args.nvb_b - (J * KTY + wy * 2);
    const uint32_t ma = la >= 4 ? 0xffffffffu : la > 0 ? (1u << (8 * (int)la)) - 1u : 0u;
    const uint32_t mb = lb >= 2 ? 0xffffu : lb > 0 ? 0xffu : 0u;
    const uint8_t *const fa = args.fa + I * KTX + wx * 4, *const fb = args.fb + J * KTY + wy * 2;
    auto flags_of = [&](int c, uint32_t &ua, uint32_t &ub) {
        ua = *reinterpret_cast<const uint32_t *>(fa + (g0 + c) * args.fs_a) & ma;
        ub = *reinterpret_cast<const uint16_t *>(fb + (g0 + c) * args.fs_b) & mb;
    };

    // this wave's blocks in the N and E planes of group g0 (blocks past the end
    // repeat the last one)
    int64_t step_a[4], step_b[2];
#pragma unroll
    for (int a = 0; a < 4; ++a)
        step_a[a] = (a < la ? a : la > 0 ? la - 1 : args.nvb_a - 1 - (I * KTX + wx * 4)) *
                    args.ngroups * KGWORDS;
#pragma unroll
    for (int b = 0; b < 2; ++b)
        step_b[b] = (b < lb ? b : lb > 0 ? lb - 1 : args.nvb_b - 1 - (J * KTY + wy * 2)) *
                    args.ngroups * KGWORDS;
    const int64_t pstride_a = args.nvb_a * args.ngroups * KGWORDS;
    const int64_t pstride_b = args.nvb_b * args.ngroups * KGWORDS;
    const uint32_t *const pside_a =
        args.pa + ((I * KTX + wx * 4) * args.ngroups + g0) * KGWORDS + lane * 4;
    const uint32_t *const pside_b =
        args.pb + ((J * KTY + wy * 2) * args.ngroups + g0) * KGWORDS + lane * 4;

    kf32x16_t acc[4][2];
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[a][b][r] = 0.0f;

    int nfast = 0;
    unsigned long long slow = 0;
#pragma unroll
    for (int c = 0; c < KNSTAGE - 1; ++c)
        if (c < ng) issue(c);
    for (int c = 0; c < ng; ++c) {
        if ((c & 63) == 0) {
            bool f = false;
            if (c + lane < ng) {
                uint32_t ua, ub;
                flags_of(c + lane, ua, ub);
                f = (ua | ub) != 0u;
            }
            slow = __builtin_amdgcn_ballot_w64(f);
        }
        // group c landed when at most the two later groups' loads are
        // outstanding (vector memory loads complete in order)
        if (c + 2 < ng)
            asm volatile("s_waitcnt vmcnt(6)" ::: "memory");
        else if (c + 1 < ng)
            asm volatile("s_waitcnt vmcnt(3)" ::: "memory");
        else
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        // every wave's part of group c is in LDS, and every wave is done with
        // group c - 1, whose stage the next issue overwrites
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (c + KNSTAGE - 1 < ng) issue(c + KNSTAGE - 1);
        if (idle) continue;
        const unsigned char *const st = smem + (c % KNSTAGE) * KSTAGE + lane * 16;
        const bool flagged = ((slow >> (c & 63)) & 1ull) != 0ull;
        uint32_t ua = 0, ub = 0, mask_a = 0x88888888u, mask_b = 0x88888888u, one = 0x22222222u;
        if (flagged) {
            // P P' + N N' + E E', twice: 0/1 on one side, 0/2 on the other
            flags_of(c, ua, ub);
            ua = __builtin_amdgcn_readfirstlane(ua);
            ub = __builtin_amdgcn_readfirstlane(ub);
            mask_a = 0x22222222u;
            mask_b = 0x44444444u;
            one = 0u;
        } else {
            ++nfast;
        }
        // one in a VGPR: v_and_or_b32 takes the mask as its only scalar
        asm("" : "+v"(one));
#pragma unroll 1
        for (int p = 0; p < (flagged ? 3 : 1); ++p) {
            u32x4_t pa[4], pb[2];
#pragma unroll
            for (int a = 0; a < 4; ++a)
                pa[a] = *reinterpret_cast<const u32x4_t *>(st + (wx * 4 + a) * (KGWORDS * 4));
#pragma unroll
            for (int b = 0; b < 2; ++b)
                pb[b] = *reinterpret_cast<const u32x4_t *>(st + (KTX + wy * 2 + b) * (KGWORDS * 4));
            if (flagged) {
                // the stored N or E words; a block whose group is not flagged
                // has N = ~P and E = 0
                if (p > 0) {
                    u32x4_t w[6];
                    load_six(pside_a + p * pstride_a + (int64_t)c * KGWORDS, step_a,
                             pside_b + p * pstride_b + (int64_t)c * KGWORDS, step_b, w);
#pragma unroll
                    for (int a = 0; a < 4; ++a)
                        pa[a] = ((ua >> (8 * a)) & 0xffu) ? w[a] : p == 1 ? ~pa[a] : (u32x4_t)0u;
#pragma unroll
                    for (int b = 0; b < 2; ++b)
                        pb[b] = ((ub >> (8 * b)) & 0xffu) ? w[4 + b] : p == 1 ? ~pb[b] : (u32x4_t)0u;
                }
#pragma unroll
                for (int a = 0; a < 4; ++a) pa[a] = (pa[a] >> 2) | (pa[a] << 30);
#pragma unroll
                for (int b = 0; b < 2; ++b) pb[b] = (pb[b] >> 1) | (pb[b] << 31);
            }
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                i32x8_t vb[2];
#pragma unroll
                for (int b = 0; b < 2; ++b) vb[b] = expand(pb[b][k], mask_b, one);
#pragma unroll
                for (int a = 0; a < 4; ++a) {
                    const i32x8_t va = expand(pa[a][k], mask_a, one);
#pragma unroll
                    for (int b = 0; b < 2; ++b) acc[a][b] = mfma_fp4(va, vb[b], acc[a][b]);
                }
                // keeps the expansions of later steps, and their registers,
                // behind this step's products
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    }
    if (idle) return;

    // acc = 2 agreeing - bits over the +-1 groups, 2 agreeing over the others.
    // 32 x 32 accumulator layout: element r of lane l is x row 8 (r / 4) +
    // 4 (l / 32) + r % 4 and y column l % 32.
    const int bits = nfast * (KGW * 32);
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int64_t x = x0 + wx * 128 + a * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                const int64_t y = y0 + wy * 64 + b * 32 + (lane & 31);
                if (x < args.na && y < args.nb && (!SYM || x >= y))
                    atomicAdd(args.count + x * args.ldc + y,
                              (unsigned long long)(((int)acc[a][b][r] + bits) >> 1));
            }
        }
}

// tau from the exact count, with the reference's arithmetic (kendall.cu:40-45);
// count == nullptr: no sample pairs (n < 2), the count is 0.  nopair: bits of
// the tiles that are no sample pair, which the count pass counted.
__global__ void kendall_finish_kernel(const unsigned long long *__restrict__ count, int64_t ldc,
                                      int64_t na, int64_t nb, int64_t n, int sym,
                                      unsigned long long nopair, double *__restrict__ tau,
                                      int64_t ldt)
{
    const int64_t total = na * nb;
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < total;
         e += (int64_t)gridDim.x * blockDim.x) {
        const int64_t x = e % na, y = e / na;
        const bool lower = !sym || x >= y;
        const unsigned long long c =
            count ? (lower ? count[x * ldc + y] : count[y * ldc + x]) - nopair : 0ull;
        const float concordant = (float)c;
        float denom = (float)n;
        denom = (denom * (denom - 1.0f)) / 2.0f;
        const float discordant = denom - concordant;
        const float numer = concordant - discordant;
        tau[y * ldt + x] = (double)numer / (double)denom;
    }
}

unsigned grid_for(int64_t total, int threads)
{
    int64_t blocks = (total + threads - 1) / threads;
    if (blocks > 65536) blocks = 65536;
    if (blocks < 1) blocks = 1;
    return (unsigned)blocks;
}

size_t align256(size_t v) { return (v + 255) / 256 * 256; }

// Workspace: planes and flags of one segment of the tiles of sample pairs,
// then the counts.  A segment takes as many tiles as keep the planes within
// three bits per sample pair and variable (blocks of 32 variables hold more
// than that when there are few variables), and at least 64 MiB; the segments
// run one after the other.
struct KendallPlan {
    int64_t tiles, seg;                  // tiles of sample pairs in all, per segment
    int64_t nvb_a, nvb_b, fs_a, fs_b;
    size_t off_pb, off_fa, off_fb, off_count, bytes;
};

KendallPlan kendall_plan(int64_t na, int64_t nb, bool same, int64_t n)
{
    KendallPlan k;
    k.tiles = pair_tiles(n);
    k.nvb_a = (na + KVB - 1) / KVB;
    k.nvb_b = same ? 0 : (nb + KVB - 1) / KVB;
    k.fs_a = (k.nvb_a + KTX - 1) / KTX * KTX;
    k.fs_b = (k.nvb_b + KTX - 1) / KTX * KTX;
    const double tile_bytes = 3.0 * KTG * KGWORDS * 4 * (double)(k.nvb_a + k.nvb_b);
    double cap = 3.0 / 8.0 * ((double)n * (double)(n - 1) / 2.0) * (double)(same ? na : na + nb);
    if (cap < 67108864.0) cap = 67108864.0;
    // a whole problem that is over by the tiles' rounding stays one segment
    const double want = cap * 1.07 / tile_bytes;
    k.seg = want < 1.0 ? 1 : want < (double)k.tiles ? (int64_t)want : k.tiles;
    size_t p = 3 * (size_t)k.nvb_a * (size_t)k.seg * KTG * KGWORDS * 4;
    k.off_pb = p;
    p += 3 * (size_t)k.nvb_b * (size_t)k.seg * KTG * KGWORDS * 4;
    k.off_fa = p;
    p += align256((size_t)k.seg * KTG * (size_t)k.fs_a);
    k.off_fb = p;
    p += align256((size_t)k.seg * KTG * (size_t)k.fs_b);
    k.off_count = p;
    k.bytes = p + align256((size_t)na * (size_t)nb * 8);
    return k;
}

// One launch for both sides, which clears the counts too: small calls take as
// long as their launches.
hipError_t launch_planes(PlanesArgs &args, int64_t begin, int64_t tiles, hipStream_t stream)
{
    const int64_t nvb = args.a.nvb + args.b.nvb;
    args.ngroups = tiles * KTG;
    args.tile_begin = begin;
    args.ntiles = tiles;
    // tiles per workgroup: as many as leave about four workgroups per CU
    args.run = nvb * tiles / 1024;
    args.run = args.run < 1 ? 1 : args.run > KRUN ? KRUN : args.run;
    args.runs = (tiles + args.run - 1) / args.run;
    hipLaunchKernelGGL(kendall_planes_kernel, dim3((unsigned)(nvb * args.runs)), dim3(256), 0,
                       stream, args);
    return hipGetLastError();
}

}  // namespace

size_t kendall_workspace_bytes(int64_t na, int64_t nb, bool same, int64_t n)
{
    if (na <= 0 || nb <= 0 || n < 2) return 0;
    return kendall_plan(na, nb, same, n).bytes;
}

hipError_t launch_kendall(const float *a, int64_t na, int64_t lda, const float *b, int64_t nb,
                          int64_t ldb, bool same, int64_t n, double *tau, int64_t ldt,
                          void *workspace, hipStream_t stream)
{
    if (na <= 0 || nb <= 0) return hipSuccess;
    hipError_t e;
    unsigned long long *count = nullptr;
    unsigned long long nopair = 0;
    if (n >= 2) {
        const KendallPlan k = kendall_plan(na, nb, same, n);
        char *ws = static_cast<char *>(workspace);
        uint32_t *pa = reinterpret_cast<uint32_t *>(ws);
        uint32_t *pb = same ? pa : reinterpret_cast<uint32_t *>(ws + k.off_pb);
        uint8_t *fa = reinterpret_cast<uint8_t *>(ws + k.off_fa);
        uint8_t *fb = same ? fa : reinterpret_cast<uint8_t *>(ws + k.off_fb);
        count = reinterpret_cast<unsigned long long *>(ws + k.off_count);
        nopair = (unsigned long long)k.tiles * KTG * KGW * 32 - (unsigned long long)n * (n - 1) / 2;
        PlanesArgs planes = {};
        planes.a = {a, na, lda, pa, fa, k.nvb_a, k.fs_a};
        if (!same) planes.b = {b, nb, ldb, pb, fb, k.nvb_b, k.fs_b};
        planes.n = n;
        planes.count = count;
        planes.ncount = na * nb;
        KendallArgs args;
        args.pa = pa;
        args.pb = pb;
        args.fa = fa;
        args.fb = fb;
        args.nvb_a = k.nvb_a;
        args.nvb_b = same ? k.nvb_a : k.nvb_b;
        args.fs_a = k.fs_a;
        args.fs_b = same ? k.fs_a : k.fs_b;
        args.na = na;
        args.nb = nb;
        args.count = count;
        args.ldc = nb;
        const int64_t ta = (na + KBX - 1) / KBX;
        args.tiles_b = (nb + KBY - 1) / KBY;
        // (self case: the last tile may lie past the last variable)
        args.ntiles = same ? ta * (ta + 1) - (args.tiles_b < 2 * ta ? 1 : 0) : ta * args.tiles_b;
        for (int64_t begin = 0; begin < k.tiles; begin += k.seg) {
            const int64_t tiles = k.tiles - begin < k.seg ? k.tiles - begin : k.seg;
            if ((e = launch_planes(planes, begin, tiles, stream)) != hipSuccess) return e;
            planes.ncount = 0;   // cleared by the first segment
            args.ngroups = tiles * KTG;
            // Ranges of groups: two workgroups run on a CU at a time (out of
            // step, so that one's barrier and LDS waits lie under the other's
            // products), so the number of workgroups is kept just under a
            // multiple of 512 (the multiple, up to 4, that leaves the fewest
            // idle), with at least 16 groups each, as long as a whole tile's
            // 32768 additions to the counts take; fewer, down to 2, where tiles
            // hold fewer pairs (43 variables x 87 samples with ties: 54 us with 16
            // groups, 14 with 2; 300 x 300 variables x 200: 53 and 77 us in all).
            int64_t splits = 1;
            double best = 0.0;
            for (int r = 1; r <= 4; ++r) {
                const int64_t s = 512 * r / args.ntiles;
                if (s < 1) continue;
                const double used = (double)(s * args.ntiles) / (512.0 * r) - 0.02 * r;
                if (used > best) {
                    best = used;
                    splits = s;
                }
            }
            int64_t least = na * nb / args.ntiles / 2048;
            least = least < 2 ? 2 : least > 16 ? 16 : least;
            if (splits > args.ngroups / least) splits = args.ngroups / least;
            if (splits < 1) splits = 1;
            args.split_g = (args.ngroups + splits - 1) / splits;
            if (args.split_g > KMAXGROUPS) args.split_g = KMAXGROUPS;
            splits = (args.ngroups + args.split_g - 1) / args.split_g;
            const int64_t ids = args.ntiles * splits;
            const int64_t max_ids = int64_t(1) << 22;
            for (int64_t off = 0; off < ids; off += max_ids) {
                args.id_offset = off;
                args.ids_this = (ids - off) < max_ids ? (ids - off) : max_ids;
                if (same)
                    hipLaunchKernelGGL(kendall_count_kernel<true>, dim3((unsigned)args.ids_this),
                                       dim3(KTHREADS), 0, stream, args);
                else
                    hipLaunchKernelGGL(kendall_count_kernel<false>, dim3((unsigned)args.ids_this),
                                       dim3(KTHREADS), 0, stream, args);
                if ((e = hipGetLastError()) != hipSuccess) return e;
            }
        }
    }
    // n < 2 leaves count null: no sample pair, tau = 0 / 0
    hipLaunchKernelGGL(kendall_finish_kernel, dim3(grid_for(na * nb, 256)), dim3(256), 0, stream,
                       count, nb, na, nb, n, same ? 1 : 0, nopair, tau, ldt);
    return hipGetLastError();
}

}  // namespace gt
