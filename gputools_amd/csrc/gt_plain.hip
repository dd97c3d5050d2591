// gt_plain.hip -- FP32 all-pairs distance tiles on the gfx950 VALU.
//
// Replaces the six *_kernel_same kernels of inst/cuda/distance.cu (and the
// unreachable cross kernels).  gputools runs one 32-thread block per pair,
// re-reads both rows from global memory for every pair and reduces through
// shared memory (distance.cu:56-69).  Here a 256-thread workgroup owns a
// square tile of pairs, 128, 64 or 32 on a side: both row blocks are staged
// through LDS in 16-feature chunks (k-major, so each lane reads float4 runs),
// and every lane keeps an 8 x 8, 4 x 4 or 2 x 2 register micro-tile of pair
// accumulators.  Each staged feature value is reused by a tile side of pairs.
//
// Summation is two-level: each 16-feature chunk is summed into a partial that
// is then added into the running total, which bounds the rounding error of a
// sum of k positive terms by about (16 + k/16) ulp instead of k ulp.
//
// The same tile also serves the FP32 form of gpuCor's Pearson correlation
// (OP_DOT: the dot product of two standardised variables).
#include "gt_common.h"
#include "gt_internal.h"

#include <math.h>

#include <type_traits>

namespace gt {
namespace {

constexpr int PBK = 16;        // features per chunk (the first level of the sums)
constexpr int PTHREADS = 256;  // 4 waves, 16 x 16 lanes

// Tile of S x S pairs, an (S / 16) x (S / 16) micro-tile per lane.  CH chunks
// are staged at a time: the small tiles do little work per chunk, so they take
// more features per pair of barriers (canberra picks its form per staged
// chunk and stays with one).
template <int OP, int S>
struct PlainTile {
    static constexpr int M = S / 16;
    static constexpr int CH = (OP == OP_CANBERRA || S == 128) ? 1 : S == 64 ? 2 : 4;
    static constexpr int BK = PBK * CH;
    static constexpr int LD = S + 4;                     // LDS row (padding against bank conflicts)
    static constexpr int LOADS = S * BK / PTHREADS;      // elements each lane stages per side
    // point of the tile that micro-tile position u of lane coordinate t holds
    static __device__ __forceinline__ int at(int t, int u)
    {
        return M == 8 ? (u < 4 ? t * 4 + u : 64 + t * 4 + (u - 4)) : t * M + u;
    }
    // the M values of a staged row that lane coordinate t uses
    static __device__ __forceinline__ void read(const float *row, int t, float (&v)[M])
    {
        if constexpr (M == 2) {
            const float2 a = *reinterpret_cast<const float2 *>(row + t * 2);
            v[0] = a.x;
            v[1] = a.y;
        } else {
#pragma unroll
            for (int h = 0; h < M / 4; ++h) {
                const float4 a = *reinterpret_cast<const float4 *>(row + h * 64 + t * 4);
                v[4 * h] = a.x;
                v[4 * h + 1] = a.y;
                v[4 * h + 2] = a.z;
                v[4 * h + 3] = a.w;
            }
        }
    }
};

struct PlainArgs {
    const float *a;  // column side (index i): self mode = x
    int64_t lda, na;
    const float *b;  // row side (index j): self mode = x
    int64_t ldb, nb;
    int64_t k;
    float *out;
    int64_t ldd;
    int64_t tiles_a;      // cross mode: tiles along A
    int64_t tile_offset;  // first logical tile of this launch
    int64_t tiles_this;   // tiles in this launch
    float p, inv_p, fk;
    int fold;             // chunks summed in `part` before it is added to `acc`
    bool vec;             // ldd and out allow 16-byte stores (pitched layouts)
};

// Canberra chunk modes.  The quotient |a-b| / |a+b| costs an IEEE divide
// (about ten instructions) unless the hardware reciprocal can stand in for it:
// when every staged value of the chunk is 0, non-finite, or of magnitude in
// [2^-100, 2^100], each nonzero finite |a+b| lies in [2^-123, 2^101] (a sum of
// such values is a multiple of 2^-123), so v_rcp_f32 (1 ulp) neither takes
// nor returns a denormal, and |a-b| * rcp(|a+b|) is within 1.5 ulp of the
// quotient with the same Inf (x/0) and NaN (0/0, Inf/Inf) results.
//   CB_CLEAN:  no 0 and no non-finite value -- no term can be NaN, so the
//              per-pair count is the chunk length, added once per chunk;
//   CB_ZEROS:  zeros but no non-finite value -- the only NaN term is 0/0
//              (a == b == 0), which max(q, 0) drops (IEEE maxNum returns the
//              non-NaN operand); the dropped terms are counted per chunk as
//              popcount(za & zb) of the two rows' 16-bit zero masks;
//   CB_RANGED: non-finite values present -- reciprocal + NaN test per term;
//   CB_IEEE:   a tiny or huge finite value present -- IEEE divide.
enum { CB_CLEAN = 0, CB_RANGED = 1, CB_IEEE = 2, CB_ZEROS = 3 };

template <int OP, int MODE = CB_IEEE>
struct Term {
    // Accumulate one feature of one pair into (part, cnt).
    static __device__ __forceinline__ void add(float &part, int &cnt, float a, float b, float p)
    {
        if (OP == OP_EUCLID) {
            const float t = a - b;
            part = fmaf(t, t, part);
        } else if (OP == OP_MAXIMUM) {
            part = fmaxf(part, fabsf(a - b));
        } else if (OP == OP_MANHATTAN) {
            part += fabsf(a - b);
        } else if (OP == OP_CANBERRA && MODE == CB_CLEAN) {
            part = fmaf(fabsf(a - b), __builtin_amdgcn_rcpf(fabsf(a + b)), part);
        } else if (OP == OP_CANBERRA && MODE == CB_ZEROS) {
            part += fmaxf(fabsf(a - b) * __builtin_amdgcn_rcpf(fabsf(a + b)), 0.0f);
        } else if (OP == OP_CANBERRA && MODE == CB_RANGED) {
            const float q = fabsf(a - b) * __builtin_amdgcn_rcpf(fabsf(a + b));
            const bool ok = (q == q);
            part += ok ? q : 0.0f;
            cnt += ok ? 1 : 0;
        } else if (OP == OP_CANBERRA) {
            // R's rule: a term with 0 numerator and 0 denominator (a == b == 0,
            // the only case where the quotient is NaN for finite input) is
            // omitted and counted as missing; a == -b != 0 gives x/0 = Inf.
            const float q = fabsf(a - b) / fabsf(a + b);
            const bool ok = (q == q);
            part += ok ? q : 0.0f;
            cnt += ok ? 1 : 0;
        } else if (OP == OP_MINK3) {
            const float t = fabsf(a - b);
            part = fmaf(t * t, t, part);
        } else if (OP == OP_DOT) {
            part = fmaf(a, b, part);
        } else {  // OP_MINKP: |t|^p = 2^(p log2|t|); log2(0) = -inf gives 0
            const float t = fabsf(a - b);
            part += exp2f(p * log2f(t));
        }
    }

    static __device__ __forceinline__ float finish(float acc, int cnt, float inv_p, float fk)
    {
        if (OP == OP_EUCLID) return sqrtf(acc);
        if (OP == OP_MAXIMUM || OP == OP_MANHATTAN || OP == OP_DOT) return acc;
        if (OP == OP_CANBERRA) {
            if (cnt == 0) return __builtin_nanf("");
            return ((float)cnt == fk) ? acc : acc / ((float)cnt / fk);
        }
        if (OP == OP_MINK3) return cbrtf(acc);
        return powf(acc, inv_p);
    }
};

// Bound: VALU issue for whole tiles (2 to 4 instructions per feature and pair).
// With few points large tiles leave CUs idle and each one's staging latency
// and arithmetic are exposed, so the tile shrinks with the number of points
// (plain_tile_side): 1000 x 64 euclidean 30.6 -> 8.4 us, 8192 x 256 446 ->
// 416 us (2080 tiles of 128 were four full rounds and a nearly empty one).
// The order of a pair's sums does not depend on the tile.
template <int OP, int LAYOUT, int S>
__global__ __launch_bounds__(PTHREADS) void plain_tile_kernel(PlainArgs args)
{
    typedef PlainTile<OP, S> T;
    constexpr int M = T::M, BK = T::BK;
    __shared__ __attribute__((aligned(16))) float lds[2][BK][T::LD];  // [0] column side (i), [1] row side (j)

    const int tid = threadIdx.x;
    const int tx = tid & 15, ty = tid >> 4;
    const int64_t t = args.tile_offset + xcd_remap(blockIdx.x, args.tiles_this);

    int I, J;
    if (LAYOUT == OUT_CROSS) {
        I = (int)(t % args.tiles_a);
        J = (int)(t / args.tiles_a);
    } else {
        tri_tile(t, I, J);
    }
    const int64_t i0 = (int64_t)I * S, j0 = (int64_t)J * S;
    const int64_t k = args.k;

    // Global -> register staging (prefetched one step ahead).
    float sc[T::LOADS], sr[T::LOADS];
    auto gload = [&](int64_t kb) {
#pragma unroll
        for (int q = 0; q < T::LOADS; ++q) {
            const int e = tid + PTHREADS * q;
            const int row = e / BK, kc = e % BK;
            const int64_t kk = kb + kc;
            const int64_t gi = i0 + row, gj = j0 + row;
            sc[q] = (gi < args.na && kk < k) ? args.a[gi * args.lda + kk] : 0.0f;
            sr[q] = (gj < args.nb && kk < k) ? args.b[gj * args.ldb + kk] : 0.0f;
        }
    };

    float acc[M][M];
    float part[M][M];
    int cnt[M][M];
#pragma unroll
    for (int r = 0; r < M; ++r)
#pragma unroll
        for (int c = 0; c < M; ++c) {
            acc[r][c] = 0.0f;
            part[r][c] = 0.0f;
            cnt[r][c] = 0;
        }

    // One chunk of PBK staged features, from kc0 on, into the micro-tile.
    auto chunk = [&](auto mode, int kc0) {
        constexpr int MODE = decltype(mode)::value;
#pragma unroll 4
        for (int kc = kc0; kc < kc0 + PBK; ++kc) {
            float cv[M], rv[M];
            T::read(lds[0][kc], tx, cv);
            T::read(lds[1][kc], ty, rv);
#pragma unroll
            for (int r = 0; r < M; ++r)
#pragma unroll
                for (int c = 0; c < M; ++c)
                    Term<OP, MODE>::add(part[r][c], cnt[r][c], cv[c], rv[r], args.p);
        }
    };

    __shared__ int cb_flags[PTHREADS / 64];  // canberra: per-wave chunk classification
    __shared__ uint32_t cb_zero[2][S];       // canberra CB_ZEROS: per-row zero masks
    int clean_terms = 0;                     // canberra: features of CB_CLEAN / CB_ZEROS chunks

    gload(0);
    int folded = 0;   // chunks in `part` since the last fold
    for (int64_t kb = 0; kb < k; kb += BK) {
        __syncthreads();
        bool unclean = false, unranged = false, nonfin = false;
#pragma unroll
        for (int q = 0; q < T::LOADS; ++q) {
            const int e = tid + PTHREADS * q;
            const int row = e / BK, kc = e % BK;
            lds[0][kc][row] = sc[q];
            lds[1][kc][row] = sr[q];
            if (OP == OP_CANBERRA) {
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    const float m = fabsf(s ? sr[q] : sc[q]);
                    const bool mid = (m >= 0x1p-100f) && (m <= 0x1p100f);
                    unclean |= !mid;
                    unranged |= !mid && m != 0.0f && m < __builtin_inff();
                    nonfin |= !(m < __builtin_inff());
                }
            }
        }
        if (OP == OP_CANBERRA) {
            const bool wu = __builtin_amdgcn_ballot_w64(unclean) != 0;
            const bool wr = __builtin_amdgcn_ballot_w64(unranged) != 0;
            const bool wn = __builtin_amdgcn_ballot_w64(nonfin) != 0;
            if ((tid & 63) == 0) cb_flags[tid >> 6] = (wu ? 1 : 0) | (wr ? 2 : 0) | (wn ? 4 : 0);
        }
        __syncthreads();
        if (kb + BK < k) gload(kb + BK);

        if (OP == OP_CANBERRA) {
            const int4 f = *reinterpret_cast<const int4 *>(cb_flags);
            const int bits = __builtin_amdgcn_readfirstlane(f.x | f.y | f.z | f.w);
            if (bits == 0) {
                chunk(std::integral_constant<int, CB_CLEAN>{}, 0);
                clean_terms += PBK;
            } else if (bits == 1) {
                // zero masks of the 2 x S staged rows, one row per thread
                if (tid < 2 * S) {
                    const int side = tid / S, row = tid % S;
                    uint32_t zm = 0;
#pragma unroll
                    for (int kc = 0; kc < PBK; ++kc) zm |= (lds[side][kc][row] == 0.0f ? 1u : 0u) << kc;
                    cb_zero[side][row] = zm;
                }
                __syncthreads();
                chunk(std::integral_constant<int, CB_ZEROS>{}, 0);
                clean_terms += PBK;
                uint32_t zc[M], zr[M];
#pragma unroll
                for (int u = 0; u < M; ++u) {
                    zc[u] = cb_zero[0][T::at(tx, u)];
                    zr[u] = cb_zero[1][T::at(ty, u)];
                }
#pragma unroll
                for (int r = 0; r < M; ++r)
#pragma unroll
                    for (int c = 0; c < M; ++c) cnt[r][c] -= __builtin_popcount(zc[c] & zr[r]);
            } else if ((bits & 2) == 0) {
                chunk(std::integral_constant<int, CB_RANGED>{}, 0);
            } else {
                chunk(std::integral_constant<int, CB_IEEE>{}, 0);
            }
        }
#pragma unroll
        for (int ch = 0; ch < T::CH; ++ch) {
            if (ch > 0 && kb + ch * PBK >= k) break;
            if (OP != OP_CANBERRA) chunk(std::integral_constant<int, CB_IEEE>{}, ch * PBK);
            // Two-level sum: `part` collects `fold` chunks (about sqrt(k)
            // features), then joins the total, so both levels add about
            // sqrt(k / 16) terms.
            if (OP != OP_MAXIMUM && (++folded == args.fold || kb + (ch + 1) * PBK >= k)) {
                folded = 0;
#pragma unroll
                for (int r = 0; r < M; ++r)
#pragma unroll
                    for (int c = 0; c < M; ++c) {
                        acc[r][c] += part[r][c];
                        part[r][c] = 0.0f;
                    }
            }
        }
    }

    auto value = [&](int r, int c) {
        return Term<OP>::finish((OP == OP_MAXIMUM) ? part[r][c] : acc[r][c], cnt[r][c] + clean_terms,
                                args.inv_p, args.fk);
    };

    // Whole tiles of the pitched layouts (cross, and the off-diagonal tiles
    // of the symmetric one) store W values at a time: the lane's i runs along
    // a row j, and its j runs along a mirrored row i.
    if (LAYOUT != OUT_PACKED && args.vec && i0 + S <= args.na && j0 + S <= args.nb &&
        (LAYOUT == OUT_CROSS || I > J)) {
        constexpr int W = M < 4 ? M : 4;
        typedef float vec_t __attribute__((ext_vector_type(W)));
        float v[M][M];
#pragma unroll
        for (int r = 0; r < M; ++r)
#pragma unroll
            for (int c = 0; c < M; ++c) v[r][c] = value(r, c);
#pragma unroll
        for (int r = 0; r < M; ++r)
#pragma unroll
            for (int h = 0; h < M / W; ++h) {
                vec_t w;
#pragma unroll
                for (int u = 0; u < W; ++u) w[u] = v[r][W * h + u];
                *reinterpret_cast<vec_t *>(args.out + (j0 + T::at(ty, r)) * args.ldd + i0 + T::at(tx, W * h)) = w;
            }
        if (LAYOUT == OUT_FULL) {
#pragma unroll
            for (int c = 0; c < M; ++c)
#pragma unroll
                for (int h = 0; h < M / W; ++h) {
                    vec_t w;
#pragma unroll
                    for (int u = 0; u < W; ++u) w[u] = v[W * h + u][c];
                    *reinterpret_cast<vec_t *>(args.out + (i0 + T::at(tx, c)) * args.ldd + j0 + T::at(ty, W * h)) = w;
                }
        }
        return;
    }

    if (LAYOUT == OUT_PACKED) {
        // Packed rows start at arbitrary offsets, so the values go out as
        // whole runs of a row instead: 32 rows of the tile at a time are
        // transposed through LDS (the staging array), then each wave writes
        // runs of 64 (32 for the 32 tile) consecutive i of a row.
        float *tr = &lds[0][0][0];   // 32 x TLD floats
        constexpr int TLD = S + 1;
        static_assert(32 * TLD * 4 <= (int)sizeof(lds), "transpose buffer");
        constexpr int RUN = S < 64 ? S : 64;             // consecutive i per run
        constexpr int PER = 64 / RUN;                    // rows a wave writes at once
        const int wv = tid >> 6, ln = tid & (RUN - 1), sub = (tid & 63) / RUN;
#pragma unroll
        for (int grp = 0; grp < S / 32; ++grp) {
            __syncthreads();
#pragma unroll
            for (int r = 0; r < M; ++r) {
                const int lr = T::at(ty, r) - grp * 32;
                if (lr >= 0 && lr < 32) {
#pragma unroll
                    for (int c = 0; c < M; ++c) tr[lr * TLD + T::at(tx, c)] = value(r, c);
                }
            }
            __syncthreads();
            const int64_t jg = j0 + grp * 32;
#pragma unroll
            for (int rr = 0; rr < 8 / PER; ++rr) {
                const int lr = (wv + (PTHREADS / 64) * rr) * PER + sub;
                const int64_t j = jg + lr;
                if (j >= args.nb) continue;
                float *orow = args.out + packed_base(args.na, j);
#pragma unroll
                for (int h = 0; h < S / RUN; ++h) {
                    const int64_t i = i0 + h * RUN + ln;
                    if (i > j && i < args.na) orow[i] = tr[lr * TLD + h * RUN + ln];
                }
            }
        }
        return;
    }
#pragma unroll
    for (int r = 0; r < M; ++r) {
        const int64_t j = j0 + T::at(ty, r);
        if (j >= args.nb) continue;
#pragma unroll
        for (int c = 0; c < M; ++c) {
            const int64_t i = i0 + T::at(tx, c);
            if (i >= args.na) continue;
            if (LAYOUT == OUT_FULL) {
                if (i > j) {
                    const float v = value(r, c);
                    args.out[j * args.ldd + i] = v;
                    args.out[i * args.ldd + j] = v;
                } else if (i == j) {
                    // a distance is 0 there; the Pearson dot product is z . z
                    args.out[i * args.ldd + i] = (OP == OP_DOT) ? value(r, c) : 0.0f;
                }
            } else {
                args.out[j * args.ldd + i] = value(r, c);
            }
        }
    }
}

int64_t tile_count(int layout, int64_t na, int64_t nb, int64_t side)
{
    const int64_t ta = (na + side - 1) / side, tb = (nb + side - 1) / side;
    return layout == OUT_CROSS ? ta * tb : ta * (ta + 1) / 2;
}

template <int OP, int S>
hipError_t launch_op(int layout, PlainArgs &args, hipStream_t stream)
{
    args.tiles_a = (args.na + S - 1) / S;
    const int64_t total = tile_count(layout, args.na, args.nb, S);
    // Keep each launch's thread count below 2^32.
    const int64_t max_tiles = int64_t(1) << 23;
    for (int64_t off = 0; off < total; off += max_tiles) {
        args.tile_offset = off;
        args.tiles_this = (total - off) < max_tiles ? (total - off) : max_tiles;
        dim3 grid((unsigned)args.tiles_this), block(PTHREADS);
        if (layout == OUT_PACKED)
            hipLaunchKernelGGL((plain_tile_kernel<OP, OUT_PACKED, S>), grid, block, 0, stream, args);
        else if (layout == OUT_FULL)
            hipLaunchKernelGGL((plain_tile_kernel<OP, OUT_FULL, S>), grid, block, 0, stream, args);
        else
            hipLaunchKernelGGL((plain_tile_kernel<OP, OUT_CROSS, S>), grid, block, 0, stream, args);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

// Tile side, from the number of tiles (times in us, packed, 64 features).
// Canberra: the 8 x 8 micro-tile of a 128 tile needs more registers than there
// are (1784 against 1175 at 8192 x 256); 32 until the 64 tiles are many
// enough that their fewer LDS reads count (6000 x 1000: 2495 with 32, 2657
// with 64; 16384 x 128: 2442 and 2361).
// The others: 32 while 64 tiles would be little more than two a CU (1000
// points: 8.4, 13.1 and 30.6 with 32, 64 and 128; 2000: 17.5, 19.6 and 31.9;
// 2500: 24.4, 24.1 and 32.4).  Above, a 128 tile does 7% less work per pair
// than four 64 tiles, but 512 of them run at once (two a CU), and a last
// round that is not full costs as much as a full one: 128 where the rounds
// are filled to 91% (16384 x 128: 913 against 971; 9000 x 512: 914 against
// 993), 64 where they are not (8192 x 256: 416 against 446; 4000: 40 against
// 62; 10000 x 512: 1183 against 1193).
int plain_tile_side(bool canberra, int layout, int64_t na, int64_t nb)
{
    const int64_t t64 = tile_count(layout, na, nb, 64);
    if (canberra) return t64 < 10000 ? 32 : 64;
    if (t64 < 600) return 32;
    const int64_t t128 = tile_count(layout, na, nb, 128), rounds = (t128 + 511) / 512;
    return t128 * 100 >= rounds * 512 * 91 ? 128 : 64;
}

template <int OP>
hipError_t launch_sized(int layout, PlainArgs &args, hipStream_t stream)
{
    const int side = plain_tile_side(OP == OP_CANBERRA, layout, args.na, args.nb);
    if (side == 32) return launch_op<OP, 32>(layout, args, stream);
    if constexpr (OP != OP_CANBERRA)
        if (side == 128) return launch_op<OP, 128>(layout, args, stream);
    return launch_op<OP, 64>(layout, args, stream);
}

}  // namespace

hipError_t launch_plain(int op, int layout, const float *a, int64_t na, int64_t lda,
                        const float *b, int64_t nb, int64_t ldb, int64_t k, float p,
                        float *out, int64_t ldd, hipStream_t stream)
{
    PlainArgs args;
    args.a = a;
    args.lda = lda;
    args.na = na;
    args.b = b;
    args.ldb = ldb;
    args.nb = nb;
    args.k = k;
    args.out = out;
    args.ldd = ldd;
    args.vec = (ldd % 4 == 0) && ((reinterpret_cast<uintptr_t>(out) & 15u) == 0);
    args.p = p;
    args.inv_p = 1.0f / p;
    args.fk = (float)k;
    {
        // chunks per fold: about sqrt(chunks), so that the partial and the
        // total each add about sqrt(k / 16) values
        const int64_t chunks = (k + PBK - 1) / PBK;
        int f = 1;
        while ((int64_t)(f + 1) * (f + 1) <= chunks) ++f;
        args.fold = f;
    }
    if (na <= 0 || nb <= 0) return hipSuccess;
    switch (op) {
    case OP_EUCLID: return launch_sized<OP_EUCLID>(layout, args, stream);
    case OP_MAXIMUM: return launch_sized<OP_MAXIMUM>(layout, args, stream);
    case OP_MANHATTAN: return launch_sized<OP_MANHATTAN>(layout, args, stream);
    case OP_CANBERRA: return launch_sized<OP_CANBERRA>(layout, args, stream);
    case OP_MINK3: return launch_sized<OP_MINK3>(layout, args, stream);
    case OP_MINKP: return launch_sized<OP_MINKP>(layout, args, stream);
    case OP_DOT: return launch_sized<OP_DOT>(layout, args, stream);
    default: return hipErrorInvalidValue;
    }
}

// ---------------------------------------------------------------------------
// Fills: k == 0 gives NA for every pair (R: no usable column -> NA_REAL).
// ---------------------------------------------------------------------------
namespace {
__global__ void fill_kernel(float *out, int64_t count, float value)
{
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < count;
         e += (int64_t)gridDim.x * blockDim.x)
        out[e] = value;
}

__global__ void fill_full_kernel(float *out, int64_t n, int64_t ldd, float offdiag)
{
    const int64_t total = n * n;
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < total;
         e += (int64_t)gridDim.x * blockDim.x) {
        const int64_t r = e / n, c = e % n;
        out[r * ldd + c] = (r == c) ? 0.0f : offdiag;
    }
}
}  // namespace

hipError_t launch_fill(float *out, int64_t count, float value, hipStream_t stream)
{
    if (count <= 0) return hipSuccess;
    int64_t blocks = (count + 255) / 256;
    if (blocks > 65536) blocks = 65536;
    hipLaunchKernelGGL(fill_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, out, count, value);
    return hipGetLastError();
}

hipError_t launch_fill_full(float *out, int64_t n, int64_t ldd, float offdiag, hipStream_t stream)
{
    if (n <= 0) return hipSuccess;
    int64_t blocks = (n * n + 255) / 256;
    if (blocks > 65536) blocks = 65536;
    hipLaunchKernelGGL(fill_full_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, out, n, ldd,
                       offdiag);
    return hipGetLastError();
}

}  // namespace gt
