// gt_hclust.hip -- the clustering stage of gpuDistClust / gpuHclust.
//
// Agglomerative clustering on a full, symmetric n x n FP32 distance matrix
// in HBM (the layout gt_dist_device_full produces), with the ten
// Lance-Williams updates of the reference (inst/cuda/hcluster.cu:106-400) and
// its merge rule (src/hcluster.cpp:40-201): each round merges the closest
// pair (sub < sup) over the lower triangle, the surviving cluster keeps index
// sup, and its row and column are rewritten with the method's formula.
//
// The reference rescans the whole lower triangle every round (find_min1,
// n/1024 launches of n^2/2 reads in total per round) and pays three kernel
// launches plus a module load per launch and round.  Here:
//   - hclust_init_kernel (many workgroups, one wave per row) puts +inf on the
//     diagonal, sets every count to 1 and computes each row's minimum over
//     columns 0..r-1 (value and column);
//   - hclust_group_kernel (32 workgroups on one XCD, or one up to 256 points, see
//     there) runs the n - 1 rounds up to 32768 points;
//   - hclust_merge_kernel (one persistent workgroup of 1024 threads) runs them
//     elsewhere, and where the 32 found no room together.  Per round: the argmin over the cached row minima, the
//     update of row and column sup (row and column sub become +inf), then the
//     cached minima are repaired: row sup is rescanned; a row r > sup takes
//     the new D[r][sup] if it beats its cached minimum, and is rescanned only
//     when that minimum sat at column sub or sup and the new value does not
//     settle it; a row sub < r < sup is rescanned only when its minimum sat
//     at column sub.  Rows whose minimum is unaffected cost one comparison.
//   - up to n = 9216 the per-row state (counts, cached minima and the new row
//     sup) stays in LDS for the whole run.  One CU issues every store, and
//     its scattered column stores (one cache line each) dominate a round, so
//     this variant writes only row and column sup: a merged-away column is
//     recognised by its negative count instead of being set to +inf.  Only
//     the end of a round waits for the stores; until then the rescans take
//     row sup and column sup from the LDS copy.  A rescanned row is split
//     over several waves when few rows need one.
// Ties are broken exactly as the reference's 32-lane reductions do
// (hcluster.cu:27-57, 67-90): smallest value, then the lane (index mod 32)
// that wins the reduction tree (bit-reversed lane order), then smallest
// index; +inf and NaN entries are never candidates.  The update
// formulas keep the reference's arithmetic types (FP32, with the FP64
// promotions its double constants cause for median, flexible and flexible
// group) and round every product separately (no FMA contraction), so merges and heights
// match the reference's loop bit for bit.  When no finite distance is left
// (undefined in the reference) the two lowest-index clusters merge at +inf.
#include "gt_common.h"
#include "gt_internal.h"

#include <type_traits>

namespace gt {
namespace {

constexpr int HTHREADS = 1024;
constexpr int HWAVES = HTHREADS / 64;
constexpr int RESCAN_CAP = 2048;   // rows listed for rescan per round (LDS)
constexpr int HB = 4;              // rows per thread per batch (repair)
constexpr int HBU = 4;             // columns per thread per batch (update)
constexpr int NO_COL = -1;         // row without a candidate
constexpr int PENDING = -2;        // row queued for a rescan
constexpr int HC_LDS_ROWS = 9216;  // largest n whose row state fits in LDS (16 B per row)

struct HclustArgs {
    float *d;
    int64_t ldd;
    int n;
    int method;
    float lambda, beta;
    float *count;      // > 0: cluster size; < 0: merged away (minus its size)
    float *minv;       // cached row minimum over columns 0..r-1
    int *minc;         // its column, NO_COL or PENDING
    int *sub, *sup;
    float *height;
    bool vec4;         // rows start 16 B aligned
    struct HcGroup *group;   // hclust_group_kernel's meeting point; null without it
    int lgp;                 // log2 of its workgroups
    int fault;               // HcFault: a failure forced by a test
};

// Meeting point of the workgroups of hclust_group_kernel (cleared by the init
// kernel).
constexpr int GP_MAX = 32;           // workgroups, all on one XCD
constexpr int GMAX_N = 32768;        // a tie key fits 15 bits
constexpr unsigned G_ABORT = 0xffffu;
struct HcGroup {
    unsigned arrive[16];             // workgroups seen, per XCD
    unsigned chosen;                 // 0 none yet, 1 + XCD, or G_ABORT
    unsigned pad[47];
    unsigned long long rec[2][GP_MAX][2];   // [round parity][workgroup]: what it found
};
static_assert(sizeof(HcGroup) + 255 <= HC_GROUP_BYTES, "workspace share, any alignment");

// Order of equal values in the reference's 32-lane reductions: lane t keeps
// the first of its indices t, t+32, ...; the tree then folds lanes t and
// t + 16, t + 8, ..., t + 1 into t, keeping t on ties, so lane priority is
// the 5-bit reversal of the lane number (even lanes before odd ones, ...).
__device__ __forceinline__ unsigned tie_key(int idx)
{
    return ((__builtin_bitreverse32((unsigned)idx) >> 27) << 26) | ((unsigned)idx >> 5);
}

// (v, i) beats (bv, bi); bv = +inf with bi = NO_COL is the empty candidate
__device__ __forceinline__ bool beats(float v, int i, float bv, int bi)
{
    return v < bv || (v == bv && bi != NO_COL && tie_key(i) < tie_key(bi));
}

// wave-wide argmin of (value, index); lanes without a candidate hold
// (+inf, NO_COL)
__device__ __forceinline__ void wave_argmin(float &v, int &i)
{
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        const float ov = __shfl_xor(v, off, 64);
        const int oi = __shfl_xor(i, off, 64);
        if (oi != NO_COL && (i == NO_COL || beats(ov, oi, v, i))) {
            v = ov;
            i = oi;
        }
    }
}

__device__ __forceinline__ void take(float v, int c, float &bv, int &bi)
{
    if (v < INFINITY && (bi == NO_COL || beats(v, c, bv, bi))) {
        bv = v;
        bi = c;
    }
}

// argmin of row r over columns 0..r-1 by one wave (all lanes return it).
// Rows that start 16 B aligned are read 16 B per lane, four loads in flight.
__device__ __forceinline__ void scan_row(const float *row, int r, bool vec4, float &bv, int &bi)
{
    const int lane = threadIdx.x & 63;
    bv = INFINITY;
    bi = NO_COL;
    int c = 0;
    if (vec4) {
        const int full = r & ~1023;   // columns covered by whole 4 x 256 blocks
        for (; c < full; c += 1024) {
            float4 q[4];
#pragma unroll
            for (int u = 0; u < 4; ++u)
                q[u] = *reinterpret_cast<const float4 *>(row + c + u * 256 + lane * 4);
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int cc = c + u * 256 + lane * 4;
                take(q[u].x, cc, bv, bi);
                take(q[u].y, cc + 1, bv, bi);
                take(q[u].z, cc + 2, bv, bi);
                take(q[u].w, cc + 3, bv, bi);
            }
        }
    }
    for (int cc = c + lane; cc < r; cc += 64) take(row[cc], cc, bv, bi);
    wave_argmin(bv, bi);
}

// This lane's argmin of row[c] over c in [c0, c1) (c0 a multiple of 4)
// among live columns (count[c] > 0: entries of merged-away clusters are not
// kept at +inf), with column rw taking fixv: the value the current round has
// stored there, which may still be in flight.
__device__ __forceinline__ void scan_cols(const float *row, int c0, int c1, int rw, float fixv,
                                          const float *count, bool vec4, float &bv, int &bi)
{
    const int lane = threadIdx.x & 63;
    auto put = [&](float v, int c) {
        if (c < c1 && count[c] > 0.0f) take(c == rw ? fixv : v, c, bv, bi);
    };
    if (!vec4) {
        for (int cc = c0 + lane; cc < c1; cc += 64) put(row[cc], cc);
        return;
    }
    // 2048 columns per batch: eight 16 B loads per lane in flight
    for (int c = c0; c < c1; c += 2048) {
        float4 q[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int cc = c + u * 256 + lane * 4;
            q[u] = make_float4(INFINITY, INFINITY, INFINITY, INFINITY);
            if (cc + 3 < c1) {
                q[u] = *reinterpret_cast<const float4 *>(row + cc);
            } else if (cc < c1) {
                q[u].x = row[cc];
                if (cc + 1 < c1) q[u].y = row[cc + 1];
                if (cc + 2 < c1) q[u].z = row[cc + 2];
            }
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int cc = c + u * 256 + lane * 4;
            put(q[u].x, cc);
            put(q[u].y, cc + 1);
            put(q[u].z, cc + 2);
            put(q[u].w, cc + 3);
        }
    }
}

// Barrier over LDS traffic only: this wave's global stores may still be in
// flight when the others pass it.
__device__ __forceinline__ void lds_barrier()
{
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// A value the compiler cannot see through: a product passed through it is
// rounded on its own and never fused into the following add (the library is
// built with -ffp-contract=fast, under which contraction pragmas are ignored).
__device__ __forceinline__ float sep(float x)
{
    asm volatile("" : "+v"(x));
    return x;
}
__device__ __forceinline__ double sep(double x)
{
    asm volatile("" : "+v"(x));
    return x;
}

// Lance-Williams update of the reference's kernels (hcluster.cu:106-400):
// bot = D[sup][c], top = D[sub][c]; nr = new size of sup, np = size of sub,
// nq = old size of sup, nk = count[c], val = this round's merge height.
// Every product is rounded separately, as the reference's unfused code does.
template <int METHOD>
__device__ __forceinline__ float lw_update(float bot, float top, float nr, float np, float nq,
                                           float nk, float val, float lambda, float beta)
{
    switch (METHOD) {
    case HC_SINGLE:
        return fminf(bot, top);
    case HC_COMPLETE:
        return fmaxf(bot, top);
    case HC_WPGMA:
    case HC_MCQUITTY:
        return (float)((double)(bot + top) / 2.0);
    case HC_AVERAGE:
        return (sep(top * np) + sep(bot * nq)) / nr;
    case HC_MEDIAN:
        return (float)((double)(bot + top) / 2.0 - (double)val / 4.0);
    case HC_CENTROID:
        return (sep(top * np) + sep(bot * nq)) / nr - (np * nq * val) / (nr * nr);
    case HC_FLEXIBLE_GROUP:
        return (float)((sep((double)bot * (1.0 - (double)lambda) * (double)np) +
                        sep((double)top * (1.0 - (double)lambda) * (double)nq)) /
                           (double)nr +
                       (double)sep(beta * val));
    case HC_FLEXIBLE:
        return (float)((sep((double)bot * (1.0 - (double)lambda)) +
                        sep((double)top * (1.0 - (double)lambda))) /
                           2.0 +
                       (double)sep(beta * val));
    case HC_WARD: {
        if (nr == -nk) return INFINITY;
        float b = (sep(bot * (np + nk)) + sep(top * (nq + nk)) - sep(val * nk));
        b /= (nr + nk);
        return isinf(b) ? INFINITY : b;
    }
    default:
        return fminf(bot, top);
    }
}

// Diagonal to +inf, counts to 1, and every row's minimum: one wave per row.
__global__ __launch_bounds__(256) void hclust_init_kernel(HclustArgs a)
{
    const int lane = threadIdx.x & 63;
    const int64_t waves = (int64_t)gridDim.x * 4;
    if (a.group && blockIdx.x == 0)
        for (unsigned t = threadIdx.x; t < sizeof(HcGroup) / 4; t += 256)
            reinterpret_cast<unsigned *>(a.group)[t] = 0u;
    for (int64_t r = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); r < a.n; r += waves) {
        float *row = a.d + r * a.ldd;
        if (lane == 0) {
            row[r] = INFINITY;
            a.count[r] = 1.0f;
        }
        float bv;
        int bi;
        scan_row(row, (int)r, a.vec4, bv, bi);
        if (lane == 0) {
            a.minv[r] = bv;
            a.minc[r] = bi;
        }
    }
}

// LDSRES: the per-row state (counts, cached minima and the rewritten row
// sup) lives in LDS for the whole run, n <= HC_LDS_ROWS; otherwise in the
// global workspace.
template <int METHOD, bool LDSRES>
__global__ __launch_bounds__(HTHREADS) void hclust_merge_kernel(HclustArgs a)
{
    extern __shared__ float hs_dyn[];
    __shared__ float red_v[HWAVES];
    __shared__ int red_i[HWAVES];
    __shared__ int s_cw, s_rw, s_nres, s_overflow;
    __shared__ float s_val;
    __shared__ int rescan[RESCAN_CAP];
    __shared__ float part_v[HWAVES];
    __shared__ int part_i[HWAVES];

    // after hclust_group_kernel: only when its workgroups did not come together
    if (a.group && a.group->chosen != G_ABORT) return;

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int n = a.n;
    const int64_t ldd = a.ldd;
    float *cntp, *minvp, *newp;
    int *mincp;
    if constexpr (LDSRES) {
        cntp = hs_dyn;
        minvp = hs_dyn + n;
        mincp = reinterpret_cast<int *>(hs_dyn + 2 * n);
        newp = hs_dyn + 3 * n;   // D[sup][c] as rewritten this round
        for (int r = tid; r < n; r += HTHREADS) {
            cntp[r] = a.count[r];
            minvp[r] = a.minv[r];
            mincp[r] = a.minc[r];
        }
        __syncthreads();
    } else {
        cntp = a.count;
        minvp = a.minv;
        mincp = a.minc;
        newp = nullptr;
    }
    for (int iter = 0; iter + 1 < n; ++iter) {
        // ---- the closest pair: argmin over the cached row minima ----------
        float bv = INFINITY;
        int bi = NO_COL;
        for (int r = tid; r < n; r += HTHREADS) {
            const float v = minvp[r];
            if (mincp[r] >= 0 && v < INFINITY && (bi == NO_COL || beats(v, r, bv, bi))) {
                bv = v;
                bi = r;
            }
        }
        wave_argmin(bv, bi);
        if (lane == 0) {
            red_v[wave] = bv;
            red_i[wave] = bi;
        }
        if constexpr (LDSRES)
            lds_barrier();
        else
            __syncthreads();
        // the waves' candidates reduced by wave 0 (the order on (value, tie
        // key) is total, so the lane order of the reduction does not matter)
        float v = INFINITY;
        int r = NO_COL;
        if (wave == 0) {
            if (lane < HWAVES) {
                v = red_v[lane];
                r = red_i[lane];
            }
            wave_argmin(v, r);
        }
        if (tid == 0) {
            int cw, rw;
            if (r != NO_COL) {
                rw = r;
                cw = mincp[r];
            } else {
                // no finite distance left: the two lowest-index clusters
                cw = -1;
                rw = -1;
                for (int i = 0; i < n && rw < 0; ++i)
                    if (cntp[i] > 0.0f) {
                        if (cw < 0)
                            cw = i;
                        else
                            rw = i;
                    }
                v = INFINITY;
            }
            a.height[iter] = v;
            a.sub[iter] = cw;
            a.sup[iter] = rw;
            cntp[rw] += cntp[cw];
            cntp[cw] *= -1.0f;
            s_cw = cw;
            s_rw = rw;
            s_val = v;
            s_nres = 0;
            s_overflow = 0;
        }
        if constexpr (LDSRES)
            lds_barrier();
        else
            __syncthreads();
        const int cw = s_cw, rw = s_rw;
        const float val = s_val;
        const float nr = cntp[rw];
        const float np = -cntp[cw];
        const float nq = nr - np;

        // ---- rewrite row/column sup; row/column sub become +inf ----------
        float *const dcw = a.d + (int64_t)cw * ldd;
        float *const drw = a.d + (int64_t)rw * ldd;
        // batches of HBU columns per thread: every load of a batch is issued
        // before its stores, which could otherwise alias them
        // (8 columns per thread in the LDS variant: one batch of loads at
        // n = 8192, none queued behind the first batch's column stores)
        constexpr int HBC = LDSRES ? 2 * HBU : HBU;
        for (int c0 = tid; c0 < n; c0 += HTHREADS * HBC) {
            float bot[HBC], top[HBC], nk[HBC];
#pragma unroll
            for (int u = 0; u < HBC; ++u) {
                const int c = c0 + u * HTHREADS;
                if (c < n && c != cw && c != rw) {
                    bot[u] = drw[c];
                    top[u] = dcw[c];
                    if constexpr (!LDSRES) nk[u] = cntp[c];
                }
            }
#pragma unroll
            for (int u = 0; u < HBC; ++u) {
                const int c = c0 + u * HTHREADS;
                if (c >= n) break;
                float v = INFINITY;
                if constexpr (LDSRES) {
                    // row and column sub are left as they are (sub is dead,
                    // and scans skip dead columns); a dead column c holds a
                    // stale value, so its new entry is +inf.  A dead row or
                    // column is never read again: only live c are stored.
                    const float nkc = cntp[c];
                    if (c != cw && c != rw && nkc > 0.0f)
                        v = lw_update<METHOD>(bot[u], top[u], nr, np, nq, nkc, val, a.lambda, a.beta);
                    newp[c] = v;
                    if (nkc > 0.0f) {
                        drw[c] = v;
                        a.d[(int64_t)c * ldd + rw] = v;
                    }
                } else {
                    if (c != cw && c != rw)
                        v = lw_update<METHOD>(bot[u], top[u], nr, np, nq, nk[u], val, a.lambda, a.beta);
                    dcw[c] = INFINITY;
                    a.d[(int64_t)c * ldd + cw] = INFINITY;
                    drw[c] = v;
                    a.d[(int64_t)c * ldd + rw] = v;
                }
            }
        }
        if constexpr (LDSRES)
            lds_barrier();
        else
            __syncthreads();

        // ---- repair the cached row minima --------------------------------
        for (int r0 = cw + tid; r0 < n; r0 += HTHREADS * HB) {
            float cnt[HB], mvs[HB], fs[HB];
            int mcs[HB];
#pragma unroll
            for (int u = 0; u < HB; ++u) {
                const int r = r0 + u * HTHREADS;
                if (r < n) {
                    cnt[u] = cntp[r];
                    mvs[u] = minvp[r];
                    mcs[u] = mincp[r];
                    fs[u] = LDSRES ? newp[r] : drw[r];
                }
            }
#pragma unroll
            for (int u = 0; u < HB; ++u) {
            const int r = r0 + u * HTHREADS;
            if (r >= n) break;
            bool redo = false;
            if (r == cw) {
                minvp[r] = INFINITY;
                mincp[r] = NO_COL;
                continue;
            }
            if (cnt[u] <= 0.0f) continue;
            const int mc = mcs[u];
            const float mv = mvs[u];
            if (r == rw) {
                redo = true;
            } else if (r < rw) {
                redo = (mc == cw);
            } else {
                const float f = fs[u];   // the new D[r][sup]
                if (mc == cw) {
                    redo = !(f < mv);
                    if (!redo) {
                        minvp[r] = f;
                        mincp[r] = rw;
                    }
                } else if (mc == rw) {
                    redo = !(f <= mv);
                    if (!redo) minvp[r] = f;
                } else if (f < INFINITY && (mc == NO_COL || beats(f, rw, mv, mc))) {
                    minvp[r] = f;
                    mincp[r] = rw;
                }
            }
            if (redo) {
                mincp[r] = PENDING;
                const int slot = atomicAdd(&s_nres, 1);
                if (slot < RESCAN_CAP)
                    rescan[slot] = r;
                else
                    s_overflow = 1;
            }
            }
        }
        if constexpr (LDSRES)
            lds_barrier();
        else
            __syncthreads();

        // ---- rescans ------------------------------------------------------
        const int nres = s_nres < RESCAN_CAP ? s_nres : RESCAN_CAP;
        if constexpr (LDSRES) {
            // This round's stores to row and column sup may still be in
            // flight: row sup is read from its LDS copy, and in other rows
            // column sup takes the LDS copy's value.  Dead columns (sub's
            // included) are skipped by their count.
            const float *const dr = a.d;
            if (nres < HWAVES) {
                // few rows: each is split over HWAVES / nres waves, whose
                // partial argmins are combined (the order of (value, tie key)
                // is total, so any grouping gives the same minimum)
                const int S = nres > 0 ? HWAVES / nres : 1;
                const int q = wave / S, sg = wave % S;
                float v = INFINITY;
                int c = NO_COL;
                if (q < nres) {
                    const int r = rescan[q];
                    const int per = (((r + 2047) >> 11) + S - 1) / S;   // 2048-column batches
                    const int c0 = min(r, sg * per * 2048), c1 = min(r, (sg + 1) * per * 2048);
                    if (r == rw) {
                        for (int cc = c0 + lane; cc < c1; cc += 64) take(newp[cc], cc, v, c);
                    } else {
                        scan_cols(dr + (int64_t)r * ldd, c0, c1, rw, newp[r], cntp, a.vec4, v, c);
                    }
                }
                wave_argmin(v, c);
                if (lane == 0) {
                    part_v[wave] = v;
                    part_i[wave] = c;
                }
                lds_barrier();
                if (tid < nres) {
                    float bv = INFINITY;
                    int bi = NO_COL;
                    for (int w = tid * S; w < tid * S + S; ++w)
                        if (part_i[w] != NO_COL && (bi == NO_COL || beats(part_v[w], part_i[w], bv, bi))) {
                            bv = part_v[w];
                            bi = part_i[w];
                        }
                    minvp[rescan[tid]] = bv;
                    mincp[rescan[tid]] = bi;
                }
            } else {
                for (int q = wave; q < nres; q += HWAVES) {
                    const int r = rescan[q];
                    float v = INFINITY;
                    int c = NO_COL;
                    if (r == rw) {
                        for (int cc = lane; cc < r; cc += 64) take(newp[cc], cc, v, c);
                    } else {
                        scan_cols(dr + (int64_t)r * ldd, 0, r, rw, newp[r], cntp, a.vec4, v, c);
                    }
                    wave_argmin(v, c);
                    if (lane == 0) {
                        minvp[r] = v;
                        mincp[r] = c;
                    }
                }
                if (s_overflow) {
                    // more rows than the list holds: find the rest by their
                    // marker (every listed row has been rescanned by now)
                    lds_barrier();
                    for (int r = cw + 1 + wave; r < n; r += HWAVES) {
                        if (mincp[r] != PENDING) continue;
                        float v = INFINITY;
                        int c = NO_COL;
                        if (r == rw) {
                            for (int cc = lane; cc < r; cc += 64) take(newp[cc], cc, v, c);
                        } else {
                            scan_cols(dr + (int64_t)r * ldd, 0, r, rw, newp[r], cntp, a.vec4, v, c);
                        }
                        wave_argmin(v, c);
                        if (lane == 0) {
                            minvp[r] = v;
                            mincp[r] = c;
                        }
                    }
                }
            }
            // this round's global stores complete before the next round
            // reads rows sup and sub
            __syncthreads();
            continue;
        }
        for (int q = wave; q < nres; q += HWAVES) {
            const int r = rescan[q];
            float v;
            int c;
            scan_row(a.d + (int64_t)r * ldd, r, a.vec4, v, c);
            if (lane == 0) {
                minvp[r] = v;
                mincp[r] = c;
            }
        }
        if (s_overflow) {
            // more rows than the list holds: find the rest by their marker
            for (int r = cw + 1 + wave; r < n; r += HWAVES) {
                if (mincp[r] != PENDING) continue;
                float v;
                int c;
                scan_row(a.d + (int64_t)r * ldd, r, a.vec4, v, c);
                if (lane == 0) {
                    minvp[r] = v;
                    mincp[r] = c;
                }
            }
        }
        __syncthreads();
    }
}

// ---------------------------------------------------------------------------
// The merge rounds on the 32 CUs of one XCD
// ---------------------------------------------------------------------------
// One workgroup's round is a chain of memory round trips with LDS work on all
// rows' state between them, and one CU issues every scattered store.  Here 32
// workgroups share the rounds.  Rows are owned in blocks of 32, round robin; a
// workgroup keeps the cached minima of its rows in LDS, and every workgroup
// keeps all sizes (each sees every merge).  Per round:
//   - wave 0 sends out the workgroup's best row and its part of the minimum of
//     the row rewritten last round as two tagged 64-bit words, reads all
//     records and comes to the same pair as the others (the order on (value,
//     tie key) is total, so the grouping does not matter), and lists its rows
//     whose cached minimum is at column sub or sup;
//   - one wave per 64 rows reads its columns of rows sup and sub, stores the
//     new values to row and column sup and lets them beat the cached minima;
//   - at the same time the other waves scan the listed rows' remaining live
//     columns (a bit each), a row over up to 16 waves; the new value in column
//     sup joins afterwards.
// The workgroups must run on one XCD: they exchange data through its L2, where
// stores complete and which loads that pass the L1 by read.  GLAUNCH are
// launched, the first XCD that has 32 of them is chosen and the others leave.
// If none has 32 in time (a busy device, masked CUs), nobody starts and
// hclust_merge_kernel, launched behind, does the work; otherwise that leaves
// at once.
// Bound: the round's latency, most of it dependent instructions of single
// waves.  Average linkage, n = 8192 (independent normal points): 3.9 us a
// round, of which 0.2 gather, 0.5 exchange, 0.4 choice of the pair, 0.35 list,
// 1.0 rewrite and 1.1 beside it where some workgroup scans a row (0.84 of the
// rounds have one).  hclust_merge_kernel took 21.6 us; whole runs 177 -> 32 ms,
// at 1000 points 8.7 -> 3.0 ms, at 32768 4680 -> 299 ms.
// Up to here one workgroup does this kernel's rounds and meets nobody (64 points:
// 3.3 us a round against 3.6 with the meetings, 256: 3.1 and 3.2, 512: 3.9 and 3.1).
constexpr int GALONE_N = 256;
constexpr int GTHREADS = 1024, GWAVES = GTHREADS / 64;
constexpr int GLAUNCH = 320;
// Polls of a partner's record before it is given up: about a second of running
// (not of the clock, which goes on while a queue is swapped out).
constexpr unsigned GPOLLS = 5000000u;
// The wait for room: 1 us per point (100 MHz clock), a tenth to a fifth of what the
// rounds take in hclust_merge_kernel (5.9 us a round at 257 points, 8.5 at 1000,
// 19 at 8192).  They come together in some us where there is room.
constexpr unsigned long long GJOIN_TICKS = 100ull;

// End of a round: also this wave's stores are complete.
__device__ __forceinline__ void round_barrier()
{
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// Loads that pass the L1 by; stores and records complete in the L2 (a store
// of agent scope would go on to memory).
__device__ __forceinline__ float load_shared(const float *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ unsigned long long load_shared(const unsigned long long *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T>
__device__ __forceinline__ void store_shared(T *p, T v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// Four 16 B loads past the L1 at byte offsets from a row, and their wait.
using f32x4 = __attribute__((ext_vector_type(4))) float;
__device__ __forceinline__ void load_four(const float *row, int o0, int o1, int o2, int o3, f32x4 (&x)[4])
{
    asm volatile("s_nop 4\n\t"   // a lane read into the address is five wait states away
                 "global_load_dwordx4 %0, %4, %8 sc1\n\t"
                 "global_load_dwordx4 %1, %5, %8 sc1\n\t"
                 "global_load_dwordx4 %2, %6, %8 sc1\n\t"
                 "global_load_dwordx4 %3, %7, %8 sc1\n\t"
                 "s_waitcnt vmcnt(0)"
                 : "=&v"(x[0]), "=&v"(x[1]), "=&v"(x[2]), "=&v"(x[3])
                 : "v"(o0), "v"(o1), "v"(o2), "v"(o3), "s"(row)
                 : "memory");
}

// Rows and columns as their tie keys in 15 bits: (value, key) then has the
// order of beats().  No candidate: (+inf, NO_KEY).
constexpr unsigned NO_KEY = 0x7fffu + 1u;
__device__ __forceinline__ unsigned key_of(int i)
{
    return ((__builtin_bitreverse32((unsigned)i) >> 27) << 10) | ((unsigned)i >> 5);
}
__device__ __forceinline__ int index_of(unsigned k)
{
    return (int)(((k & 1023u) << 5) | (__builtin_bitreverse32(k >> 10) >> 27));
}

// One step of a wave-wide reduction in registers: lanes without a source, or
// in rows that the mask leaves out, keep their value.  A DPP read needs two
// wait states after the write of its source.
#define GT_DPP_STEP(op, x, ctrl) "s_nop 1\n\t" op " " x ", " x ", " x " " ctrl "\n\t"
#define GT_DPP_STEPS(op, x)                                                                        \
    GT_DPP_STEP(op, x, "row_shr:1 row_mask:0xf bank_mask:0xf")                                     \
    GT_DPP_STEP(op, x, "row_shr:2 row_mask:0xf bank_mask:0xf")                                     \
    GT_DPP_STEP(op, x, "row_shr:4 row_mask:0xf bank_mask:0xf")                                     \
    GT_DPP_STEP(op, x, "row_shr:8 row_mask:0xf bank_mask:0xf")                                     \
    GT_DPP_STEP(op, x, "row_bcast:15 row_mask:0xa bank_mask:0xf")                                  \
    GT_DPP_STEP(op, x, "row_bcast:31 row_mask:0xc bank_mask:0xf")                                  \
    "s_nop 1"

__device__ __forceinline__ float lane_of(float v, int lane)
{
    return __uint_as_float((unsigned)__builtin_amdgcn_readlane((int)__float_as_uint(v), lane));
}

// The lane that wins among those with (v, k) at the wave's minimum m; -1
// when m is +inf.
__device__ __forceinline__ int winner(float v, unsigned k, float m)
{
    unsigned long long at = __builtin_amdgcn_ballot_w64(v == m);
    if (!(m < INFINITY)) return -1;
    if (at & (at - 1)) {
        const unsigned own = v == m ? k : ~0u;
        unsigned q = own;
        asm volatile(GT_DPP_STEPS("v_min_u32_dpp", "%0") : "+v"(q));
        at = __builtin_amdgcn_ballot_w64(own == (unsigned)__builtin_amdgcn_readlane((int)q, 63));
    }
    return __builtin_ctzll(at);
}

// Wave-wide minimum.  (fminf would bring each step's operands into canonical
// form first.)  No candidate is a NaN.
__device__ __forceinline__ float wave_min(float v)
{
    asm volatile(GT_DPP_STEPS("v_min_f32_dpp", "%0") : "+v"(v));
    return lane_of(v, 63);
}

// two at once: each fills the other's wait states
#define GT_DPP_STEP2(ctrl)                                                                         \
    "s_nop 0\n\tv_min_f32_dpp %0, %0, %0 " ctrl "\n\tv_min_f32_dpp %1, %1, %1 " ctrl "\n\t"
__device__ __forceinline__ void wave_min2(float v, float w, float &mv, float &mw)
{
    asm volatile("s_nop 0\n\t"
                 GT_DPP_STEP2("row_shr:1 row_mask:0xf bank_mask:0xf")
                 GT_DPP_STEP2("row_shr:2 row_mask:0xf bank_mask:0xf")
                 GT_DPP_STEP2("row_shr:4 row_mask:0xf bank_mask:0xf")
                 GT_DPP_STEP2("row_shr:8 row_mask:0xf bank_mask:0xf")
                 GT_DPP_STEP2("row_bcast:15 row_mask:0xa bank_mask:0xf")
                 GT_DPP_STEP2("row_bcast:31 row_mask:0xc bank_mask:0xf")
                 "s_nop 1"
                 : "+v"(v), "+v"(w));
    mv = lane_of(v, 63);
    mw = lane_of(w, 63);
}

// rows per workgroup, a multiple of 32
__host__ __device__ __forceinline__ int group_rows(int n, int lgp) { return (((n + 31) / 32 - 1 >> lgp) + 1) * 32; }

template <int METHOD>
__global__ __launch_bounds__(GTHREADS) void hclust_group_kernel(HclustArgs a)
{
    extern __shared__ __attribute__((aligned(16))) float hs_dyn[];   // (mink is read 16 B at a time)
    __shared__ int s_g, s_nres, s_rw, s_cw;
    __shared__ float s_val, s_np, s_nq;
    // per wave: its rows' best (value, row and column), its part of row sup's
    // minimum, its part of a rescan
    __shared__ float best_v[GWAVES], sup_v[GWAVES], scan_v[GWAVES];
    __shared__ unsigned best_k[GWAVES], best_c[GWAVES], sup_k[GWAVES], scan_k[GWAVES];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    HcGroup *const grp = a.group;
    const int lgp = a.lgp, gp = 1 << lgp;
    if (tid == 0) s_g = 0;   // a workgroup alone meets nobody
    if (tid == 0 && lgp > 0) {
        const unsigned xcc = __builtin_amdgcn_s_getreg(20 | (0 << 6) | (3 << 11)) & 15u;   // HW_REG_XCC_ID
        const unsigned t = atomicAdd(&grp->arrive[xcc], 1u);
        if (t == (unsigned)gp - 1 && a.fault != HC_FAULT_JOIN) atomicCAS(&grp->chosen, 0u, xcc + 1u);
        const unsigned long long began = wall_clock64();
        unsigned c = 0u;
        while (c == 0u) {
            const bool late = wall_clock64() - began > GJOIN_TICKS * (unsigned long long)a.n;
            c = atomicCAS(&grp->chosen, 0u, late ? G_ABORT : 0u);
            if (late) break;
            __builtin_amdgcn_s_sleep(4);
        }
        s_g = (c == xcc + 1u && t < (unsigned)gp) ? (int)t : -1;
    }
    __syncthreads();
    const int g = s_g;
    if (g < 0) return;

    const int n = a.n, rows = group_rows(n, lgp), words = (n + 31) / 32;
    const int64_t ldd = a.ldd;
    float *const minv = hs_dyn;                                   // own rows: cached minimum,
    unsigned *const mink = reinterpret_cast<unsigned *>(minv + rows);   // its column's key,
    float *const newv = minv + 2 * rows;                          // D[sup][row] as rewritten,
    int *const list = reinterpret_cast<int *>(minv + 3 * rows);   // rows to rescan
    float *const scanv = minv + 4 * rows;                         // and what each scan found
    unsigned *const scank = reinterpret_cast<unsigned *>(minv + 5 * rows);
    unsigned *const live = reinterpret_cast<unsigned *>(minv + 6 * rows);   // bit per cluster, sup's off
    float *const cnt = reinterpret_cast<float *>(live + words);   // sizes of all clusters
    auto row_of = [&](int l) { return (((l >> 5) << lgp) + g) * 32 + (l & 31); };
    auto mine = [&](int r) { return ((r >> 5) & (gp - 1)) == g; };
    auto local = [&](int r) { return (r >> (5 + lgp)) * 32 + (r & 31); };
    for (int c = tid; c < n; c += GTHREADS) cnt[c] = 1.0f;
    for (int w = tid; w < words; w += GTHREADS)
        live[w] = n - w * 32 >= 32 ? ~0u : (1u << (n - w * 32)) - 1;
    for (int l = tid; l < rows; l += GTHREADS) {
        const int r = row_of(l);
        const int c = r < n ? a.minc[r] : NO_COL;
        minv[l] = c >= 0 ? a.minv[r] : INFINITY;
        mink[l] = c >= 0 ? key_of(c) : NO_KEY;
    }
    __syncthreads();

    if (tid < GWAVES) best_v[tid] = sup_v[tid] = INFINITY;
    __syncthreads();

    const unsigned lane_key = (__builtin_bitreverse32((unsigned)lane) >> 27) << 10;
    const bool updates = wave * 64 < rows;      // 64 rows each
    const int first = rows <= 256 ? 8 : 0;      // waves that rescan
    // the best of this wave's rows and its part of row sup, to LDS
    auto publish = [&](float v, unsigned k, unsigned c, float pv, unsigned pk) {
        float m, pm;
        wave_min2(v, pv, m, pm);
        const int w = winner(v, k, m), pw = winner(pv, pk, pm);
        if (lane == 0) {
            best_v[wave] = w < 0 ? INFINITY : lane_of(v, w & 63);
            best_k[wave] = (unsigned)__builtin_amdgcn_readlane((int)k, w & 63);
            best_c[wave] = (unsigned)__builtin_amdgcn_readlane((int)c, w & 63);
            sup_v[wave] = pw < 0 ? INFINITY : lane_of(pv, pw & 63);
            sup_k[wave] = (unsigned)__builtin_amdgcn_readlane((int)pk, pw & 63);
        }
    };
    if (updates) {
        const int l = wave * 64 + lane;
        const bool in = l < rows;
        publish(in ? minv[l] : INFINITY, key_of(row_of(l)), in ? mink[l] : NO_KEY, INFINITY, NO_KEY);
    }
    __syncthreads();

    int last = -1;      // the row rewritten last round
    float rv = INFINITY;                      // best of the rows rescanned last round
    unsigned rk = NO_KEY, rc = NO_KEY;
    for (int iter = 0; iter + 1 < n; ++iter) {
        if (wave == 0) {
            const unsigned tag = (unsigned)(iter >> 1) % 3u + 1u;
            // ---- this workgroup's best row, and its part of row `last` ------
            float bv = rv, pv = INFINITY;
            unsigned bk = rk, bc = rc, pk = NO_KEY;
            if (lane < GWAVES) {
                pv = sup_v[lane];
                pk = sup_k[lane];
                const float v = best_v[lane];
                const unsigned k = best_k[lane], c = best_c[lane];
                const bool t = v < bv || (v == bv && k < bk && v < INFINITY);
                bv = t ? v : bv;
                bk = t ? k : bk;
                bc = t ? c : bc;
            }
            if (last >= 0 && lane == 0) atomicOr(&live[last >> 5], 1u << (last & 31));
            // (the last round's stores are complete, so the record may go out)
            unsigned long long w0, w1;   // best row; part of row `last`
            {
                float mb, mp;
                wave_min2(bv, pv, mb, mp);
                const int wb = winner(bv, bk, mb), wp = winner(pv, pk, mp);
                const unsigned k = (unsigned)__builtin_amdgcn_readlane((int)bk, wb & 63) & 0x7fffu;
                const unsigned c = (unsigned)__builtin_amdgcn_readlane((int)bc, wb & 63) & 0x7fffu;
                const unsigned q = (unsigned)__builtin_amdgcn_readlane((int)pk, wp & 63) & 0x7fffu;
                const float v = wb < 0 ? INFINITY : lane_of(bv, wb & 63);
                const float qv = wp < 0 ? INFINITY : lane_of(pv, wp & 63);
                w0 = ((unsigned long long)__float_as_uint(v) << 32) | (k << 17 | c << 2 | tag);
                w1 = ((unsigned long long)__float_as_uint(qv) << 32) | (q << 2 | tag);
            }
            // ---- all records ---------------------------------------------------
            bool failed = false;
            if (lgp > 0) {
                unsigned long long *const rec = grp->rec[iter & 1][0];
                if (lane < 2) store_shared(rec + g * 2 + lane, lane == 0 ? w0 : w1);
                for (unsigned spin = 0;; ++spin) {
                    w0 = load_shared(rec + (lane & (gp - 1)) * 2);
                    w1 = load_shared(rec + (lane & (gp - 1)) * 2 + 1);
                    if (__builtin_amdgcn_ballot_w64((w0 & 3u) != tag || (w1 & 3u) != tag) == 0) break;
                    if (spin == (a.fault == HC_FAULT_PARTNER ? 0u : GPOLLS)) {
                        failed = true;
                        break;
                    }
                }
            }
            asm volatile("" ::: "memory");
            if (failed) {
                // a partner is gone; d is half rewritten, so what is left is marked
                // as no merge (sub == sup, NaN), which host callers get as an error
                for (int i = iter + lane; g == 0 && i + 1 < n; i += 64) {
                    a.height[i] = __builtin_nanf("");
                    a.sub[i] = a.sup[i] = 0;
                }
                if (lane == 0) s_nres = -1;
            } else {
                const float v = lane < gp ? __uint_as_float((unsigned)(w0 >> 32)) : INFINITY;
                const float lv = lane < gp ? __uint_as_float((unsigned)(w1 >> 32)) : INFINITY;
                const unsigned k = (unsigned)w0 >> 17, kc = ((unsigned)w0 >> 2) & 0x7fffu;
                const unsigned lk = ((unsigned)w1 >> 2) & 0x7fffu;
                float mv, ml;
                wave_min2(v, lv, mv, ml);
                const int wr = winner(v, k, mv);
                float val = INFINITY;
                unsigned krw = NO_KEY, kcw = NO_KEY;
                if (wr >= 0) {
                    val = lane_of(v, wr);
                    krw = (unsigned)__builtin_amdgcn_readlane((int)k, wr);
                    kcw = (unsigned)__builtin_amdgcn_readlane((int)kc, wr);
                }
                if (last >= 0) {
                    const int wl = winner(lv, lk, ml);
                    float lval = INFINITY;
                    unsigned lkey = NO_KEY;
                    if (wl >= 0) {
                        lval = lane_of(lv, wl);
                        lkey = (unsigned)__builtin_amdgcn_readlane((int)lk, wl);
                        const unsigned kl = key_of(last);
                        if (lval < val || (lval == val && kl < krw)) {
                            val = lval;
                            krw = kl;
                            kcw = lkey;
                        }
                    }
                    if (mine(last) && lane == 0) {
                        minv[local(last)] = lval;
                        mink[local(last)] = lkey;
                    }
                }
                int cw = -1, rw = -1;
                if (krw != NO_KEY) {
                    rw = index_of(krw);
                    cw = index_of(kcw);
                } else {
                    // no finite distance left: the two lowest-index clusters
                    for (int i = 0; i < words && rw < 0; ++i) {
                        unsigned m = live[i];
                        if (m && cw < 0) {
                            cw = i * 32 + __builtin_ctz(m);
                            m &= m - 1;
                        }
                        if (m && cw >= 0) rw = i * 32 + __builtin_ctz(m);
                    }
                    rw = __builtin_amdgcn_readfirstlane(rw);
                    cw = __builtin_amdgcn_readfirstlane(cw);
                    krw = key_of(rw);
                    kcw = key_of(cw);
                }
                last = rw;
                // the other waves are past the last round's reads
                const float nq = cnt[rw], np = cnt[cw];
                // rows whose cached minimum is at column sub or sup: their
                // other columns are scanned while row and column sup are made
                int nres = 0;
                const int own = mine(rw) ? local(rw) : -1;
                for (int l0 = 0; l0 < rows; l0 += 256) {
                    const int l = l0 + lane * 4;
                    uint4 mk = make_uint4(NO_KEY, NO_KEY, NO_KEY, NO_KEY);
                    if (l < rows) mk = *reinterpret_cast<const uint4 *>(mink + l);   // (rows: of 32)
                    auto hit = [&](unsigned k, int at) { return (k == kcw || k == krw) && at != own; };
                    const bool h0 = hit(mk.x, l), h1 = hit(mk.y, l + 1), h2 = hit(mk.z, l + 2), h3 = hit(mk.w, l + 3);
                    if (__builtin_amdgcn_ballot_w64(h0 || h1 || h2 || h3) == 0) continue;
                    auto add = [&](bool h, int at) {
                        const unsigned long long who = __builtin_amdgcn_ballot_w64(h);
                        if (h)
                            list[nres + (int)__builtin_amdgcn_mbcnt_hi(
                                            (unsigned)(who >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)who, 0u))] = at;
                        nres += __popcll(who);
                    };
                    add(h0, l);
                    add(h1, l + 1);
                    add(h2, l + 2);
                    add(h3, l + 3);
                }
                if (lane == 0) {
                    s_val = val;
                    s_cw = cw;
                    s_rw = rw;
                    s_np = np;
                    s_nq = nq;
                    s_nres = nres;
                    cnt[rw] = nq + np;
                    cnt[cw] = 0.0f;
                    atomicAnd(&live[cw >> 5], ~(1u << (cw & 31)));
                    atomicAnd(&live[rw >> 5], ~(1u << (rw & 31)));
                    if (g == 0) {
                        a.height[iter] = val;
                        a.sub[iter] = cw;
                        a.sup[iter] = rw;
                    }
                }
            }
        }
        lds_barrier();
        const int listed_row = list[min(lane, rows - 1)];
        const int nres = __builtin_amdgcn_readfirstlane(s_nres);
        if (nres < 0) return;
        const int rw = __builtin_amdgcn_readfirstlane(s_rw);
        const unsigned krw = key_of(rw);
        if (updates) {
            // ---- row and column sup at 64 of this workgroup's rows -------------
            const int cw = __builtin_amdgcn_readfirstlane(s_cw);
            const unsigned kcw = key_of(cw);
            const float np = s_np, nq = s_nq, val = s_val;
            const float *const dcw = a.d + (int64_t)cw * ldd;
            float *const drw = a.d + (int64_t)rw * ldd;
            const int l = wave * 64 + lane, c = row_of(l);
            const bool in = l < rows && c < n;
            float bot = 0.0f, top = 0.0f, nk = 0.0f, m = INFINITY;
            unsigned mk = NO_KEY;
            if (in) {
                bot = load_shared(drw + c);
                top = load_shared(dcw + c);
                nk = cnt[c];
                m = minv[l];
                mk = mink[l];
            }
            const float nr = nq + np;
            const bool alive = nk > 0.0f, other = alive && c != rw;
            float f = lw_update<METHOD>(bot, top, nr, np, nq, nk, val, a.lambda, a.beta);
            f = other ? f : INFINITY;
            if (alive) {
                store_shared(drw + c, f);
                store_shared(a.d + (int64_t)c * ldd + rw, f);
            }
            const bool part = other && c < rw && f < INFINITY;
            const unsigned kc = lane_key | ((unsigned)c >> 5);
            // ---- the cached minimum of each row: the new value may beat it.  Row
            // sup's is put together from all parts; listed rows follow below.
            const bool drop = c == rw || c == cw;
            const bool listed = (mk == kcw || mk == krw) && !drop;
            if (other && c > rw && f < INFINITY && (f < m || (f == m && krw < mk))) {
                m = f;
                mk = krw;
            }
            m = drop ? INFINITY : m;
            mk = drop ? NO_KEY : mk;
            if (in) newv[l] = f;
            if (in && !listed) {
                minv[l] = m;
                mink[l] = mk;
            }
            publish(listed ? INFINITY : m, kc, mk, part ? f : INFINITY, kc);
        }
        // ---- listed rows: the live columns but sup, a row over several waves ----
        const int lgw = first ? 3 : 4;
        const int lgs = nres <= 1 ? lgw : max(lgw - (32 - __builtin_clz(nres - 1)), 0), S = 1 << lgs;
        for (int q = (wave - first) >> lgs; wave >= first && q < nres; q += 1 << (lgw - lgs)) {
            const int l = q < 64 ? __builtin_amdgcn_readlane(listed_row, q & 63)
                                 : __builtin_amdgcn_readfirstlane(list[q]);
            const int r = row_of(l), sg = (wave - first) & (S - 1);
            const float *const row = a.d + (int64_t)r * ldd;
            const int r4 = r & ~3, per = ((((r + 255) >> 8) + S - 1) >> lgs) * 256;
            const int c0 = min(r4, sg * per), c1 = min(r4, (sg + 1) * per);
            float v = INFINITY;
            unsigned k = NO_KEY;
            // 1024 columns at a time, 4 x 4 per lane
            for (int cb = c0; cb < c1; cb += 1024) {
                const int cc = cb + lane * 4;
                f32x4 x[4];
                float best;
                int first_at;
                // the lane's first minimum over `units` of its four 16 B units, in
                // key order: columns 0, 2, 1, 3 of four, each over the units (four
                // short chains, then two)
                auto scan = [&](auto units) {
                    constexpr int NU = decltype(units)::value;
                    unsigned open[NU];   // bits of the live columns
#pragma unroll
                    for (int u = 0; u < NU; ++u) {
                        const int cu = cc + u * 256;
                        const unsigned w = live[min(cu >> 5, words - 1)];
                        open[u] = cu < c1 ? w >> (cu & 31) : 0u;
                    }
                    load_four(row, min(cc, c1 - 4) * 4, min(cc + 256, c1 - 4) * 4, min(cc + 512, c1 - 4) * 4,
                              min(cc + 768, c1 - 4) * 4, x);
                    float bv[4];
                    int bo[4];
#pragma unroll
                    for (int c = 0; c < 4; ++c) {
                        const int e = (c >> 1) | ((c << 1) & 2);
                        bv[c] = INFINITY;
                        bo[c] = -1;
#pragma unroll
                        for (int u = 0; u < NU; ++u) {
                            const unsigned on = (unsigned)((int)(open[u] << (31 - e)) >> 31);   // all bits or none
                            const float y = __uint_as_float((__float_as_uint(x[u][e]) & on) | (0x7f800000u & ~on));
                            const bool t = y < bv[c];   // (passes NaN over)
                            bv[c] = t ? y : bv[c];
                            bo[c] = t ? c * 4 + u : bo[c];
                        }
                    }
#pragma unroll
                    for (int c = 0; c < 4; c += 2) {
                        const bool t = bv[c + 1] < bv[c];
                        bv[c] = t ? bv[c + 1] : bv[c];
                        bo[c] = t ? bo[c + 1] : bo[c];
                    }
                    const bool hi = bv[2] < bv[0];
                    best = hi ? bv[2] : bv[0];
                    first_at = hi ? bo[2] : bo[0];
                };
                if (c1 - cb <= 256)
                    scan(std::integral_constant<int, 1>());
                else
                    scan(std::integral_constant<int, 4>());
                const float m = wave_min(best);
                if (m < INFINITY && m <= v) {
                    const int at = best == m ? first_at : -1;
                    const unsigned bk =
                        at < 0 ? NO_KEY : key_of(cc) + ((unsigned)(at >> 2) << 13) + ((unsigned)(at & 3) << 3);
                    const int w = winner(at < 0 ? INFINITY : m, bk, m);
                    const unsigned wk = (unsigned)__builtin_amdgcn_readlane((int)bk, w);
                    if (m < v || wk < k) {
                        v = m;
                        k = wk;
                        if (m == 0.0f) v = load_shared(row + index_of(wk));   // its sign
                    }
                }
            }
            if (sg == S - 1 && r4 < r) {
                // the last one to three columns
                const int c = min(r4 + lane, r - 1);
                float x = load_shared(row + c);
                x = (live[c >> 5] >> (c & 31)) & 1u && r4 + lane < r && x < INFINITY ? x : INFINITY;
                const unsigned ck = key_of(c);
                const float m = wave_min(x);
                const int w = winner(x, ck, m);
                if (w >= 0) {
                    const unsigned wk = (unsigned)__builtin_amdgcn_readlane((int)ck, w);
                    if (m < v || (m == v && wk < k)) {
                        v = lane_of(x, w);
                        k = wk;
                    }
                }
            }
            if (lane == 0) {
                scanv[q * S + sg] = v;
                scank[q * S + sg] = k;
            }
        }
        round_barrier();
        if (wave == 0) {
            rv = INFINITY;
            if (nres > 0) {
                float sv = INFINITY;
                unsigned sk = NO_KEY;
                if (S > 1) {
                    // (at most 8 rows, 16 parts)
                    const float ov = lane < nres * S ? scanv[lane] : INFINITY;
                    const unsigned ok = lane < nres * S ? scank[lane] : NO_KEY;
                    for (int q = 0; q < nres; ++q) {
                        const float v = (lane >> lgs) == q ? ov : INFINITY;
                        const int w = winner(v, ok, wave_min(v));
                        if (lane == q && w >= 0) {
                            sv = lane_of(ov, w);
                            sk = (unsigned)__builtin_amdgcn_readlane((int)ok, w);
                        }
                    }
                }
                for (int q = lane; q < nres; q += 64) {
                    const int l = list[q], r = row_of(l);
                    float m = S > 1 ? sv : scanv[q];
                    unsigned mk = S > 1 ? sk : scank[q];
                    const float f = newv[l];
                    if (r > rw && f < INFINITY && (f < m || (f == m && krw < mk))) {
                        m = f;
                        mk = krw;
                    }
                    minv[l] = m;
                    mink[l] = mk;
                    const unsigned k = key_of(r);
                    if (m < rv || (m == rv && m < INFINITY && k < rk)) {
                        rv = m;
                        rk = k;
                        rc = mk;
                    }
                }
            }
        }
    }
}

unsigned group_lds(int n, int lgp) { return (unsigned)((n + 31) / 32 * 4 + 4 * n + 24 * group_rows(n, lgp)); }

}  // namespace

hipError_t launch_hclust(float *d, int64_t n, int64_t ldd, int method, float lambda, float beta,
                         float *count, float *minv, int *minc, void *group, int *sub, int *sup,
                         float *height, int state, int fault, hipStream_t stream)
{
    if (n < 2) return hipSuccess;
    HclustArgs a;
    a.d = d;
    a.ldd = ldd;
    a.n = (int)n;
    a.method = method;
    a.lambda = lambda;
    a.beta = beta;
    a.count = count;
    a.minv = minv;
    a.minc = minc;
    a.sub = sub;
    a.sup = sup;
    a.height = height;
    a.vec4 = (ldd % 4 == 0) && ((reinterpret_cast<uintptr_t>(d) & 15) == 0);
    a.group = nullptr;
    a.fault = fault;
    a.lgp = n <= GALONE_N ? 0 : 5;
    // up to what 15-bit tie keys and the LDS hold (32768 points: 9.1 us a round,
    // one workgroup of hclust_merge_kernel 143)
    if (state == HC_STATE_AUTO && group && n <= GMAX_N)
        a.group = reinterpret_cast<HcGroup *>((reinterpret_cast<uintptr_t>(group) + 255) & ~(uintptr_t)255);
    int64_t blocks = (n + 3) / 4;
    if (blocks > 65536) blocks = 65536;
    hipLaunchKernelGGL(hclust_init_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, a);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    // 16 B of LDS per row (count, cached minimum and its column, the new row
    // sup) next to the 8 KB of static LDS: 155 KB at the largest n
    static_assert(HC_LDS_ROWS == HC_LDS_MAX_N, "LDS row limit");
    if (state == HC_STATE_LDS && n > HC_LDS_ROWS) return hipErrorInvalidValue;
    const bool lds = state == HC_STATE_LDS || (state == HC_STATE_AUTO && n <= HC_LDS_ROWS);
    const unsigned shm = lds ? (unsigned)(16 * n) : 0u;
    switch (method) {
#define GT_HC_CASE(m)                                                                          \
    case m:                                                                                    \
        if (a.group) {                                                                         \
            const unsigned gl = group_lds((int)n, a.lgp);                                      \
            e = hipFuncSetAttribute(reinterpret_cast<const void *>(hclust_group_kernel<m>),    \
                                    hipFuncAttributeMaxDynamicSharedMemorySize, (int)gl);      \
            if (e != hipSuccess) return e;                                                     \
            hipLaunchKernelGGL(hclust_group_kernel<m>, dim3(a.lgp ? GLAUNCH : 1),              \
                               dim3(GTHREADS), gl, stream, a);                                 \
            if ((e = hipGetLastError()) != hipSuccess || a.lgp == 0) return e;                 \
        }                                                                                      \
        if (lds) {                                                                             \
            e = hipFuncSetAttribute(reinterpret_cast<const void *>(hclust_merge_kernel<m, true>), \
                                    hipFuncAttributeMaxDynamicSharedMemorySize, (int)shm);     \
            if (e != hipSuccess) return e;                                                     \
            hipLaunchKernelGGL((hclust_merge_kernel<m, true>), dim3(1), dim3(HTHREADS), shm,   \
                               stream, a);                                                     \
        } else {                                                                               \
            hipLaunchKernelGGL((hclust_merge_kernel<m, false>), dim3(1), dim3(HTHREADS), 0,    \
                               stream, a);                                                     \
        }                                                                                      \
        break;
    GT_HC_CASE(HC_SINGLE)
    GT_HC_CASE(HC_COMPLETE)
    GT_HC_CASE(HC_WPGMA)
    GT_HC_CASE(HC_AVERAGE)
    GT_HC_CASE(HC_MEDIAN)
    GT_HC_CASE(HC_CENTROID)
    GT_HC_CASE(HC_FLEXIBLE_GROUP)
    GT_HC_CASE(HC_FLEXIBLE)
    GT_HC_CASE(HC_WARD)
    GT_HC_CASE(HC_MCQUITTY)
#undef GT_HC_CASE
    default:
        return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace gt
