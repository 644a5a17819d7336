// Gustavson SpGEMM (symbolic + numeric), masked SpGEMM and the fused
// masked-SpGEMM + SUM used for triangle counting, for gfx950.
//
// What is computed is what the reference's workspace lowering computes
// (lib/Dialect/IndexTree/Transforms/SymbolicCompute.cpp:215-339,
// lib/Conversion/IndexTreeToSCF/SymbolicDomainConversion.cpp:81-340,
// lib/Dialect/IndexTree/Transforms/WorkspaceTransforms.cpp:97-276,
// lib/Conversion/TensorAlgebraToSCF/SparseTensorConversionPass.cpp:595-638,
// 982-1159; masks: lib/Conversion/IndexTreeToSCF/IndexTreeToSCF.cpp:1083-1148,
// 1327-1448): every structurally reachable (i,j) is kept, columns come out
// ascending.  How it is computed is different: one 1024-lane workgroup owns a
// row at a time and keeps the row's column set as a bitmap in LDS (128 KiB
// covers 2^20 columns), so counting is a popcount, "sort the touched columns"
// (the reference's comet_sort call) is reading the bitmap in order, and the
// mark array / mark value bookkeeping disappears.  Values accumulate with
// fp64 atomics, in one of three places chosen by the number of products of the
// row: a dense per-workgroup slab in HBM (few products, every masked product and
// every semiring other than plus-times; the extraction step reads it back and
// re-zeroes it with an atomic exchange, so every access to the slab is performed
// at the L2 and no stale L1 line can be seen), a compact array in LDS indexed by
// the rank of the column among the row's columns (spgemm_numeric_span_kernel),
// or LDS accumulators for one block of 16384 columns at a time
// (spgemm_numeric_dense_kernel, the widest rows).
// The order in which the products of one (i,j) are added is therefore not the
// reference's ascending-k order: values agree to rounding, structure exactly.
#include <algorithm>
#include <cstring>
#include <type_traits>

#include "common.h"

namespace comet {

// Coalesced stores of C go out as streaming (non-temporal) stores: C is written once and never read here, and
// its 289 GB at scale 20 would otherwise push the rows of B out of the L2 (-7 ms in the block kernel, -7 ms in
// the span kernel).  Stores that scatter, a few bytes per lane - the span kernel's columns - stay ordinary:
// as streaming stores they reach memory unmerged (span kernel 144 -> 411 ms).
template <typename T>
__device__ __forceinline__ void store_streaming(T *p, T v)
{
    __builtin_nontemporal_store(v, p);
}

constexpr int SG_T = 1024;                 // lanes per workgroup
constexpr int SG_WAVES = SG_T / 64;
constexpr int SG_LDS_MAX_W = 32;           // words per lane that still fit LDS (33 * 1024 * 4 B = 132 KiB)

__device__ inline int64_t readlane_i64(int64_t v, int lane)
{
    int lo = (int)(v & 0xffffffff), hi = (int)(v >> 32);
    lo = __builtin_amdgcn_readlane(lo, lane);
    hi = __builtin_amdgcn_readlane(hi, lane);
    return ((int64_t)hi << 32) | (uint32_t)lo;
}

__device__ inline int64_t uniform_i64_sg(int64_t v)
{
    return ((int64_t)__builtin_amdgcn_readfirstlane((int)(v >> 32)) << 32) |
           (uint32_t)__builtin_amdgcn_readfirstlane((int)(v & 0xffffffff));
}

__device__ inline double readlane_d(double v, int lane)
{
    int lo = __double2loint(v), hi = __double2hiint(v);
    lo = __builtin_amdgcn_readlane(lo, lane);
    hi = __builtin_amdgcn_readlane(hi, lane);
    return __hiloint2double(hi, lo);
}

// Bitmap layout: word w = j/32 sits at address w + w/W, i.e. one padding word
// after every W words, W = words per lane.  Random probes of neighbouring
// columns land in neighbouring LDS banks, and the extraction sweep, in which
// lane t reads its own words t*W .. t*W+W-1 at addresses t*(W+1)+k, is
// conflict-free too because W+1 is odd.
struct BmAddr {
    int logW;
    __device__ inline int word(int j) const
    {
        const int w = j >> 5;
        return w + (w >> logW);
    }
    __device__ inline uint32_t bit(int j) const { return 1u << (j & 31); }
};

// Visit every product of output row i: f(j, q, a, p, s) for k = Acrd[p] in A_i,
// q over the entries [s, e) of B_k, j = Bcrd[q], a = A's value (the visitor
// loads Bval[q] itself, and only if it needs it).  The entries of A_i are dealt to the 16 wavefronts
// one at a time (entry p goes to wavefront p mod 16), because in a sorted row
// the neighbours with long rows sit next to each other and would otherwise all
// land on one wavefront.  A wavefront fetches 64 of its entries at once (one per
// lane).  Rows of B with at least FEP_SHORT entries are then walked one by one
// with all lanes striding over B_k; shorter ones go to the four 16-lane quarters,
// four rows at a time.  A wavefront runs these turns one after the other and a
// turn costs about one trip to memory, so each turn issues all of its loads (up
// to four per lane; a load no lane needs is skipped) before the visitor runs.
constexpr int FEP_SHORT = 32, FEP_SHORT_LOADS = FEP_SHORT / 16, FEP_LONG_LOADS = 4;
constexpr int FEP_WIDE_DEPTH = 4;       // turns of a long row a wavefront takes at a time (WIDE walks)
// what the look-up and fetch steps of a masked product's visitor hand to the visit itself: where the column's
// value lives (negative: the mask does not hold the column) and B's value, fetched for hits only
struct MaskHit {
    int at;
    double b;
};
// four consecutive entries of an index array that lies at any 4-byte boundary
typedef int sg_i4u __attribute__((ext_vector_type(4), aligned(4)));
// With WIDE, a lane takes four consecutive entries in a turn in which every lane has all its entries - one 16-byte
// load instead of four loads 64 entries apart - and f4(j, q, a, p, s) visits the entries q .. q + 3 of B_k at once
// (their columns in j).  That pays where the visitor can treat neighbouring columns together (the symbolic phase:
// 78 -> 64 ms on A*A of an R-MAT graph of scale 20); a visitor that probes a hash table per product is slower with
// it (masked numeric phase, 247 -> 300 ms).
// A visitor that looks its column up in LDS first (a mask's bitmap or hash table) and fetches B's value only on a
// hit hands these two steps in as pre(j) and mid(j, q, what pre returned), and f gets what mid returned as a sixth
// argument.  The walk runs pre for all the entries of a turn together, then mid for all of them (inside f each
// step would sit behind the branch of the entry before it: four trips to LDS and four to memory per turn, one
// after the other) - and it visits a turn's entries one turn late, after the next turn's columns have arrived and
// its look-ups are out, so that the trip to memory for the values of the hits overlaps with the next turn's instead
// of standing alone (a wavefront runs its turns one after the other, and nothing else hides that trip).  The
// look-ups of a turn therefore run before the visits of the turn before it: they must not depend on them.
template <bool VALUES, bool WIDE, typename PRE, typename MID, typename F, typename F4>
__device__ inline void for_each_product_impl(int64_t as, int64_t ae, const int32_t *__restrict__ Acrd,
                                             const double *__restrict__ Aval, const int64_t *__restrict__ Bpos,
                                             const int32_t *__restrict__ Bcrd, PRE pre, MID mid, F f, F4 f4)
{
    using T1 = decltype(pre(0));
    using T2 = decltype(mid(0, (int64_t)0, T1()));
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int quarter = lane >> 4, sub = lane & 15;
    // the entries of the turn before: visited once the next turn's look-ups are out
    constexpr int NP = FEP_LONG_LOADS > FEP_SHORT_LOADS ? FEP_LONG_LOADS : FEP_SHORT_LOADS;
    bool w_ok[NP];
    int w_j[NP];
    int64_t w_q[NP], w_p[NP], w_s[NP];
    double w_a[NP];
    T2 w_md[NP];
#pragma unroll
    for (int x = 0; x < NP; ++x)
        w_ok[x] = false;
    const auto visit_pending = [&]() {
#pragma unroll
        for (int x = 0; x < NP; ++x)
            if (w_ok[x])
                f(w_j[x], w_q[x], w_a[x], w_p[x], w_s[x], w_md[x]);
    };
    // one turn: up to N entries per lane (ok[x]: the lane has entry x), columns j, places q in B
    const auto turn = [&](auto n_tag, const bool *ok, const int *j, const int64_t *q, double at, int64_t p, int64_t s) {
        constexpr int N = decltype(n_tag)::value;
        T1 tk[N];
#pragma unroll
        for (int x = 0; x < N; ++x)
            tk[x] = ok[x] ? pre(j[x]) : T1();
        visit_pending();
#pragma unroll
        for (int x = 0; x < NP; ++x) {
            w_ok[x] = x < N ? ok[x] : false;
            if (x < N) {
                w_j[x] = j[x];
                w_q[x] = q[x];
                w_a[x] = at;
                w_p[x] = p;
                w_s[x] = s;
                w_md[x] = ok[x] ? mid(j[x], q[x], tk[x]) : T2();
            }
        }
    };
    for (int64_t base = as + wave; base < ae; base += (int64_t)SG_WAVES * 64) {
        const int64_t left = (ae - base + SG_WAVES - 1) / SG_WAVES;     // my entries from here on
        const int cnt = (int)(left < 64 ? left : 64);
        int64_t bs = 0, be = 0;
        double a = 0.0;
        if (lane < cnt) {
            const int64_t p = base + (int64_t)lane * SG_WAVES;
            const int k = Acrd[p];
            bs = Bpos[k];
            be = Bpos[k + 1];
            if (VALUES)
                a = Aval[p];
        }
        unsigned long long big = __ballot(be - bs >= FEP_SHORT);
        unsigned long long todo = __ballot(bs < be && be - bs < FEP_SHORT);
        while (big) {
            const int t = __builtin_ctzll(big);
            big &= big - 1;
            const int64_t s = readlane_i64(bs, t), len = readlane_i64(be, t) - s;
            const double at = VALUES ? readlane_d(a, t) : 0.0;
            const int64_t p = base + (int64_t)t * SG_WAVES;
            int64_t o = lane;
            if (WIDE && len >= 64 * FEP_LONG_LOADS) {
                // Turns in which every lane has all its entries: a lane takes four consecutive ones, a single
                // 16-byte load, and the loads of the next turn are in flight while the visitor works on this one.
                static_assert(FEP_LONG_LOADS == 4, "a lane's entries of a full turn are one 16-byte load");
                int64_t c = s + 4 * (int64_t)lane;
                int64_t done = 0;
                // A wavefront with one or two kilobytes on their way from memory waits most of the time (a row of
                // B comes from beyond the L2 as a rule, two microseconds away): rows long enough are taken
                // FEP_WIDE_DEPTH turns at a time with as many again in flight behind them, then two at a time
                // (symbolic phase of A*A on an R-MAT graph of scale 20: 64.7 -> 46.8 ms; eight at a time gains
                // nothing over four).
                constexpr int64_t TURN = 64 * FEP_LONG_LOADS;
                const auto deep = [&](auto dtag) {
                    constexpr int D = decltype(dtag)::value;
                    if (len - done < 2 * D * TURN)
                        return;
                    sg_i4u jd[D];
#pragma unroll
                    for (int d = 0; d < D; ++d)
                        jd[d] = *reinterpret_cast<const sg_i4u *>(Bcrd + c + d * TURN);
                    for (int64_t full = done + D * TURN; full + D * TURN <= len; full += D * TURN) {
                        sg_i4u jn[D];
#pragma unroll
                        for (int d = 0; d < D; ++d)
                            jn[d] = *reinterpret_cast<const sg_i4u *>(Bcrd + c + (D + d) * TURN);
#pragma unroll
                        for (int d = 0; d < D; ++d)
                            f4(jd[d], c + d * TURN, at, p, s);
#pragma unroll
                        for (int d = 0; d < D; ++d)
                            jd[d] = jn[d];
                        c += D * TURN;
                        done += D * TURN;
                    }
#pragma unroll
                    for (int d = 0; d < D; ++d)
                        f4(jd[d], c + d * TURN, at, p, s);
                    c += D * TURN;
                    done += D * TURN;
                };
                deep(std::integral_constant<int, FEP_WIDE_DEPTH>());
                deep(std::integral_constant<int, 2>());
                if (len - done >= TURN) {
                sg_i4u j = *reinterpret_cast<const sg_i4u *>(Bcrd + c);
                for (int64_t full = done + 64 * FEP_LONG_LOADS; full + 64 * FEP_LONG_LOADS <= len;
                     full += 64 * FEP_LONG_LOADS) {
                    const sg_i4u jn = *reinterpret_cast<const sg_i4u *>(Bcrd + c + 64 * FEP_LONG_LOADS);
                    f4(j, c, at, p, s);
                    j = jn;
                    c += 64 * FEP_LONG_LOADS;
                    done += 64 * FEP_LONG_LOADS;
                }
                f4(j, c, at, p, s);
                done += 64 * FEP_LONG_LOADS;
                }
                o += done;
            }
            if (!WIDE && len >= 64 * FEP_LONG_LOADS) {
                // Turns in which every lane has all its entries: no predicates, and the loads of the next such
                // turn are in flight while this one's look-ups and the visits of the turn before it run.
                bool all[FEP_LONG_LOADS];
                int j[FEP_LONG_LOADS];
                int64_t q[FEP_LONG_LOADS];
#pragma unroll
                for (int x = 0; x < FEP_LONG_LOADS; ++x) {
                    all[x] = true;
                    j[x] = Bcrd[s + o + 64 * x];
                }
                for (int64_t full = 64 * FEP_LONG_LOADS; full + 64 * FEP_LONG_LOADS <= len;
                     full += 64 * FEP_LONG_LOADS) {
                    int jn[FEP_LONG_LOADS];
#pragma unroll
                    for (int x = 0; x < FEP_LONG_LOADS; ++x)
                        jn[x] = Bcrd[s + o + 64 * (FEP_LONG_LOADS + x)];
#pragma unroll
                    for (int x = 0; x < FEP_LONG_LOADS; ++x)
                        q[x] = s + o + 64 * x;
                    turn(std::integral_constant<int, FEP_LONG_LOADS>(), all, j, q, at, p, s);
#pragma unroll
                    for (int x = 0; x < FEP_LONG_LOADS; ++x)
                        j[x] = jn[x];
                    o += 64 * FEP_LONG_LOADS;
                }
#pragma unroll
                for (int x = 0; x < FEP_LONG_LOADS; ++x)
                    q[x] = s + o + 64 * x;
                turn(std::integral_constant<int, FEP_LONG_LOADS>(), all, j, q, at, p, s);
                o += 64 * FEP_LONG_LOADS;
            }
            if (o < len) {          // the rest of the row: fewer than 64 * FEP_LONG_LOADS entries
                bool ok[FEP_LONG_LOADS];
                int j[FEP_LONG_LOADS];
                int64_t q[FEP_LONG_LOADS];
#pragma unroll
                for (int x = 0; x < FEP_LONG_LOADS; ++x) {
                    ok[x] = o + 64 * x < len;
                    q[x] = s + o + 64 * x;
                }
#pragma unroll
                for (int x = 0; x < FEP_LONG_LOADS; ++x)
                    j[x] = ok[x] ? Bcrd[q[x]] : 0;
                turn(std::integral_constant<int, FEP_LONG_LOADS>(), ok, j, q, at, p, s);
            }
        }
        while (todo) {
            int pick = -1;
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int t = todo ? __builtin_ctzll(todo) : -1;
                todo = todo ? (todo & (todo - 1)) : 0;
                pick = quarter == g ? t : pick;
            }
            const int src = pick < 0 ? lane : pick;
            const int64_t s = ((int64_t)__shfl((int)(bs >> 32), src, 64) << 32) |
                              (uint32_t)__shfl((int)(bs & 0xffffffff), src, 64);
            const int64_t e = ((int64_t)__shfl((int)(be >> 32), src, 64) << 32) |
                              (uint32_t)__shfl((int)(be & 0xffffffff), src, 64);
            const double at =
                VALUES ? __hiloint2double(__shfl(__double2hiint(a), src, 64), __shfl(__double2loint(a), src, 64)) : 0.0;
            const int64_t p = base + (int64_t)src * SG_WAVES;
            bool ok[FEP_SHORT_LOADS];
            int j[FEP_SHORT_LOADS];
            int64_t q[FEP_SHORT_LOADS];
#pragma unroll
            for (int x = 0; x < FEP_SHORT_LOADS; ++x) {
                ok[x] = pick >= 0 && s + sub + 16 * x < e;
                q[x] = s + sub + 16 * x;
            }
#pragma unroll
            for (int x = 0; x < FEP_SHORT_LOADS; ++x)
                j[x] = ok[x] ? Bcrd[q[x]] : 0;
            turn(std::integral_constant<int, FEP_SHORT_LOADS>(), ok, j, q, at, p, s);
        }
    }
    visit_pending();
}

template <bool VALUES, typename F>
__device__ inline void for_each_product(int64_t as, int64_t ae, const int32_t *__restrict__ Acrd,
                                        const double *__restrict__ Aval, const int64_t *__restrict__ Bpos,
                                        const int32_t *__restrict__ Bcrd, F f)
{
    for_each_product_impl<VALUES, false>(
        as, ae, Acrd, Aval, Bpos, Bcrd, [](int) { return 0u; }, [](int, int64_t, uint32_t) { return 0u; },
        [&](int j, int64_t q, double a, int64_t p, int64_t s, uint32_t) { f(j, q, a, p, s); },
        [](sg_i4u, int64_t, double, int64_t, int64_t) {});
}
template <bool VALUES, typename PRE, typename MID, typename F>
__device__ inline void for_each_product_probed(int64_t as, int64_t ae, const int32_t *__restrict__ Acrd,
                                               const double *__restrict__ Aval, const int64_t *__restrict__ Bpos,
                                               const int32_t *__restrict__ Bcrd, PRE pre, MID mid, F f)
{
    for_each_product_impl<VALUES, false>(as, ae, Acrd, Aval, Bpos, Bcrd, pre, mid, f,
                                         [](sg_i4u, int64_t, double, int64_t, int64_t) {});
}
template <bool VALUES, typename F, typename F4>
__device__ inline void for_each_product(int64_t as, int64_t ae, const int32_t *__restrict__ Acrd,
                                        const double *__restrict__ Aval, const int64_t *__restrict__ Bpos,
                                        const int32_t *__restrict__ Bcrd, F f, F4 f4)
{
    for_each_product_impl<VALUES, true>(
        as, ae, Acrd, Aval, Bpos, Bcrd, [](int) { return 0u; }, [](int, int64_t, uint32_t) { return 0u; },
        [&](int j, int64_t q, double a, int64_t p, int64_t s, uint32_t) { f(j, q, a, p, s); }, f4);
}

__device__ inline int wave_sum_i32(int v)
{
    for (int d = 32; d > 0; d >>= 1)
        v += __shfl_down(v, d, 64);
    return v;
}

__device__ inline double wave_sum_f64(double v)
{
    for (int d = 32; d > 0; d >>= 1)
        v += __shfl_down(v, d, 64);
    return v;
}

// Rows are handed out through a global ticket counter, because row costs differ
// by six orders of magnitude and follow the bit pattern of the row id in R-MAT
// graphs (a fixed row -> workgroup map leaves some workgroups with ten times the
// work of others).  Lane 0 draws the ticket, LDS broadcasts it, and the value is
// read back through readfirstlane so that it lives in scalar registers: every
// branch on the row index is then a uniform scalar branch.  That matters because
// the row loop contains workgroup barriers.  The loop must also keep a single
// back edge with the draw at its end (no `continue`): with a draw at the top and
// a `continue` below it the compiler splits the loop per lane and parks lanes
// 1..1023 in a barrier loop that never draws again, which hangs the workgroup.
// What a ticket indexes is a list of the rows that have work, heaviest first
// (RowList): empty rows and rows another kernel serves cost no ticket, and the
// rows that take milliseconds start first instead of forming the tail.
struct RowList {
    const int32_t *rows;       // row - row_begin, by descending number of products
    const int64_t *bounds;     // [0] rows with >= dense_threshold products, [1] rows with any product,
                               // [2] rows with >= wide_threshold products (a prefix of [0]),
                               // [3] rows with >= mid_threshold products ([0] is a prefix of it),
                               // [4] rows with >= few_threshold products ([3] is a prefix of it)
    int64_t counts[5];         // the same on the host where it has them, else -1
    // whether the host knows that there are none such (unknown counts are all -1, hence equal)
    bool only_heavy() const { return counts[1] >= 0 && counts[1] == counts[0]; }
    bool none_small() const { return counts[1] >= 0 && counts[1] == counts[3]; }
    bool none_mid() const { return counts[0] >= 0 && counts[0] == counts[3]; }
};
// Which of a list's rows a kernel takes: from one of the bounds (-1: the list's begin) to another.  A number of both, so
// that a kernel reads two words in place of a chain of branches (values of 60000 rows of 20 entries, us: 316, now 296).
constexpr int list_part(int first, int end) { return (first + 1) | end << 4; }
constexpr int LIST_LIGHT = list_part(0, 1), LIST_ALL = list_part(-1, 1);
constexpr int LIST_WIDEST = list_part(-1, 2), LIST_SPAN = list_part(2, 0);                // the heavy rows
constexpr int LIST_MID = list_part(0, 3), LIST_SMALL = list_part(3, 1);                   // the light ones
constexpr int LIST_SMALL_MORE = list_part(3, 4), LIST_FEW = list_part(4, 1);              // the small ones
constexpr int LIST_NOT_FEW = list_part(-1, 4);
__device__ inline void list_range(const RowList &l, int part, int64_t *first, int64_t *end)
{
    *first = (part & 15) ? l.bounds[(part & 15) - 1] : 0;
    *end = l.bounds[part >> 4];
}
// A workgroup barrier that orders LDS traffic only.  __syncthreads() also makes every wavefront wait until its
// global stores have been acknowledged, a microsecond that a kernel whose stores nobody reads back (the rows
// of C going out) need not spend at every barrier.
__device__ __forceinline__ void lds_barrier()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}
// Inclusive prefix sum over the 64 lanes of a wavefront through the cross-lane data path of the vector ALU
// (shifts within a row of 16 lanes, then the last lane of a row broadcast to the rows after it): no LDS round
// trips, unlike a shuffle.  A lane whose source lies outside its row, or whose row is masked, adds 0.
__device__ __forceinline__ int wave_inclusive_scan(int v)
{
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);    // row_shr:1
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);    // row_shr:2
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);    // row_shr:4
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);    // row_shr:8
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);    // row_bcast:15 into rows 1 and 3
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);    // row_bcast:31 into rows 2 and 3
    return v;
}
__device__ __forceinline__ int lane_value(int v, int from) { return __builtin_amdgcn_ds_bpermute(from << 2, v); }
// orders a wavefront's own LDS accesses for the compiler; the hardware keeps their order
__device__ __forceinline__ void wave_lds_order()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
}

template <bool LDS_ONLY = false>
__device__ inline int64_t draw_row(unsigned long long *ticket, int64_t first, int64_t *slot)
{
    if (threadIdx.x == 0)
        *slot = first + (int64_t)atomicAdd(ticket, 1ull);
    if (LDS_ONLY)
        lds_barrier();
    else
        __syncthreads();
    const int64_t r = *slot;
    if (LDS_ONLY)
        lds_barrier();
    else
        __syncthreads();
    const int lo = __builtin_amdgcn_readfirstlane((int)(r & 0xffffffff));
    const int hi = __builtin_amdgcn_readfirstlane((int)(r >> 32));
    return ((int64_t)hi << 32) | (uint32_t)lo;
}

// Two kernels that share one list, one taking rows from its front and one from its back until they meet: the
// ticket word holds both counts (front in the low half, back in the high half), so the value an atomic add
// returns tells the claimant how many rows were taken from either end before it, and a claim is good while
// their sum is below n.  Every row is claimed once, and the meeting point settles where both kernels finish.
__device__ inline int64_t draw_front(unsigned long long *ticket, int64_t n, int64_t *slot)
{
    if (threadIdx.x == 0) {
        const unsigned long long old = atomicAdd(ticket, 1ull);
        const int64_t f = (int64_t)(old & 0xffffffffull), b = (int64_t)(old >> 32);
        *slot = f + b < n ? f : n;
    }
    __syncthreads();
    const int64_t r = *slot;
    __syncthreads();
    const int lo = __builtin_amdgcn_readfirstlane((int)(r & 0xffffffff));
    const int hi = __builtin_amdgcn_readfirstlane((int)(r >> 32));
    return ((int64_t)hi << 32) | (uint32_t)lo;
}

// Semiring operators of C = A @(reduce, mult) B.  The codes are the C ABI's.
enum { SR_PLUS = 0, SR_MIN = 1, SR_MAX = 2, SR_ANY = 3 };
__device__ inline double semiring_mult(int op, double a, double b)
{
    switch (op) {
    case 0: return a * b;
    case 1: return a;
    case 2: return b;
    case 3: return 1.0;
    case 4: return a + b;
    case 5: return a - b;
    case 6: return a < b ? a : b;
    case 7: return a > b ? a : b;
    default: return a / b;
    }
}
// Order-preserving map of a double onto an unsigned integer and back: min and
// max become integer atomics whose result does not depend on the order of the
// products, and an all-zero slot can stand for "nothing stored yet".
__device__ inline unsigned long long f64_key(double x)
{
    const unsigned long long u = (unsigned long long)__double_as_longlong(x);
    return (u >> 63) ? ~u : (u | 0x8000000000000000ull);
}
__device__ inline double key_f64(unsigned long long k)
{
    const unsigned long long u = (k >> 63) ? (k & 0x7fffffffffffffffull) : ~k;
    return __longlong_as_double((long long)u);
}
// One product of a semiring into an accumulator in LDS.  plus adds; min, max and any keep a 64-bit key and take the
// larger one, so the result does not depend on the order of the products: min the complement of the value's key,
// max the key, any the place (pa, q) of the product - pa counts the entries of the row of A from 1, q is the place
// in B - so that the product the reference's sequential loop reaches last wins.  An accumulator that received
// nothing is all-zero whatever the semiring.
__device__ __forceinline__ void semiring_lds_add(double *slot, int reduce_op, int mult_op, double a, double b, int pa,
                                                 int64_t q)
{
    unsigned long long *key = reinterpret_cast<unsigned long long *>(slot);
    if (reduce_op == SR_ANY) {
        __hip_atomic_fetch_max(key, ((unsigned long long)(uint32_t)pa << 32) | (unsigned long long)(uint32_t)q,
                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    } else {
        const double e = semiring_mult(mult_op, a, b);
        if (reduce_op == SR_PLUS)
            __hip_atomic_fetch_add(slot, e, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        else
            __hip_atomic_fetch_max(key, reduce_op == SR_MIN ? ~f64_key(e) : f64_key(e), __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_WORKGROUP);
    }
}
// The value such an accumulator stands for (as = where the row of A begins).  max starts from 0, as the reference's
// accumulator does, and so never returns less.
__device__ __forceinline__ double semiring_lds_value(unsigned long long v, int reduce_op, int mult_op, int64_t as,
                                                     const double *__restrict__ Aval, const double *__restrict__ Bval)
{
    if (reduce_op == SR_PLUS)
        return __longlong_as_double((long long)v);
    if (reduce_op == SR_MIN)
        return key_f64(~v);
    if (reduce_op == SR_MAX)
        return v < f64_key(0.0) ? 0.0 : key_f64(v);
    return semiring_mult(mult_op, Aval[as + (int64_t)(v >> 32) - 1], Bval[(int64_t)(v & 0xffffffffull)]);
}
// Every kernel here carves its dynamic LDS into 32-bit words and fp64 regions (ds_add_f64 and 64-bit reads fault on
// an address that is not a multiple of 8): the array itself starts 16-byte aligned, and every fp64 region begins an
// even number of words into it - asserted where each layout is defined.
extern __shared__ __align__(16) uint32_t sg_dyn_lds[];
// Hash table of a masked product's mask row (see spgemm_numeric_kernel): values first (8-byte aligned), keys after.
constexpr int SG_HASH_LOG = 13, SG_HASH_SLOTS = 1 << SG_HASH_LOG;
static_assert((2 * SG_HASH_SLOTS) % 2 == 0 && SG_HASH_SLOTS % 2 == 0, "hash table: values at word 0, keys an even number of words in");
#ifndef COMET_SG_HASH_FILL
#define COMET_SG_HASH_FILL (SG_HASH_SLOTS * 3 / 4)
#endif
constexpr int SG_HASH_FILL = COMET_SG_HASH_FILL;          // longest mask row that goes into the table
constexpr size_t SG_HASH_LDS = (size_t)SG_HASH_SLOTS * (8 + 4);
// The first slot a column is looked for in.  (Keeping groups of 32 neighbouring columns together, so that the
// look-ups of a wavefront walking a sorted row fall into neighbouring LDS banks, was slower: 370 against 240 ms on
// A*A masked by A at R-MAT scale 20 - a miss that lands in such a group walks to its end.)
__device__ inline uint32_t sg_hash_slot(int j)
{
    return ((uint32_t)j * 2654435761u) >> (32 - SG_HASH_LOG);
}

// ---------------------------------------------------------------------------
// Symbolic phase.  Unmasked: set the bit of every reachable column, count the
// bits that were new.  Masked: the bitmap starts as the mask row; a product
// clears its bit, and the bits that were still set are the output entries.
// ---------------------------------------------------------------------------
template <bool BM_LDS, bool MASKED>
__global__ __launch_bounds__(SG_T) void spgemm_symbolic_kernel(
    int64_t nrows, const int64_t *__restrict__ Apos, const int32_t *__restrict__ Acrd,
    const int64_t *__restrict__ Bpos, const int32_t *__restrict__ Bcrd, const int64_t *__restrict__ Mpos,
    const int32_t *__restrict__ Mcrd, int logW, uint32_t *__restrict__ gbm, unsigned long long *ticket,
    RowList list, int part, int64_t *__restrict__ rowcount)
{
    __shared__ int64_t row_slot;
    __shared__ int wave_cnt[SG_WAVES];
    uint32_t *bm;
    if constexpr (BM_LDS)
        bm = sg_dyn_lds;
    else
        bm = gbm + (size_t)blockIdx.x * (size_t)(SG_T * ((1 << logW) + 1));
    const BmAddr ad{logW};
    const int nwords = SG_T * ((1 << logW) + 1);
    if constexpr (BM_LDS) {
        for (int w = threadIdx.x; w < nwords; w += SG_T)
            bm[w] = 0;
    }
    __syncthreads();
    int64_t t_first, t_end;
    list_range(list, part, &t_first, &t_end);
    int64_t t = draw_row(ticket, t_first, &row_slot);
    while (t < t_end) {
        const int64_t i = list.rows[t];       // rows outside the list keep the zero the host put there
        const int64_t as = Apos[i], ae = Apos[i + 1];
        int64_t ms = 0, me = 1;
        if constexpr (MASKED) {
            ms = Mpos[i];
            me = Mpos[i + 1];
        }
        const bool work = as != ae && ms != me;
        if (work) {
        if constexpr (MASKED) {
            for (int64_t t = ms + threadIdx.x; t < me; t += SG_T)
                atomicOr(&bm[ad.word(Mcrd[t])], ad.bit(Mcrd[t]));
            __syncthreads();
        }
        int count = 0;
        for_each_product<false>(as, ae, Acrd, nullptr, Bpos, Bcrd, [&](int j, int64_t, double, int64_t, int64_t) {
            const uint32_t b = ad.bit(j);
            if constexpr (MASKED) {
                const uint32_t old = atomicAnd(&bm[ad.word(j)], ~b);
                count += (old & b) ? 1 : 0;
            } else if constexpr (BM_LDS) {
                atomicOr(&bm[ad.word(j)], b);       // nothing comes back, so the walk never waits for LDS:
            } else {                                // the bits are counted when the bitmap is cleared
                const uint32_t old = atomicOr(&bm[ad.word(j)], b);
                count += (old & b) ? 0 : 1;
            }
        }, [&](sg_i4u j, int64_t, double, int64_t, int64_t) {
            // four consecutive entries of a sorted row: the bits that fall into one word go there together
            if constexpr (BM_LDS && !MASKED) {
                int w = ad.word(j.x);
                uint32_t b = ad.bit(j.x);
                const int js[3] = {j.y, j.z, j.w};
#pragma unroll
                for (int x = 0; x < 3; ++x) {
                    const int wx = ad.word(js[x]);
                    if (wx != w) {
                        atomicOr(&bm[w], b);
                        w = wx;
                        b = 0u;
                    }
                    b |= ad.bit(js[x]);
                }
                atomicOr(&bm[w], b);
            } else {
                const int js[4] = {j.x, j.y, j.z, j.w};
#pragma unroll
                for (int x = 0; x < 4; ++x) {
                    const uint32_t b = ad.bit(js[x]);
                    if constexpr (MASKED) {
                        const uint32_t old = atomicAnd(&bm[ad.word(js[x])], ~b);
                        count += (old & b) ? 1 : 0;
                    } else {
                        const uint32_t old = atomicOr(&bm[ad.word(js[x])], b);
                        count += (old & b) ? 0 : 1;
                    }
                }
            }
        });
        if constexpr (BM_LDS && !MASKED) {
            __syncthreads();
            for (int w = threadIdx.x; w < nwords; w += SG_T) {
                count += __popc(bm[w]);
                bm[w] = 0;
            }
        }
        count = wave_sum_i32(count);
        if ((threadIdx.x & 63) == 0)
            wave_cnt[threadIdx.x >> 6] = count;
        __syncthreads();
        if (threadIdx.x == 0) {
            int total = 0;
            for (int w = 0; w < SG_WAVES; ++w)
                total += wave_cnt[w];
            rowcount[i] = total;
        }
        // leave the bitmap all-zero for the next row
        if constexpr (MASKED) {
            for (int64_t t = Mpos[i] + threadIdx.x; t < Mpos[i + 1]; t += SG_T)
                atomicAnd(&bm[ad.word(Mcrd[t])], 0u);
        } else if constexpr (!BM_LDS) {
            for_each_product<false>(as, ae, Acrd, nullptr, Bpos, Bcrd,
                                    [&](int j, int64_t, double, int64_t, int64_t) { atomicAnd(&bm[ad.word(j)], 0u); });
        }
        }   // work
        t = draw_row(ticket, t_first, &row_slot);     // its barriers also close this row's bitmap clean-up
    }
}

// ---------------------------------------------------------------------------
// Numeric phase for rows [row_begin,row_end).
// ---------------------------------------------------------------------------
// SEMI: any reduction/multiplication pair.  plus adds with the same fp64 atomic;
// min, max and any keep an integer key in the slab instead of a double and
// combine with an atomic max, so their results are independent of the order in
// which the products arrive: min stores the complement of the value's key, max
// the key itself (and, like the reference, never returns less than 0), any the
// position (p, q) of the product and so keeps the one a sequential traversal
// would reach last.  A slot is back to all-zero after extraction in every case.
template <bool BM_LDS, bool MASKED, bool SEMI>
__global__ __launch_bounds__(SG_T) void spgemm_numeric_kernel(
    int64_t row_begin, int64_t row_end, int64_t ncols, const int64_t *__restrict__ Apos,
    const int32_t *__restrict__ Acrd, const double *__restrict__ Aval, const int64_t *__restrict__ Bpos,
    const int32_t *__restrict__ Bcrd, const double *__restrict__ Bval, const int64_t *__restrict__ Mpos,
    const int32_t *__restrict__ Mcrd, int logW, uint32_t *__restrict__ gbm, uint32_t *__restrict__ gmask,
    double *__restrict__ slabs, unsigned long long *ticket, RowList list, int part,
    int reduce_op, int mult_op, const int64_t *__restrict__ Cpos,
    int32_t *__restrict__ Ccrd, double *__restrict__ Cval)
{
    __shared__ int64_t row_slot;
    __shared__ int wave_tot[SG_WAVES];
    // Two bitmaps: the columns of the output row (bm) and, for a masked product, the mask row (mbm).  One of
    // them fits LDS.  Unmasked, that is bm.  Masked, it is the mask: every product probes it, while only the
    // products that fall on a mask entry touch bm, which then lives in HBM with the slab and, like the slab,
    // is reached through L2 atomics only.
    constexpr bool OUT_LDS = BM_LDS && !MASKED, MASK_LDS = BM_LDS && MASKED;
    uint32_t *bm, *mbm = nullptr;
    if constexpr (OUT_LDS)
        bm = sg_dyn_lds;
    else
        bm = gbm + (size_t)blockIdx.x * (size_t)(SG_T * ((1 << logW) + 1));
    if constexpr (MASK_LDS)
        mbm = sg_dyn_lds;
    else if constexpr (MASKED)
        mbm = gmask + (size_t)blockIdx.x * (size_t)(SG_T * ((1 << logW) + 1));
    double *slab = slabs + (size_t)blockIdx.x * (size_t)ncols;
    const BmAddr ad{logW};
    const int W = 1 << logW;
    const int nwords = SG_T * ((1 << logW) + 1);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if constexpr (BM_LDS) {
        // the bitmap and, for a masked product, the hash table that shares its place
        const int lds_words = MASKED && nwords < (int)(SG_HASH_LDS / 4) ? (int)(SG_HASH_LDS / 4) : nwords;
        for (int w = threadIdx.x; w < lds_words; w += SG_T)
            sg_dyn_lds[w] = 0;
    }
    __syncthreads();
    const int64_t out0 = Cpos[row_begin];
    int64_t t_first, t_end;
    list_range(list, part, &t_first, &t_end);      // rows with many products are left to spgemm_numeric_dense_kernel
    int64_t t = draw_row(ticket, t_first, &row_slot);
    while (t < t_end) {
        const int64_t i = row_begin + list.rows[t];
        const int64_t as = Apos[i], ae = Apos[i + 1];
        const int64_t ob = Cpos[i], oe = Cpos[i + 1];
        bool hashed = false;
        if constexpr (MASK_LDS)
            hashed = __builtin_amdgcn_readfirstlane((int)(Mpos[i + 1] - Mpos[i] <= SG_HASH_FILL)) != 0;
        if (as != ae && ob != oe && hashed) {
            // A mask row of at most SG_HASH_FILL entries (nearly every row) goes into a hash table in LDS, column
            // -> slot, and the slot holds the value: a product probes the table (one LDS read for the 96 % that
            // miss), a product that falls on a mask entry adds into the slot with an LDS atomic, and nothing of
            // the row touches the L2.  A slot's key is column + 1, bit 31 says that a product has arrived.
            uint32_t *hkey = sg_dyn_lds + 2 * SG_HASH_SLOTS;
            double *hval = reinterpret_cast<double *>(sg_dyn_lds);
            unsigned long long *hbits = reinterpret_cast<unsigned long long *>(sg_dyn_lds);
            const auto slot_of = [&](int j) -> int {          // the slot that holds column j, or -1
                uint32_t sl = sg_hash_slot(j);
                for (;;) {
                    const uint32_t k = hkey[sl];
                    if ((k & 0x7fffffffu) == (uint32_t)j + 1u)
                        return (int)sl;
                    if (k == 0u)
                        return -1;
                    sl = (sl + 1) & (SG_HASH_SLOTS - 1);
                }
            };
            const int64_t ms = Mpos[i], mlen = Mpos[i + 1] - ms;
            for (int64_t e = ms + threadIdx.x; e < ms + mlen; e += SG_T) {
                const uint32_t key = (uint32_t)Mcrd[e] + 1u;
                uint32_t sl = sg_hash_slot(Mcrd[e]);
                for (;;) {
                    const uint32_t old = atomicCAS(&hkey[sl], 0u, key);
                    if (old == 0u || old == key)
                        break;
                    sl = (sl + 1) & (SG_HASH_SLOTS - 1);
                }
            }
            __syncthreads();
            const auto first_slot = [](int j) { return sg_hash_slot(j); };
            for_each_product_probed<true>(as, ae, Acrd, Aval, Bpos, Bcrd, [&](int j) { return hkey[first_slot(j)]; },
                                          [&](int j, int64_t q, uint32_t k0) {
                // k0 = the key in the column's first slot: nearly always that settles it
                MaskHit h{-1, 0.0};
                if (k0 != 0u)
                    h.at = (k0 & 0x7fffffffu) == (uint32_t)j + 1u ? (int)first_slot(j) : slot_of(j);
                if (h.at >= 0 && !(SEMI && reduce_op == SR_ANY))
                    h.b = Bval[q];
                return h;
            }, [&](int j, int64_t q, double a, int64_t p, int64_t bs, MaskHit h) {
                const int sl = h.at;
                if (sl < 0)
                    return;
                if (!(hkey[sl] >> 31))
                    atomicOr(&hkey[sl], 0x80000000u);
                if constexpr (SEMI) {
                    if (reduce_op == SR_ANY) {
                        const unsigned long long key = ((unsigned long long)(p - as + 1) << 32) | (unsigned long long)(q - bs);
                        __hip_atomic_fetch_max(&hbits[sl], key, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                    } else {
                        const double e = semiring_mult(mult_op, a, h.b);
                        if (reduce_op == SR_PLUS)
                            __hip_atomic_fetch_add(&hval[sl], e, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                        else
                            __hip_atomic_fetch_max(&hbits[sl], reduce_op == SR_MIN ? ~f64_key(e) : f64_key(e),
                                                   __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                    }
                } else {
                    __hip_atomic_fetch_add(&hval[sl], a * h.b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                }
            });
            __syncthreads();
            // the mask row is sorted: thread t takes a run of its entries, counts the ones a product reached, and
            // after a prefix sum over the workgroup writes them in place
            const int64_t per = (mlen + SG_T - 1) / SG_T;
            const int64_t e0 = ms + (int64_t)threadIdx.x * per;
            const int64_t e1 = e0 + per < ms + mlen ? e0 + per : ms + mlen;
            int mine = 0;
            for (int64_t e = e0; e < e1; ++e) {
                const int j = Mcrd[e];
                if (e > ms && Mcrd[e - 1] == j)
                    continue;          // a column stored twice in the mask row is one output entry
                mine += (int)(hkey[slot_of(j)] >> 31);
            }
            const int inc = wave_inclusive_scan(mine);
            if (lane == 63)
                wave_tot[wave] = inc;
            __syncthreads();
            int64_t off = ob - out0 + (inc - mine);
            for (int w = 0; w < wave; ++w)
                off += wave_tot[w];
            for (int64_t e = e0; e < e1; ++e) {
                const int j = Mcrd[e];
                if (e > ms && Mcrd[e - 1] == j)
                    continue;
                const int sl = slot_of(j);
                if (!(hkey[sl] >> 31))
                    continue;
                Ccrd[off] = j;
                double out = hval[sl];
                if (SEMI && reduce_op != SR_PLUS) {
                    const unsigned long long v = hbits[sl];
                    if (reduce_op == SR_MIN) {
                        out = key_f64(~v);
                    } else if (reduce_op == SR_MAX) {
                        out = v < f64_key(0.0) ? 0.0 : key_f64(v);
                    } else {
                        const int64_t pp = as + (int64_t)(v >> 32) - 1;
                        const int64_t qq = Bpos[Acrd[pp]] + (int64_t)(v & 0xffffffffull);
                        out = semiring_mult(mult_op, Aval[pp], Bval[qq]);
                    }
                }
                Cval[off] = out;
                ++off;
            }
            __syncthreads();           // everybody has found its slots: now they are emptied (keys last used above)
            for (int sl = threadIdx.x; sl < SG_HASH_SLOTS; sl += SG_T)
                if (hkey[sl]) {
                    hkey[sl] = 0u;
                    hbits[sl] = 0ull;
                }
        }
        if (as != ae && ob != oe && !hashed) {
        if constexpr (MASKED) {
            for (int64_t t = Mpos[i] + threadIdx.x; t < Mpos[i + 1]; t += SG_T)
                atomicOr(&mbm[ad.word(Mcrd[t])], ad.bit(Mcrd[t]));
            __syncthreads();
        }
        for_each_product_probed<true>(as, ae, Acrd, Aval, Bpos, Bcrd, [&](int j) {
            if constexpr (MASK_LDS)
                return mbm[ad.word(j)];      // the mask row was set before the barrier above and does not change
            else
                return 0u;
        }, [&](int j, int64_t q, uint32_t mword) {
            MaskHit h{0, 0.0};
            if constexpr (MASK_LDS)
                h.at = (mword & ad.bit(j)) ? 0 : -1;
            else if constexpr (MASKED)
                h.at = (atomicOr(&mbm[ad.word(j)], 0u) & ad.bit(j)) ? 0 : -1;
            if (h.at >= 0 && !(SEMI && reduce_op == SR_ANY))
                h.b = Bval[q];
            return h;
        }, [&](int j, int64_t q, double a, int64_t p, int64_t bs, MaskHit h) {
            if (h.at < 0)
                return;
            const int w = ad.word(j);
            const uint32_t b = ad.bit(j);
            atomicOr(&bm[w], b);
            if constexpr (SEMI) {
                unsigned long long *slot = (unsigned long long *)&slab[j];
                if (reduce_op == SR_ANY) {
                    const unsigned long long key = ((unsigned long long)(p - as + 1) << 32) | (unsigned long long)(q - bs);
                    __hip_atomic_fetch_max(slot, key, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                } else {
                    const double e = semiring_mult(mult_op, a, h.b);
                    if (reduce_op == SR_PLUS)
                        __hip_atomic_fetch_add(&slab[j], e, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                    else
                        __hip_atomic_fetch_max(slot, reduce_op == SR_MIN ? ~f64_key(e) : f64_key(e),
                                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                }
            } else {
                __hip_atomic_fetch_add(&slab[j], a * h.b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            }
        });
        __syncthreads();
        if constexpr (MASK_LDS) {
            // (rows whose mask row fits the hash table never come here: see below)
            // The output row is a subset of the mask row: walk that (it is sorted) instead of the bitmap.  Thread t
            // takes a run of consecutive mask entries, counts those whose bit a product has set, and after a prefix
            // sum over the workgroup writes them in place; value and bit are fetched and cleared on the way.
            const int64_t ms = Mpos[i], mlen = Mpos[i + 1] - ms;
            const int64_t per = (mlen + SG_T - 1) / SG_T;
            const int64_t e0 = ms + (int64_t)threadIdx.x * per;
            const int64_t e1 = e0 + per < ms + mlen ? e0 + per : ms + mlen;
            int mine = 0;
            for (int64_t e = e0; e < e1; ++e) {
                const int j = Mcrd[e];
                if (e > ms && Mcrd[e - 1] == j)
                    continue;          // a column stored twice in the mask row is one output entry
                mine += (atomicOr(&bm[ad.word(j)], 0u) & ad.bit(j)) ? 1 : 0;
            }
            int inc = wave_inclusive_scan(mine);
            if (lane == 63)
                wave_tot[wave] = inc;
            __syncthreads();           // also: every bit has been read before the first one is cleared below
            int64_t off = ob - out0 + (inc - mine);
            for (int w = 0; w < wave; ++w)
                off += wave_tot[w];
            for (int64_t e = e0; e < e1; ++e) {
                const int j = Mcrd[e];
                if ((e > ms && Mcrd[e - 1] == j) || !(atomicOr(&bm[ad.word(j)], 0u) & ad.bit(j)))
                    continue;
                Ccrd[off] = j;
                if (SEMI && reduce_op != SR_PLUS) {
                    const unsigned long long v = __hip_atomic_exchange((unsigned long long *)&slab[j], 0ull,
                                                                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                    double out;
                    if (reduce_op == SR_MIN) {
                        out = key_f64(~v);
                    } else if (reduce_op == SR_MAX) {
                        out = v < f64_key(0.0) ? 0.0 : key_f64(v);
                    } else {
                        const int64_t pp = as + (int64_t)(v >> 32) - 1;
                        const int64_t qq = Bpos[Acrd[pp]] + (int64_t)(v & 0xffffffffull);
                        out = semiring_mult(mult_op, Aval[pp], Bval[qq]);
                    }
                    Cval[off] = out;
                } else {
                    Cval[off] = __hip_atomic_exchange(&slab[j], 0.0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                }
                ++off;
            }
            __syncthreads();           // all reads of the bits are done
            for (int64_t e = e0; e < e1; ++e) {
                const int j = Mcrd[e];
                atomicAnd(&bm[ad.word(j)], ~ad.bit(j));
                atomicAnd(&mbm[ad.word(j)], 0u);
            }
        } else {
        // extraction: my words hold my columns in ascending order
        int mine = 0;
        for (int k = 0; k < W; ++k)
            mine += __popc(OUT_LDS ? bm[threadIdx.x * (W + 1) + k] : atomicOr(&bm[threadIdx.x * (W + 1) + k], 0u));
        int inc = mine;
        for (int d = 1; d < 64; d <<= 1) {
            const int o = __shfl_up(inc, d, 64);
            if (lane >= d)
                inc += o;
        }
        if (lane == 63)
            wave_tot[wave] = inc;
        __syncthreads();
        int64_t off = ob - out0 + (inc - mine);
        for (int w = 0; w < wave; ++w)
            off += wave_tot[w];
        for (int k = 0; k < W; ++k) {
            uint32_t word;
            if constexpr (OUT_LDS) {
                word = bm[threadIdx.x * (W + 1) + k];
                bm[threadIdx.x * (W + 1) + k] = 0;
            } else {
                word = atomicAnd(&bm[threadIdx.x * (W + 1) + k], 0u);
            }
            const int jbase = (((int)threadIdx.x << logW) + k) << 5;
            while (word) {
                const int b = __ffs(word) - 1;
                word &= word - 1;
                const int j = jbase + b;
                Ccrd[off] = j;
                if (SEMI && reduce_op != SR_PLUS) {
                    const unsigned long long v = __hip_atomic_exchange((unsigned long long *)&slab[j], 0ull,
                                                                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                    double out;
                    if (reduce_op == SR_MIN) {
                        out = key_f64(~v);
                    } else if (reduce_op == SR_MAX) {
                        out = v < f64_key(0.0) ? 0.0 : key_f64(v);
                    } else {
                        const int64_t pp = as + (int64_t)(v >> 32) - 1;
                        const int64_t qq = Bpos[Acrd[pp]] + (int64_t)(v & 0xffffffffull);
                        out = semiring_mult(mult_op, Aval[pp], Bval[qq]);
                    }
                    Cval[off] = out;
                } else {
                    Cval[off] = __hip_atomic_exchange(&slab[j], 0.0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                }
                ++off;
            }
        }
        if constexpr (MASKED) {
            for (int64_t t = Mpos[i] + threadIdx.x; t < Mpos[i + 1]; t += SG_T)
                atomicAnd(&mbm[ad.word(Mcrd[t])], 0u);
        }
        }   // extraction over the bitmap
        }   // row with output
        t = draw_row(ticket, t_first, &row_slot);     // its barriers also close this row's clean-up
    }
}

// ---------------------------------------------------------------------------
// Numeric phase for rows with many products: the L2 performs only ~20 G atomic
// line operations per second, so the slab path above costs one of those per
// product.  Here a row is swept in blocks of 16384 columns whose accumulators
// (128 KiB of doubles) and bitmap live in LDS; the products of one block are
// found through the per-row block pointers of B's plan.  Blocks are visited in
// ascending order and each is emitted in bitmap order, so the row still comes
// out sorted.
// ---------------------------------------------------------------------------
constexpr int SG_CB_LOG = 14;
constexpr int SG_CB = 1 << SG_CB_LOG;                                 // columns per block
typedef uint16_t emit_t;                                              // a column of the block being written out
constexpr int SG_EMIT = 8192;                                         // entries written out per turn of the emit
constexpr size_t SG_DENSE_LDS = (size_t)SG_CB * 8 + (size_t)SG_CB / 8 + (size_t)SG_EMIT * sizeof(emit_t) +
                                2 * (size_t)SG_CB / 8;               // accumulators, bitmap, list of the columns being
                                                                      // written out, the mask row's bits (two blocks)
// the accumulators (fp64) come first; what follows them is 32- and 16-bit data and starts on a word
static_assert(((size_t)SG_CB * 8) % 8 == 0 && ((size_t)SG_CB / 8) % 4 == 0 && ((size_t)SG_EMIT * sizeof(emit_t)) % 4 == 0,
              "the one-block kernel's LDS regions are aligned for their types");

// products[i - row_begin] = sum over k in A_i of nnz(B_k); one wavefront per row.
__global__ __launch_bounds__(256) void spgemm_row_products(int64_t row_begin, int64_t row_end,
                                                           const int64_t *__restrict__ Apos,
                                                           const int32_t *__restrict__ Acrd,
                                                           const int64_t *__restrict__ Bpos,
                                                           int64_t *__restrict__ products)
{
    const int64_t i = row_begin + (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (i >= row_end)
        return;
    const int lane = threadIdx.x & 63;
    int64_t s = 0;
    for (int64_t p = Apos[i] + lane; p < Apos[i + 1]; p += 64) {
        const int k = Acrd[p];
        s += Bpos[k + 1] - Bpos[k];
    }
    for (int d = 32; d > 0; d >>= 1)
        s += __shfl_down(s, d, 64);
    if (lane == 0)
        products[i - row_begin] = s;
}

// blkptr[k * (nblk + 1) + cb] = position in crd/val of the first entry of row k whose column is >= cb * SG_CB
// (cb = nblk gives the end of the row): the slice of row k inside block cb is one 16-byte load away.
// crd16[q] = the column of entry q inside its block of SG_CB columns
__global__ void spgemm_block_columns(int64_t nnz, const int32_t *__restrict__ crd, uint16_t *__restrict__ crd16)
{
    const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q < nnz)
        crd16[q] = (uint16_t)(crd[q] & (SG_CB - 1));
}

__global__ void spgemm_block_pointers(int64_t nrows, const int64_t *__restrict__ pos,
                                      const int32_t *__restrict__ crd, int nblk, int64_t *__restrict__ blkptr)
{
    const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= nrows)
        return;
    const int64_t s = pos[k], e = pos[k + 1];
    int64_t *out = blkptr + k * (nblk + 1);
    int64_t lo = s;
    out[0] = s;
    for (int cb = 1; cb <= nblk; ++cb) {
        const int64_t bound = (int64_t)cb << SG_CB_LOG;
        int64_t hi = e;
        while (lo < hi) {
            const int64_t mid = (lo + hi) >> 1;
            if (crd[mid] < bound)
                lo = mid + 1;
            else
                hi = mid;
        }
        out[cb] = lo;
    }
}

// One barrier tells every wavefront of the workgroup whether any of them had work in this visit.  The answer is
// made scalar, so that a branch on it is uniform (the branches taken on it hold barriers).  Three flags take
// turns: a wavefront may be a whole visit ahead of the slowest one, which is still to read this visit's flag
// when the fast one raises the next; the flag of the visit after that is cleared here, before the barrier,
// when everybody has long read its last use (they all came through the previous visit's barrier since).
__device__ __forceinline__ int visit_flag(int *flags, int visit, int touched, int lane)
{
    if (threadIdx.x == 0)
        flags[visit == 2 ? 0 : visit + 1] = 0;
    if (touched && lane == 0)
        flags[visit] = 1;
    lds_barrier();
    return __builtin_amdgcn_readfirstlane(flags[visit]);
}

// Visits the products of one slice per lane: f(j, a, b, pa, q) for the entries [lo, hi) of a row of B (the part of
// it inside the column block or blocks being swept), j the column, a the entry of A (and pa the tag the caller
// gave it: its place in the row of A, which only the `any` semiring needs), b the entry of B and q its place there;
// f4(j, a, v0, v1, pa, q) for four consecutive entries q .. q + 3 of one row of B, columns j, values v0.x, v0.y, v1.x,
// v1.y.  Returns whether this wavefront had anything to visit.

constexpr int SG_SHORT = 32;          // slices shorter than this are laid end to end, the others take turns of their own
constexpr int SG_SHORT_LOADS = 2;                 // entries of the short slices per lane and batch
constexpr int SG_LONG_LOADS = 4;                  // entries of a long slice per lane and turn

// One turn of a wavefront over a slice that starts at entry s of B and has len entries: lane l visits the
// entries o + 64 x < len, x < SG_LONG_LOADS (o = l for the first turn of a slice).  All loads are issued before
// the first visit, and a load that no lane needs is skipped.
// The columns of B come as 32-bit numbers or (COL = uint16_t) as the 16-bit numbers inside their block of SG_CB
// columns that the right-hand operand's plan keeps for the kernel that takes one block per visit: a third of the
// bytes of an entry it only needs the column of.
typedef unsigned short sg_h4u __attribute__((ext_vector_type(4), aligned(2)));
typedef double sg_d2u __attribute__((ext_vector_type(2), aligned(8)));
template <typename COL>
struct SgCol4;
template <>
struct SgCol4<int32_t> {
    typedef sg_i4u type;
};
template <>
struct SgCol4<uint16_t> {
    typedef sg_h4u type;
};

template <typename COL, typename F>
__device__ __forceinline__ void turn_of_slice(int64_t s, int64_t o, int64_t len, double at, int pt,
                                              const COL *__restrict__ Bcrd, const double *__restrict__ Bval, F f)
{
    int64_t q[SG_LONG_LOADS];
    bool ok[SG_LONG_LOADS];
#pragma unroll
    for (int x = 0; x < SG_LONG_LOADS; ++x) {
        ok[x] = o + 64 * x < len;
        q[x] = ok[x] ? s + o + 64 * x : 0;
    }
    int j[SG_LONG_LOADS];
    double v[SG_LONG_LOADS];
#pragma unroll
    for (int x = 0; x < SG_LONG_LOADS; ++x)
        j[x] = ok[x] ? (int)Bcrd[q[x]] : 0;
#pragma unroll
    for (int x = 0; x < SG_LONG_LOADS; ++x)
        v[x] = ok[x] ? Bval[q[x]] : 0.0;
#pragma unroll
    for (int x = 0; x < SG_LONG_LOADS; ++x)
        if (ok[x])
            f(j[x], at, v[x], pt, q[x]);
}

template <typename COL, typename F, typename F4>
__device__ __forceinline__ int for_each_in_slices(int64_t lo, int64_t hi, double a, int pa, int lane,
                                                  const COL *__restrict__ Bcrd,
                                                  const double *__restrict__ Bval, F f, F4 f4)
{
    typedef typename SgCol4<COL>::type col4;
    // Long slices take the whole wavefront, one at a time; short ones (a slice of one block often holds a
    // dozen entries) are laid end to end and dealt to the lanes entry by entry (below).  A wavefront runs its
    // turns one after the other (there is room for one workgroup per CU, so nobody else hides the latency), and
    // a turn costs about one trip to memory: so every turn issues all of its loads before the first LDS
    // operation waits for one, and a load that no lane needs is skipped.  Measured on A*A of an R-MAT
    // graph of scale 20: two loads per lane and turn of a long slice instead of four, +18 % time in this
    // kernel, eight +2 %; two long slices per turn, +2..8 %; slices of up to 4 or 8 entries left to their own
    // lane (64 slices per turn, but every lane a cache line of its own), +4..6 %; the short slices one to a
    // 16-lane quarter, four at a time, +1.7 % (up to 64 or 128 entries that way, +1..5 % more); laid end to
    // end up to 128 or 256 entries instead of 32, +6 % and +22 %.
    unsigned long long big = __ballot(hi - lo >= SG_SHORT);
    unsigned long long todo = __ballot(lo < hi && hi - lo < SG_SHORT);
    const int touched = (big | todo) != 0;
    while (big) {               // one long slice per turn, up to SG_LONG_LOADS entries of it per lane
        const int t = __builtin_ctzll(big);
        big &= big - 1;
        const int64_t s = readlane_i64(lo, t), len = readlane_i64(hi, t) - s;
        const double at = readlane_d(a, t);
        const int pt = __builtin_amdgcn_readlane(pa, t);
        int64_t o = lane;
        if (len >= 64 * SG_LONG_LOADS) {
            // turns in which every lane has all its entries run without predicates, and the loads of the next
            // such turn are in flight while this one's products go into LDS
            // In a full turn a lane takes SG_LONG_LOADS consecutive entries: one 16-byte load of columns and two of
            // values per lane instead of four loads of each, a stride of 64 entries apart.  (Entries of B lie at any
            // 4- and 8-byte boundary: the loads are declared unaligned.)
            static_assert(SG_LONG_LOADS == 4, "a lane's entries of a full turn are one 16-byte load of columns");
            int64_t c = s + 4 * (int64_t)lane;          // this lane's first entry of the turn
            col4 j = *reinterpret_cast<const col4 *>(Bcrd + c);
            sg_d2u v0 = *reinterpret_cast<const sg_d2u *>(Bval + c), v1 = *reinterpret_cast<const sg_d2u *>(Bval + c + 2);
            int64_t done = 0;
            for (int64_t full = 64 * SG_LONG_LOADS; full + 64 * SG_LONG_LOADS <= len; full += 64 * SG_LONG_LOADS) {
                const int64_t cn = c + 64 * SG_LONG_LOADS;
                const col4 jn = *reinterpret_cast<const col4 *>(Bcrd + cn);
                const sg_d2u v0n = *reinterpret_cast<const sg_d2u *>(Bval + cn);
                const sg_d2u v1n = *reinterpret_cast<const sg_d2u *>(Bval + cn + 2);
                f4(j, at, v0, v1, pt, c);
                j = jn;
                v0 = v0n;
                v1 = v1n;
                c = cn;
                done += 64 * SG_LONG_LOADS;
            }
            f4(j, at, v0, v1, pt, c);
            done += 64 * SG_LONG_LOADS;
            o += done;
        }
        if (o < len)
            turn_of_slice<COL>(s, o, len, at, pt, Bcrd, Bval, f);
    }
    // The short slices are laid end to end and dealt to the lanes entry by entry, 64 at a time, so that every load
    // and every LDS operation has all its lanes (a quarter-wavefront per slice left two thirds of them idle: a
    // slice of one block holds a dozen entries).  The lane that holds the slice an entry belongs to is found by
    // bisection over the running sum of the slices' lengths.
    if (todo) {
        const int mylen = (todo >> lane) & 1ull ? (int)(hi - lo) : 0;
        const int upto = wave_inclusive_scan(mylen);           // entries of the short slices of lanes 0..lane
        const int total = __builtin_amdgcn_readlane(upto, 63);
        // the entries e0 + 64 x + lane: where they lie in B, whose they are, and their loads
        const auto fetch = [&](int e0, bool *ok, int64_t *q, double *at, int *pt, int *j, double *v) {
#pragma unroll
            for (int x = 0; x < SG_SHORT_LOADS; ++x) {
                const int e = e0 + 64 * x + lane;
                ok[x] = e < total;
                int l = 0, h = 63;                  // the first lane whose running sum exceeds e
#pragma unroll
                for (int step = 0; step < 6; ++step) {
                    const int mid = (l + h) >> 1;
                    const bool right = __shfl(upto, mid, 64) <= e;
                    l = right ? mid + 1 : l;
                    h = right ? h : mid;
                }
                const int t = ok[x] ? l : lane;
                const int before = __shfl(upto - mylen, t, 64);
                const int64_t s = ((int64_t)__shfl((int)(lo >> 32), t, 64) << 32) |
                                  (uint32_t)__shfl((int)(lo & 0xffffffff), t, 64);
                q[x] = ok[x] ? s + (e - before) : 0;
                at[x] = __hiloint2double(__shfl(__double2hiint(a), t, 64), __shfl(__double2loint(a), t, 64));
                pt[x] = __shfl(pa, t, 64);
            }
#pragma unroll
            for (int x = 0; x < SG_SHORT_LOADS; ++x)
                j[x] = ok[x] ? (int)Bcrd[q[x]] : 0;
#pragma unroll
            for (int x = 0; x < SG_SHORT_LOADS; ++x)
                v[x] = ok[x] ? Bval[q[x]] : 0.0;
        };
        bool ok[SG_SHORT_LOADS];
        int64_t q[SG_SHORT_LOADS];
        double at[SG_SHORT_LOADS], v[SG_SHORT_LOADS];
        int pt[SG_SHORT_LOADS], j[SG_SHORT_LOADS];
        fetch(0, ok, q, at, pt, j, v);
        for (int e0 = 0; e0 < total; e0 += 64 * SG_SHORT_LOADS) {
            // the next batch's loads are in flight while this one's products go into LDS
            bool okn[SG_SHORT_LOADS];
            int64_t qn[SG_SHORT_LOADS];
            double atn[SG_SHORT_LOADS], vn[SG_SHORT_LOADS];
            int ptn[SG_SHORT_LOADS], jn[SG_SHORT_LOADS];
            const bool more = e0 + 64 * SG_SHORT_LOADS < total;
            if (more)
                fetch(e0 + 64 * SG_SHORT_LOADS, okn, qn, atn, ptn, jn, vn);
#pragma unroll
            for (int x = 0; x < SG_SHORT_LOADS; ++x) {
                if (ok[x]) {
                    f(j[x], at[x], v[x], pt[x], q[x]);
                }
            }
            if (more) {
#pragma unroll
                for (int x = 0; x < SG_SHORT_LOADS; ++x) {
                    ok[x] = okn[x];
                    q[x] = qn[x];
                    at[x] = atn[x];
                    v[x] = vn[x];
                    pt[x] = ptn[x];
                    j[x] = jn[x];
                }
            }
        }
    }
    return touched;
}

// One product a * b for column j of the block that begins at column col0 (j counts from there with 16-bit columns):
// its bit is set and it is added to the column's accumulator in LDS.
template <bool SEMI, typename COL>
__device__ __forceinline__ void dense_add(double *acc, uint32_t *bm, int col0, int j, double a, double b, int pa,
                                          int64_t q, int reduce_op, int mult_op)
{
    if constexpr (sizeof(COL) == 4)
        j -= col0;
    atomicOr(&bm[j >> 5], 1u << (j & 31));
    if constexpr (SEMI)
        semiring_lds_add(&acc[j], reduce_op, mult_op, a, b, pa, q);
    else
        __hip_atomic_fetch_add(&acc[j], a * b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
// Four consecutive entries of a row of B at once (columns ascending): the bits that fall into one word of the bitmap
// go there together - lanes that walk a dense slice otherwise pile up on that word, four times each.
template <bool SEMI, typename COL, typename J4, typename V2>
__device__ __forceinline__ void dense_add4(double *acc, uint32_t *bm, int col0, J4 j4, double a, V2 v0, V2 v1, int pa,
                                           int64_t q, int reduce_op, int mult_op)
{
    int j[4] = {(int)j4.x, (int)j4.y, (int)j4.z, (int)j4.w};
    const double b[4] = {v0.x, v0.y, v1.x, v1.y};
    if constexpr (sizeof(COL) == 4) {
#pragma unroll
        for (int x = 0; x < 4; ++x)
            j[x] -= col0;
    }
    int w = j[0] >> 5;
    uint32_t bits = 1u << (j[0] & 31);
#pragma unroll
    for (int x = 1; x < 4; ++x) {
        if ((j[x] >> 5) != w) {
            atomicOr(&bm[w], bits);
            w = j[x] >> 5;
            bits = 0u;
        }
        bits |= 1u << (j[x] & 31);
    }
    atomicOr(&bm[w], bits);
#pragma unroll
    for (int x = 0; x < 4; ++x) {
        if constexpr (SEMI)
            semiring_lds_add(&acc[j[x]], reduce_op, mult_op, a, b[x], pa, q + x);
        else
            __hip_atomic_fetch_add(&acc[j[x]], a * b[x], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
}
// the block's value of column j, which is cleared (as: where the row of A begins, for the semirings that keep places)
template <bool SEMI>
__device__ __forceinline__ double dense_take(double *acc, int j, int reduce_op, int mult_op, int64_t as,
                                             const double *__restrict__ Aval, const double *__restrict__ Bval)
{
    double out;
    if constexpr (SEMI)
        out = semiring_lds_value(reinterpret_cast<unsigned long long *>(acc)[j], reduce_op, mult_op, as, Aval, Bval);
    else
        out = acc[j];
    acc[j] = 0.0;
    return out;
}

// Writes out the block of SG_CB columns a workgroup holds in LDS (bitmap bm, accumulators read and cleared through
// take) as sorted entries of C and leaves the bitmap clean; returns how many.  place(total), which every thread
// calls once the number of entries is known, says where in Ccrd / Cval the first of them goes.  With MASKED the
// columns that are not set in mb are dropped and mb is cleared as well.
template <bool MASKED, typename TAKE, typename PLACE>
__device__ __forceinline__ int dense_emit_block(uint32_t *bm, uint32_t *mb, double *acc, emit_t *emit_col,
                                                int *wave_tot, int lane, int wave, int col0,
                                                int32_t *__restrict__ Ccrd, double *__restrict__ Cval, TAKE take,
                                                PLACE place)
{
    // Thread t owns the columns [8t, 8t + 8) and [8192 + 8t, 8192 + 8t + 8): one byte from each half of the bitmap,
    // so that the dense low columns of a half (the columns of a power-law graph thin out with the number of set
    // bits of the id) are spread over all the wavefronts.  The counts of the two bytes are scanned together,
    // packed into one word.
    static_assert(SG_T * 16 == SG_CB && SG_WAVES <= 64, "one byte of each half of the bitmap per thread");
    const uint8_t *bm8 = reinterpret_cast<const uint8_t *>(bm);
    uint32_t bits_a = bm8[threadIdx.x], bits_b = bm8[SG_CB / 16 + threadIdx.x];
    const int jbase = (int)threadIdx.x << 3;
    if constexpr (MASKED) {          // columns outside the mask row are dropped here
        const uint8_t *mb8 = reinterpret_cast<const uint8_t *>(mb);
        const uint32_t keep_a = mb8[threadIdx.x], keep_b = mb8[SG_CB / 16 + threadIdx.x];
        for (uint32_t w = bits_a & ~keep_a; w; w &= w - 1)
            acc[jbase + __ffs(w) - 1] = 0.0;
        for (uint32_t w = bits_b & ~keep_b; w; w &= w - 1)
            acc[SG_CB / 2 + jbase + __ffs(w) - 1] = 0.0;
        bits_a &= keep_a;
        bits_b &= keep_b;
    }
    const int mine = __popc(bits_a) | (__popc(bits_b) << 16);
    const int inc = wave_inclusive_scan(mine);
    if (lane == 63)
        wave_tot[wave] = inc;
    lds_barrier();
    const int tots = wave_inclusive_scan(lane < SG_WAVES ? wave_tot[lane] : 0);
    const int all = __builtin_amdgcn_readlane(tots, SG_WAVES - 1);
    const int before = (wave ? __builtin_amdgcn_readlane(tots, wave - 1) : 0) + inc - mine;
    const int total_a = all & 0xffff, total = total_a + (all >> 16);
    const int first_a = before & 0xffff, first_b = total_a + (before >> 16);
    const int64_t off = place(total);
    if (threadIdx.x < SG_CB / 32) {    // everybody has read its bytes: the bitmap is clean for the next block,
        bm[threadIdx.x] = 0;           // which nobody enters before the barrier below
        if constexpr (MASKED)
            mb[threadIdx.x] = 0;
    }
    // The owner of a byte knows where its columns go, but writing them from there would scatter every store over
    // 64 cache lines.  So the columns are listed in LDS, SG_EMIT at a time, and then every lane writes the entry
    // at its own place in the list: coalesced stores.
    if (total <= SG_EMIT) {         // the usual case: the whole block fits the list
        int at = first_a;
        for (uint32_t w = bits_a; w; w &= w - 1, ++at)
            emit_col[at] = (emit_t)(jbase + __ffs(w) - 1);
        at = first_b;
        for (uint32_t w = bits_b; w; w &= w - 1, ++at)
            emit_col[at] = (emit_t)(SG_CB / 2 + jbase + __ffs(w) - 1);
        lds_barrier();
        for (int q = threadIdx.x; q < total; q += SG_T) {
            const int j = emit_col[q];
            store_streaming(&Ccrd[off + q], col0 + j);
            store_streaming(&Cval[off + q], take(j));
        }
        lds_barrier();
    } else {
        for (int c0 = 0; c0 < total; c0 += SG_EMIT) {
            int at = first_a - c0;
            for (uint32_t w = bits_a; w; w &= w - 1, ++at)
                if (at >= 0 && at < SG_EMIT)
                    emit_col[at] = (emit_t)(jbase + __ffs(w) - 1);
            at = first_b - c0;
            for (uint32_t w = bits_b; w; w &= w - 1, ++at)
                if (at >= 0 && at < SG_EMIT)
                    emit_col[at] = (emit_t)(SG_CB / 2 + jbase + __ffs(w) - 1);
            lds_barrier();
            const int n = total - c0 < SG_EMIT ? total - c0 : SG_EMIT;
            for (int q = threadIdx.x; q < n; q += SG_T) {
                const int j = emit_col[q];
                store_streaming(&Ccrd[off + c0 + q], col0 + j);
                store_streaming(&Cval[off + c0 + q], take(j));
            }
            lds_barrier();
        }
    }
    return total;
}

// MASKED (C<M> = A*B, for the rows whose mask row is too long for the slab kernel's hash table): every product is
// added as without a mask - the LDS adds are not what this kernel waits for - and the mask row decides what leaves:
// before a block's products are walked, the mask row's entries inside the block are set in a bitmap of their own
// (the row is sorted, so they start where the block before ended), and when the block is written out the columns
// outside it are dropped and their accumulators cleared.
// COL: B's columns as 32-bit numbers, or as 16-bit numbers inside their block (see turn_of_slice).
template <bool SEMI, bool MASKED, typename COL>
__global__ __launch_bounds__(SG_T) void spgemm_numeric_dense_kernel(
    int64_t row_begin, int64_t row_end, const int64_t *__restrict__ Apos, const int32_t *__restrict__ Acrd,
    const double *__restrict__ Aval, const COL *__restrict__ Bcrd, const double *__restrict__ Bval,
    const int64_t *__restrict__ Mpos, const int32_t *__restrict__ Mcrd,
    const int64_t *__restrict__ blkptr, int nblk,
    unsigned long long *ticket, RowList list,
    const int64_t *__restrict__ Cpos, int32_t *__restrict__ Ccrd, double *__restrict__ Cval, int reduce_op,
    int mult_op)
{
    __shared__ int64_t row_slot;
    __shared__ int wave_tot[SG_WAVES];
    __shared__ int block_touched[3];            // see visit_flag
    __shared__ unsigned long long mask_next[2]; // where the mask row's entries of a block begin; blocks take turns
    double *acc = reinterpret_cast<double *>(sg_dyn_lds);
    uint32_t *bm = sg_dyn_lds + SG_CB * 2;
    emit_t *emit_col = reinterpret_cast<emit_t *>(bm + SG_CB / 32);
    uint32_t *mbits = reinterpret_cast<uint32_t *>(emit_col + SG_EMIT);
    if constexpr (MASKED) {
        for (int w = threadIdx.x; w < 2 * (SG_CB / 32); w += SG_T)
            mbits[w] = 0;
    }
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    for (int j = threadIdx.x; j < SG_CB; j += SG_T)
        acc[j] = 0.0;
    if (threadIdx.x < SG_CB / 32)
        bm[threadIdx.x] = 0;
    if (threadIdx.x < 3)
        block_touched[threadIdx.x] = 0;
    lds_barrier();
    int visit = 0;
    const int64_t out0 = Cpos[row_begin];
    int64_t t_first, t_end;
    list_range(list, LIST_WIDEST, &t_first, &t_end);     // the other heavy rows go to spgemm_numeric_span_kernel
    int64_t t = draw_row<true>(ticket, t_first, &row_slot);
    while (t < t_end) {
        const int64_t i = row_begin + list.rows[t];
        const int64_t as = Apos[i], ae = Apos[i + 1];
        int64_t me = 0;
        if constexpr (MASKED) {
            me = Mpos[i + 1];
            if (threadIdx.x == 0)
                mask_next[0] = mask_next[1] = (unsigned long long)Mpos[i];
            lds_barrier();
        }
        if (as != ae) {
            int64_t off = Cpos[i] - out0;
            // A row of at most one entry of A per lane (nearly all rows) keeps its entries in registers over
            // the blocks: the end of a slice in one block is its start in the next, so a block costs one
            // pointer load per lane, and that load is issued a block ahead.
            const int held = __builtin_amdgcn_readfirstlane((int)(ae - as <= SG_T));
            int64_t h_lo = 0, h_hi = 0;
            double h_a = 0.0;
            int h_pa = 0;
            const int64_t *h_bp = nullptr;
            if (held) {
                const int64_t p = as + wave + (int64_t)lane * SG_WAVES;
                if (p < ae) {
                    h_bp = blkptr + (int64_t)Acrd[p] * (nblk + 1);
                    h_lo = h_bp[0];
                    h_hi = h_bp[1];
                    h_a = Aval[p];
                    h_pa = (int)(p - as + 1);
                }
            }
            for (int cb = 0; cb < nblk; ++cb) {
                const int col0 = cb << SG_CB_LOG;
                uint32_t *mb = mbits + (cb & 1) * (SG_CB / 32);
                if constexpr (MASKED) {
                    // The mask row's entries inside this block: they begin at mask_next[cb & 1], and where they end
                    // goes to the other slot, for the next block (a slot is read in one block and written in the
                    // next one, with the block's barrier in between; it only ever grows along a row).
                    const int64_t lo = (int64_t)mask_next[cb & 1];
                    const int col_end = col0 + SG_CB;
                    if (threadIdx.x == 0)
                        atomicMax(&mask_next[(cb + 1) & 1], (unsigned long long)lo);
                    for (int64_t e = lo + threadIdx.x; e < me; e += SG_T) {
                        const int j = Mcrd[e];
                        if (j >= col_end)
                            break;
                        atomicOr(&mb[(j - col0) >> 5], 1u << ((j - col0) & 31));
                        if (e + 1 == me || Mcrd[e + 1] >= col_end)
                            atomicMax(&mask_next[(cb + 1) & 1], (unsigned long long)(e + 1));
                    }
                }
                int touched = 0;     // did this wavefront add anything to the block
                const auto add = [&](int j, double a, double b, int pa, int64_t q) {
                    dense_add<SEMI, COL>(acc, bm, col0, j, a, b, pa, q, reduce_op, mult_op);
                };
                const auto add4 = [&](auto j, double a, auto v0, auto v1, int pa, int64_t q) {
                    dense_add4<SEMI, COL>(acc, bm, col0, j, a, v0, v1, pa, q, reduce_op, mult_op);
                };
                const auto take = [&](int j) { return dense_take<SEMI>(acc, j, reduce_op, mult_op, as, Aval, Bval); };
                if (held) {
                    int64_t next = h_hi;
                    if (h_bp && cb + 1 < nblk)
                        next = h_bp[cb + 2];
                    touched = for_each_in_slices(h_lo, h_hi, h_a, h_pa, lane, Bcrd, Bval, add, add4);
                    h_lo = h_hi;
                    h_hi = next;
                }
                for (int64_t base = as + wave; !held && base < ae; base += (int64_t)SG_WAVES * 64) {
                    const int64_t left = (ae - base + SG_WAVES - 1) / SG_WAVES;
                    const int cnt = (int)(left < 64 ? left : 64);
                    int64_t lo = 0, hi = 0;
                    double a = 0.0;
                    int pa = 0;
                    if (lane < cnt) {
                        const int64_t p = base + (int64_t)lane * SG_WAVES;
                        const int64_t *bp = blkptr + (int64_t)Acrd[p] * (nblk + 1) + cb;
                        lo = bp[0];
                        hi = bp[1];
                        a = Aval[p];
                        pa = (int)(p - as + 1);
                    }
                    touched |= for_each_in_slices(lo, hi, a, pa, lane, Bcrd, Bval, add, add4);
                }
                const int any = visit_flag(block_touched, visit, touched, lane);
                visit = visit == 2 ? 0 : visit + 1;
                if (any) {
                    off += dense_emit_block<MASKED>(bm, mb, acc, emit_col, wave_tot, lane, wave, col0, Ccrd, Cval,
                                                    take, [&](int) { return off; });
                } else if constexpr (MASKED) {   // the block received no product
                    if (threadIdx.x < SG_CB / 32)        // (the next block's bits go to the other half; the one after
                        mb[threadIdx.x] = 0;             // that comes after the next block's barrier)
                }
            }
        }
        t = draw_row<true>(ticket, t_first, &row_slot);
    }
}

// ---------------------------------------------------------------------------
// The same rows, block by block: the kernel above takes a row through its column blocks, so at any time the
// workgroups of an XCD read the slices of every block and the long rows of B, which most products come from,
// never stay in its L2 (a few hundred rows of an R-MAT graph make over half of the products, but they hold
// tens of megabytes).  Here the tickets go over (column block, row) with the block outermost: all workgroups
// are in the same block at the same time and what they share is that block's slices of the long rows only.
// A row's entries inside a block then leave before the blocks ahead of it are counted, so where they go is
// handed from block to block: before[r * nblk + cb] = the row's entries ahead of block cb, written by the
// workgroup that counted block cb - 1 and awaited by the one that writes block cb.  That one holds a later
// ticket, and a workgroup only ever waits for earlier tickets, which running workgroups hold: the one with the
// earliest unfinished ticket waits for nobody.  The wait is bounded all the same (`patience` polls, after
// which *gave_up is set and the row is wrong: the host then fails the call).
// A ticket is up to DB_ROWS consecutive rows of the list, so that the loads which lead to a row's slices (its entries
// of A, their block pointers) are issued while the row before is walked.
// ---------------------------------------------------------------------------
struct DenseRow {
    int64_t as;         // first entry of the row of A
    int64_t coff;       // first entry of the row of C, counted from the row block's
    int32_t cnt;        // entries of the row of A
    int32_t pad;
};
constexpr int DB_ROWS = 8;
// A matrix of fewer columns than a block.  The columns there are are shared out to the wavefronts, or one writes out what all
// have added; and where there are rows enough (nine to two CUs) two workgroups of half the lanes share a CU, one adding while
// the other starts on a row or writes it out.  us, A*A, R-MAT, a block of 16384 columns / its own / two workgroups, and the rows
// here: 1024 vertices, edge factor 8, min-plus 61.9 / 57.8 / 60.5 (114), 2048 and 16 95.0 / 85.7 / 94.7 (724), 4000 and 10 122 /
// 112 / 120 (1105); plus-times 3000 and 12 107 / 99 / 98 (1121), 8000 and 5 119 / 115 / 111 (1171), 4096 and 16 136 / 126 / 120
// (1766), 8000 and 10 177 / 168 / 158 (2639), 6000 and 16 236 / 232 / 184 (3096), 8192 and 16 268 / 264 / 218 (3776).
constexpr int64_t DB_TWO_ROWS = 9;
constexpr int DB_PATIENCE = 1 << 24;

// Where the rows come from: the first of the list, as rows of A and C.
struct RowSource {
    const int32_t *list;
    int64_t row_begin;
    const int64_t *Apos, *Cpos;
};
__device__ __forceinline__ DenseRow dense_row(const RowSource &s, int64_t x)
{
    const int64_t i = s.row_begin + s.list[x];
    DenseRow r;
    r.as = s.Apos[i];
    r.cnt = (int32_t)(s.Apos[i + 1] - r.as);         // (the host sends matrices of under 2^30 entries here)
    r.coff = s.Cpos[i] - s.Cpos[s.row_begin];
    r.pad = 0;
    return r;
}

// rows[r] for the nd first rows of the list and before[] in its initial state: nothing ahead of block 0, the rest open
__global__ void spgemm_dense_rows(RowSource source, int64_t nd, int nblk, DenseRow *__restrict__ rows,
                                  int32_t *__restrict__ before)
{
    const int64_t x = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (x < nd * nblk)
        before[x] = x % nblk == 0 ? 0 : -1;
    if (x < nd)
        rows[x] = dense_row(source, x);
}

// The slices of a row of the product inside a block lie in LDS for all wavefronts: 64 to a batch, the batch's own slices
// that are not empty in front, and they are streamed end to end.  A batch is cut into quads of four entries wherever its
// slices end, 64 quads are a turn, and the turns of all batches go to the wavefronts one by one: every wavefront has its
// share of the row whatever the lengths are, and the loads of two turns (5 KiB a wavefront) are under way while a third
// goes into LDS.  (A slice at a time to the wavefront that holds its entry of A waited for memory at every slice and for
// the wavefront with the longest ones at the end.)
// Bound by the LDS, two thirds of the time busy: 36 clocks for 64 additions of doubles, 14 of them bank conflicts.  A*A of
// R-MAT graphs, whole product: 65536 vertices, edge factor 16 5.31 -> 4.76 ms (with the walk alone, accumulators beside a
// bitmap as before, 5.23), 30000 and 10 1.74 -> 1.47; 2^20 and 16 349 -> 329 ms.
constexpr int64_t SLICE_NNZ_MOST = 1ll << 32;    // a place in B and the end of 64 slices fit a word
struct alignas(16) SliceRec {
    int64_t where;                   // first entry less 4 x quads before it << END_BITS + 6 | lane that brought it << END_BITS | end
    double a;                        // A's value
};
// ENTRIES of A at a time; slices of MOST entries at most are staged: longer ones only with repeated columns
template <int ENTRIES, int MOST_, int END_BITS_, int WAVES_ = SG_WAVES>
struct SliceStage {
    static constexpr int SLICES = ENTRIES, MOST = MOST_, END_BITS = END_BITS_, WAVES = WAVES_;
    static_assert(64ll * MOST < 1ll << END_BITS && END_BITS + 6 + 34 <= 64, "the end of a batch's last slice fits, and a place");
    SliceRec rec[ENTRIES];
    int first[ENTRIES];              // quads of its batch before a slice
    uint32_t marks[WAVES][2];        // zero between turns
    int turns[ENTRIES / 64];         // of each batch
};
template <int T>
using BlockStage = SliceStage<T, SG_CB, 21, T / 64>;
// of workgroups of T lanes whose wavefronts each have 64 * ROWS columns
template <int T, int ROWS>
constexpr size_t DB_LDS = (size_t)T * ROWS * 8 + sizeof(BlockStage<T>);
static_assert(DB_LDS<SG_T, 16> + 256 <= 160 * 1024, "accumulators and slices fit LDS");
static_assert(512 * 16 == SG_CB / 2 && 2 * (DB_LDS<512, 16> + 256) <= 160 * 1024, "so do two workgroups' of a matrix of half a block");

template <typename COL>
struct SliceTurn {
    typename SgCol4<COL>::type j;
    sg_d2u v0, v1;
    double a;
    int64_t q;                       // the place in B of the four entries
    uint32_t mask;                   // which of them are the slice's
    int pa;                          // the place of a among the row's staged entries
};

// a lane's slice [lo, hi) of this pass and its entry of A; the wavefronts of the entries that are staged call it
template <typename STAGE>
__device__ __forceinline__ void slice_put(STAGE &st, int64_t lo, int64_t hi, double a, int lane, int wave)
{
    constexpr int DB_END_BITS = STAGE::END_BITS;
    const int len = hi - lo > STAGE::MOST ? STAGE::MOST : (int)(hi - lo);
    const unsigned long long has = __ballot(len > 0);
    const int below = __builtin_amdgcn_mbcnt_hi((uint32_t)(has >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)has, 0));
    const int slot = wave * 64 + (len > 0 ? below : __popcll(has) + lane - below);
    const int quads = (len + 3) >> 2, inc = wave_inclusive_scan(quads), pre = inc - quads;
    SliceRec r;
    r.where = (lo - 4 * pre) << (DB_END_BITS + 6) | (int64_t)lane << DB_END_BITS | (int64_t)(len + 4 * pre);
    r.a = a;
    st.rec[slot] = r;
    st.first[slot] = len > 0 ? pre : 1 << 30;
    if (lane == 63)
        st.turns[wave] = (inc + 63) >> 6;
}

// four(turn) for this wavefront's turns of the staged slices (without VALUES B's are not read); returns the number of turns
// of all wavefronts
// LEAN: fewer copies of `four`, where it is long
template <bool VALUES, bool LEAN, typename COL, typename STAGE, typename FOUR>
__device__ __forceinline__ int slice_walk(STAGE &st, const COL *__restrict__ Bcrd, const double *__restrict__ Bval,
                                          int64_t nnz, int lane, int wave, FOUR four)
{
    typedef typename SgCol4<COL>::type col4;
    constexpr int DB_END_BITS = STAGE::END_BITS;
    const int own = lane < STAGE::SLICES / 64 ? st.turns[lane] : 0;
    const int upto = wave_inclusive_scan(own);
    const int total = __builtin_amdgcn_readlane(upto, 63);
    uint32_t *marks = st.marks[wave];
    int batch = -1, pre = 0;
    const auto issue = [&](SliceTurn<COL> &t, int i) {          // the wavefront's turn i
        const int g = wave + i * STAGE::WAVES, b = __builtin_ctzll(__ballot(upto > g));
        const int base = (g - (__builtin_amdgcn_readlane(upto, b) - __builtin_amdgcn_readlane(own, b))) * 64;
        if (b != batch) {
            batch = b;
            pre = st.first[b * 64 + lane];
        }
        // a slice that begins at quad s > base sets bit s - 1 - base: the bits below a quad are the slices up to its own
        const uint32_t bit = (uint32_t)(pre - 1 - base);
        if (bit < 64u)
            atomicOr(&marks[bit >> 5], 1u << (bit & 31u));
        const int before = __popcll(__ballot(pre <= base)) - 1;
        wave_lds_order();
        const uint2 m = *reinterpret_cast<const uint2 *>(marks);
        wave_lds_order();
        if (lane < 2)
            marks[lane] = 0;
        const int owner = (int)__builtin_amdgcn_mbcnt_hi(m.y, __builtin_amdgcn_mbcnt_lo(m.x, (uint32_t)before));
        const SliceRec r = st.rec[b * 64 + owner];
        const int q4 = 4 * (base + lane);
        const int left = (int)(r.where & ((1 << DB_END_BITS) - 1)) - q4;
        int64_t q = (r.where >> (DB_END_BITS + 6)) + q4;
        t.a = r.a;
        t.pa = b * 64 + ((int)(r.where >> DB_END_BITS) & 63);
        const int n = left < 0 ? 0 : left < 4 ? left : 4;
        t.mask = (1u << n) - 1u;
        if (n == 0)
            q = 0;
        if (q > nnz - 4) {               // the last entries of B
            t.mask <<= (int)(q - (nnz - 4));
            q = nnz - 4;
        }
        t.q = q;
        t.j = *reinterpret_cast<const col4 *>(Bcrd + q);
        if constexpr (VALUES) {
            t.v0 = *reinterpret_cast<const sg_d2u *>(Bval + q);
            t.v1 = *reinterpret_cast<const sg_d2u *>(Bval + q + 2);
        }
        wave_lds_order();
    };
    // No turn inside the loop is issued on a condition: where loads under way may or may not have been followed by others,
    // the compiler waits for all of them, and every second turn then waited for loads just issued.  us, kernel of whole
    // blocks and of several: 65536 vertices, edge factor 16 2282 + 867 -> 2145 + 834, 30000 and 10 340 + 315 -> 323 + 306.
    const int n = (total - wave + STAGE::WAVES - 1) / STAGE::WAVES;
    if (n <= 0)
        return total;
    SliceTurn<COL> x, y;
    issue(x, 0);
    if (n > 1) {
        issue(y, 1);
        int i = 2;
        for (; i + 1 < n; i += 2) {
            four(x);
            issue(x, i);
            four(y);
            issue(y, i + 1);
        }
        if constexpr (!LEAN) {
            four(x);
            if (i == n) {
                four(y);
                return total;
            }
            issue(x, i);
            four(y);
            four(x);
            return total;
        }
    } else {
        y.mask = 0;
    }
    four(x);
    if constexpr (LEAN) {
        x.mask = 0;
        if (n > 1 && n % 2 != 0)
            issue(x, n - 1);
        four(y);
        four(x);
    }
    return total;
}

// An accumulator of the block that has received nothing holds a value that no sum and no key can be, and so the block
// needs no bitmap: -0.0 where products are added (every product is made +0.0 if it is -0.0 first, as an accumulator
// that starts at +0.0 would have it; a sum of others is never -0.0), 0 where keys are kept (the one NaN whose key is 0
// takes the next one's).  The product and the +0.0 must stay two operations: fused, a negative product that underflows gives
// -0.0, and its entry, counted in the structure, would be missing from the row.
__device__ __forceinline__ unsigned long long block_empty(int reduce_op)
{
    return reduce_op == SR_PLUS ? 0x8000000000000000ull : 0ull;
}
template <bool SEMI>
__device__ __forceinline__ void block_add(double *slot, double a, double b, int pa, int64_t q, int reduce_op, int mult_op)
{
#pragma clang fp contract(off)
    if constexpr (SEMI) {
        unsigned long long *key = reinterpret_cast<unsigned long long *>(slot);
        if (reduce_op == SR_ANY) {
            semiring_lds_add(slot, reduce_op, mult_op, a, b, pa, q);
        } else {
            const double e = semiring_mult(mult_op, a, b);
            if (reduce_op == SR_PLUS) {
                __hip_atomic_fetch_add(slot, e + 0.0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            } else {
                const unsigned long long k = reduce_op == SR_MIN ? ~f64_key(e) : f64_key(e);
                __hip_atomic_fetch_max(key, k ? k : 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            }
        }
    } else {
        __hip_atomic_fetch_add(slot, a * b + 0.0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
}

// Writes out what the accumulators of a block hold, in order of the columns, and leaves them empty; place(total) as in
// dense_emit_block.  A wavefront has 64 * ROWS columns to itself: it takes them into registers, and its part of acc becomes
// the list, half of the columns at a time, from which every lane writes the entry at its own place.
template <bool SEMI, int WAVES, int ROWS, typename VALUE, typename PLACE>
__device__ __forceinline__ void block_emit(double *acc, int *wave_tot, int lane, int wave, int col0, int reduce_op,
                                           int32_t *__restrict__ Ccrd, double *__restrict__ Cval, VALUE value, PLACE place)
{
    constexpr int MINE = 64 * ROWS, HALF = ROWS / 2;
    static_assert(MINE / 2 * (8 + 2) <= MINE * 8, "the list of half the columns fits their accumulators");
    const unsigned long long empty = block_empty(SEMI ? reduce_op : SR_PLUS);
    unsigned long long *own = reinterpret_cast<unsigned long long *>(acc) + wave * MINE;
    uint16_t *own_col = reinterpret_cast<uint16_t *>(own + MINE / 2);
    unsigned long long v[ROWS], held[ROWS];
    int cnt = 0;
#pragma unroll
    for (int r = 0; r < ROWS; ++r)
        v[r] = own[r * 64 + lane];
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
        held[r] = __ballot(v[r] != empty);
        cnt += __popcll(held[r]);
    }
    if (lane == 0)
        wave_tot[wave] = cnt;
    lds_barrier();
    const int tots = wave_inclusive_scan(lane < WAVES ? wave_tot[lane] : 0);
    const int total = __builtin_amdgcn_readlane(tots, WAVES - 1);
    int64_t off = place(total) + (wave ? __builtin_amdgcn_readlane(tots, wave - 1) : 0);
    const int first = col0 + wave * MINE;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        int n = 0;
#pragma unroll
        for (int r = h * HALF; r < (h + 1) * HALF; ++r) {
            const unsigned long long m = held[r];
            const int at = n + (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0));
            if (m >> lane & 1ull) {
                own[at] = v[r];
                own_col[at] = (uint16_t)(r * 64 + lane);
            }
            n += __popcll(m);
        }
        wave_lds_order();
        for (int q = lane; q < n; q += 64) {
            store_streaming(&Ccrd[off + q], first + (int)own_col[q]);
            store_streaming(&Cval[off + q], value(own[q]));
        }
        wave_lds_order();
        off += n;
    }
    const ulonglong2 none = make_ulonglong2(empty, empty);
#pragma unroll
    for (int r = 0; r < ROWS / 2; ++r)
        reinterpret_cast<ulonglong2 *>(own)[r * 64 + lane] = none;
}

// ALONE: the matrix is one block wide, a row's entries leave at once; nobody has listed the rows (rows is null then).
// T lanes, 64 * ROWS columns to a wavefront.
template <bool SEMI, typename COL, bool ALONE, int T, int ROWS>
__global__ __launch_bounds__(T, 4) void spgemm_numeric_dense_blocks_kernel(
    const DenseRow *__restrict__ rows, RowSource source, int64_t nd, const int32_t *__restrict__ Acrd, const double *__restrict__ Aval,
    const COL *__restrict__ Bcrd, const double *__restrict__ Bval, int64_t Bnnz, const int64_t *__restrict__ blkptr, int nblk,
    unsigned long long *ticket, int32_t *before, int rows_each, int patience, int *gave_up, int32_t *__restrict__ Ccrd,
    double *__restrict__ Cval, int reduce_op, int mult_op)
{
    __shared__ int64_t row_slot;
    __shared__ int wave_tot[T / 64];
    __shared__ int ahead_slot;                  // the row's entries ahead of the block
    double *acc = reinterpret_cast<double *>(sg_dyn_lds);
    BlockStage<T> &st = *reinterpret_cast<BlockStage<T> *>(acc + T * ROWS);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    for (int j = threadIdx.x; j < T * ROWS; j += T)
        reinterpret_cast<unsigned long long *>(acc)[j] = block_empty(SEMI ? reduce_op : SR_PLUS);
    if (lane < 2)
        st.marks[wave][lane] = 0;
    lds_barrier();
    const int64_t nchunks = (nd + rows_each - 1) / rows_each;
    const int64_t u_end = ALONE ? nchunks : nchunks * nblk;
    // (ALONE: the first by number - 256 draws from one word take 3 us; the others' order is what lets a block wait for the
    // one before it)
    int64_t u = ALONE ? (int64_t)blockIdx.x : draw_row<true>(ticket, 0, &row_slot);
    while (u < u_end) {
        const int cb = ALONE ? 0 : (int)(u / nchunks);
        const int64_t r0 = (u - cb * nchunks) * rows_each;
        const int nr = (int)(nd - r0 < rows_each ? nd - r0 : rows_each);
        const int col0 = cb << SG_CB_LOG;
        DenseRow mine;
        mine.as = mine.coff = 0;
        mine.cnt = 0;
        if (lane < nr) {
            if constexpr (ALONE)
                mine = dense_row(source, r0 + lane);
            else
                mine = rows[r0 + lane];
        }
        // the entry of A a lane holds of row x of the ticket (of its first T entries: a longer row loads the others
        // as it goes), and the slice of its row of B inside the block
        const auto load_entry = [&](int x, int &k, double &a) {
            k = -1;
            a = 0.0;
            if (x < nr) {
                const int cnt = __builtin_amdgcn_readlane(mine.cnt, x);
                const int p = (int)threadIdx.x;
                if (p < cnt) {
                    const int64_t as = ((int64_t)__builtin_amdgcn_readlane((int)(mine.as >> 32), x) << 32) |
                                       (uint32_t)__builtin_amdgcn_readlane((int)mine.as, x);
                    k = Acrd[as + p];
                    a = Aval[as + p];
                }
            }
        };
        const auto load_slice = [&](int k, int64_t &lo, int64_t &hi) {
            lo = hi = 0;
            if (k >= 0) {
                const int64_t *bp = blkptr + (ALONE ? 2 * (int64_t)k : (int64_t)k * (nblk + 1) + cb);
                lo = bp[0];
                hi = bp[1];
            }
        };
        int k0, k1, k2;
        double a0, a1, a2;
        int64_t lo0, hi0, lo1, hi1;
        load_entry(0, k0, a0);
        load_entry(1, k1, a1);
        load_slice(k0, lo0, hi0);
        slice_put(st, lo0, hi0, a0, lane, wave);
        lds_barrier();
        for (int x = 0; x < nr; ++x) {
            load_slice(k1, lo1, hi1);
            load_entry(x + 2, k2, a2);
            const int cnt = __builtin_amdgcn_readlane(mine.cnt, x);
            const int64_t as = ((int64_t)__builtin_amdgcn_readlane((int)(mine.as >> 32), x) << 32) |
                               (uint32_t)__builtin_amdgcn_readlane((int)mine.as, x);
            const int64_t coff = ((int64_t)__builtin_amdgcn_readlane((int)(mine.coff >> 32), x) << 32) |
                                 (uint32_t)__builtin_amdgcn_readlane((int)mine.coff, x);
            const int from0 = sizeof(COL) == 4 ? col0 : 0;
            // the staged slices; what of a slice with repeated columns is not staged is its lane's
            const auto walk = [&](int pa0, int64_t lo, int64_t hi, double a) {
                const int turns = slice_walk<true, SEMI, COL>(st, Bcrd, Bval, Bnnz, lane, wave, [&](const SliceTurn<COL> &t) {
                    const int j[4] = {(int)t.j.x, (int)t.j.y, (int)t.j.z, (int)t.j.w};
                    const double b[4] = {t.v0.x, t.v0.y, t.v1.x, t.v1.y};
#pragma unroll
                    for (int x = 0; x < 4; ++x)
                        if (t.mask >> x & 1u)
                            block_add<SEMI>(&acc[j[x] - from0], t.a, b[x], pa0 + t.pa + 1, t.q + x, reduce_op, mult_op);
                });
                for (int64_t q = lo + BlockStage<T>::MOST; q < hi; ++q)
                    block_add<SEMI>(&acc[(int)Bcrd[q] - from0], a, Bval[q], pa0 + (int)threadIdx.x + 1, q, reduce_op, mult_op);
                return turns;
            };
            // What lies ahead of this block comes from whoever counted the block before it.  That was many tickets
            // ago as a rule, so the answer is asked for before the walk and the trip to memory it takes is over by
            // the time the walk is; only if it was not there yet is it waited for, behind the walk.
            int32_t *mark = ALONE ? nullptr : before + (r0 + x) * nblk + cb;
            int early = 0;
            if (!ALONE && threadIdx.x == 0 && cb > 0)
                early = __hip_atomic_fetch_max(mark, -1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            int turns;
            if (cnt <= T) {
                turns = walk(0, lo0, hi0, a0);
                lds_barrier();
            } else {
                // the entries of A beyond the first T, T at a time: a pass's entries are loaded two passes
                // ahead and its slices one, so that a walk does not begin with two trips to memory
                const auto load_more = [&](int base, int &k, double &a) {
                    k = -1;
                    a = 0.0;
                    if (base + (int)threadIdx.x < cnt) {
                        k = Acrd[as + base + threadIdx.x];
                        a = Aval[as + base + threadIdx.x];
                    }
                };
                int kn;
                double ab = a0, an;
                int64_t lob = lo0, hib = hi0;
                load_more(T, kn, an);
                turns = 0;
                for (int base = 0; base < cnt; base += T) {
                    int64_t lon, hin;
                    load_slice(kn, lon, hin);
                    int kf;
                    double af;
                    load_more(base + 2 * T, kf, af);
                    turns += walk(base, lob, hib, ab);
                    lds_barrier();
                    lob = lon;
                    hib = hin;
                    ab = an;
                    kn = kf;
                    an = af;
                    if (base + T < cnt) {
                        slice_put(st, lob, hib, ab, lane, wave);
                        lds_barrier();
                    }
                }
            }
            // the next row's slices, read behind the barriers of the write-out
            slice_put(st, lo1, hi1, a1, lane, wave);
            const int any = turns;          // every wavefront counts the same
            const auto await = [&]() {
                int ahead = early;
                if constexpr (ALONE)
                    return 0;
                for (int polls = 1; ahead < 0 && polls < patience; ++polls) {
                    __builtin_amdgcn_s_sleep(4);
                    ahead = __hip_atomic_fetch_max(mark, -1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
                if (ahead < 0) {
                    __hip_atomic_store(gave_up, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);          // in host memory
                    ahead = 0;
                }
                return ahead;
            };
            const auto hand_on = [&](int ahead) {
                if (!ALONE && cb + 1 < nblk)
                    __hip_atomic_exchange(mark + 1, ahead, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            };
            if (any) {
                if (threadIdx.x == 0)
                    ahead_slot = await();          // (read behind the first barrier of the write-out)
                block_emit<SEMI, T / 64, ROWS>(acc, wave_tot, lane, wave, col0, reduce_op, Ccrd, Cval,
                                 [&](unsigned long long v) {
                                     return SEMI ? semiring_lds_value(v, reduce_op, mult_op, as, Aval, Bval)
                                                 : __longlong_as_double((long long)v);
                                 },
                                 [&](int total) {
                                     const int ahead = ahead_slot;
                                     if (threadIdx.x == 0)
                                         hand_on(ahead + total);
                                     return coff + ahead;
                                 });
            } else if (threadIdx.x == 0) {
                hand_on(await());
            }
            lds_barrier();
            k0 = k1;
            a0 = a1;
            lo0 = lo1;
            hi0 = hi1;
            k1 = k2;
            a1 = a2;
        }
        u = draw_row<true>(ticket, ALONE ? gridDim.x : 0, &row_slot);
    }
}

// ---------------------------------------------------------------------------
// Heavy rows that are not wide: a row with 10^4..10^5 products is the union of a few long rows of B with hardly
// a column in common, so each of its 64 column blocks receives a few hundred products and a block visit of the
// kernel above costs more in barriers and write-out than in products.  Here a visit spans up to SP_BLOCKS column
// blocks and keeps the values compact: a first pass over the products sets the span's bitmap in LDS, a prefix
// sum over the bitmap gives every column its rank, and a second pass adds each product at the rank of its column
// (two LDS reads and one fp64 LDS atomic).  The values then leave in rank order, which is column order, and the
// columns come from the bitmap.  The compact array holds SP_CAP = 16384 entries; a span that holds more is cut
// at the last block boundary that fits (one block always does), so the kernel is right for any row and merely
// slow for wide ones.
// ---------------------------------------------------------------------------
constexpr int SP_BLOCKS = 8;                              // column blocks per visit at most
constexpr int SP_BLOCK_WORDS = SG_CB / 32;                // bitmap words of one block
constexpr int SP_WORDS = SP_BLOCKS * SP_BLOCK_WORDS;      // bitmap words of a span
constexpr int SP_WPT = SP_WORDS / SG_T;                   // consecutive bitmap words per thread
constexpr int SP_CAP = SG_CB;                             // entries of C per visit at most
constexpr int SP_ENTRIES = 256;                           // entries of A that are staged at a time
typedef SliceStage<SP_ENTRIES, SP_BLOCKS * SG_CB, 24> SpanStage;
constexpr size_t SG_SPAN_LDS = (size_t)SP_CAP * 8 + (size_t)SP_WORDS * 4 + (size_t)SP_WORDS * 2 +       // values, bitmap, ranks
                               sizeof(SpanStage);
static_assert(((size_t)SP_WORDS * 6) % 16 == 0, "the values (fp64) come first, the staged slices begin on 16 bytes");
static_assert(SG_SPAN_LDS + 512 <= 160 * 1024, "all of it fits LDS");
static_assert(SP_WORDS % SG_T == 0 && SP_BLOCK_WORDS % SP_WPT == 0 && SP_CAP >= SG_CB && SP_CAP <= 65535,
              "a thread's words lie in one block, one block fits the value array, ranks fit 16 bits");

template <bool SEMI>
__global__ __launch_bounds__(SG_T) void spgemm_numeric_span_kernel(
    int64_t row_begin, const int64_t *__restrict__ Apos, const int32_t *__restrict__ Acrd,
    const double *__restrict__ Aval, const int32_t *__restrict__ Bcrd, const double *__restrict__ Bval, int64_t Bnnz,
    const int64_t *__restrict__ blkptr, int nblk, RowList list,
    const int64_t *__restrict__ Cpos, int32_t *__restrict__ Ccrd, double *__restrict__ Cval, int reduce_op,
    int mult_op)
{
    __shared__ int wave_tot[SG_WAVES];
    __shared__ int blk_pre[SP_BLOCKS + 1];      // entries of the span before each of its blocks, and in all
    double *val = reinterpret_cast<double *>(sg_dyn_lds);
    uint32_t *bm = sg_dyn_lds + SP_CAP * 2;
    uint16_t *pre = reinterpret_cast<uint16_t *>(bm + SP_WORDS);
    SpanStage &st = *reinterpret_cast<SpanStage *>(pre + SP_WORDS);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    for (int j = threadIdx.x; j < SP_CAP; j += SG_T)
        val[j] = 0.0;
    for (int w = threadIdx.x; w < SP_WORDS; w += SG_T)
        bm[w] = 0;
    if (lane < 2)
        st.marks[wave][lane] = 0;
    lds_barrier();
    const int64_t out0 = Cpos[row_begin];
    int64_t t_first, t_end;
    list_range(list, LIST_SPAN, &t_first, &t_end);
    // Rows dealt out in advance: the list goes down by products, so every workgroup gets about the same, and what leads to
    // a row's slices can be fetched ahead - the bounds of 64 rows at a time, a row's first entries of A two rows ahead and
    // their slices one.
    int64_t l_as = 0, l_coff = 0;
    int l_cnt = 0, l_out = 0;
    const auto load_entry = [&](int r, int base, int &k, double &a) {
        k = -1;
        a = 0.0;
        const int cnt = __builtin_amdgcn_readlane(l_cnt, r & 63);
        if (r < 64 && (int)threadIdx.x < SP_ENTRIES && base + (int)threadIdx.x < cnt) {
            const int64_t p = readlane_i64(l_as, r & 63) + base + threadIdx.x;
            k = Acrd[p];
            a = Aval[p];
        }
    };
    const auto load_slice = [&](int k, int cbf, int cbt, int64_t &lo, int64_t &hi) {
        lo = hi = 0;
        if (k >= 0) {
            const int64_t *bp = blkptr + (int64_t)k * (nblk + 1);
            lo = bp[cbf];
            hi = bp[cbt];
        }
    };
    const auto put = [&](int64_t lo, int64_t hi, double a) {
        if (wave < SP_ENTRIES / 64)
            slice_put(st, lo, hi, a, lane, wave);
    };
    const int span0 = nblk < SP_BLOCKS ? nblk : SP_BLOCKS;
    for (int64_t t0 = t_first + blockIdx.x; t0 < t_end; t0 += 64 * (int64_t)gridDim.x) {
    const int64_t t = t0 + lane * (int64_t)gridDim.x;
    l_cnt = 0;
    if (t < t_end) {
        const int64_t i = row_begin + list.rows[t];
        l_as = Apos[i];
        l_cnt = (int)(Apos[i + 1] - l_as);               // (the host sends matrices of under 2^30 entries here)
        l_coff = Cpos[i] - out0;
        l_out = (int)(Cpos[i + 1] - Cpos[i]);
    }
    const int64_t left = (t_end - 1 - t0) / gridDim.x + 1;
    const int nr = __builtin_amdgcn_readfirstlane((int)(left < 64 ? left : 64));
    int k0, k1;
    double a0, a1;
    int64_t lo0, hi0;
    load_entry(0, 0, k0, a0);
    load_entry(1, 0, k1, a1);
    load_slice(k0, 0, span0, lo0, hi0);
    for (int r = 0; r < nr; ++r) {
        int k2;
        double a2;
        int64_t lo1, hi1;
        load_slice(k1, 0, span0, lo1, hi1);
        load_entry(r + 2, 0, k2, a2);
        const int64_t as = readlane_i64(l_as, r), coff = readlane_i64(l_coff, r);
        const int cnt = __builtin_amdgcn_readlane(l_cnt, r);
        bool copy = false;
        if (cnt == 1) {          // and the row of B holds no column twice
            const int64_t *bp = blkptr + (int64_t)Acrd[as] * (nblk + 1);
            copy = __builtin_amdgcn_readfirstlane((int)(bp[nblk] - bp[0])) == __builtin_amdgcn_readlane(l_out, r);
        }
        if (copy) {
            // one entry of A: the row of C is that row of B times the entry (0 + a * b, as an accumulator that
            // starts at zero gives it).  70,000 rows of the R-MAT product at scale 20 are like that, each the
            // copy of a hub's row.
            const int64_t *bp = blkptr + (int64_t)Acrd[as] * (nblk + 1);
            const int64_t bs = bp[0], len = bp[nblk] - bs, off = coff;
            const double a = Aval[as];
            for (int64_t q = threadIdx.x; q < len; q += SG_T) {
                store_streaming(&Ccrd[off + q], Bcrd[bs + q]);
                if constexpr (SEMI) {        // what the reference's accumulator holds after this one product
                    const double e = semiring_mult(mult_op, a, Bval[bs + q]);
                    store_streaming(&Cval[off + q], reduce_op == SR_PLUS  ? 0.0 + e
                                                    : reduce_op == SR_MAX ? (f64_key(e) < f64_key(0.0) ? 0.0 : e)
                                                                          : e);
                } else {
                    store_streaming(&Cval[off + q], 0.0 + a * Bval[bs + q]);
                }
            }
        } else if (cnt > 0) {
            int64_t off = coff;
            int cb = 0;
            while (cb < nblk) {
                const int nbv = nblk - cb < SP_BLOCKS ? nblk - cb : SP_BLOCKS;
                const int col0 = cb << SG_CB_LOG;
                // f4(columns, mask, ...) over the products whose columns lie in the blocks [cb, cbt), SP_ENTRIES entries
                // of A at a time; staged: the slices of the one pass there is are in LDS already.  Returns the turns.
                const auto walk = [&](int cbt, bool staged, auto values, auto f) -> int {
                    constexpr bool VALUES = decltype(values)::value;
                    int turns = 0;
                    for (int base = 0; base < cnt; base += SP_ENTRIES) {
                        int k = k0;
                        double a = a0;
                        int64_t lo = lo0, hi = hi0;
                        if (base > 0)
                            load_entry(r, base, k, a);
                        if (base > 0 || cb > 0 || cbt != span0)
                            load_slice(k, cb, cbt, lo, hi);
                        if (!staged || base > 0) {
                            put(lo, hi, a);
                            lds_barrier();
                        }
                        turns += slice_walk<VALUES, VALUES && SEMI, int32_t>(st, Bcrd, Bval, Bnnz, lane, wave, [&](const SliceTurn<int32_t> &u) {
                            const int j[4] = {u.j.x - col0, u.j.y - col0, u.j.z - col0, u.j.w - col0};
                            f(j, u.mask, u.a, u.v0, u.v1, base + u.pa + 1, u.q);
                        });
                        // what of a slice with repeated columns is not staged is its lane's, one entry at a time
                        for (int64_t q = lo + SpanStage::MOST; q < hi; ++q) {
                            const int j[4] = {Bcrd[q] - col0, 0, 0, 0};
                            f(j, 1u, a, sg_d2u{Bval[q], 0.0}, sg_d2u{0.0, 0.0}, base + (int)threadIdx.x + 1, q);
                        }
                        lds_barrier();
                    }
                    return turns;
                };
                const int any = walk(cb + nbv, false, std::false_type{},
                                     [&](const int (&j)[4], uint32_t mask, double, sg_d2u, sg_d2u, int, int64_t) {
                    // entries of a sorted row: the bits that fall into one word go there together
                    int w = 0;
                    uint32_t bits = 0u;
#pragma unroll
                    for (int x = 0; x < 4; ++x)
                        if (mask >> x & 1u) {
                            if (bits && (j[x] >> 5) != w) {
                                atomicOr(&bm[w], bits);
                                bits = 0u;
                            }
                            w = j[x] >> 5;
                            bits |= 1u << (j[x] & 31);
                        }
                    if (bits)
                        atomicOr(&bm[w], bits);
                });
                int nb = nbv;
                if (any) {
                    // ranks: thread t owns the words [SP_WPT * t, SP_WPT * (t + 1))
                    uint32_t w[SP_WPT];
                    int mine = 0;
#pragma unroll
                    for (int k = 0; k < SP_WPT; ++k) {
                        w[k] = bm[threadIdx.x * SP_WPT + k];
                        mine += __popc(w[k]);
                    }
                    const int inc = wave_inclusive_scan(mine);
                    if (lane == 63)
                        wave_tot[wave] = inc;
                    lds_barrier();
                    const int tots = wave_inclusive_scan(lane < SG_WAVES ? wave_tot[lane] : 0);
                    const int all = __builtin_amdgcn_readlane(tots, SG_WAVES - 1);
                    const int before = (wave ? __builtin_amdgcn_readlane(tots, wave - 1) : 0) + inc - mine;
                    int run = before;
#pragma unroll
                    for (int k = 0; k < SP_WPT; ++k) {
                        pre[threadIdx.x * SP_WPT + k] = (uint16_t)(run < 65535 ? run : 65535);    // exact below the cut
                        run += __popc(w[k]);
                    }
                    if (threadIdx.x % (SP_BLOCK_WORDS / SP_WPT) == 0)
                        blk_pre[threadIdx.x / (SP_BLOCK_WORDS / SP_WPT)] = before;
                    if (threadIdx.x == SG_T - 1)
                        blk_pre[SP_BLOCKS] = all;
                    lds_barrier();
                    // the cut: as many blocks as fit the value array (blocks the span does not have are empty)
                    nb = 1;
                    for (int b = 2; b <= nbv; ++b)
                        nb = __builtin_amdgcn_readfirstlane(blk_pre[b]) <= SP_CAP ? b : nb;
                    const int total = __builtin_amdgcn_readfirstlane(blk_pre[nb]);
                    // (a cut visit ends, and the next span starts, at block cb + nb)
                    const auto add_at_rank = [&](int j, double a, double b, int pa, int64_t q) {
                        const uint32_t below = bm[j >> 5] & ((1u << (j & 31)) - 1u);
                        const int r = pre[j >> 5] + __popc(below);
                        if constexpr (SEMI)
                            semiring_lds_add(&val[r], reduce_op, mult_op, a, b, pa, q);
                        else
                            __hip_atomic_fetch_add(&val[r], a * b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                    };
                    walk(cb + nb, cnt <= SP_ENTRIES && nb == nbv, std::true_type{},
                         [&](const int (&j)[4], uint32_t mask, double a, sg_d2u v0, sg_d2u v1, int pa, int64_t q) {
                        const double b[4] = {v0.x, v0.y, v1.x, v1.y};
#pragma unroll
                        for (int x = 0; x < 4; ++x)
                            if (mask >> x & 1u)
                                add_at_rank(j[x], a, b[x], pa, q + x);
                    });
                    for (int q = threadIdx.x; q < total; q += SG_T) {
                        if constexpr (SEMI)
                            store_streaming(&Cval[off + q],
                                            semiring_lds_value(reinterpret_cast<unsigned long long *>(val)[q], reduce_op,
                                                               mult_op, as, Aval, Bval));
                        else
                            store_streaming(&Cval[off + q], val[q]);
                    }
                    lds_barrier();
                    // the values are out: their array now takes the list of the columns, so that these leave
                    // through coalesced stores too (from their owners they would scatter, four bytes per lane)
                    uint32_t *cols = reinterpret_cast<uint32_t *>(val);
                    int at = before;
#pragma unroll
                    for (int k = 0; k < SP_WPT; ++k) {
                        const int wi = threadIdx.x * SP_WPT + k;
                        if (wi < nb * SP_BLOCK_WORDS)
                            for (uint32_t bits = w[k]; bits; bits &= bits - 1)
                                cols[at++] = (uint32_t)(wi * 32 + __ffs(bits) - 1);
                        bm[wi] = 0;             // also the words beyond the cut: the next visit sets them again
                    }
                    lds_barrier();
                    for (int q = threadIdx.x; q < total; q += SG_T)
                        store_streaming(&Ccrd[off + q], col0 + (int)cols[q]);
                    lds_barrier();
                    for (int q = threadIdx.x; q < total; q += SG_T)
                        val[q] = 0.0;           // nobody adds into it before the next visit's three barriers
                    off += total;
                }
                cb += nb;
            }
        }
        k0 = k1;
        a0 = a1;
        lo0 = lo1;
        hi0 = hi1;
        k1 = k2;
        a1 = a2;
    }
    }
}

// ---------------------------------------------------------------------------
// Masked SpGEMM + SUM without the output: rowsum[i] = sum over products of row
// i that fall on a stored entry of mask row i.  Per-lane partial sums are
// combined in a fixed order, so the result does not depend on scheduling.
// ---------------------------------------------------------------------------
template <bool BM_LDS>
__global__ __launch_bounds__(SG_T) void spgemm_masked_sum_kernel(
    int64_t nrows, const int64_t *__restrict__ Apos, const int32_t *__restrict__ Acrd,
    const double *__restrict__ Aval, const int64_t *__restrict__ Bpos, const int32_t *__restrict__ Bcrd,
    const double *__restrict__ Bval, const int64_t *__restrict__ Mpos, const int32_t *__restrict__ Mcrd,
    int logW, uint32_t *__restrict__ gbm, unsigned long long *ticket, RowList list, double *__restrict__ rowsum)
{
    // takes the rows with work from the heavy end of the list; spgemm_masked_sum_small_kernel comes from the other
    __shared__ int64_t row_slot;
    __shared__ double wave_part[SG_WAVES];
    uint32_t *bm;
    if constexpr (BM_LDS)
        bm = sg_dyn_lds;
    else
        bm = gbm + (size_t)blockIdx.x * (size_t)(SG_T * ((1 << logW) + 1));
    const BmAddr ad{logW};
    const int nwords = SG_T * ((1 << logW) + 1);
    if constexpr (BM_LDS) {
        for (int w = threadIdx.x; w < nwords; w += SG_T)
            bm[w] = 0;
    }
    __syncthreads();
    int64_t t_first, t_end;
    list_range(list, LIST_ALL, &t_first, &t_end);
    int64_t tk = draw_front(ticket, t_end, &row_slot);
    while (tk < t_end) {
        const int64_t i = list.rows[tk];      // rows outside the list keep the zero the host put there
        const int64_t as = Apos[i], ae = Apos[i + 1];
        const int64_t ms = Mpos[i], me = Mpos[i + 1];
        const bool work = as != ae && ms != me;
        if (work) {
        for (int64_t t = ms + threadIdx.x; t < me; t += SG_T)
            atomicOr(&bm[ad.word(Mcrd[t])], ad.bit(Mcrd[t]));
        __syncthreads();
        double part = 0.0;
        for_each_product_probed<true>(as, ae, Acrd, Aval, Bpos, Bcrd, [&](int j) {
            if constexpr (BM_LDS)
                return bm[ad.word(j)];
            else
                return atomicOr(&bm[ad.word(j)], 0u);
        }, [&](int j, int64_t q, uint32_t word) {
            MaskHit h{-1, 0.0};
            if (word & ad.bit(j)) {      // the value is fetched for hits only
                h.at = 0;
                h.b = Bval[q];
            }
            return h;
        }, [&](int, int64_t, double a, int64_t, int64_t, MaskHit h) {
            if (h.at >= 0)
                part += a * h.b;
        });
        part = wave_sum_f64(part);
        if ((threadIdx.x & 63) == 0)
            wave_part[threadIdx.x >> 6] = part;
        __syncthreads();
        if (threadIdx.x == 0) {
            double total = 0.0;
            for (int w = 0; w < SG_WAVES; ++w)
                total += wave_part[w];
            rowsum[i] = total;
        }
        for (int64_t t = ms + threadIdx.x; t < me; t += SG_T)
            atomicAnd(&bm[ad.word(Mcrd[t])], 0u);
        }   // work
        tk = draw_front(ticket, t_end, &row_slot);     // its barriers also close this row's bitmap clean-up
    }
}

// ---------------------------------------------------------------------------
// The same sum for rows with few products: one wavefront per row, no workgroup
// barrier anywhere.  A row of a thousand products spends more time on the
// ticket, bitmap and reduction barriers of the kernel above than on its
// products.  Here the mask row goes into a small hash table in LDS that belongs
// to the wavefront; the neighbours of the row are taken one at a time and the
// lanes walk along that neighbour's row of B, probing the table.  A mask row too
// long for the table is searched by bisection in memory instead.
// ---------------------------------------------------------------------------
constexpr int SM_WAVES = 4;                    // wavefronts per workgroup
constexpr int SM_SLOTS = 256;                  // hash slots per wavefront (1 KB: four such workgroups fit a CU beside
                                               // one workgroup of the kernel above and its 132 KB bitmap)
constexpr int SM_MASK_MAX = 96;                // longest mask row that goes into the table
constexpr int SM_BATCH = 16;                   // rows a wavefront claims at a time in the lighter half of the list

__device__ inline int sm_hash(int j) { return (int)(((uint32_t)j * 2654435761u) >> 24) & (SM_SLOTS - 1); }

__global__ __launch_bounds__(SM_WAVES * 64) void spgemm_masked_sum_small_kernel(
    const int64_t *__restrict__ Apos, const int32_t *__restrict__ Acrd, const double *__restrict__ Aval,
    const int64_t *__restrict__ Bpos, const int32_t *__restrict__ Bcrd, const double *__restrict__ Bval,
    const int64_t *__restrict__ Mpos, const int32_t *__restrict__ Mcrd, unsigned long long *ticket, RowList list,
    double *__restrict__ rowsum)
{
    __shared__ int table[SM_WAVES][SM_SLOTS];
    const int lane = threadIdx.x & 63;
    int *tab = table[threadIdx.x >> 6];
    for (int s = lane; s < SM_SLOTS; s += 64)
        tab[s] = -1;
    int64_t t_first, t_end;
    list_range(list, LIST_ALL, &t_first, &t_end);
    int take = SM_BATCH;
    int64_t mine_next = 0, mine_end = 0;     // the rows t_end - 1 - b, b in [mine_next, mine_end), are this wavefront's
    for (;;) {
        if (mine_next == mine_end) {
            // rows from the light end of the list (see draw_front): SM_BATCH at a time in the lighter half of the
            // list - rows of a few thousand products at most, and 600,000 draws on one word are what the L2 does
            // in the time the whole count takes - a quarter of that in the next quarter, then one by one: a
            // batch of rows near the meeting point would keep one wavefront for long
            unsigned long long drawn = 0;
            if (lane == 0)
                drawn = atomicAdd(ticket, (unsigned long long)take << 32);
            const int64_t f = (int64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(drawn & 0xffffffffu));
            const int64_t b = (int64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(drawn >> 32));
            if (f + b >= t_end)
                break;
            mine_next = b;
            mine_end = b + take < t_end - f ? b + take : t_end - f;     // what the front had not reached
            const int64_t taken = b + take;
            take = taken < t_end / 2 ? SM_BATCH : taken < t_end - t_end / 4 ? SM_BATCH / 4 : 1;
        }
        const int64_t tk = t_end - 1 - mine_next;
        ++mine_next;
        const int64_t i = list.rows[tk];
        const int64_t as = Apos[i], ae = Apos[i + 1], ms = Mpos[i], me = Mpos[i + 1];
        if (as == ae || ms == me)
            continue;               // rowsum[i] keeps the zero the host put there
        const bool hashed = me - ms <= SM_MASK_MAX;
        if (hashed)
            for (int64_t t = ms + lane; t < me; t += 64) {
                const int j = Mcrd[t];
                int h = sm_hash(j);
                while (atomicCAS(&tab[h], -1, j) != -1)
                    h = (h + 1) & (SM_SLOTS - 1);
            }
        double part = 0.0;
        for (int64_t p0 = as; p0 < ae; p0 += 64) {
            // up to 64 neighbours at a time: lane l holds neighbour p0 + l, its value and its row of B
            const int cnt = (int)(ae - p0 < 64 ? ae - p0 : 64);
            int64_t bs = 0, be = 0;
            double a = 0.0;
            if (lane < cnt) {
                const int k = Acrd[p0 + lane];
                bs = Bpos[k];
                be = Bpos[k + 1];
                a = Aval[p0 + lane];
            }
            auto probe = [&](int j, int64_t q, double al) {
                bool hit = false;
                if (hashed) {
                    int h = sm_hash(j);
                    for (int v = tab[h]; v != -1; v = tab[h]) {
                        if (v == j) {
                            hit = true;
                            break;
                        }
                        h = (h + 1) & (SM_SLOTS - 1);
                    }
                } else {
                    int64_t lo = ms, hi = me;
                    while (lo < hi) {
                        const int64_t mid = (lo + hi) >> 1;
                        if (Mcrd[mid] < j)
                            lo = mid + 1;
                        else
                            hi = mid;
                    }
                    hit = lo < me && Mcrd[lo] == j;
                }
                if (hit)
                    part += al * Bval[q];
            };
            // rows of B with 64 entries and more take the whole wavefront, one at a time; shorter ones (a row
            // of the lower triangle holds 15 entries on average) go to the four 16-lane quarters, four at a time.
            // (Laying all products of the row end to end, lane x taking product x after a bisection over the
            // running totals, fills every lane and was slower: 11.0 against 10.0 ms - the kernel is bound by
            // instructions per product, not by idle lanes.)
            unsigned long long big = __ballot(be - bs >= 64);
            unsigned long long todo = __ballot(bs < be && be - bs < 64);
            while (big) {
                const int l = __builtin_ctzll(big);
                big &= big - 1;
                const int64_t s = readlane_i64(bs, l), e = readlane_i64(be, l);
                const double al = readlane_d(a, l);
                for (int64_t q = s + lane; q < e; q += 256) {      // all loads of a turn first, then the probes
                    int j[4];
#pragma unroll
                    for (int x = 0; x < 4; ++x)
                        j[x] = q + 64 * x < e ? Bcrd[q + 64 * x] : 0;
#pragma unroll
                    for (int x = 0; x < 4; ++x)
                        if (q + 64 * x < e)
                            probe(j[x], q + 64 * x, al);
                }
            }
            const int quarter = lane >> 4, sub = lane & 15;
            while (todo) {
                int pick = -1;
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const int l = todo ? __builtin_ctzll(todo) : -1;
                    todo = todo ? (todo & (todo - 1)) : 0;
                    pick = quarter == g ? l : pick;
                }
                const int src = pick < 0 ? lane : pick;
                const int64_t s = ((int64_t)__shfl((int)(bs >> 32), src, 64) << 32) |
                                  (uint32_t)__shfl((int)(bs & 0xffffffff), src, 64);
                const int64_t e = ((int64_t)__shfl((int)(be >> 32), src, 64) << 32) |
                                  (uint32_t)__shfl((int)(be & 0xffffffff), src, 64);
                const double al = __hiloint2double(__shfl(__double2hiint(a), src, 64),
                                                   __shfl(__double2loint(a), src, 64));
                int j[4];                   // a row here has fewer than 64 entries: four per lane cover it
#pragma unroll
                for (int x = 0; x < 4; ++x)
                    j[x] = pick >= 0 && s + sub + 16 * x < e ? Bcrd[s + sub + 16 * x] : 0;
#pragma unroll
                for (int x = 0; x < 4; ++x)
                    if (pick >= 0 && s + sub + 16 * x < e)
                        probe(j[x], s + sub + 16 * x, al);
            }
        }
        part = wave_sum_f64(part);
        if (lane == 0)
            rowsum[i] = part;
        if (hashed)
            for (int s = lane; s < SM_SLOTS; s += 64)
                tab[s] = -1;
    }
}

// ---------------------------------------------------------------------------
// CSR .* CSR -> CSR, one lane per row, two-pointer merge of the sorted rows
// (lib/Conversion/IndexTreeToSCF/IndexTreeToSCF.cpp:864-1053).
// ---------------------------------------------------------------------------
template <bool FILL>
__global__ void eltwise_mult_kernel(int64_t nrows, const int64_t *__restrict__ Apos,
                                    const int32_t *__restrict__ Acrd, const double *__restrict__ Aval,
                                    const int64_t *__restrict__ Bpos, const int32_t *__restrict__ Bcrd,
                                    const double *__restrict__ Bval, int64_t *__restrict__ rowcount,
                                    const int64_t *__restrict__ Cpos, int32_t *__restrict__ Ccrd,
                                    double *__restrict__ Cval)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nrows)
        return;
    int64_t p = Apos[i], q = Bpos[i];
    const int64_t pe = Apos[i + 1], qe = Bpos[i + 1];
    int64_t n = 0;
    int64_t o = FILL ? Cpos[i] : 0;
    while (p < pe && q < qe) {
        const int ca = Acrd[p], cb = Bcrd[q];
        if (ca == cb) {
            if (FILL) {
                Ccrd[o] = ca;
                Cval[o] = Aval[p] * Bval[q];
                ++o;
            }
            ++n;
        }
        p += (ca <= cb);
        q += (cb <= ca);
    }
    if (!FILL)
        rowcount[i] = n;
}

// CSR (op) Dense, op = * for the plain elementwise product and any other COMET_OP_* for the monoid forms
// A @(op) B of test/integration/semiring/eltwise_monoid*_COOxDense_oCOO.ta: the stored entries of A combined
// with the dense values under them.  TO_DENSE writes them into a dense
// output at their positions and leaves every other element as it was (the nest only visits the entries of
// A, test/integration/ops/eltwise_mult_CSRxDense_oDense.ta); otherwise they become the values of a CSR with
// A's structure (eltwise_mult_CSRxDense_oCSR.ta).
template <bool TO_DENSE>
__global__ void eltwise_mult_dense_kernel(int64_t nrows, const int64_t *__restrict__ pos,
                                          const int32_t *__restrict__ crd, const double *__restrict__ val,
                                          const double *__restrict__ D, int64_t ldd, double *__restrict__ out,
                                          int64_t ldo, int op)
{
    // one 16-lane group per row
    const int64_t i = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 4;
    if (i >= nrows)
        return;
    for (int64_t p = pos[i] + (threadIdx.x & 15); p < pos[i + 1]; p += 16) {
        const double v = semiring_mult(op, val[p], D[i * ldd + crd[p]]);
        if (TO_DENSE)
            out[i * ldo + crd[p]] = v;
        else
            out[p] = v;
    }
}

// ------------------------------------------------------------------ host side
// ---------------------------------------------------------------------------
// Masked products as dot products over the mask (the reference's masked Gustavson nest,
// lib/Conversion/IndexTreeToSCF/IndexTreeToSCF.cpp:1083-1148 and :1327-1448, walks every product of row i and tests
// its column against the mask row's mark array; C keeps the mask's entries that received a product, in mask order -
// what comes out here is the same set and, per entry, the same sum).  C<M>[i][j] = sum over k of A[i][k] * B[k][j] is the dot product of
// row i of A and column j of B; walking the products of row i (every entry of every B_k, k in A_i) costs |B_k|
// look-ups per entry of A_i whatever the mask holds, the dot product of a stored pair (i, j) costs the shorter of
// its two lists when that one is streamed against a table of the longer one.  So the pairs of the mask are split
// by which list is longer, and for every row x of a matrix of pairs P the list T_x goes into a table that the lists
// L_y of the pairs (x, y) of that half are streamed against (masked_dots.h).
//   the row's half:     P = M,   T = A (rows),            L = B^T (columns of B);  pair (i, j) when |B^T_j| <= |A_i|
//   the column's half:  P = M^T, T = B^T (columns of B),  L = A (rows);            pair (j, i) when |A_i| < |B^T_j|
// ---------------------------------------------------------------------------
// rowcount[i - rb] = stored pairs of mask row i that met a product
__global__ __launch_bounds__(256) void spgemm_dot_count(int64_t rb, int64_t re, const int64_t *__restrict__ Mpos,
                                                        const uint8_t *__restrict__ pair_hit,
                                                        int64_t *__restrict__ rowcount)
{
    const int64_t i = rb + (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (i >= re)
        return;
    const int lane = threadIdx.x & 63;
    const int64_t out0 = Mpos[rb];
    int n = 0;
    for (int64_t p = Mpos[i] + lane; p < Mpos[i + 1]; p += 64)
        n += pair_hit[p - out0];
    n = wave_sum_i32(n);
    if (lane == 0)
        rowcount[i - rb] = n;
}

// What a matrix is like, looked at once.  Of its structure (rows are sorted): some row holds a column twice, some entry lies
// on or above the diagonal, some lies on or below it, some row is much longer than the mean; of its values: they are not all
// the same, and the first one.
struct CsrTraits {
    int twice, above, below, uneven, differ, unused;
    double first;
};
// crd or val null: that part is not looked at.  A lane to every entry and to every row: of the few entries whose right
// neighbour has the same column it is looked up whether a row ends between them.  (A wavefront to a row took 293 us for the
// 15.7 M entries of the scale-20 R-MAT graph's lower triangle, the longest rows' way from turn to turn; now 60 us with the
// values.)
__global__ __launch_bounds__(256) void csr_traits(int64_t nrows, int64_t nnz, const int64_t *__restrict__ pos,
                                                  const int32_t *__restrict__ crd, const double *__restrict__ val,
                                                  int64_t even, CsrTraits *__restrict__ out)
{
    const int64_t most = nnz > nrows ? nnz : nrows;
    const double first = val ? val[0] : 0.0;
    bool twice = false, above = false, below = false, uneven = false, differ = false;
    for (int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x; t < most; t += (int64_t)gridDim.x * 256) {
        if (val && t < nnz)
            differ = differ || val[t] != first;
        if (!crd)
            continue;
        if (t < nrows) {
            const int64_t s = pos[t], e = pos[t + 1];
            above = above || (s < e && crd[e - 1] >= t);
            below = below || (s < e && crd[s] <= t);
            uneven = uneven || e - s > even;
        }
        if (t + 1 < nnz && crd[t] == crd[t + 1]) {
            int64_t lo = 0, hi = nrows;          // the first row that begins behind entry t
            while (lo < hi) {
                const int64_t mid = (lo + hi) >> 1;
                if (pos[mid] <= t)
                    lo = mid + 1;
                else
                    hi = mid;
            }
            twice = twice || pos[lo] != t + 1;
        }
    }
    const bool any[5] = {__any(twice) != 0, __any(above) != 0, __any(below) != 0, __any(uneven) != 0, __any(differ) != 0};
    if ((threadIdx.x & 63) == 0) {
        int *flags = &out->twice;
        for (int k = 0; k < 5; ++k)
            if (any[k])
                flags[k] = 1;
    }
    if (blockIdx.x == 0 && threadIdx.x == 0)
        out->first = first;
}

__global__ void fill_iota_f64(int64_t n, double *__restrict__ out)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n)
        out[i] = (double)i;
}

// ---------------------------------------------------------------------------
// Rows with few products, SM_PRODUCTS at most, of matrices of few columns: a row is over in a handful of loads that wait
// for each other, so what counts is how few they are and how many rows are under way.  A workgroup of four wavefronts has
// the row's bitmap, with the number of columns before every word of it, and a value for every product it can have: 26 to
// 38 KiB of LDS, four to six to a CU.  A lane looks up one entry of A, the products are laid end to end over the lanes,
// eight to a lane, which finds the entry of each by counting the beginnings before it: five loads one after the other
// whatever the row looks like, and the products stay in registers for the second time they are needed.  (With sixteen
// lanes to an entry a row of two hundred entries was thirteen times three loads one after the other, twice.)  us, structure
// and values: A*A of R-MAT graphs of 65536 vertices, edge factor 16 96 + 379 -> 56 + 95, 30000 and 10 47 + 156 -> 26 + 48,
// 16000 and 8 24 + 84 -> 17 + 34, 5000 and 12 17 + 36 -> 10 + 21.
// Rows of a product a lane at most - all there are in products of meshes, bands and other graphs of a few edges a vertex -
// are bound by instructions and barriers.  Up to 64 entries of A are therefore held by every wavefront, which finds its
// products' entries by itself; the structure counts the columns that found their bit clear instead of going over the bitmap;
// and where there are enough of them their values have a launch of their own, with half the registers.  us, structure and
// values, sixteen lanes to an entry / eight products a lane / so: 65536 rows of 8 uniform entries 129 + 246 / 210 + 282 / 59 +
// 194, 60000 rows of a band of 9 125 + 230 / 199 + 260 / 63 + 181, a mesh of 22500 18 + 48 / 44 + 70 / 22 + 35, 20000 rows of
// a band of 15 32 + 63 / 54 + 74 / 31 + 48.  (Only these rows have their structure found here: SG_FEW_TOGETHER.)
// ---------------------------------------------------------------------------
constexpr int SM_PER = 8;                           // products of a lane
constexpr int SM_T = 256, SM_COLS = 1 << 16;
constexpr int SM_MID_T = 512;                       // the lanes of a workgroup for twice as many
constexpr int64_t SM_FEW_ROWS = 2048;               // rows of few products that are worth a launch beside others' (4 us)
constexpr int SM_FEW_PRODUCTS = SM_T, SM_PRODUCTS = SM_PER * SM_T, SM_MID_PRODUCTS = SM_PER * SM_MID_T;
template <int T>
struct SmallStage {
    int64_t start[T];                    // of the entries of A that have any: where their products begin in B, less their
    double a[T];                         // place among the products; A's value; the entry's place in the row
    int place[T];
    unsigned long long marks[SM_PER * T / 64];       // a bit where an entry's products begin; zero between passes
    uint32_t own_marks[T / 64][2];       // the same for a wavefront that works by itself
    int tot[2][T / 64];
};
template <int T, int PER>
struct SmallRowLds {                     // behind the bitmap
    double val[PER * T];
    SmallStage<T> stage;
    uint16_t col[PER * T];
    int wave_tot[T / 64];
};
template <bool VALUES, int PER>
struct SmallProducts {
    int col[PER];                        // -1: none
    double a[VALUES ? PER : 1], b[VALUES ? PER : 1];
    int place[VALUES ? PER : 1];
    int64_t q[VALUES ? PER : 1];         // the place in B
};

// A lane's entry of A: its row of B, or no products.
struct SmallEntry {
    int64_t start = 0;                   // in B
    int len = 0, place = 0;              // products; the entry's place in its row, from 1 on
    double a = 0.0;
};
template <bool VALUES>
__device__ __forceinline__ SmallEntry small_entry(int64_t as, int64_t p, int64_t ae, const int32_t *__restrict__ Acrd,
                                                  const double *__restrict__ Aval, const int64_t *__restrict__ Bpos)
{
    SmallEntry e;
    if (p < ae) {
        const int k = Acrd[p];
        e.start = Bpos[k];
        e.len = (int)(Bpos[k + 1] - e.start);
        if constexpr (VALUES) {
            e.a = Aval[p];
            e.place = (int)(p - as) + 1;
        }
    }
    return e;
}

// Of a row whose entries of A every wavefront holds, lane by lane, and of T products at most: the lane's one.  No wavefront
// waits for another.
template <bool VALUES, int T, int PER>
__device__ __forceinline__ void small_few(SmallStage<T> &st, const SmallEntry &e, const int32_t *__restrict__ Bcrd,
                                          const double *__restrict__ Bval, SmallProducts<VALUES, PER> &out)
{
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), base = 64 * wave;
    const int inc = wave_inclusive_scan(e.len), total = __builtin_amdgcn_readlane(inc, 63);
    out.col[0] = -1;
    if (base >= total)
        return;
    const int off = inc - e.len;
    const unsigned long long has = __ballot(e.len > 0);
    const int below = (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(has >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)has, 0));
    // entry number x of those with products is that of lane by_rank[x]
    const int by_rank = __builtin_amdgcn_ds_permute((e.len > 0 ? below : (int)__popcll(has) + lane - below) << 2, lane);
    // an entry that begins at product s > base sets bit s - 1 - base: the bits below a lane are the entries up to its own
    uint32_t *marks = st.own_marks[wave];
    const uint32_t bit = (uint32_t)(off - 1 - base);
    if (e.len > 0 && bit < 64u)
        atomicOr(&marks[bit >> 5], 1u << (bit & 31u));
    const int before = __popcll(__ballot(e.len > 0 && off <= base)) - 1;
    wave_lds_order();
    const uint2 m = *reinterpret_cast<const uint2 *>(marks);
    wave_lds_order();
    if (lane < 2)
        marks[lane] = 0;
    const int owner = lane_value(by_rank, (int)__builtin_amdgcn_mbcnt_hi(m.y, __builtin_amdgcn_mbcnt_lo(m.x, (uint32_t)before)));
    const int64_t start = e.start - off;
    const int64_t q = ((int64_t)lane_value((int)(start >> 32), owner) << 32 | (uint32_t)lane_value((int)start, owner)) + base + lane;
    double a = 0.0;
    int place = 0;
    if constexpr (VALUES) {
        a = __hiloint2double(lane_value(__double2hiint(e.a), owner), lane_value(__double2loint(e.a), owner));
        place = lane_value(e.place, owner);
    }
    if (base + lane < total) {
        out.col[0] = Bcrd[q];
        if constexpr (VALUES) {
            out.q[0] = q;
            out.b[0] = Bval[q];
            out.a[0] = a;
            out.place[0] = place;
        }
    }
}

// Lays out the products of T entries of a row of A, one to a lane, and returns how many there are.  The marks are left set:
// small_clear behind the next barrier.
template <bool VALUES, int T>
__device__ __forceinline__ int small_stage(SmallStage<T> &st, const SmallEntry &e)
{
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), len = e.len;
    const int inc = wave_inclusive_scan(len);
    const unsigned long long has = __ballot(len > 0);
    if (lane == 63) {
        st.tot[0][wave] = inc;
        st.tot[1][wave] = __popcll(has);
    }
    lds_barrier();
    int off = inc - len, slot = (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(has >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)has, 0));
    int total = 0;
#pragma unroll
    for (int w = 0; w < T / 64; ++w) {
        off += w < wave ? st.tot[0][w] : 0;
        slot += w < wave ? st.tot[1][w] : 0;
        total += st.tot[0][w];
    }
    if (len > 0) {
        st.start[slot] = e.start - off;
        if constexpr (VALUES) {
            st.a[slot] = e.a;
            st.place[slot] = e.place;
        }
        atomicOr(&st.marks[off >> 6], 1ull << (off & 63));
    }
    lds_barrier();
    return __builtin_amdgcn_readfirstlane(total);
}
// The lane's products of those laid out, PER at most.
template <bool VALUES, int T, int PER>
__device__ __forceinline__ void small_products(SmallStage<T> &st, int total, const int32_t *__restrict__ Bcrd,
                                               const double *__restrict__ Bval, SmallProducts<VALUES, PER> &out)
{
    const int tid = threadIdx.x, lane = tid & 63;
    static_assert(PER * T / 64 <= 64, "a word of marks to a lane");
    const unsigned long long word = lane < PER * T / 64 ? st.marks[lane] : 0;
    const int before = wave_inclusive_scan(__popcll(word)) - __popcll(word);
#pragma unroll
    for (int x = 0; x < PER; ++x) {
        const int t = tid + T * x, w = t >> 6;
        const unsigned lo = (unsigned)lane_value((int)word, w), hi = (unsigned)lane_value((int)(word >> 32), w);
        const int c = lane_value(before, w);
        out.col[x] = -1;
        if (t < total) {
            const int owner = c + __popcll(((unsigned long long)hi << 32 | lo) & ((2ull << (t & 63)) - 1ull)) - 1;
            const int64_t q = st.start[owner] + t;
            out.col[x] = Bcrd[q];
            if constexpr (VALUES) {
                out.q[x] = q;
                out.b[x] = Bval[q];
                out.a[x] = st.a[owner];
                out.place[x] = st.place[owner];
            }
        }
    }
}
template <int T>
__device__ __forceinline__ void small_clear(SmallStage<T> &st)
{
    if (threadIdx.x < SM_PER * T / 64)
        st.marks[threadIdx.x] = 0;
}
// before[w] = set bits in front of word w, for a thread's share of the words; returns how many there are
template <int T>
__device__ __forceinline__ int small_row_ranks(const uint32_t *bm, uint16_t *before, int words, int *wave_tot)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int per = (words + T - 1) / T, w0 = threadIdx.x * per;
    int mine = 0;
    for (int w = w0; w < w0 + per && w < words; ++w)
        mine += __popc(bm[w]);
    const int inc = wave_inclusive_scan(mine);
    if (lane == 63)
        wave_tot[wave] = inc;
    lds_barrier();
    int run = inc - mine, all = 0;
    for (int x = 0; x < T / 64; ++x) {
        run += x < wave ? wave_tot[x] : 0;
        all += wave_tot[x];
    }
    if (before)
        for (int w = w0; w < w0 + per && w < words; ++w) {
            before[w] = (uint16_t)run;
            run += __popc(bm[w]);
        }
    return all;
}
// the rows a workgroup takes, their bounds fetched while the row before is worked on
struct SmallRows {
    const RowList &list;
    const int64_t *Apos;
    int64_t row_begin, t, t_end;
    int64_t r, rn, as, ae;               // this row (counted from row_begin), the next one, this one's entries of A
    __device__ __forceinline__ SmallRows(const RowList &l, int part, const int64_t *pos, int64_t begin)
        : list(l), Apos(pos), row_begin(begin)
    {
        int64_t t_first;
        list_range(list, part, &t_first, &t_end);
        t = t_first + blockIdx.x;
        r = t < t_end ? list.rows[t] : 0;
        rn = t + gridDim.x < t_end ? list.rows[t + gridDim.x] : r;
        as = Apos[row_begin + r];
        ae = Apos[row_begin + r + 1];
    }
    __device__ __forceinline__ bool more() const { return t < t_end; }
};

// The row counters of a phase's kernels, one each.  0-3: a phase's own, which clears them; 4-7: the numeric phase's where the
// symbolic one of the same call has cleared them.
constexpr int SG_TICKETS = 8;
// What the symbolic phase's first kernel over a row list clears for the ones behind it: those counters, and the counts of the
// rows without products, which the list has at its end and no kernel takes.
__device__ __forceinline__ void sg_clear_rest(const RowList &list, int64_t nrows, unsigned long long *__restrict__ tickets,
                                              int64_t *__restrict__ rowcount)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < SG_TICKETS)
        tickets[i] = 0;
    for (int64_t t = list.bounds[1] + i; t < nrows; t += (int64_t)gridDim.x * blockDim.x)
        rowcount[list.rows[t]] = 0;
}

// tickets: null, or what it clears first (sg_clear_rest)
__global__ __launch_bounds__(SM_T) void spgemm_symbolic_small_kernel(
    int64_t row_begin, RowList list, int words, const int64_t *__restrict__ Apos, const int32_t *__restrict__ Acrd,
    const int64_t *__restrict__ Bpos, const int32_t *__restrict__ Bcrd, int64_t nrows, unsigned long long *__restrict__ tickets,
    int64_t *__restrict__ rowcount)
{
    if (tickets)
        sg_clear_rest(list, nrows, tickets, rowcount);
    uint32_t *bm = sg_dyn_lds;
    __shared__ SmallStage<SM_T> stage;
    __shared__ int wave_tot[SM_T / 64];
    for (int w = threadIdx.x; w < words; w += SM_T)
        bm[w] = 0;
    small_clear(stage);
    if ((threadIdx.x & 63) < 2)
        stage.own_marks[threadIdx.x >> 6][threadIdx.x & 63] = 0;
    lds_barrier();
    SmallRows rows(list, LIST_FEW, Apos, row_begin);
    while (rows.more()) {
        const int64_t r = rows.r, as = rows.as, ae = rows.ae;
        rows.t += gridDim.x;
        rows.r = rows.rn;
        rows.as = Apos[row_begin + rows.rn];
        rows.ae = Apos[row_begin + rows.rn + 1];
        rows.rn = rows.t + gridDim.x < rows.t_end ? list.rows[rows.t + gridDim.x] : rows.rn;
        const int held = __builtin_amdgcn_readfirstlane((int)(ae - as <= 64));          // by every wavefront
        SmallEntry e = small_entry<false>(as, as + (held ? threadIdx.x & 63 : threadIdx.x), ae, Acrd, nullptr, Bpos);
        const int products = __builtin_amdgcn_readlane(wave_inclusive_scan(e.len), 63);
        if (held && products <= SM_T) {
            // a product to a lane: the columns are those that found their bit clear
            SmallProducts<false, 1> it;
            small_few<false, SM_T>(stage, e, Bcrd, nullptr, it);
            const int j = it.col[0];
            const uint32_t bit = 1u << (j & 31);
            bool fresh = false;
            if (j >= 0)
                fresh = !(atomicOr(&bm[j >> 5], bit) & bit);
            const int n = (int)__popcll(__ballot(fresh));
            if ((threadIdx.x & 63) == 0)
                wave_tot[threadIdx.x >> 6] = n;
            lds_barrier();
            if (threadIdx.x == 0) {
                int all = 0;
                for (int w = 0; w < SM_T / 64; ++w)
                    all += wave_tot[w];
                rowcount[r] = all;
            }
            if (j >= 0)
                bm[j >> 5] = 0;
        } else {
            if (held && threadIdx.x >= 64)
                e.len = 0;
            for (int64_t p0 = as; p0 < ae; p0 += SM_T) {
                if (p0 > as)
                    e = small_entry<false>(as, p0 + threadIdx.x, ae, Acrd, nullptr, Bpos);
                SmallProducts<false, 1> it;
                small_products<false, SM_T, 1>(stage, small_stage<false, SM_T>(stage, e), Bcrd, nullptr, it);
                if (it.col[0] >= 0)
                    atomicOr(&bm[it.col[0] >> 5], 1u << (it.col[0] & 31));
                lds_barrier();
                small_clear(stage);
            }
            const int n = small_row_ranks<SM_T>(bm, nullptr, words, wave_tot);
            if (threadIdx.x == 0)
                rowcount[r] = n;
            const int per = (words + SM_T - 1) / SM_T;
            for (int w = threadIdx.x * per; w < (int)(threadIdx.x + 1) * per && w < words; ++w)          // its own words
                bm[w] = 0;
        }
        lds_barrier();
    }
}

// The structure of the other rows of such a matrix, of more than a product a lane there: eight wavefronts to a row, its rows of B streamed as staged slices, and
// as many workgroups as make 32 wavefronts a CU.  (Sixteen wavefronts, all that a
// CU then held, a row of B at a time took, us, A*A of 65536 vertices, edge factor 16 971, 30000 and 10 240, 16000 and 8 86,
// 5000 and 12 48, so 739, 168, 66, 38.)
constexpr int SMID_T = 512, SMID_WAVES = SMID_T / 64;
typedef SliceStage<SMID_T, SM_COLS, 23, SMID_WAVES> RowStage;
// The longest rows of B, a sixty-fourth of the columns and more, are taken as bitmaps, 16 bytes to a lane, which keeps its
// words of the row in registers: of A*A of 65536 vertices, edge factor 16, 137 of them hold 834 of 1236 M products.  us, this
// phase without them, with rows from a 32nd, a 64th and a 128th of the columns on: 65536 and 16 736, 565, 472, 514; 30000
// and 10 158, 150, 134, 157; 20000 and 12 152, 129, 131, 141; 16000 and 8 62, 60, 61, 76.
constexpr int SMID_HUB_PART = 64, SMID_HUBS = 4;          // so many at a time
static_assert(SM_COLS / 32 <= SMID_T * 4, "a lane has four words of a bitmap");
__global__ void spgemm_hub_rows(int64_t nrows, const int64_t *__restrict__ Bpos, int64_t least, int32_t *__restrict__ slot,
                                int32_t *__restrict__ hub, int32_t *__restrict__ hubs)
{
    const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= nrows)
        return;
    int s = -1;
    if (Bpos[k + 1] - Bpos[k] >= least) {
        s = atomicAdd(hubs, 1);
        hub[s] = (int32_t)k;
    }
    slot[k] = s;
}
__global__ __launch_bounds__(256) void spgemm_hub_bits(const int64_t *__restrict__ Bpos, const int32_t *__restrict__ Bcrd,
                                                       const int32_t *__restrict__ hub, const int32_t *__restrict__ hubs,
                                                       int words, uint32_t *__restrict__ bits)
{
    __shared__ uint32_t bm[SM_COLS / 32];
    const int n = *hubs;
    for (int s = blockIdx.x; s < n; s += gridDim.x) {
        for (int w = threadIdx.x; w < words; w += 256)
            bm[w] = 0;
        __syncthreads();
        const int64_t end = Bpos[hub[s] + 1];
        for (int64_t q = Bpos[hub[s]] + threadIdx.x; q < end; q += 256)
            atomicOr(&bm[Bcrd[q] >> 5], 1u << (Bcrd[q] & 31));
        __syncthreads();
        for (int w = threadIdx.x; w < words; w += 256)
            bits[(int64_t)s * words + w] = bm[w];
        __syncthreads();
    }
}

// HUBS: with such bitmaps (hub_slot, hub_bits; else null).  part: the list's rows that are taken; tickets: null, or what it
// clears first (sg_clear_rest)
template <bool HUBS>
__global__ __launch_bounds__(SMID_T, 8) void spgemm_symbolic_rows_kernel(
    int64_t row_begin, RowList list, int part, int words, const int64_t *__restrict__ Apos, const int32_t *__restrict__ Acrd,
    const int64_t *__restrict__ Bpos, const int32_t *__restrict__ Bcrd, int64_t Bnnz, const int32_t *__restrict__ hub_slot,
    const uint4 *__restrict__ hub_bits, int64_t nrows, unsigned long long *__restrict__ tickets, int64_t *__restrict__ rowcount)
{
    uint32_t *bm = sg_dyn_lds;
    if (tickets)
        sg_clear_rest(list, nrows, tickets, rowcount);
    __shared__ RowStage st;
    __shared__ int wave_cnt[SMID_WAVES], hub[HUBS ? SMID_T : 1], hubs[2];
    const bool mine = (int)threadIdx.x < words / 4;          // four words of a bitmap
    int pass = 0;
    if (threadIdx.x < 2)
        hubs[threadIdx.x] = 0;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    for (int w = threadIdx.x; w < words; w += SMID_T)
        bm[w] = 0;
    if (lane < 2)
        st.marks[wave][lane] = 0;
    lds_barrier();          // the first pass counts its hubs before its own
    int64_t t_first, t_end;
    list_range(list, part, &t_first, &t_end);
    // rows dealt out in advance, heaviest first; the bounds of 64 at a time, entries of A and their rows of B ahead
    for (int64_t t0 = t_first + blockIdx.x; t0 < t_end; t0 += 64 * (int64_t)gridDim.x) {
        const int64_t t = t0 + lane * (int64_t)gridDim.x;
        int64_t l_as = 0;
        int l_cnt = 0, l_row = 0;
        if (t < t_end) {
            l_row = list.rows[t];
            l_as = Apos[row_begin + l_row];
            l_cnt = (int)(Apos[row_begin + l_row + 1] - l_as);
        }
        const int64_t left = (t_end - 1 - t0) / gridDim.x + 1;
        const int nr = __builtin_amdgcn_readfirstlane((int)(left < 64 ? left : 64));
        const auto load_entry = [&](int r, int base) {
            const int cnt = __builtin_amdgcn_readlane(l_cnt, r & 63);
            return r < 64 && base + (int)threadIdx.x < cnt ? Acrd[readlane_i64(l_as, r & 63) + base + threadIdx.x] : -1;
        };
        const auto load_row = [&](int k, int64_t &lo, int64_t &hi, int &slot) {
            lo = hi = 0;
            slot = -1;
            if (k >= 0) {
                lo = Bpos[k];
                hi = Bpos[k + 1];
                if constexpr (HUBS)
                    slot = hub_slot[k];
            }
        };
        int k0 = load_entry(0, 0), k1 = load_entry(1, 0), slot0;
        int64_t lo0, hi0;
        load_row(k0, lo0, hi0, slot0);
        for (int r = 0; r < nr; ++r) {
            int64_t lo1, hi1;
            int slot1;
            load_row(k1, lo1, hi1, slot1);
            const int k2 = load_entry(r + 2, 0);
            const int cnt = __builtin_amdgcn_readlane(l_cnt, r);
            uint4 own = make_uint4(0, 0, 0, 0);
            for (int base = 0; base < cnt; base += SMID_T) {
                int64_t lo = lo0, hi = hi0;
                int slot = slot0;
                if (base > 0)
                    load_row(load_entry(r, base), lo, hi, slot);
                if (slot >= 0)
                    hi = lo;
                slice_put(st, lo, hi, 0.0, lane, wave);
                if constexpr (HUBS) {
                    const unsigned long long has = __ballot(slot >= 0);
                    if (has) {
                        int first = 0;
                        if (lane == 0)
                            first = atomicAdd(&hubs[pass], __popcll(has));
                        first = __builtin_amdgcn_readfirstlane(first);
                        if (slot >= 0)
                            hub[__builtin_amdgcn_mbcnt_hi((uint32_t)(has >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)has, first))] = slot;
                    }
                }
                lds_barrier();
                if constexpr (HUBS) {
                    const int nh = __builtin_amdgcn_readfirstlane(hubs[pass]);
                    pass ^= 1;
                    if (threadIdx.x == 0)
                        hubs[pass] = 0;
                    for (int h = 0; h < nh; h += SMID_HUBS) {
                        const int which = hub[h + (lane < SMID_HUBS && h + lane < nh ? lane : 0)];          // past the last one, h again
                        uint4 v[SMID_HUBS];
    #pragma unroll
                        for (int x = 0; x < SMID_HUBS; ++x)
                            v[x] = hub_bits[(int64_t)__builtin_amdgcn_readlane(which, x) * (words / 4) + (mine ? threadIdx.x : 0)];
    #pragma unroll
                        for (int x = 0; x < SMID_HUBS; ++x) {
                            own.x |= v[x].x;
                            own.y |= v[x].y;
                            own.z |= v[x].z;
                            own.w |= v[x].w;
                        }
                    }
                }
                slice_walk<false, false, int32_t>(st, Bcrd, nullptr, Bnnz, lane, wave, [&](const SliceTurn<int32_t> &u) {
                    const int j[4] = {u.j.x, u.j.y, u.j.z, u.j.w};
                    int w = 0;
                    uint32_t bits = 0u;
#pragma unroll
                    for (int x = 0; x < 4; ++x)
                        if (u.mask >> x & 1u) {
                            if (bits && (j[x] >> 5) != w) {
                                atomicOr(&bm[w], bits);
                                bits = 0u;
                            }
                            w = j[x] >> 5;
                            bits |= 1u << (j[x] & 31);
                        }
                    if (bits)
                        atomicOr(&bm[w], bits);
                });
                for (int64_t q = lo + RowStage::MOST; q < hi; ++q)          // a row of B with repeated columns
                    atomicOr(&bm[Bcrd[q] >> 5], 1u << (Bcrd[q] & 31));
                lds_barrier();
            }
            int n = 0;
            if (mine) {
                uint4 &at = reinterpret_cast<uint4 *>(bm)[threadIdx.x];
                const uint4 b = at;
                at = make_uint4(0, 0, 0, 0);
                n = __popc(b.x | own.x) + __popc(b.y | own.y) + __popc(b.z | own.z) + __popc(b.w | own.w);
            }
            n = wave_sum_i32(n);
            if (lane == 0)
                wave_cnt[wave] = n;
            lds_barrier();
            if (threadIdx.x == 0) {
                int all = 0;
                for (int w = 0; w < SMID_WAVES; ++w)
                    all += wave_cnt[w];
                rowcount[__builtin_amdgcn_readlane(l_row, r)] = all;
            }
            k0 = k1;
            lo0 = lo1;
            hi0 = hi1;
            slot0 = slot1;
            k1 = k2;
        }
    }
}

// PER: products of a lane; part: the list's rows that are taken (PER = 1: of at most T products)
template <bool SEMI, int T, int PER>
__global__ __launch_bounds__(T) void spgemm_numeric_small_kernel(
    int64_t row_begin, RowList list, int part, int words, const int64_t *__restrict__ Apos, const int32_t *__restrict__ Acrd,
    const double *__restrict__ Aval, const int64_t *__restrict__ Bpos, const int32_t *__restrict__ Bcrd,
    const double *__restrict__ Bval, const int64_t *__restrict__ Cpos, int32_t *__restrict__ Ccrd,
    double *__restrict__ Cval, int reduce_op, int mult_op)
{
    uint32_t *bm = sg_dyn_lds;
    uint16_t *before = reinterpret_cast<uint16_t *>(bm + words);
    SmallRowLds<T, PER> &sh = *reinterpret_cast<SmallRowLds<T, PER> *>(bm + words + words / 2);
    for (int w = threadIdx.x; w < words + words / 2 + (int)(sizeof sh / 4); w += T)
        bm[w] = 0;
    lds_barrier();
    const int64_t c0 = Cpos[row_begin];
    SmallRows rows(list, part, Apos, row_begin);
    while (rows.more()) {
        const int64_t as = rows.as, ae = rows.ae, coff = Cpos[row_begin + rows.r] - c0;
        rows.t += gridDim.x;
        rows.r = rows.rn;
        rows.as = Apos[row_begin + rows.rn];
        rows.ae = Apos[row_begin + rows.rn + 1];
        rows.rn = rows.t + gridDim.x < rows.t_end ? list.rows[rows.t + gridDim.x] : rows.rn;
        SmallProducts<true, PER> it;
        const int held = PER == 1 ? __builtin_amdgcn_readfirstlane((int)(ae - as <= 64)) : 0;          // by every wavefront
        const auto products = [&](int64_t p0) {
            if (held) {
                const SmallEntry e = small_entry<true>(as, as + (threadIdx.x & 63), ae, Acrd, Aval, Bpos);
                small_few<true, T>(sh.stage, e, Bcrd, Bval, it);
            } else {
                const int n = small_stage<true, T>(sh.stage, small_entry<true>(as, p0 + threadIdx.x, ae, Acrd, Aval, Bpos));
                small_products<true, T, PER>(sh.stage, n, Bcrd, Bval, it);
            }
        };
        for (int64_t p0 = as; p0 < ae; p0 += T) {
            products(p0);
#pragma unroll
            for (int x = 0; x < PER; ++x)
                if (it.col[x] >= 0)
                    atomicOr(&bm[it.col[x] >> 5], 1u << (it.col[x] & 31));
            lds_barrier();
            small_clear(sh.stage);
        }
        const int total = small_row_ranks<T>(bm, before, words, sh.wave_tot);
        lds_barrier();
        for (int64_t p0 = as; p0 < ae; p0 += T) {
            if (ae - as > T) {          // more entries than lanes: their products once more
                products(p0);
                lds_barrier();
                small_clear(sh.stage);
            }
#pragma unroll
            for (int x = 0; x < PER; ++x)
                if (it.col[x] >= 0) {
                    const int j = it.col[x], r = before[j >> 5] + __popc(bm[j >> 5] & ((1u << (j & 31)) - 1u));
                    sh.col[r] = (uint16_t)j;
                    if constexpr (SEMI)
                        semiring_lds_add(&sh.val[r], reduce_op, mult_op, it.a[x], it.b[x], it.place[x], it.q[x]);
                    else
                        __hip_atomic_fetch_add(&sh.val[r], it.a[x] * it.b[x], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                }
        }
        lds_barrier();
        for (int q = threadIdx.x; q < total; q += T) {
            const int j = sh.col[q];
            Ccrd[coff + q] = j;
            Cval[coff + q] = dense_take<SEMI>(sh.val, q, reduce_op, mult_op, as, Aval, Bval);
            bm[j >> 5] = 0;
        }
        lds_barrier();
    }
}

struct SgScratch {
    Workspace ticket;     // SG_TICKETS 64-bit row counters
    Workspace rowcount;   // int64[nrows] / double[nrows]
    Workspace gbm;        // global bitmaps (only when the bitmap does not fit LDS)
    Workspace gmask;      // global mask bitmaps (masked numeric)
    Workspace slabs;      // dense accumulators, zero between calls
    Workspace dense_rows;     // DenseRow[] and before[] of spgemm_numeric_dense_blocks_kernel
    Workspace dense_before;
};
static SgScratch g_sg;

struct SgGeom {
    int logW;
    bool lds;
    int groups;
    size_t lds_bytes;
    size_t bm_words;      // words per workgroup bitmap
};

static int sg_geometry(int64_t ncols, SgGeom *g)
{
    const int64_t words = ceil_div(ncols > 0 ? ncols : 1, 32);
    int logW = 0;
    while (((int64_t)SG_T << logW) < words)
        ++logW;
    if (logW > 20)
        return set_error(COMET_HIP_ERR_SIZE, "too many columns (%lld)", (long long)ncols);
    g->logW = logW;
    g->lds = (1 << logW) <= SG_LDS_MAX_W;
    g->bm_words = (size_t)SG_T * ((size_t)(1 << logW) + 1);
    g->lds_bytes = g->lds ? g->bm_words * sizeof(uint32_t) : 0;
    g->groups = num_cus() > 0 ? num_cus() : 256;
    if (g->lds && g->lds_bytes <= 48 * 1024)
        g->groups *= 2;          // two workgroups of 16 wavefronts fit a CU when the bitmap is small
    return COMET_HIP_OK;
}

template <typename K>
static int sg_allow_lds(K kernel, size_t bytes)
{
    if (bytes > 0)
        COMET_HIPCHK(hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes));
    return COMET_HIP_OK;
}

__global__ __launch_bounds__(256) void sg_clear(unsigned long long *__restrict__ tickets, int64_t *__restrict__ rowcount, int64_t n)
{
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < SG_TICKETS)
        tickets[i] = 0;
    if (i < n)
        rowcount[i] = 0;
}
static unsigned long long *sg_ticket(int k) { return (unsigned long long *)g_sg.ticket.ptr + k; }
static int sg_reset_ticket()
{
    COMET_CHK(g_sg.ticket.ensure(SG_TICKETS * sizeof(unsigned long long), false));
    COMET_HIPCHK(hipMemsetAsync(g_sg.ticket.ptr, 0, SG_TICKETS * sizeof(unsigned long long), stream()));
    return COMET_HIP_OK;
}

static int check_product_shapes(const Csr *a, const Csr *b, const Csr *m, const char *who)
{
    if (a->ncols != b->nrows)
        return set_error(COMET_HIP_ERR_ARG, "%s: A is %lld x %lld but B is %lld x %lld", who, (long long)a->nrows,
                         (long long)a->ncols, (long long)b->nrows, (long long)b->ncols);
    if (m && (m->nrows != a->nrows || m->ncols != b->ncols))
        return set_error(COMET_HIP_ERR_ARG, "%s: mask is %lld x %lld, product is %lld x %lld", who,
                         (long long)m->nrows, (long long)m->ncols, (long long)a->nrows, (long long)b->ncols);
    return COMET_HIP_OK;
}

// keys that order rows by descending products; rows without products sort to the very end
// With a mask (Mpos, already offset to the first row of the list), the rows whose mask row holds more than `fill`
// entries sort in front of all others (keys below 2^61), whatever their number of products.
__global__ void sg_row_keys(int64_t n, const int64_t *__restrict__ rowprod, const int64_t *__restrict__ Mpos,
                            int64_t fill, uint64_t *__restrict__ keys, uint32_t *__restrict__ idx)
{
    const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (r < n) {
        const int64_t p = rowprod[r];
        uint64_t key = p > 0 ? (uint64_t)((1ll << 62) - p) : ~0ull >> 1;
        if (Mpos && p > 0 && Mpos[r + 1] - Mpos[r] > fill)
            key = (uint64_t)((1ll << 61) - (p < (1ll << 61) ? p : (1ll << 61) - 1));
        keys[r] = key;
        idx[r] = (uint32_t)r;
    }
}

// bounds[0] = rows with >= threshold products, bounds[1] = rows with any, bounds[2] = rows with >= wide products,
// in the sorted key array
__global__ void sg_row_bounds(int64_t n, const uint64_t *__restrict__ keys, int64_t threshold, int64_t wide, int64_t middle,
                              int64_t few, int64_t *__restrict__ bounds)
{
    if (threadIdx.x > 4 || blockIdx.x > 0)
        return;
    // first key that is larger than the limit: keys ascend as products descend
    const uint64_t limit = threadIdx.x == 1 ? (uint64_t)((1ll << 62) - 1)
                                            : (uint64_t)((1ll << 62) - (threadIdx.x == 0   ? threshold
                                                                        : threadIdx.x == 2 ? wide
                                                                        : threadIdx.x == 3 ? middle
                                                                                           : few));
    int64_t lo = 0, hi = n;
    while (lo < hi) {
        const int64_t mid = (lo + hi) >> 1;
        if (keys[mid] <= limit)
            lo = mid + 1;
        else
            hi = mid;
    }
    bounds[threadIdx.x] = lo;
}

struct SgRowLists {
    Workspace rowprod, keys_in, keys_out, idx_in, idx_out, bounds;
};
static SgRowLists g_rl;

// Products per row of rows [rb, re) of A*B and the list of those rows by descending products.
// The list depends on the two structures, the range and the thresholds only: it is kept in A's handle and found
// again by the uids of the matrices it was made from (a matrix gets a new uid when it is invalidated), so a
// product that is taken again, or taken in row blocks, sorts nothing.  COMET_HIP_SPGEMM_NO_LIST_CACHE turns the
// keeping off (the tests compare both).
constexpr size_t SG_ROW_LISTS_KEPT = 24;
static int sg_row_list(const Csr *a, const Csr *b, int64_t rb, int64_t re, int64_t dense_threshold,
                       int64_t wide_threshold, RowList *out, const Csr *long_mask = nullptr,
                       int64_t mask_fill = 0, bool want_counts = false, int64_t mid_threshold = -1, int64_t few_threshold = -1)
{
    for (int64_t &c : out->counts)
        c = -1;
    if (mid_threshold < 0)
        mid_threshold = dense_threshold;
    if (few_threshold < 0)
        few_threshold = mid_threshold;
    const int64_t n = re - rb;
    const bool keep = getenv("COMET_HIP_SPGEMM_NO_LIST_CACHE") == nullptr;
    Csr *owner = const_cast<Csr *>(a);
    RowListEntry key;
    key.b_uid = b->uid;
    key.mask_uid = long_mask ? long_mask->uid : 0;
    key.rb = rb;
    key.re = re;
    key.dense_threshold = dense_threshold;
    key.wide_threshold = wide_threshold;
    key.mid_threshold = mid_threshold;
    key.few_threshold = few_threshold;
    key.mask_fill = mask_fill;
    if (keep)
        for (const RowListEntry &e : owner->row_lists)
            if (e.b_uid == key.b_uid && e.mask_uid == key.mask_uid && e.rb == rb && e.re == re &&
                e.dense_threshold == dense_threshold && e.wide_threshold == wide_threshold &&
                e.mid_threshold == mid_threshold && e.few_threshold == few_threshold && e.mask_fill == mask_fill) {
                out->rows = e.rows;
                out->bounds = e.bounds;
                std::copy(e.counts, e.counts + 5, out->counts);
                return COMET_HIP_OK;
            }
    COMET_CHK(g_rl.rowprod.ensure(sizeof(int64_t) * (size_t)n, false));
    COMET_CHK(g_rl.keys_in.ensure(8 * (size_t)n, false));
    COMET_CHK(g_rl.keys_out.ensure(8 * (size_t)n, false));
    COMET_CHK(g_rl.idx_in.ensure(4 * (size_t)n, false));
    COMET_CHK(g_rl.idx_out.ensure(4 * (size_t)n, false));
    COMET_CHK(g_rl.bounds.ensure(40, false));
    int64_t *rowprod = (int64_t *)g_rl.rowprod.ptr;
    {
        KernelTimer t("spgemm_row_products");
        spgemm_row_products<<<dim3((unsigned)ceil_div(n, 4)), dim3(256), 0, stream()>>>(
            rb, re, a->pos, a->crd, b->pos, rowprod);
        sg_row_keys<<<dim3((unsigned)ceil_div(n, 256)), dim3(256), 0, stream()>>>(
            n, rowprod, long_mask ? long_mask->pos + rb : nullptr, mask_fill, (uint64_t *)g_rl.keys_in.ptr,
            (uint32_t *)g_rl.idx_in.ptr);
    }
    COMET_HIPCHK(hipGetLastError());
    COMET_CHK(sort_pairs_u64_u32((const uint64_t *)g_rl.keys_in.ptr, (uint64_t *)g_rl.keys_out.ptr,
                                 (const uint32_t *)g_rl.idx_in.ptr, (uint32_t *)g_rl.idx_out.ptr, n, 63));
    sg_row_bounds<<<dim3(1), dim3(64), 0, stream()>>>(n, (const uint64_t *)g_rl.keys_out.ptr, dense_threshold,
                                                      wide_threshold, mid_threshold, few_threshold, (int64_t *)g_rl.bounds.ptr);
    COMET_HIPCHK(hipGetLastError());
    out->rows = (const int32_t *)g_rl.idx_out.ptr;
    out->bounds = (const int64_t *)g_rl.bounds.ptr;
    if (keep && n > 0) {
        // a copy of its own; failing to get the memory only means that the list is built again next time
        if (owner->row_lists.size() >= SG_ROW_LISTS_KEPT) {
            COMET_CHK(stream_wait());        // a kernel may still be reading the oldest one
            (void)dev_free(owner->row_lists.front().rows);
            (void)dev_free(owner->row_lists.front().bounds);
            owner->row_lists.erase(owner->row_lists.begin());
        }
        if (dev_malloc((void **)&key.rows, 4 * (size_t)n) != hipSuccess ||
            dev_malloc((void **)&key.bounds, 40) != hipSuccess) {
            (void)hipGetLastError();
            (void)dev_free(key.rows);
            return COMET_HIP_OK;
        }
        COMET_HIPCHK(hipMemcpyAsync(key.rows, g_rl.idx_out.ptr, 4 * (size_t)n, hipMemcpyDeviceToDevice, stream()));
        COMET_HIPCHK(hipMemcpyAsync(key.bounds, g_rl.bounds.ptr, 40, hipMemcpyDeviceToDevice, stream()));
        if (want_counts) {          // once per list instead of once per product
            int64_t *word = nullptr;
            COMET_CHK(mailbox((void **)&word));
            COMET_HIPCHK(hipMemcpyAsync(word, key.bounds, 40, hipMemcpyDeviceToHost, stream()));
            COMET_CHK(stream_wait());
            std::copy(word, word + 5, key.counts);
            std::copy(word, word + 5, out->counts);
        }
        owner->row_lists.push_back(key);
        out->rows = key.rows;
        out->bounds = key.bounds;
    }
    return COMET_HIP_OK;
}

constexpr int64_t SG_NO_DENSE = 1ll << 61;     // a threshold no row reaches: every row stays on the slab path

static int dot_form_fits(const Csr *a, const Csr *b, const Csr *m, bool *fits);
static int pair_dot_values(Csr *a, Csr *b, Csr *m, int64_t rb, int64_t re, double **pair_val, uint8_t **pair_hit,
                           int64_t *pairs, int reduce_op, int mult_op);

constexpr int SG_DENSE_MAX_BLOCKS = 64;        // the dense path serves matrices of up to 2^20 columns
// Rows with at least this many products per column block of the matrix keep their values in LDS (the span or
// the block kernel); the others add into a slab in HBM through L2 atomics.  Measured as above, ms per product
// with the span kernel in place: 128 per block 555, 64: 533, 32: 519, 16: 514, 8: 513.5, 4: 513, 1: 515.
constexpr int64_t SG_DENSE_PER_BLOCK = 8;

// Heavy rows with at least this many products per column block of the matrix stay with the block kernel, the
// others go to the span kernel (measured on A*A of an R-MAT graph of scale 20, 64 blocks, ms per product:
// 512 per block 583, 1024 572, 2048 559, 4096 557, 8192 570, every heavy row to the span kernel 604, none 613;
// with the kernels as they are now 1024 per block 437, 2048 402, 4096 386, 6144 381, 8192 382, 12288 382, 16384 389).
// COMET_HIP_SPGEMM_WIDE, a number of products per row, overrides the rule: either kernel is right for any row,
// so the tests use it to send the same rows through both.
// With one or two blocks the line lies higher, us by products per block, 6144 / 10240: 10000 vertices, edge factor 16 572 /
// 536, 16000 and 16 849 / 809, 30000 and 10 1379 / 1239 (three blocks: 45000 and 12 2990 / 3064).  A matrix that fills no
// more than half a block sends all its heavy rows there, a launch less: 1024 and 8 117 / 97, 4096 and 8 178 / 153, 8000 and
// 4 162 / 139, 8192 and 16 346 / 331.
constexpr int64_t SG_WIDE_PER_BLOCK = 6144, SG_WIDE_PER_BLOCK_FEW = 10240;
constexpr int64_t SG_NARROW = SG_CB / 2;
static int64_t sg_wide_threshold(int64_t ncols, int nblk)
{
    const char *e = getenv("COMET_HIP_SPGEMM_WIDE");
    return e && *e ? atoll(e) : ncols <= SG_NARROW ? 0 : (nblk <= 2 ? SG_WIDE_PER_BLOCK_FEW : SG_WIDE_PER_BLOCK) * nblk;
}

// From how many products on a row's values are kept in LDS by the large workgroups, and from how many on block by block.
// small: the matrix has few enough columns for the kernels of rows with few products; mid and more products are too many
// for a workgroup of 256 lanes.  Rows of mid up to dense products go to one of 512 lanes: 7000 of the rows of a product of
// 65536 rows (R-MAT, 16 edges a row), 74 us there and 127 less in the kernel that visits the blocks, 12 and 40 of 980 us
// in all with 30000 rows.  A matrix of half a block has no such rows: the kernel of whole blocks visits it once.
struct SgClasses { int64_t few, mid, dense, wide; };
static SgClasses sg_row_classes(int64_t ncols, bool small)
{
    const int nblk = (int)ceil_div(ncols > 0 ? ncols : 1, SG_CB);
    SgClasses c;
    c.dense = !small ? SG_DENSE_PER_BLOCK * nblk : ncols <= SG_NARROW ? SM_PRODUCTS + 1 : SM_MID_PRODUCTS + 1;
    c.mid = small ? SM_PRODUCTS + 1 : c.dense;
    c.few = small ? SM_FEW_PRODUCTS + 1 : c.mid;
    c.wide = std::max(sg_wide_threshold(ncols, nblk), c.dense);
    return c;
}
static int sm_words(int64_t ncols) { return (int)ceil_div(ceil_div(ncols > 0 ? ncols : 1, 32), 4) * 4; }
static dim3 sm_grid(int64_t rows, int per_cu)          // rows < 0: how many is not known
{
    const int64_t most = (int64_t)num_cus() * per_cu;          // workgroups that fit the CUs
    return dim3((unsigned)(rows < 0 ? most : std::min(most, rows)));
}

// The bitmaps of b's long rows, words to each; a matrix of few columns or none such rows goes without, and so does one for
// which there is no memory.  (The host waits once for how many there are: a bound on them from the entries alone is 8 bytes
// of bitmaps for every one, also where no row is long.)
static int sg_plan_hubs(Csr *b, int words)
{
    const int64_t least = ceil_div(b->ncols, SMID_HUB_PART);
    if (b->sg_hub_state != 0 || b->ncols <= SG_NARROW || b->nrows >= 1ll << 31 || b->nnz < least)
        return COMET_HIP_OK;
    b->sg_hub_state = 1;
    const int64_t most = std::min(b->nnz / least, b->nrows);
    int32_t *slot = nullptr, *n = nullptr;
    uint32_t *bits = nullptr;
    COMET_CHK(mailbox((void **)&n));
    KernelTimer t("spgemm_hub_bits");
    const auto run = [&]() -> int {
        COMET_HIPCHK(dev_malloc((void **)&slot, sizeof(int32_t) * (size_t)(b->nrows + most + 1)));
        int32_t *hub = slot + b->nrows, *hubs = hub + most;
        COMET_HIPCHK(hipMemsetAsync(hubs, 0, sizeof(int32_t), stream()));
        spgemm_hub_rows<<<dim3((unsigned)ceil_div(b->nrows, 256)), dim3(256), 0, stream()>>>(b->nrows, b->pos, least, slot, hub,
                                                                                           hubs);
        COMET_HIPCHK(hipMemcpyAsync(n, hubs, sizeof(int32_t), hipMemcpyDeviceToHost, stream()));
        COMET_CHK(stream_wait());
        const int64_t found = *(volatile int32_t *)n;
        if (found == 0)
            return COMET_HIP_OK;
        COMET_HIPCHK(dev_malloc((void **)&bits, sizeof(uint32_t) * (size_t)words * (size_t)found));
        spgemm_hub_bits<<<dim3((unsigned)std::min<int64_t>(found, 2 * (int64_t)num_cus())), dim3(256), 0, stream()>>>(
            b->pos, b->crd, hub, hubs, words, bits);
        COMET_HIPCHK(hipGetLastError());
        b->sg_hub_slot = slot;
        b->sg_hub_bits = bits;
        b->sg_hub_state = 2;
        return COMET_HIP_OK;
    };
    const int rc = run();
    if (b->sg_hub_state != 2) {
        (void)dev_free(slot);
        (void)dev_free(bits);
    }
    return rc;
}

// Rows of at most SM_FEW_PRODUCTS products go to a kernel of 256 lanes a row, the others to one of 512 that streams slices of
// B; so few of the former join the latter instead, since a launch (4 us) costs more.  us, A*A, R-MAT graphs, apart / together:
// 1024 vertices, edge factor 8 65 / 62, 4000 and 10 126 / 122, 8000 and 5 123 / 120, 65000 and 4 832 / 837 with 16384 rows;
// 20000 rows of 8 entries and 8 hubs 179 / 191, 60000 of 4 326 / 392.  (Rows of up to 2048 products to the first: 60000 rows
// of 20 entries 504 in place of 454, a band of 27 697 in place of 548; the counters and counts cleared by a launch of their
// own: 2.2 more for every product.)
constexpr int64_t SG_FEW_TOGETHER = 4096;
static int symbolic_counts(const Csr *a, const Csr *b, const Csr *m, int64_t *rowcount)
{
    bool dots = false;
    COMET_CHK(dot_form_fits(a, b, m, &dots));
    if (dots) {         // a masked product: which stored pairs of the mask meet a product
        double *pair_val = nullptr;
        uint8_t *pair_hit = nullptr;
        int64_t pairs = 0;
        COMET_CHK(pair_dot_values(const_cast<Csr *>(a), const_cast<Csr *>(b), const_cast<Csr *>(m), 0, a->nrows, &pair_val,
                                  &pair_hit, &pairs, COMET_SR_PLUS, COMET_OP_TIMES));
        KernelTimer t("spgemm_symbolic_dot_count");
        spgemm_dot_count<<<dim3((unsigned)ceil_div(a->nrows, 4)), dim3(256), 0, stream()>>>(0, a->nrows, m->pos, pair_hit,
                                                                                            rowcount);
        COMET_HIPCHK(hipGetLastError());
        return COMET_HIP_OK;
    }
    SgGeom g;
    COMET_CHK(sg_geometry(b->ncols, &g));
    RowList list;
    const bool small = !m && b->ncols <= SM_COLS;
    const SgClasses classes = sg_row_classes(b->ncols, small);
    if (small)          // the list the numeric phase takes
        COMET_CHK(sg_row_list(a, b, 0, a->nrows, classes.dense, classes.wide, &list, nullptr, 0, true, classes.mid, classes.few));
    else
        COMET_CHK(sg_row_list(a, b, 0, a->nrows, SG_NO_DENSE, SG_NO_DENSE, &list));
    COMET_CHK(g_sg.ticket.ensure(SG_TICKETS * sizeof(unsigned long long), false));
    const bool known = list.counts[0] >= 0;
    const bool rows_fit = small && b->nnz >= 4 && b->nnz < SLICE_NNZ_MOST && a->nnz < (1ll << 30);
    const int64_t few = known ? list.counts[1] - list.counts[4] : -1;
    const bool together = rows_fit && known && list.counts[4] > 0 && few <= SG_FEW_TOGETHER;
    const bool small_rows = small && !together && few != 0, other_rows = rows_fit && list.counts[4] != 0;
    // the first of these launches clears for itself and the others
    unsigned long long *clears = small_rows || other_rows ? sg_ticket(0) : nullptr;
    if (!clears) {
        const int64_t words = std::max<int64_t>(a->nrows, SG_TICKETS);
        sg_clear<<<dim3((unsigned)ceil_div(words, 256)), dim3(256), 0, stream()>>>(sg_ticket(0), rowcount, a->nrows);
    }
    if (small_rows) {
        const int words = sm_words(b->ncols);
        KernelTimer t("spgemm_symbolic_small");
        const dim3 grid = sm_grid(few, 7);
        spgemm_symbolic_small_kernel<<<grid, dim3(SM_T), sizeof(uint32_t) * (size_t)words, stream()>>>(
            0, list, words, a->pos, a->crd, b->pos, b->crd, a->nrows, clears, rowcount);
        clears = nullptr;
    }
    if (rows_fit) {
        if (other_rows) {
            const int words = sm_words(b->ncols);
            Csr *right = const_cast<Csr *>(b);           // what is kept in a handle is not part of the matrix
            (void)plan_made([&] { return sg_plan_hubs(right, words); });
            KernelTimer t("spgemm_symbolic");
            const auto kernel = b->sg_hub_bits ? spgemm_symbolic_rows_kernel<true> : spgemm_symbolic_rows_kernel<false>;
            kernel<<<sm_grid(list.counts[together ? 1 : 4], 4), dim3(SMID_T), sizeof(uint32_t) * (size_t)words, stream()>>>(
                0, list, together ? LIST_ALL : LIST_NOT_FEW, words, a->pos, a->crd, b->pos, b->crd, b->nnz, b->sg_hub_slot,
                (const uint4 *)b->sg_hub_bits, a->nrows, clears, rowcount);
        }
        COMET_HIPCHK(hipGetLastError());
        return COMET_HIP_OK;
    }
    if (small && list.counts[4] == 0) {
        COMET_HIPCHK(hipGetLastError());
        return COMET_HIP_OK;
    }
    uint32_t *gbm = nullptr;
    if (!g.lds) {
        COMET_CHK(g_sg.gbm.ensure(sizeof(uint32_t) * g.bm_words * (size_t)g.groups, true));
        gbm = (uint32_t *)g_sg.gbm.ptr;
    }
    const dim3 grid((unsigned)g.groups), block(SG_T);
#define LAUNCH_SYM(L, M)                                                                                   \
    do {                                                                                                   \
        COMET_CHK(sg_allow_lds(spgemm_symbolic_kernel<L, M>, g.lds_bytes));                                \
        KernelTimer t(M ? "spgemm_symbolic_masked" : "spgemm_symbolic");                                   \
        spgemm_symbolic_kernel<L, M><<<grid, block, g.lds_bytes, stream()>>>(                              \
            a->nrows, a->pos, a->crd, b->pos, b->crd, m ? m->pos : nullptr, m ? m->crd : nullptr, g.logW,  \
            gbm, (unsigned long long *)g_sg.ticket.ptr, list, small ? LIST_NOT_FEW : LIST_ALL, rowcount);              \
    } while (0)
    if (g.lds) {
        if (m) LAUNCH_SYM(true, true); else LAUNCH_SYM(true, false);
    } else {
        if (m) LAUNCH_SYM(false, true); else LAUNCH_SYM(false, false);
    }
#undef LAUNCH_SYM
    COMET_HIPCHK(hipGetLastError());
    return COMET_HIP_OK;
}

// Per-row block pointers of the right-hand operand, built once per matrix.
static int sg_plan_blocks(Csr *b)
{
    const int nblk = (int)ceil_div(b->ncols > 0 ? b->ncols : 1, SG_CB);
    if (b->sg_blkptr && b->sg_nblk == nblk)
        return COMET_HIP_OK;
    if (b->sg_blkptr) {
        COMET_CHK(stream_wait());
        COMET_HIPCHK(dev_free(b->sg_blkptr));
        (void)dev_free(b->sg_crd16);
        b->sg_blkptr = nullptr;
        b->sg_crd16 = nullptr;
    }
    static_assert(SG_CB <= 65536, "a column inside its block fits 16 bits");
    if (dev_malloc((void **)&b->sg_crd16, sizeof(uint16_t) * (size_t)(b->nnz > 0 ? b->nnz : 1)) != hipSuccess) {
        (void)hipGetLastError();        // an allocation that may fail: its error must not reach the next check
        b->sg_crd16 = nullptr;          // the kernel then reads the 32-bit columns
    } else if (b->nnz > 0) {
        spgemm_block_columns<<<dim3((unsigned)ceil_div(b->nnz, 256)), dim3(256), 0, stream()>>>(b->nnz, b->crd,
                                                                                                 b->sg_crd16);
        COMET_HIPCHK(hipGetLastError());
    }
    COMET_HIPCHK(dev_malloc((void **)&b->sg_blkptr,
                           sizeof(int64_t) * (size_t)(nblk + 1) * (size_t)(b->nrows > 0 ? b->nrows : 1)));
    b->sg_nblk = nblk;
    if (b->nrows > 0) {
        KernelTimer t("spgemm_block_pointers");
        spgemm_block_pointers<<<dim3((unsigned)ceil_div(b->nrows, 256)), dim3(256), 0, stream()>>>(
            b->nrows, b->pos, b->crd, nblk, b->sg_blkptr);
    }
    COMET_HIPCHK(hipGetLastError());
    return COMET_HIP_OK;
}

// ---- masked products as dot products over the mask: the host side ----
static Workspace g_dot_val, g_dot_hit, g_dot_flag;

static int dot_transposed(const Csr *x, Csr **out)
{
    Csr *m = const_cast<Csr *>(x);           // what is kept in a handle is not part of the matrix
    if (!m->transposed) {
        m->transposed = csr_transposed_copy(m);
        if (!m->transposed)
            return COMET_HIP_ERR_HIP;
    }
    *out = m->transposed;
    return COMET_HIP_OK;
}

// the transpose of the structure of x whose values say where each entry lies in x
static int dot_transposed_index(const Csr *x, Csr **out)
{
    Csr *m = const_cast<Csr *>(x);
    if (!m->transposed_index) {
        double *iota = nullptr;
        COMET_HIPCHK(dev_malloc((void **)&iota, sizeof(double) * (size_t)(m->nnz > 0 ? m->nnz : 1)));
        if (m->nnz > 0)
            fill_iota_f64<<<dim3((unsigned)ceil_div(m->nnz, 256)), dim3(256), 0, stream()>>>(m->nnz, iota);
        Csr view;
        view.nrows = m->nrows;
        view.ncols = m->ncols;
        view.nnz = m->nnz;
        view.pos = m->pos;
        view.crd = m->crd;
        view.val = iota;
        m->transposed_index = csr_transposed_copy(&view);
        const hipError_t e = hipStreamSynchronize(stream());
        (void)dev_free(iota);
        if (!m->transposed_index || e != hipSuccess)
            return set_error(COMET_HIP_ERR_HIP, "transposing the mask failed");
    }
    *out = m->transposed_index;
    return COMET_HIP_OK;
}

// rows are even where none is longer than this and this many times the mean
constexpr int64_t CSR_EVEN_ROW = 24, CSR_EVEN_FACTOR = 8;

// fills in what is not known yet of the two states; both together take one look and one wait
static int csr_look(const Csr *x, bool structure, bool values)
{
    Csr *m = const_cast<Csr *>(x);
    structure = structure && m->dup_state == 0;
    values = values && m->iso_state == 0;
    if (!structure && !values)
        return COMET_HIP_OK;
    CsrTraits *seen = nullptr;
    COMET_CHK(mailbox((void **)&seen));
    *seen = CsrTraits{0, 0, 0, 0, 1, 0, 0.0};
    if (m->nnz > 0) {
        COMET_CHK(g_dot_flag.ensure(sizeof *seen, false));
        COMET_HIPCHK(hipMemsetAsync(g_dot_flag.ptr, 0, sizeof *seen, stream()));
        const int64_t blocks = ceil_div(std::max(m->nnz, m->nrows), 256);
        csr_traits<<<dim3((unsigned)std::min<int64_t>(blocks, 1 << 16)), dim3(256), 0, stream()>>>(
            m->nrows, m->nnz, m->pos, structure ? m->crd : nullptr, values ? m->val : nullptr,
            CSR_EVEN_ROW + CSR_EVEN_FACTOR * (m->nnz / m->nrows), (CsrTraits *)g_dot_flag.ptr);
        COMET_HIPCHK(hipGetLastError());
        COMET_HIPCHK(hipMemcpyAsync(seen, g_dot_flag.ptr, sizeof *seen, hipMemcpyDeviceToHost, stream()));
        COMET_CHK(stream_wait());
    }
    const volatile CsrTraits *t = seen;
    if (structure) {
        m->sides = (t->above ? 1 : 0) | (t->below ? 2 : 0);
        m->uneven = t->uneven != 0;
        m->dup_state = t->twice ? 2 : 1;
    }
    if (values) {
        m->iso_value = t->first;
        m->iso_state = t->differ ? 2 : 1;
    }
    return COMET_HIP_OK;
}

// whether no row of x holds a column twice
static int dot_no_duplicates(const Csr *x, bool *ok)
{
    COMET_CHK(csr_look(x, true, false));
    *ok = x->dup_state == 1;
    return COMET_HIP_OK;
}

static int csr_is_iso(const Csr *x, bool *iso)
{
    COMET_CHK(csr_look(x, false, true));
    *iso = x->iso_state == 1;
    return COMET_HIP_OK;
}

#include "masked_pairs.h"
#include "masked_dots.h"
#include "triangles.h"

// A masked product runs as dot products when the table over k fits LDS and no list that goes into a table holds a
// column twice.  COMET_HIP_SPGEMM_NO_DOT keeps the walk over the products of every row (the tests run both).
static int dot_form_fits(const Csr *a, const Csr *b, const Csr *m, bool *fits)
{
    *fits = false;
    if (!m || a->ncols > (1ll << 20) || a->nrows >= (1ll << 31) || b->ncols >= (1ll << 31) || m->nnz > PAIR_NNZ_MAX || a->nnz > PAIR_NNZ_MAX ||
        b->nnz > PAIR_NNZ_MAX ||
        getenv("COMET_HIP_SPGEMM_NO_DOT") != nullptr)
        return COMET_HIP_OK;
    bool ok_a = false, ok_b = false, ok_m = false;
    COMET_CHK(dot_no_duplicates(a, &ok_a));
    COMET_CHK(dot_no_duplicates(b, &ok_b));
    COMET_CHK(dot_no_duplicates(m, &ok_m));
    *fits = ok_a && ok_b && ok_m;
    return COMET_HIP_OK;
}

static int numeric_rows(const Csr *a, Csr *b, const Csr *m, const int64_t *Cpos, int64_t rb, int64_t re,
                        int32_t *Ccrd, double *Cval, int reduce_op, int mult_op, bool tickets_clear = false)
{
    if (reduce_op < 0 || reduce_op > COMET_SR_ANY || mult_op < 0 || mult_op > COMET_OP_DIV)
        return set_error(COMET_HIP_ERR_ARG, "unknown semiring (reduce %d, mult %d)", reduce_op, mult_op);
    const bool semi = reduce_op != COMET_SR_PLUS || mult_op != COMET_OP_TIMES;
    if (m && reduce_op != COMET_SR_ANY && re > rb) {
        bool dots = false;
        COMET_CHK(dot_form_fits(a, b, m, &dots));
        if (dots) {
            double *pair_val = nullptr;
            uint8_t *pair_hit = nullptr;
            int64_t pairs = 0, *before = nullptr, chunks = 0;
            COMET_CHK(pair_dot_values(const_cast<Csr *>(a), b, const_cast<Csr *>(m), rb, re, &pair_val, &pair_hit, &pairs,
                                      reduce_op, mult_op));
            COMET_CHK(dot_chunks(pairs, pair_hit, &before, &chunks));
            KernelTimer t("spgemm_numeric_dot_compact");
            if (chunks > 0)
                dot_chunk_compact<<<dim3((unsigned)chunks), dim3(256), 0, stream()>>>(rb, re, m->pos, m->crd, pair_val, pair_hit,
                                                                                      before, nullptr, Ccrd, Cval);
            COMET_HIPCHK(hipGetLastError());
            return COMET_HIP_OK;
        }
    }
    SgGeom g;
    COMET_CHK(sg_geometry(b->ncols, &g));
    if (!tickets_clear)
        COMET_CHK(sg_reset_ticket());
    unsigned long long *tickets = sg_ticket(tickets_clear ? SG_TICKETS / 2 : 0);
    // rows with many products go to the LDS-accumulator kernel (unmasked products only)
    const int nblk = (int)ceil_div(b->ncols > 0 ? b->ncols : 1, SG_CB);
    // (the `any` semiring keeps a product's place in B in 32 bits of its accumulator)
    const bool lds_rows = nblk <= SG_DENSE_MAX_BLOCKS && (reduce_op != COMET_SR_ANY || b->nnz < (1ll << 32));
    const bool dense = !m && lds_rows;
    // masked: the rows whose mask row does not fit the slab kernel's hash table take the one-block kernel
    const bool mdense = m && lds_rows && g.lds && getenv("COMET_HIP_SPGEMM_NO_MASKED_DENSE") == nullptr;
    const bool small = dense && b->ncols <= SM_COLS;
    SgClasses classes = sg_row_classes(b->ncols, small);
    // the kernels that stream staged slices take four entries of B at a time and keep a place in B and an end in a word
    const bool slices = dense && a->nnz < (1ll << 30) && b->nnz >= 4 && b->nnz < SLICE_NNZ_MOST;
    if (!slices)                 // every heavy row to the kernel that takes the widest block by block
        classes.wide = classes.dense;
    if (dense || mdense)
        COMET_CHK(sg_plan_blocks(b));
    RowList list;
    if (mdense)         // those rows sort in front (sg_row_keys): bounds[0] = bounds[2] = their number
        COMET_CHK(sg_row_list(a, b, rb, re, 1ll << 61, 1ll << 61, &list, m, SG_HASH_FILL));
    else
        COMET_CHK(sg_row_list(a, b, rb, re, dense ? classes.dense : SG_NO_DENSE, dense ? classes.wide : SG_NO_DENSE, &list, nullptr,
                              0, dense, dense ? classes.mid : -1, dense ? classes.few : -1));
    uint32_t *gbm = nullptr, *gmask = nullptr;
    if (!small) {
        if (!g.lds || m) {          // the output row's bitmap is in HBM when LDS holds the mask row instead
            COMET_CHK(g_sg.gbm.ensure(sizeof(uint32_t) * g.bm_words * (size_t)g.groups, true));
            gbm = (uint32_t *)g_sg.gbm.ptr;
        }
        if (m && !g.lds) {
            COMET_CHK(g_sg.gmask.ensure(sizeof(uint32_t) * g.bm_words * (size_t)g.groups, true));
            gmask = (uint32_t *)g_sg.gmask.ptr;
        }
        COMET_CHK(g_sg.slabs.ensure(sizeof(double) * (size_t)(b->ncols > 0 ? b->ncols : 1) * (size_t)g.groups, true));
    }
    const dim3 grid((unsigned)g.groups), block(SG_T);
    // a masked product keeps either the mask row's bitmap or its hash table in LDS, whichever the row needs
    const size_t num_lds = m && g.lds && g.lds_bytes < SG_HASH_LDS ? SG_HASH_LDS : g.lds_bytes;
#define LAUNCH_NUM(L, M, S)                                                                                \
    do {                                                                                                   \
        COMET_CHK(sg_allow_lds(spgemm_numeric_kernel<L, M, S>, num_lds));                                  \
        KernelTimer t(S ? "spgemm_numeric_semiring" : M ? "spgemm_numeric_masked" : "spgemm_numeric");    \
        spgemm_numeric_kernel<L, M, S><<<grid, block, num_lds, stream()>>>(                                \
            rb, re, b->ncols, a->pos, a->crd, a->val, b->pos, b->crd, b->val, m ? m->pos : nullptr,        \
            m ? m->crd : nullptr, g.logW, gbm, gmask, (double *)g_sg.slabs.ptr,                            \
            tickets, list, LIST_LIGHT, reduce_op, mult_op, Cpos, Ccrd, Cval);                               \
    } while (0)
#define LAUNCH_NUM_S(L, M)                                                                                 \
    do {                                                                                                   \
        if (semi) LAUNCH_NUM(L, M, true); else LAUNCH_NUM(L, M, false);                                    \
    } while (0)
    if (small) {
        const int words = sm_words(b->ncols);
        const bool known = list.counts[0] >= 0;
        const auto launch = [&](auto kernel, int part, int lanes, size_t behind, int64_t rows, int per_cu) -> int {
            const size_t lds = sizeof(uint32_t) * (size_t)(words + words / 2) + behind;
            KernelTimer t(semi ? "spgemm_numeric_semiring" : "spgemm_numeric");
            COMET_CHK(sg_allow_lds(kernel, lds));
            kernel<<<sm_grid(known ? rows : -1, per_cu), dim3(lanes), lds, stream()>>>(
                rb, list, part, words, a->pos, a->crd, a->val, b->pos, b->crd, b->val, Cpos, Ccrd, Cval, reduce_op, mult_op);
            return COMET_HIP_OK;
        };
        // rows of few products by a launch of their own, unless they are too few beside others to be worth it
        const int64_t few = known ? list.counts[1] - list.counts[4] : 0;
        const bool apart = few >= SM_FEW_ROWS || (few > 0 && list.counts[4] == list.counts[3]);
        if (apart)
            COMET_CHK(launch(semi ? spgemm_numeric_small_kernel<true, SM_T, 1> : spgemm_numeric_small_kernel<false, SM_T, 1>,
                             LIST_FEW, SM_T, sizeof(SmallRowLds<SM_T, 1>), few, 7));
        if (!list.none_small() && !(apart && list.counts[4] == list.counts[3]))
            COMET_CHK(launch(semi ? spgemm_numeric_small_kernel<true, SM_T, SM_PER> : spgemm_numeric_small_kernel<false, SM_T, SM_PER>,
                             apart ? LIST_SMALL_MORE : LIST_SMALL, SM_T, sizeof(SmallRowLds<SM_T, SM_PER>),
                             list.counts[apart ? 4 : 1] - list.counts[3], 7));
        if (classes.mid < classes.dense && !list.none_mid())
            COMET_CHK(launch(semi ? spgemm_numeric_small_kernel<true, SM_MID_T, SM_PER> : spgemm_numeric_small_kernel<false, SM_MID_T, SM_PER>,
                             LIST_MID, SM_MID_T, sizeof(SmallRowLds<SM_MID_T, SM_PER>), list.counts[3] - list.counts[0], 2));
    } else if (list.only_heavy()) {
        // nothing for these kernels
    } else if (g.lds) {
        if (m) LAUNCH_NUM_S(true, true); else LAUNCH_NUM_S(true, false);
    } else {
        if (m) LAUNCH_NUM_S(false, true); else LAUNCH_NUM_S(false, false);
    }
#undef LAUNCH_NUM_S
#undef LAUNCH_NUM
    COMET_HIPCHK(hipGetLastError());
    // the rows of the one-block kernel block by block (COMET_HIP_SPGEMM_ROW_MAJOR keeps them row by row; the
    // tests run both)
    const bool by_blocks = slices && getenv("COMET_HIP_SPGEMM_ROW_MAJOR") == nullptr;
    bool ran_blocks = false;
    int64_t *word = nullptr;
    COMET_CHK(mailbox((void **)&word));
    int *gave_up = (int *)(word + 1);
    if (by_blocks) {
        int64_t nd = list.counts[2];
        if (nd < 0) {
            COMET_HIPCHK(hipMemcpyAsync(word, list.bounds + 2, sizeof(int64_t), hipMemcpyDeviceToHost, stream()));
            COMET_CHK(stream_wait());
            nd = *(volatile int64_t *)word;
        }
        if (nd > 0) {
            ran_blocks = true;
            const bool alone = nblk == 1;
            if (!alone) {
                COMET_CHK(g_sg.dense_rows.ensure(sizeof(DenseRow) * (size_t)nd, false));
                COMET_CHK(g_sg.dense_before.ensure(sizeof(int32_t) * (size_t)nd * (size_t)nblk, false));
            }
            const RowSource source{list.rows, rb, a->pos, Cpos};
            gave_up[0] = 0;
            int patience = DB_PATIENCE;
            if (const char *e = getenv("COMET_HIP_SPGEMM_PATIENCE"))
                patience = atoi(e);
            KernelTimer t("spgemm_numeric_dense_blocks");
            const dim3 cus((unsigned)(num_cus() > 0 ? num_cus() : 256));
            if (!alone)
                spgemm_dense_rows<<<dim3((unsigned)ceil_div(nd * nblk, 256)), dim3(256), 0, stream()>>>(
                    source, nd, nblk, (DenseRow *)g_sg.dense_rows.ptr, (int32_t *)g_sg.dense_before.ptr);
            const auto launch = [&](auto kernel, const auto *crd, int lanes, size_t lds, unsigned a_cu) -> int {
                // as many rows to a ticket as leave every workgroup some four of them (8 to each of 50 CUs: 78 us for a
                // graph of 1024 vertices, the others idle)
                const dim3 grid(a_cu * cus.x);
                const int rows_each = (int)std::max<int64_t>(1, std::min<int64_t>(DB_ROWS, nd * nblk / (4 * (int64_t)grid.x)));
                COMET_CHK(sg_allow_lds(kernel, lds));
                kernel<<<grid, dim3(lanes), lds, stream()>>>(
                    (const DenseRow *)g_sg.dense_rows.ptr, source, nd, a->crd, a->val, crd, b->val, b->nnz, b->sg_blkptr, nblk,
                    tickets + 1, (int32_t *)g_sg.dense_before.ptr, rows_each, patience, gave_up, Ccrd, Cval, reduce_op, mult_op);
                return COMET_HIP_OK;
            };
            const auto by_shape = [&](auto semiring) -> int {
                constexpr bool S = decltype(semiring)::value;
                if (!b->sg_crd16 || getenv("COMET_HIP_SPGEMM_WIDE_COLUMNS") != nullptr)
                    return alone ? launch(spgemm_numeric_dense_blocks_kernel<S, int32_t, true, SG_T, 16>, b->crd, SG_T, DB_LDS<SG_T, 16>, 1)
                                 : launch(spgemm_numeric_dense_blocks_kernel<S, int32_t, false, SG_T, 16>, b->crd, SG_T, DB_LDS<SG_T, 16>, 1);
                if (!alone)
                    return launch(spgemm_numeric_dense_blocks_kernel<S, uint16_t, false, SG_T, 16>, b->sg_crd16, SG_T, DB_LDS<SG_T, 16>, 1);
#define LAUNCH_ALONE(T, ROWS, A_CU)                                                                                     \
    return launch(spgemm_numeric_dense_blocks_kernel<S, uint16_t, true, T, ROWS>, b->sg_crd16, T, DB_LDS<T, ROWS>, A_CU)
                if (b->ncols <= SG_NARROW && nd >= DB_TWO_ROWS * (int64_t)cus.x / 2) {
                    if (b->ncols <= 512 * 4)
                        LAUNCH_ALONE(512, 4, 2);
                    if (b->ncols <= 512 * 8)
                        LAUNCH_ALONE(512, 8, 2);
                    LAUNCH_ALONE(512, 16, 2);
                }
                if (b->ncols <= SG_T * 2)
                    LAUNCH_ALONE(SG_T, 2, 1);
                if (b->ncols <= SG_T * 4)
                    LAUNCH_ALONE(SG_T, 4, 1);
                if (b->ncols <= SG_T * 8)
                    LAUNCH_ALONE(SG_T, 8, 1);
                LAUNCH_ALONE(SG_T, 16, 1);
#undef LAUNCH_ALONE
            };
            COMET_CHK(semi ? by_shape(std::true_type()) : by_shape(std::false_type()));
            COMET_HIPCHK(hipGetLastError());
        }
    }
    if ((dense && !by_blocks) || mdense) {
        KernelTimer t(mdense ? "spgemm_numeric_dense_masked" : "spgemm_numeric_dense");
        const dim3 cus((unsigned)(num_cus() > 0 ? num_cus() : 256));
#define LAUNCH_DENSE_C(S, M, COL, CRD)                                                                     \
    do {                                                                                                   \
        COMET_CHK(sg_allow_lds(spgemm_numeric_dense_kernel<S, M, COL>, SG_DENSE_LDS));                     \
        spgemm_numeric_dense_kernel<S, M, COL><<<cus, block, SG_DENSE_LDS, stream()>>>(                    \
            rb, re, a->pos, a->crd, a->val, CRD, b->val, m ? m->pos : nullptr, m ? m->crd : nullptr,       \
            b->sg_blkptr, nblk, tickets + 1, list, Cpos, Ccrd, Cval, reduce_op, mult_op);                                                                                      \
    } while (0)
#define LAUNCH_DENSE(S, M)                                                                                 \
    do {                                                                                                   \
        if (b->sg_crd16 && getenv("COMET_HIP_SPGEMM_WIDE_COLUMNS") == nullptr)                             \
            LAUNCH_DENSE_C(S, M, uint16_t, b->sg_crd16);                                                   \
        else                                                                                               \
            LAUNCH_DENSE_C(S, M, int32_t, b->crd);                                                         \
    } while (0)
        if (mdense) {
            if (semi) LAUNCH_DENSE(true, true); else LAUNCH_DENSE(false, true);
        } else {
            if (semi) LAUNCH_DENSE(true, false); else LAUNCH_DENSE(false, false);
        }
#undef LAUNCH_DENSE_C
#undef LAUNCH_DENSE
        COMET_HIPCHK(hipGetLastError());
    }
    if (dense && (list.counts[0] < 0 || list.counts[0] > list.counts[2])) {
        KernelTimer t("spgemm_numeric_span");
        const dim3 cus((unsigned)(num_cus() > 0 ? num_cus() : 256));
        if (semi) {
            COMET_CHK(sg_allow_lds(spgemm_numeric_span_kernel<true>, SG_SPAN_LDS));
            spgemm_numeric_span_kernel<true><<<cus, block, SG_SPAN_LDS, stream()>>>(
                rb, a->pos, a->crd, a->val, b->crd, b->val, b->nnz, b->sg_blkptr, nblk, list, Cpos, Ccrd, Cval, reduce_op, mult_op);
        } else {
            COMET_CHK(sg_allow_lds(spgemm_numeric_span_kernel<false>, SG_SPAN_LDS));
            spgemm_numeric_span_kernel<false><<<cus, block, SG_SPAN_LDS, stream()>>>(
                rb, a->pos, a->crd, a->val, b->crd, b->val, b->nnz, b->sg_blkptr, nblk, list, Cpos, Ccrd, Cval, reduce_op, mult_op);
        }
        COMET_HIPCHK(hipGetLastError());
    }
    if (ran_blocks) {           // did a workgroup stop waiting for the block before its own
        COMET_CHK(stream_wait());
        if (*(volatile int *)gave_up)
            return set_error(COMET_HIP_ERR_HIP, "spgemm numeric: a column block's place in its row never arrived");
    }
    return COMET_HIP_OK;
}

}  // namespace comet

using namespace comet;

extern "C" int comet_hip_spgemm_csr_symbolic(int64_t ah, int64_t bh, int64_t mh, int64_t pos_dptr, int64_t *nnz_out)
{
    COMET_CHK(ensure_init());
    Csr *a = csr_from_handle(ah), *b = csr_from_handle(bh), *m = mh ? csr_from_handle(mh) : nullptr;
    if (!a || !b || (mh && !m))
        return COMET_HIP_ERR_HANDLE;
    if (!pos_dptr)
        return set_error(COMET_HIP_ERR_ARG, "null pos passed to comet_hip_spgemm_csr_symbolic");
    COMET_CHK(check_product_shapes(a, b, m, "spgemm symbolic"));
    int64_t *pos = (int64_t *)pos_dptr;
    if (a->nrows > 0) {
        COMET_CHK(g_sg.rowcount.ensure(sizeof(int64_t) * (size_t)a->nrows, false));
        COMET_CHK(symbolic_counts(a, b, m, (int64_t *)g_sg.rowcount.ptr));
    }
    int64_t *word = nullptr;
    if (nnz_out)
        COMET_CHK(mailbox((void **)&word));
    COMET_CHK(exclusive_scan_i64((const int64_t *)g_sg.rowcount.ptr, a->nrows, pos, word));
    if (nnz_out) {
        COMET_CHK(stream_wait());
        *nnz_out = *(volatile int64_t *)word;
    }
    return COMET_HIP_OK;
}

extern "C" int comet_hip_spgemm_csr_numeric(int64_t ah, int64_t bh, int64_t mh, int64_t pos_dptr, int64_t row_begin,
                                            int64_t row_end, int64_t crd_dptr, int64_t val_dptr)
{
    return comet_hip_spgemm_csr_numeric_semiring(ah, bh, mh, pos_dptr, row_begin, row_end, crd_dptr, val_dptr,
                                                 COMET_SR_PLUS, COMET_OP_TIMES);
}

extern "C" int comet_hip_spgemm_csr_numeric_semiring(int64_t ah, int64_t bh, int64_t mh, int64_t pos_dptr,
                                                     int64_t row_begin, int64_t row_end, int64_t crd_dptr,
                                                     int64_t val_dptr, int reduce_op, int mult_op)
{
    COMET_CHK(ensure_init());
    Csr *a = csr_from_handle(ah), *b = csr_from_handle(bh), *m = mh ? csr_from_handle(mh) : nullptr;
    if (!a || !b || (mh && !m))
        return COMET_HIP_ERR_HANDLE;
    COMET_CHK(check_product_shapes(a, b, m, "spgemm numeric"));
    if (row_begin < 0 || row_end < row_begin || row_end > a->nrows)
        return set_error(COMET_HIP_ERR_ARG, "row range [%lld,%lld) outside [0,%lld]", (long long)row_begin,
                         (long long)row_end, (long long)a->nrows);
    if (!pos_dptr || !crd_dptr || !val_dptr)
        return set_error(COMET_HIP_ERR_ARG, "null output array passed to comet_hip_spgemm_csr_numeric");
    if (row_begin == row_end)
        return COMET_HIP_OK;
    return numeric_rows(a, b, m, (const int64_t *)pos_dptr, row_begin, row_end, (int32_t *)crd_dptr,
                        (double *)val_dptr, reduce_op, mult_op);
}

extern "C" int64_t comet_hip_spgemm_csr(int64_t ah, int64_t bh, int64_t mh)
{
    return comet_hip_spgemm_csr_semiring(ah, bh, mh, COMET_SR_PLUS, COMET_OP_TIMES);
}

// C<M> = A*B in one pass over the pairs of the mask: their values and which of them met a product come out of
// the same walk, so the row pointers need no symbolic phase of their own.  *done says whether this form applied.
static int64_t masked_product_one_pass(const Csr *a, const Csr *b, const Csr *m, int reduce_op, int mult_op, bool *done)
{
    *done = false;
    bool dots = false;
    if (dot_form_fits(a, b, m, &dots) != COMET_HIP_OK)
        return 0;
    if (!dots || a->nrows == 0)
        return 0;
    *done = true;
    double *pair_val = nullptr;
    uint8_t *pair_hit = nullptr;
    int64_t pairs = 0, *before = nullptr, chunks = 0;
    void *word = nullptr;
    if (mailbox(&word) != COMET_HIP_OK ||
        pair_dot_values(const_cast<Csr *>(a), const_cast<Csr *>(b), const_cast<Csr *>(m), 0, a->nrows, &pair_val, &pair_hit,
                        &pairs, reduce_op, mult_op) != COMET_HIP_OK ||
        dot_chunks(pairs, pair_hit, &before, &chunks, (int64_t *)word) != COMET_HIP_OK)
        return 0;
    Csr *c = new Csr();
    c->nrows = a->nrows;
    c->ncols = b->ncols;
    c->owns = true;
    const auto fail = [&](const char *what) -> int64_t {
        if (what)
            set_error(COMET_HIP_ERR_HIP, "%s", what);
        csr_release(c);
        return 0;
    };
    if (stream_wait() != COMET_HIP_OK)
        return fail("reading the size of the product failed");
    c->nnz = *(volatile int64_t *)word;
    if (dev_malloc((void **)&c->pos, sizeof(int64_t) * (size_t)(a->nrows + 1)) != hipSuccess ||
        dev_malloc((void **)&c->crd, sizeof(int32_t) * (size_t)(c->nnz > 0 ? c->nnz : 1)) != hipSuccess ||
        dev_malloc((void **)&c->val, sizeof(double) * (size_t)(c->nnz > 0 ? c->nnz : 1)) != hipSuccess)
        return fail("output allocation failed");
    if (chunks == 0 && hipMemsetAsync(c->pos, 0, sizeof(int64_t) * (size_t)(a->nrows + 1), stream()) != hipSuccess)
        return fail("clearing the row pointers failed");
    if (chunks > 0) {
        KernelTimer t("spgemm_numeric_dot_compact");
        dot_chunk_compact<<<dim3((unsigned)chunks), dim3(256), 0, stream()>>>(0, a->nrows, m->pos, m->crd, pair_val, pair_hit,
                                                                              before, c->pos, c->crd, c->val);
    }
    if (hipGetLastError() != hipSuccess)
        return fail("launching the compaction failed");
    return csr_register(c);
}

extern "C" int64_t comet_hip_spgemm_csr_semiring(int64_t ah, int64_t bh, int64_t mh, int reduce_op, int mult_op)
{
    if (ensure_init() != COMET_HIP_OK)
        return 0;
    Csr *a = csr_from_handle(ah), *b = csr_from_handle(bh), *m = mh ? csr_from_handle(mh) : nullptr;
    if (!a || !b || (mh && !m))
        return 0;
    if (check_product_shapes(a, b, m, "spgemm") != COMET_HIP_OK)
        return 0;
    if (m && reduce_op >= 0 && reduce_op < COMET_SR_ANY && mult_op >= 0 && mult_op <= COMET_OP_DIV) {
        bool done = false;
        const int64_t h = masked_product_one_pass(a, b, m, reduce_op, mult_op, &done);
        if (done)
            return h;
    }
    int64_t *pos = nullptr;
    if (dev_malloc((void **)&pos, sizeof(int64_t) * (size_t)(a->nrows + 1)) != hipSuccess) {
        set_error(COMET_HIP_ERR_HIP, "row pointer allocation failed");
        return 0;
    }
    int64_t nnz = 0;
    if (comet_hip_spgemm_csr_symbolic(ah, bh, mh, (int64_t)pos, &nnz) != COMET_HIP_OK) {
        (void)dev_free(pos);
        return 0;
    }
    Csr *c = new Csr();
    c->nrows = a->nrows;
    c->ncols = b->ncols;
    c->nnz = nnz;
    c->pos = pos;
    c->owns = true;
    if (dev_malloc((void **)&c->crd, sizeof(int32_t) * (size_t)(nnz > 0 ? nnz : 1)) != hipSuccess ||
        dev_malloc((void **)&c->val, sizeof(double) * (size_t)(nnz > 0 ? nnz : 1)) != hipSuccess) {
        set_error(COMET_HIP_ERR_HIP, "output allocation of %lld entries failed", (long long)nnz);
        (void)dev_free(c->crd);
        (void)dev_free(pos);
        delete c;
        return 0;
    }
    if (nnz > 0 && numeric_rows(a, b, m, pos, 0, a->nrows, c->crd, c->val, reduce_op, mult_op, !m) != COMET_HIP_OK) {
        (void)dev_free(c->crd);
        (void)dev_free(c->val);
        (void)dev_free(pos);
        delete c;
        return 0;
    }
    return csr_register(c);
}

extern "C" int comet_hip_spgemm_masked_sum(int64_t ah, int64_t bh, int64_t mh, double *out)
{
    COMET_CHK(ensure_init());
    Csr *a = csr_from_handle(ah), *b = csr_from_handle(bh), *m = csr_from_handle(mh);
    if (!a || !b || !m)
        return COMET_HIP_ERR_HANDLE;
    if (!out)
        return set_error(COMET_HIP_ERR_ARG, "null result pointer");
    COMET_CHK(check_product_shapes(a, b, m, "masked sum"));
    if (a->nrows == 0) {
        *out = 0.0;
        return COMET_HIP_OK;
    }
    SgGeom g;
    COMET_CHK(sg_geometry(b->ncols, &g));
    bool iso = false;
    if (g.lds && a == b && a == m)
        COMET_CHK(csr_look(a, true, true));
    if (g.lds)
        COMET_CHK(csr_is_iso(b, &iso));
    bool pairs = false;
    if (iso)
        COMET_CHK(pair_form_fits(a, b, m, &pairs));
    if (pairs && a == b && a == m) {
        if (a->tri_state == 0)
            (void)plan_made([&] { return tri_plan(a, pair_only()); });
        if (a->tri_state == 2)
            return tri_count(a, out);
    }
    if (pairs)
        return pair_masked_sum(a, b, m, out);
    COMET_CHK(sg_reset_ticket());
    COMET_CHK(g_sg.rowcount.ensure(sizeof(double) * (size_t)a->nrows, false));
    uint32_t *gbm = nullptr;
    if (!g.lds) {
        COMET_CHK(g_sg.gbm.ensure(sizeof(uint32_t) * g.bm_words * (size_t)g.groups, true));
        gbm = (uint32_t *)g_sg.gbm.ptr;
    }
    double *rowsum = (double *)g_sg.rowcount.ptr;
    RowList list;
    // rows whose mask row is too long for the wavefront kernel's table sort to the front, whatever their products:
    // the workgroup kernel, which starts there, looks a column up in one LDS read; the wavefront kernel would
    // bisect the mask row in memory for every product
    COMET_CHK(sg_row_list(a, b, 0, a->nrows, SG_NO_DENSE, SG_NO_DENSE, &list, m, SM_MASK_MAX));
    COMET_HIPCHK(hipMemsetAsync(rowsum, 0, sizeof(double) * (size_t)a->nrows, stream()));
    const dim3 grid((unsigned)g.groups), block(SG_T);
    // Two kernels side by side, the second on the auxiliary stream: a workgroup per row from the heavy end of
    // the list, a wavefront per row from the light end, until they meet.  A row of a thousand products costs
    // the first kernel more in barriers than in products; a row of a million would keep one wavefront of the
    // second busy for a millisecond.  Triangle count of the scale-20 R-MAT graph: 29.2 ms with the first
    // kernel alone, 22.1 ms one after the other with a fixed split at 65536 products, 17.6 ms side by side with
    // the best fixed split (49152 products), 18.9 ms with the two ends meeting by themselves (the difference is
    // the last wavefront-rows near the meeting point; looking at the ticket word before drawing from it, to keep
    // the wavefronts away from those rows, or drawing 16 rows at a time, costs more on that one word than it saves).
    // COMET_HIP_MASKED_SUM_ONLY=workgroup|wavefront launches one of the two kernels only, which then takes every
    // row: the tests send each class of rows through both
    const char *only = getenv("COMET_HIP_MASKED_SUM_ONLY");
    const bool run_wg = !only || strcmp(only, "wavefront") != 0, run_wave = !only || strcmp(only, "workgroup") != 0;
    COMET_CHK(aux_fork());
    if (!run_wg) {
    } else if (g.lds) {
        COMET_CHK(sg_allow_lds(spgemm_masked_sum_kernel<true>, g.lds_bytes));
        KernelTimer t("spgemm_masked_sum");
        spgemm_masked_sum_kernel<true><<<grid, block, g.lds_bytes, stream()>>>(
            a->nrows, a->pos, a->crd, a->val, b->pos, b->crd, b->val, m->pos, m->crd, g.logW, gbm,
            (unsigned long long *)g_sg.ticket.ptr, list, rowsum);
    } else {
        KernelTimer t("spgemm_masked_sum");
        spgemm_masked_sum_kernel<false><<<grid, block, 0, stream()>>>(
            a->nrows, a->pos, a->crd, a->val, b->pos, b->crd, b->val, m->pos, m->crd, g.logW, gbm,
            (unsigned long long *)g_sg.ticket.ptr, list, rowsum);
    }
    if (run_wave) {   // eight workgroups of four wavefronts per CU: four fit beside the kernel above, the rest follow it
        KernelTimer t("spgemm_masked_sum_small", aux_stream());
        spgemm_masked_sum_small_kernel<<<dim3((unsigned)(num_cus() * 8)), dim3(SM_WAVES * 64), 0, aux_stream()>>>(
            a->pos, a->crd, a->val, b->pos, b->crd, b->val, m->pos, m->crd,
            (unsigned long long *)g_sg.ticket.ptr, list, rowsum);
    }
    COMET_HIPCHK(hipGetLastError());
    COMET_CHK(aux_join());
    return reduce_sum_device(rowsum, a->nrows, out);
}

extern "C" int64_t comet_hip_eltwise_mult_csr(int64_t ah, int64_t bh)
{
    if (ensure_init() != COMET_HIP_OK)
        return 0;
    Csr *a = csr_from_handle(ah), *b = csr_from_handle(bh);
    if (!a || !b)
        return 0;
    if (a->nrows != b->nrows || a->ncols != b->ncols) {
        set_error(COMET_HIP_ERR_ARG, "element-wise product of %lld x %lld and %lld x %lld", (long long)a->nrows,
                  (long long)a->ncols, (long long)b->nrows, (long long)b->ncols);
        return 0;
    }
    const int64_t n = a->nrows;
    int64_t *pos = nullptr;
    if (dev_malloc((void **)&pos, sizeof(int64_t) * (size_t)(n + 1)) != hipSuccess) {
        set_error(COMET_HIP_ERR_HIP, "row pointer allocation failed");
        return 0;
    }
    auto fail = [&](Csr *c) -> int64_t {
        if (c) {
            (void)dev_free(c->crd);
            (void)dev_free(c->val);
            delete c;
        }
        (void)dev_free(pos);
        return 0;
    };
    if (g_sg.rowcount.ensure(sizeof(int64_t) * (size_t)(n > 0 ? n : 1), false) != COMET_HIP_OK)
        return fail(nullptr);
    int64_t *rowcount = (int64_t *)g_sg.rowcount.ptr;
    const dim3 grid((unsigned)ceil_div(n > 0 ? n : 1, 256)), block(256);
    if (n > 0) {
        KernelTimer t("eltwise_mult_count");
        eltwise_mult_kernel<false><<<grid, block, 0, stream()>>>(n, a->pos, a->crd, a->val, b->pos, b->crd, b->val,
                                                                 rowcount, nullptr, nullptr, nullptr);
    }
    if (exclusive_scan_i64(rowcount, n, pos) != COMET_HIP_OK)
        return fail(nullptr);
    int64_t nnz = 0;
    if (hipMemcpyAsync(&nnz, pos + n, sizeof(int64_t), hipMemcpyDeviceToHost, stream()) != hipSuccess ||
        stream_wait() != COMET_HIP_OK) {
        set_error(COMET_HIP_ERR_HIP, "reading nnz failed");
        return fail(nullptr);
    }
    Csr *c = new Csr();
    c->nrows = n;
    c->ncols = a->ncols;
    c->nnz = nnz;
    c->pos = pos;
    c->owns = true;
    if (dev_malloc((void **)&c->crd, sizeof(int32_t) * (size_t)(nnz > 0 ? nnz : 1)) != hipSuccess ||
        dev_malloc((void **)&c->val, sizeof(double) * (size_t)(nnz > 0 ? nnz : 1)) != hipSuccess) {
        set_error(COMET_HIP_ERR_HIP, "output allocation failed");
        return fail(c);
    }
    if (n > 0 && nnz > 0) {
        KernelTimer t("eltwise_mult_fill");
        eltwise_mult_kernel<true><<<grid, block, 0, stream()>>>(n, a->pos, a->crd, a->val, b->pos, b->crd, b->val,
                                                                nullptr, pos, c->crd, c->val);
    }
    if (hipGetLastError() != hipSuccess) {
        set_error(COMET_HIP_ERR_HIP, "element-wise kernel launch failed");
        return fail(c);
    }
    return csr_register(c);
}

extern "C" int64_t comet_hip_eltwise_csr_dense_csr(int64_t ah, int64_t d_dptr, int64_t ldd, int op)
{
    if (ensure_init() != COMET_HIP_OK)
        return 0;
    Csr *a = csr_from_handle(ah);
    if (!a)
        return 0;
    if (ldd < a->ncols || (a->nnz > 0 && !d_dptr) || op < 0 || op > COMET_OP_DIV) {
        set_error(COMET_HIP_ERR_ARG, "bad dense operand or operator passed to comet_hip_eltwise_csr_dense_csr");
        return 0;
    }
    Csr *c = new Csr();
    if (csr_alloc(c, a->nrows, a->ncols, a->nnz) != COMET_HIP_OK) {
        delete c;
        return 0;
    }
    bool ok = hipMemcpyAsync(c->pos, a->pos, sizeof(int64_t) * (size_t)(a->nrows + 1), hipMemcpyDeviceToDevice,
                             stream()) == hipSuccess;
    if (ok && a->nnz > 0) {
        ok = hipMemcpyAsync(c->crd, a->crd, sizeof(int32_t) * (size_t)a->nnz, hipMemcpyDeviceToDevice, stream()) ==
             hipSuccess;
        KernelTimer t("eltwise_mult_dense");
        eltwise_mult_dense_kernel<false><<<dim3((unsigned)ceil_div(a->nrows * 16, 256)), dim3(256), 0, stream()>>>(
            a->nrows, a->pos, a->crd, a->val, (const double *)d_dptr, ldd, c->val, 0, op);
    }
    if (!ok || hipGetLastError() != hipSuccess) {
        set_error(COMET_HIP_ERR_HIP, "CSR .* Dense failed");
        csr_release(c);
        return 0;
    }
    return csr_register(c);
}

extern "C" int comet_hip_eltwise_csr_dense_dense(int64_t ah, int64_t d_dptr, int64_t ldd, int64_t c_dptr,
                                                 int64_t ldc, int op)
{
    COMET_CHK(ensure_init());
    Csr *a = csr_from_handle(ah);
    if (!a)
        return COMET_HIP_ERR_HANDLE;
    if (ldd < a->ncols || ldc < a->ncols || (a->nnz > 0 && (!d_dptr || !c_dptr)) || op < 0 || op > COMET_OP_DIV)
        return set_error(COMET_HIP_ERR_ARG, "bad dense operand or operator passed to comet_hip_eltwise_csr_dense_dense");
    if (a->nnz == 0)
        return COMET_HIP_OK;
    KernelTimer t("eltwise_mult_dense");
    eltwise_mult_dense_kernel<true><<<dim3((unsigned)ceil_div(a->nrows * 16, 256)), dim3(256), 0, stream()>>>(
        a->nrows, a->pos, a->crd, a->val, (const double *)d_dptr, ldd, (double *)c_dptr, ldc, op);
    COMET_HIPCHK(hipGetLastError());
    return COMET_HIP_OK;
}

// Dense (op) Dense over n elements (test/integration/semiring/eltwise_monoid*_DensexDense_oDense.ta).
__global__ void eltwise_dense_kernel(int64_t n, const double *__restrict__ a, const double *__restrict__ b,
                                     double *__restrict__ c, int op)
{
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t step = (int64_t)gridDim.x * blockDim.x;
    for (; i < n; i += step)
        c[i] = semiring_mult(op, a[i], b[i]);
}

extern "C" int comet_hip_eltwise_dense_f64(int64_t n, int64_t a_dptr, int64_t b_dptr, int64_t c_dptr, int op)
{
    COMET_CHK(ensure_init());
    if (n < 0 || (n > 0 && (!a_dptr || !b_dptr || !c_dptr)) || op < 0 || op > COMET_OP_DIV)
        return set_error(COMET_HIP_ERR_ARG, "bad arguments to comet_hip_eltwise_dense_f64");
    if (n == 0)
        return COMET_HIP_OK;
    KernelTimer t("eltwise_dense");
    const unsigned blocks = (unsigned)std::min<int64_t>(ceil_div(n, 256), (int64_t)num_cus() * 32);
    eltwise_dense_kernel<<<dim3(blocks), dim3(256), 0, stream()>>>(n, (const double *)a_dptr, (const double *)b_dptr,
                                                                  (double *)c_dptr, op);
    COMET_HIPCHK(hipGetLastError());
    return COMET_HIP_OK;
}

// Diagnostic: the vector registers per lane of the two kernels of the pattern-matrix masked sum, as the loaded code
// object has them.  The workgroup kernel (16 wavefronts, four to a SIMD) and one wavefront of the other kernel
// share a SIMD's 512 registers, allotted in eights: what a test holds them to.
extern "C" int comet_hip_debug_masked_sum_registers(int *workgroup_kernel, int *wavefront_kernel)
{
    COMET_CHK(ensure_init());
    if (!workgroup_kernel || !wavefront_kernel)
        return set_error(COMET_HIP_ERR_ARG, "null result pointer");
    hipFuncAttributes at;
    COMET_HIPCHK(hipFuncGetAttributes(&at, reinterpret_cast<const void *>(pair_sum_heavy_kernel<true>)));
    *workgroup_kernel = at.numRegs;
    COMET_HIPCHK(hipFuncGetAttributes(&at, reinterpret_cast<const void *>(pair_sum_light_kernel<true>)));
    *wavefront_kernel = at.numRegs;
    return COMET_HIP_OK;
}

// Diagnostic: where the fp64 sums of the dot-product kernel begin in its LDS, in 32-bit words, for a bitmap of
// `words` words (the counts beside it included); lets a CPU-side test sweep the invariant "even".
extern "C" int comet_hip_debug_tri_bucket(int group, int attempt, int log_buckets)
{
    return tri_bucket((uint32_t)group << 16, tri_multiplier(attempt), log_buckets);
}

extern "C" int comet_hip_debug_dot_table_words(int words)
{
    return dot_table_words(32 * (int64_t)(words < 1 ? 1 : words));
}
