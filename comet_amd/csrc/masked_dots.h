// C<M> = A*B as dot products, pair by pair (included by spgemm.hip after masked_pairs.h): for every stored (i, j) of M
// the sum over the columns that row i of A and column j of B share.  The shorter of the two is streamed, its columns and
// values together - a quarter of the look-ups of a power-law graph hit, so nearly every cache line of the values is
// needed anyway - against a table of the longer one in LDS that turns a column into its place in the row.

typedef double pair_d2 __attribute__((ext_vector_type(2), aligned(8)));

// One row of 64 quads is a turn: 3 KiB a wavefront, twice that under way, which 16 wavefronts a CU make enough; two rows
// need more registers than there are (4.3 ms for the long rows of 200003 vertices, edge factor 16, instead of 3.3).
struct DotTurn {
    sg_i4u q;
    pair_d2 lo, hi;
    uint32_t mask;                       // bits 0-3: which of the four columns are the list's
    int owner;                           // the list's lane
    unsigned long long ends;             // bit l: lane l has its list's last quad in this turn (the same in all lanes)
};

// 64 lists, one per lane, streamed end to end as in quad_walk
struct DotLists {
    int a0, end, first, Q;
    uint32_t before;
    __device__ __forceinline__ void take(uint32_t start, int len)
    {
        const int quads = (len + 3) >> 2;
        const int inc = wave_inclusive_scan(quads), pre = inc - quads;
        Q = __builtin_amdgcn_readlane(inc, 63);
        a0 = (int)(start - 4u * (uint32_t)pre);
        end = (int)(start + (uint32_t)len);
        first = len > 0 ? pre - 1 : -1;          // -1: sets no mark
        before = 0;
    }
    // the loads of the turn that begins at quad `base`; past the last quad they name no columns
    __device__ __forceinline__ void issue(DotTurn &t, int base, const PairSide &s, uint32_t *marks, int lane)
    {
        const uint32_t bit = (uint32_t)(first - base);
        if (bit < 64u)
            atomicOr(&marks[bit >> 5], 1u << (bit & 31u));
        wave_lds_order();
        uint2 m = *reinterpret_cast<const uint2 *>(marks);
        wave_lds_order();
        if (lane < 2)
            marks[lane] = 0;
        m.x = (uint32_t)__builtin_amdgcn_readfirstlane((int)m.x);
        m.y = (uint32_t)__builtin_amdgcn_readfirstlane((int)m.y);
        uint32_t from;
        quad_place(m, before, a0, end, 4u * (uint32_t)(base + lane), s.Lnnz - 4u, t.owner, from, t.mask);
        // a mark at a quad is the beginning of the next list behind it
        t.ends = (unsigned long long)m.y << 32 | m.x | 1ull << 63;
        t.q = *reinterpret_cast<const sg_i4u *>(s.Lcrd + from);
        t.lo = *reinterpret_cast<const pair_d2 *>(s.Lval + from);
        t.hi = *reinterpret_cast<const pair_d2 *>(s.Lval + from + 2);
        wave_lds_order();
    }
};

// v summed over the lanes of one list (ends: their last lanes), complete in the last of them.  Which lanes take part in a
// step is the same for the whole wavefront and costs its vector unit, the busiest part of these kernels, nothing: a bit of
// a scalar register selects what is added.
__device__ __forceinline__ double list_sum_f64(double v, unsigned long long ends)
{
    const unsigned long long starts = ends << 1;
    const auto below = [](uint32_t x) { return (x - 1u) & ~x; };          // the bits below the lowest one that is set
    // bit l: the 1, 2, 4, 8 lanes up to l go on with the list of the lane before each, in the same row of 16 lanes
    const unsigned long long m1 = ~starts & 0xfffefffefffefffeull, m2 = m1 & m1 << 1, m4 = m2 & m2 << 2, m8 = m4 & m4 << 4;
    // so do all lanes up to l of an odd row; of the upper half
    const unsigned long long m16 = (unsigned long long)(below((uint32_t)(starts >> 48)) & 0xffffu) << 48 |
                                   (unsigned long long)(below((uint32_t)starts >> 16) & 0xffffu) << 16;
    const unsigned long long m32 = (unsigned long long)below((uint32_t)(starts >> 32)) << 32;
#define COMET_LIST_STEP(ctrl, lanes)                                                                           \
    {                                                                                                          \
        const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), ctrl, 0xf, 0xf, true);                \
        const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), ctrl, 0xf, 0xf, true);                \
        v += __builtin_amdgcn_inverse_ballot_w64(lanes) ? __hiloint2double(hi, lo) : 0.0;                      \
    }
    COMET_LIST_STEP(0x111, m1)
    COMET_LIST_STEP(0x112, m2)
    COMET_LIST_STEP(0x114, m4)
    COMET_LIST_STEP(0x118, m8)
    COMET_LIST_STEP(0x142, m16)
    COMET_LIST_STEP(0x143, m32)
#undef COMET_LIST_STEP
    return v;
}

struct DotSemiring {
    int reduce_op, mult_op;
};

// What the look-ups of a turn give, added to the lists' results acc[64] and hit[64] (the wavefront's own).
// SEMI: another semiring than plus-times; acc holds sums or keys, and every product is added by itself.
template <bool SEMI, typename PROBE>
__device__ __forceinline__ void dot_turn(const DotTurn &t, const PROBE &probe, double *acc, int *hit, DotSemiring op,
                                         bool swapped)
{
    const int j[4] = {t.q.x, t.q.y, t.q.z, t.q.w};
    const double lv[4] = {t.lo.x, t.lo.y, t.hi.x, t.hi.y};
    bool met[4];
    int at[4];
    probe.find(j, t.mask, met, at);
    const bool any = met[0] | met[1] | met[2] | met[3];
    if (__any(any)) {
        double tv[4];
        probe.values(at, tv);
        if constexpr (SEMI) {
#pragma unroll
            for (int c = 0; c < 4; ++c)
                if (met[c]) {
                    const double e = swapped ? semiring_mult(op.mult_op, lv[c], tv[c]) : semiring_mult(op.mult_op, tv[c], lv[c]);
                    if (op.reduce_op == SR_PLUS)
                        __hip_atomic_fetch_add(&acc[t.owner], e, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                    else
                        __hip_atomic_fetch_max(reinterpret_cast<unsigned long long *>(&acc[t.owner]),
                                               op.reduce_op == SR_MIN ? ~f64_key(e) : f64_key(e), __ATOMIC_RELAXED,
                                               __HIP_MEMORY_SCOPE_WORKGROUP);
                }
        } else {
            double p = 0.0;
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const double e = tv[c] * lv[c];
                p += met[c] ? e : 0.0;
            }
            p = list_sum_f64(p, t.ends);
            if (__builtin_amdgcn_inverse_ballot_w64(t.ends))
                acc[t.owner] += p;
        }
        if (any)
            hit[t.owner] = 1;
        wave_lds_order();
    }
}

// The lists' quads, the loads of a turn issued before the look-ups of the one before it.
template <bool SEMI, typename PROBE>
__device__ __forceinline__ void dot_walk(DotLists &lists, const PairSide &s, uint32_t *marks, int lane, const PROBE &probe,
                                         double *acc, int *hit, DotSemiring op, bool swapped)
{
    DotTurn a, b;
    lists.issue(a, 0, s, marks, lane);
    if (lists.Q <= 64) {
        dot_turn<SEMI>(a, probe, acc, hit, op, swapped);
        return;
    }
    int base = 0;
    do {
        lists.issue(b, base + 64, s, marks, lane);
        dot_turn<SEMI>(a, probe, acc, hit, op, swapped);
        lists.issue(a, base + 128, s, marks, lane);
        dot_turn<SEMI>(b, probe, acc, hit, op, swapped);
        base += 128;
    } while (base < lists.Q);
}

// ---------------------------------------------------------------------------
// Rows of long tables: a workgroup per part of a row.  Large graphs are bound by the lists' way from the memory-side cache:
// 200003 vertices, edge factor 16, 23.5 GB past the L2s in 3.2 ms, 7.3 TB/s, while parts took every so many'th list of a row.
// A part has the lists of a stretch of memory now (pair_ranges), and the parts are taken in the order of their stretches, an
// eighth of them by every XCD, so that its workgroups read about the same lists at about the same time: 36 % of the lines are
// in the L2 where 13 % were, 17.8 GB in 2.67 ms, the vector unit busy in three quarters of it.  Whole product, us, every
// so many'th list / by stretches: 200003 and 16 3505 / 2930, 260000 and 14 3085 / 2650, 120000 and 16 1565 / 1250, 90000 and 16
// 1295 / 1020, 260000 and 5 757 / 712, 60000 and 12 467 / 455.  (Without the order, a part of the lists for every XCD: eight
// times the tables, 4.0 ms.)  Smaller ones, whose lists the L2 holds, by the vector
// unit, busy two thirds of the time.  The first item of a workgroup is its own, not drawn: with one word to draw from, the
// last of 256 began 3 us after the first.  Whole product: n = 200003 21.7 -> 3.6 ms, 20351 0.70 -> 0.24.  With values
// read from LDS rather than by flat loads, sums over the lanes of a list by scalar masks, and two workgroups to a CU, us:
// 200003 and 16 3624 -> 3513, 60000 and 12 623 -> 473, 30000 and 8 228 -> 166, 16000 and 16 236 -> 169.
// The table is a bitmap in LDS with, beside every word (BIG: for
// every 8 words), the number of entries before it, so that a column's place in the row is that and the bits below; the
// row's values lie in LDS as well where they fit, behind the table.
// ---------------------------------------------------------------------------
typedef const __attribute__((address_space(3))) uint32_t dot_lds_word;
typedef const __attribute__((address_space(3))) uint64_t dot_lds_pair;
typedef const __attribute__((address_space(3))) double dot_lds_f64;

// IN_LDS: the row's values lie at byte vals_at of the LDS, else in memory.  (One pointer to either made every look at a
// value a flat load, which waits for all loads under way, the next turn's among them.)
template <bool BIG, bool IN_LDS>
struct RankProbe {                       // the table at address 0 of the LDS
    const uint32_t *before;              // BIG: of every 8 words
    uint32_t vals_at;
    const double *Tval;
    __device__ __forceinline__ void find(const int (&j)[4], uint32_t valid, bool (&met)[4], int (&at)[4]) const
    {
        uint32_t w[4], b[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            if constexpr (BIG) {
                w[c] = *reinterpret_cast<dot_lds_word *>((uint32_t)j[c] >> 5 << 2);
                b[c] = 0;
            } else {
                const uint64_t e = *reinterpret_cast<dot_lds_pair *>((uint32_t)j[c] >> 5 << 3);
                w[c] = (uint32_t)e;
                b[c] = (uint32_t)(e >> 32);
            }
        }
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const uint32_t k = (uint32_t)j[c] & 31u;
            met[c] = ((w[c] >> k) & (valid >> c) & 1u) != 0;
            int rank = (int)b[c] + __popc(w[c] & ((1u << k) - 1u));
            if constexpr (BIG) {
                if (met[c]) {
                    const uint32_t word = (uint32_t)j[c] >> 5, group = word >> 3;
                    rank += (int)before[group];
                    for (uint32_t x = group << 3; x < word; ++x)
                        rank += __popc(*reinterpret_cast<dot_lds_word *>(x << 2));
                }
            }
            at[c] = met[c] ? rank : 0;
        }
    }
    __device__ __forceinline__ void values(const int (&at)[4], double (&tv)[4]) const
    {
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            if constexpr (IN_LDS)
                tv[c] = *reinterpret_cast<dot_lds_f64 *>(vals_at + 8u * (uint32_t)at[c]);
            else
                tv[c] = Tval[at[c]];
        }
    }
};

template <int T>
struct DotHeavyShared {                  // in LDS behind the table
    double acc[T / 64][64];
    uint32_t marks[T / 64][2];
    int hit[T / 64][64];
    PairItem slot[2];
    int batch_next;
};

constexpr size_t DOT_LDS_MOST = 160 * 1024 - 256;
// words of LDS the table of ncols columns takes, and whether it is the one with a count for every 8 words only: where the
// other leaves no room for what lies behind it (from 0.6 M columns on).  fp64 values follow: an even number of words.
constexpr int dot_table_words(int64_t ncols, bool big)
{
    const int64_t words = (ncols + 31) / 32, groups = (words + 7) / 8;
    return (int)(big ? groups * 8 + (groups + 3) / 4 * 4 : (2 * words + 3) / 4 * 4);
}
constexpr bool dot_table_big(int64_t ncols)
{
    return sizeof(uint32_t) * (size_t)dot_table_words(ncols, false) + sizeof(DotHeavyShared<SG_T>) > DOT_LDS_MOST;
}
constexpr int dot_table_words(int64_t ncols) { return dot_table_words(ncols, dot_table_big(ncols)); }
static_assert(dot_table_words(1 << 20) * sizeof(uint32_t) + sizeof(DotHeavyShared<SG_T>) <= DOT_LDS_MOST,
              "the table of 2^20 columns fits LDS");

// Two workgroups of half the wavefronts to a CU, one building or clearing its table while the other looks up, where tables
// are small enough to leave the rows' values room in half the LDS and there are items enough for both.  us of the long
// rows, two / one: 100000 vertices, edge factor 8 394 / 433, 60000 and 16 524 / 555, 30000 and 8 110 / 128, 16000 and 16
// 128 / 150; 140000 and 10 1233 / 1088, 200003 and 16 3922 / 3192; few items: 8000 and 6 34 / 29, 5000 and 12 45 / 43.
constexpr int DOT_TWO_T = 512;
constexpr int64_t DOT_TWO_COLS = PAIR_RANGED_COLS;
constexpr size_t DOT_TWO_LDS_MOST = 80 * 1024 - 256;
static_assert(dot_table_words(DOT_TWO_COLS) * sizeof(uint32_t) + sizeof(DotHeavyShared<DOT_TWO_T>) <= DOT_TWO_LDS_MOST / 2,
              "half of a workgroup's LDS is left for values");

// pair_val, pair_hit: the result of a pair and whether a product met it, at the pair's place.
// nvals: values of a row that fit LDS behind the shared part
template <int T, bool BIG, bool SEMI>
__global__ __launch_bounds__(T, 4) void pair_dot_heavy_kernel(PairSide s0, PairSide s1, int table_words, int before_at, int nvals,
                                                              unsigned queues, unsigned long long *__restrict__ tickets,
                                                              double *__restrict__ pair_val,
                                                              uint8_t *__restrict__ pair_hit, DotSemiring op)
{
    uint32_t *tab = sg_dyn_lds;
    DotHeavyShared<T> &sh = *reinterpret_cast<DotHeavyShared<T> *>(sg_dyn_lds + table_words);
    double *vals = reinterpret_cast<double *>(&sh + 1);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    uint32_t *marks = sh.marks[wave];
    double *acc = sh.acc[wave];
    int *hit = sh.hit[wave];
    for (int w = threadIdx.x; w < table_words + (int)(sizeof sh / 4); w += T)
        sg_dyn_lds[w] = 0;
    __syncthreads();
    const uint32_t n0 = (uint32_t)(s0.counts[0] & 0xffffffff), n1 = (uint32_t)(s1.counts[0] & 0xffffffff);
    // the items in eighths, one to an XCD, whose workgroups draw from the others' when theirs are gone
    const unsigned long long items = (unsigned long long)n0 + n1;
    unsigned queue = blockIdx.x % queues;
    const auto begin = [&](unsigned q) { return items * q / queues; };
    const auto draw = [&]() -> PairItem {
        for (unsigned tries = 0; tries < queues; ++tries) {
            const unsigned long long own = (gridDim.x + queues - 1u - queue) / queues;
            const unsigned long long at = begin(queue) + own + atomicAdd(&tickets[queue], 1ull);
            if (at < begin(queue + 1))
                return pair_item<true>(s0, s1, n0, n1, at);
            queue = (queue + 1u) % queues;
        }
        return pair_item<true>(s0, s1, n0, n1, items);
    };
    if (threadIdx.x == 0) {
        const unsigned long long at = begin(queue) + blockIdx.x / queues;
        sh.slot[0] = at < begin(queue + 1) ? pair_item<true>(s0, s1, n0, n1, at) : draw();
    }
    __syncthreads();
    PairItem it = pair_item_read(sh.slot[0]);
    int cur = 0;
    uint32_t *before = tab + before_at;          // BIG
    while (it.index >= 0) {
        const PairSide s = it.side ? s1 : s0;
        const bool in_lds = it.tlen <= nvals;
        for (int t = threadIdx.x; t < it.tlen; t += T) {
            const int k = s.Tcrd[it.ts + t], prev = t > 0 ? s.Tcrd[it.ts + t - 1] : -1;
            if constexpr (BIG) {
                atomicOr(&tab[k >> 5], 1u << (k & 31));
                if (k >> 8 != prev >> 8)
                    before[k >> 8] = (uint32_t)t;
            } else {
                atomicOr(&tab[k >> 5 << 1], 1u << (k & 31));
                if (k >> 5 != prev >> 5)
                    tab[(k >> 5 << 1) + 1] = (uint32_t)t;
            }
            if (in_lds)
                vals[t] = s.Tval[it.ts + t];
        }
        if (threadIdx.x == 0)
            sh.batch_next = T / 64;
        lds_barrier();
        if (threadIdx.x == 0)
            sh.slot[cur ^ 1] = draw();
        const int mine = (it.kn + it.parts - 1) / it.parts;          // pairs of a part, about
        int B = mine / (4 * (T / 64));
        B = B > 64 ? 64 : B < 4 ? 4 : B;          // four lists fill a turn or two
        const int nb = (it.kn + B - 1) / B;
        PairEnt e;
        uint32_t place;
        const auto fetch = [&](int j) {          // past the last pair, that one: take() leaves it out
            const int64_t p = (int64_t)(it.part + it.parts * j) * B + lane;
            const int64_t q = it.ks + (p < it.kn ? p : it.kn - 1);
            e = s.ent[q];
            place = s.place[q];
        };
        const auto walk = [&](const auto &probe) {
            int j = wave;
            fetch(j);
            while (it.part + it.parts * j < nb) {
                const bool own = lane < B && (int64_t)(it.part + it.parts * j) * B + lane < it.kn;
                const uint32_t at = place;
                DotLists lists;
                lists.take(e.start, own ? (int)e.len : 0);
                int d = 0;
                if (lane == 0)
                    d = atomicAdd(&sh.batch_next, 1);
                j = __builtin_amdgcn_readfirstlane(d);
                fetch(j);          // the next batch's pairs arrive while this one is walked
                dot_walk<SEMI>(lists, s, marks, lane, probe, acc, hit, op, it.side != 0);
                if (own) {
                    pair_hit[at] = (uint8_t)hit[lane];
                    pair_val[at] = SEMI ? semiring_lds_value(reinterpret_cast<unsigned long long *>(acc)[lane], op.reduce_op,
                                                             op.mult_op, 0, nullptr, nullptr)
                                        : acc[lane];
                }
                acc[lane] = 0.0;
                hit[lane] = 0;
                wave_lds_order();
            }
        };
        const uint32_t vals_at = (uint32_t)sizeof(uint32_t) * (uint32_t)table_words + (uint32_t)sizeof sh;
        if (it.kn == 0) {          // no list of the row begins there
        } else if (in_lds)
            walk(RankProbe<BIG, true>{before, vals_at, nullptr});
        else
            walk(RankProbe<BIG, false>{before, 0, s.Tval + it.ts});
        lds_barrier();
        for (int t = threadIdx.x; t < it.tlen; t += T) {
            const int k = s.Tcrd[it.ts + t];
            tab[BIG ? k >> 5 : k >> 5 << 1] = 0;
        }
        cur ^= 1;
        it = pair_item_read(sh.slot[cur]);
        lds_barrier();
    }
}

// ---------------------------------------------------------------------------
// Rows of short tables: a wavefront per row, the row in buckets of four words (column + 1 and, above 21 bits, its place
// in the row); a full bucket's columns go on to the next.  A chain of look-ups of one wavefront, like the short rows of
// the summed form, with the next row's entries and pairs fetched ahead.
// ---------------------------------------------------------------------------
constexpr int DOT_LIGHT_WAVES = 4, DOT_LIGHT_OCC = 4;
static_assert(PAIR_LIGHT_MAX <= 1 << 11, "a place takes 11 bits");

struct PlaceProbe {
    const int *tab;
    int shift;               // 32 - log2 of the buckets
    const double *vals;
    __device__ __forceinline__ static int bucket(int j, int shift)
    {
        return (int)((uint32_t)__umul24((uint32_t)j, 0x9E3779u) >> shift);
    }
    __device__ __forceinline__ void find(const int (&j)[4], uint32_t valid, bool (&met)[4], int (&at)[4]) const
    {
        si_bucket k[4];
        int b[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            b[c] = bucket(j[c], shift);
            k[c] = *reinterpret_cast<const si_bucket *>(tab + 4 * b[c]);
        }
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const uint32_t key = (uint32_t)(j[c] + 1) << 11;
            const auto look = [&](si_bucket x) {
                const bool m0 = (uint32_t)x.x << 11 == key, m1 = (uint32_t)x.y << 11 == key, m2 = (uint32_t)x.z << 11 == key,
                           m3 = (uint32_t)x.w << 11 == key;
                at[c] = (int)((uint32_t)(m0 ? x.x : m1 ? x.y : m2 ? x.z : x.w) >> 21);
                met[c] = m0 | m1 | m2 | m3;
            };
            look(k[c]);
            bool on = !met[c] && k[c].w != 0 && (valid >> c & 1u);
            while (__any(on)) {
                if (on) {
                    b[c] = (b[c] + 1) & ((1 << (32 - shift)) - 1);
                    const si_bucket x = *reinterpret_cast<const si_bucket *>(tab + 4 * b[c]);
                    look(x);
                    on = !met[c] && x.w != 0;
                }
            }
            met[c] = met[c] && (valid >> c & 1u);
            at[c] = met[c] ? at[c] : 0;
        }
    }
    __device__ __forceinline__ void values(const int (&at)[4], double (&tv)[4]) const
    {
#pragma unroll
        for (int c = 0; c < 4; ++c)
            tv[c] = vals[at[c]];
    }
};

struct DotLightShared {
    int tab[4 << PAIR_LIGHT_LOG];
    double vals[PAIR_LIGHT_MAX];
    double acc[64];
    uint32_t marks[2];
    int hit[64];
};

// tickets: null, or those of the long rows' launch in front of this one, which it clears
template <bool SEMI>
__global__ __launch_bounds__(DOT_LIGHT_WAVES * 64, DOT_LIGHT_OCC) void pair_dot_light_kernel(
    PairSide s0, PairSide s1, unsigned long long *__restrict__ tickets, double *__restrict__ pair_val,
    uint8_t *__restrict__ pair_hit, DotSemiring op)
{
    if (tickets && blockIdx.x == 0 && threadIdx.x < 8)
        tickets[threadIdx.x] = 0;
    __shared__ __align__(16) DotLightShared all[DOT_LIGHT_WAVES];
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    DotLightShared &sh = all[wv];
    for (int b = lane; b < 1 << PAIR_LIGHT_LOG; b += 64)
        reinterpret_cast<si_bucket *>(sh.tab)[b] = si_bucket{0, 0, 0, 0};
    if (lane < 2)
        sh.marks[lane] = 0;
    sh.acc[lane] = 0.0;
    sh.hit[lane] = 0;
    wave_lds_order();
    const uint32_t n0 = (uint32_t)(s0.counts[0] >> 32), n1 = (uint32_t)(s1.counts[0] >> 32);
    const unsigned long long n = (unsigned long long)n0 + n1;
    // dealt out in advance, row i to wavefront i mod `waves`, which looks at 64 of its rows at a time
    const unsigned long long waves = (unsigned long long)gridDim.x * DOT_LIGHT_WAVES;
    const unsigned long long wave_id = blockIdx.x + (unsigned long long)gridDim.x * wv;
    for (unsigned long long tk = wave_id; tk < n; tk += 64 * waves) {
        const unsigned long long left = (n - 1 - tk) / waves + 1;
        const int nr = (int)(left < 64 ? left : 64);
        int64_t l_ts = 0, l_ks = 0;
        int l_tlen = 0, l_kn = 0;
        if (lane < nr) {
            const unsigned long long i = tk + lane * waves;
            const bool one = i >= n0;
            const int64_t *Tpos = one ? s1.Tpos : s0.Tpos, *kpos = one ? s1.kpos : s0.kpos;
            const int x = (one ? s1.light : s0.light)[one ? i - n0 : i];
            l_ts = Tpos[x];
            l_tlen = (int)(Tpos[x + 1] - l_ts);
            l_ks = kpos[x];
            l_kn = (int)(kpos[x + 1] - l_ks);
        }
        // the columns, the values and the first 64 pairs of the next row arrive while this one is walked
        constexpr int PER = (PAIR_LIGHT_MAX + 63) / 64;
        int jn[PER];
        double vn[PER];
        PairEnt en{0, 0};
        uint32_t pn = 0;
        const auto ahead = [&](int r) {
            const PairSide &s = tk + r * waves >= n0 ? s1 : s0;
            const int64_t ts = readlane_i64(l_ts, r), ks = readlane_i64(l_ks, r);
            const int tlen = __builtin_amdgcn_readlane(l_tlen, r), kn = __builtin_amdgcn_readlane(l_kn, r);
#pragma unroll
            for (int u = 0; u < PER; ++u) {
                const bool in = 64 * u + lane < tlen;
                jn[u] = in ? s.Tcrd[ts + 64 * u + lane] : -1;
                vn[u] = in ? s.Tval[ts + 64 * u + lane] : 0.0;
            }
            const int p = lane < kn ? lane : kn - 1;
            en = s.ent[ks + p];
            pn = s.place[ks + p];
        };
        ahead(0);
        for (int r = 0; r < nr; ++r) {
            const bool second = tk + r * waves >= n0;
            const PairSide s = second ? s1 : s0;
            const int64_t ks = readlane_i64(l_ks, r);
            const int tlen = __builtin_amdgcn_readlane(l_tlen, r), kn = __builtin_amdgcn_readlane(l_kn, r);
            PairEnt e = en;
            uint32_t place = pn;
            // as many buckets as keep them three quarters of a column full, 64 at least
            int log_nb = 6;
            while (log_nb < PAIR_LIGHT_LOG && tlen > (1 << log_nb) * 3 / 4)
                ++log_nb;
            const int shift = 32 - log_nb;
#pragma unroll
            for (int u = 0; u < PER; ++u) {
                if (jn[u] >= 0) {
                    const int place_in_row = 64 * u + lane, word = (jn[u] + 1) | place_in_row << 21;
                    sh.vals[place_in_row] = vn[u];
                    int b = PlaceProbe::bucket(jn[u], shift), x = 0;
                    while (atomicCAS(&sh.tab[4 * b + x], 0, word) != 0) {
                        x = (x + 1) & 3;
                        b = x == 0 ? (b + 1) & ((1 << log_nb) - 1) : b;
                    }
                }
            }
            wave_lds_order();
            if (r + 1 < nr)
                ahead(r + 1);
            const PlaceProbe probe{sh.tab, shift, sh.vals};
            for (int b = 0; b < kn; b += 64) {
                const bool own = b + lane < kn;
                const uint32_t at = place;
                DotLists lists;
                lists.take(e.start, own ? (int)e.len : 0);
                const int64_t q = ks + (b + 64 + lane < kn ? b + 64 + lane : kn - 1);
                e = s.ent[q];
                place = s.place[q];
                dot_walk<SEMI>(lists, s, sh.marks, lane, probe, sh.acc, sh.hit, op, second);
                if (own) {
                    pair_hit[at] = (uint8_t)sh.hit[lane];
                    pair_val[at] = SEMI ? semiring_lds_value(reinterpret_cast<unsigned long long *>(sh.acc)[lane],
                                                             op.reduce_op, op.mult_op, 0, nullptr, nullptr)
                                        : sh.acc[lane];
                }
                sh.acc[lane] = 0.0;
                sh.hit[lane] = 0;
                wave_lds_order();
            }
            for (int b = lane; b < 1 << log_nb; b += 64)
                reinterpret_cast<si_bucket *>(sh.tab)[b] = si_bucket{0, 0, 0, 0};
            wave_lds_order();
        }
    }
}

// pair_hit[p - Mpos[rb]] and, where it is set, pair_val for every stored pair p of the mask rows [rb, re),
// *pairs of them.
static int pair_dot_values(Csr *a, Csr *b, Csr *m, int64_t rb, int64_t re, double **pair_val, uint8_t **pair_hit, int64_t *pairs,
                           int reduce_op, int mult_op)
{
    const bool semi = reduce_op != COMET_SR_PLUS || mult_op != COMET_OP_TIMES;
    Csr *bt = nullptr;
    COMET_CHK(dot_transposed(b, &bt));
    PairPlan key;
    key.b_uid = b->uid;
    key.mask_uid = m->uid;
    key.kind = 0;
    key.first = rb;
    key.last = re;
    bool found = false;
    PairPlan *plan = pair_plan_slot(a, key, &found);
    if (!found) {
        const auto build = [&]() -> int {
            Csr *mt = nullptr;
            COMET_CHK(dot_transposed_index(m, &mt));
            int64_t *word = nullptr, ends[2];
            COMET_CHK(mailbox((void **)&word));
            COMET_CHK(pair_ends(m, rb, re, word, ends));
            plan->out0 = ends[0];
            plan->outs = ends[1] - ends[0];
            COMET_CHK(pair_side_plan(a, m, bt, rb, re, 0, 0, 1ll << 62, 0, PAIR_LIGHT_MAX, false, 1.0, true, nullptr, ends[0],
                                     &plan->side[0]));
            return pair_side_plan(bt, mt, a, 0, mt->nrows, 1, rb, re, 0, PAIR_LIGHT_MAX, false, 1.0, true, mt->val, ends[0],
                                  &plan->side[1]);
        };
        const int rc = build();
        if (rc != COMET_HIP_OK) {
            pair_plan_free(a->pair_plans.back());
            a->pair_plans.pop_back();
            return rc;
        }
    }
    const size_t outs = (size_t)(plan->outs > 0 ? plan->outs : 1);
    *pairs = plan->outs;
    COMET_CHK(g_dot_hit.ensure(outs, false));
    COMET_CHK(g_dot_val.ensure(sizeof(double) * outs, false));
    *pair_hit = (uint8_t *)g_dot_hit.ptr;
    *pair_val = (double *)g_dot_val.ptr;
    if (plan->outs == 0)
        return COMET_HIP_OK;
    if (plan->side[0].pairs + plan->side[1].pairs < plan->outs)          // pairs of an empty row or column are of no side
        COMET_HIPCHK(hipMemsetAsync(*pair_hit, 0, outs, stream()));
    const PairSide s0 = pair_side(plan->side[0], a, bt), s1 = pair_side(plan->side[1], bt, a);
    const int64_t nheavy = plan->side[0].nheavy + plan->side[1].nheavy, nlight = plan->side[0].nlight + plan->side[1].nlight;
    const DotSemiring op{reduce_op, mult_op};
    const bool beside = nheavy > 0 && nlight > 0 && plan->side[0].pairs + plan->side[1].pairs >= PAIR_BESIDE;
    if (beside)
        COMET_CHK(aux_fork());
    unsigned long long *kept = nullptr, *tickets = nullptr;
    if (nheavy > 0) {
        COMET_CHK(pair_tickets(&kept));
        tickets = kept;
        const bool big = dot_table_big(a->ncols);
        const int words = dot_table_words(a->ncols);
        const int before_at = (int)ceil_div(a->ncols, 256) * 8;
        const bool two = a->ncols <= DOT_TWO_COLS && nheavy >= 4 * (int64_t)num_cus();
        const size_t fixed = sizeof(uint32_t) * (size_t)words + (two ? sizeof(DotHeavyShared<DOT_TWO_T>) : sizeof(DotHeavyShared<SG_T>));
        const int nvals = (int)(((two ? DOT_TWO_LDS_MOST : DOT_LDS_MOST) - fixed) / sizeof(double)) & ~1;
        const size_t lds = fixed + sizeof(double) * (size_t)nvals;
        const dim3 grid((unsigned)std::min<int64_t>(nheavy, (int64_t)num_cus() * (two ? 2 : 1))), block(two ? DOT_TWO_T : SG_T);
        const unsigned queues = s0.ranged || s1.ranged ? 8 : 1;
        KernelTimer t("spgemm_numeric_dot");
#define LAUNCH_DOT(T, BIG, SEMI)                                                                                       \
    do {                                                                                                               \
        COMET_CHK(sg_allow_lds(pair_dot_heavy_kernel<T, BIG, SEMI>, lds));                                             \
        pair_dot_heavy_kernel<T, BIG, SEMI><<<grid, block, lds, stream()>>>(s0, s1, words, before_at, nvals, queues, tickets,  \
                                                                            *pair_val, *pair_hit, op);                 \
    } while (0)
        if (two && semi)
            LAUNCH_DOT(DOT_TWO_T, false, true);
        else if (two)
            LAUNCH_DOT(DOT_TWO_T, false, false);
        else if (big && semi)
            LAUNCH_DOT(SG_T, true, true);
        else if (big)
            LAUNCH_DOT(SG_T, true, false);
        else if (semi)
            LAUNCH_DOT(SG_T, false, true);
        else
            LAUNCH_DOT(SG_T, false, false);
#undef LAUNCH_DOT
        if (nlight == 0 || beside) {          // else the launch behind this one clears them
            COMET_HIPCHK(hipMemsetAsync(tickets, 0, 8 * sizeof *tickets, stream()));
            tickets = nullptr;
        }
    }
    if (nlight > 0) {
        const dim3 grid((unsigned)std::min<int64_t>(ceil_div(nlight, DOT_LIGHT_WAVES), (int64_t)num_cus() * DOT_LIGHT_OCC)),
            block(DOT_LIGHT_WAVES * 64);
        const hipStream_t on = beside ? aux_stream() : stream();
        KernelTimer t("spgemm_numeric_dot_small", on);
        if (semi)
            pair_dot_light_kernel<true><<<grid, block, 0, on>>>(s0, s1, tickets, *pair_val, *pair_hit, op);
        else
            pair_dot_light_kernel<false><<<grid, block, 0, on>>>(s0, s1, tickets, *pair_val, *pair_hit, op);
    }
    if (beside)
        COMET_CHK(aux_join());
    return pair_launched(kept);
}

// ---------------------------------------------------------------------------
// The pairs that met a product become the result, PAIR_CHUNK of the mask's entries at a time wherever its rows end (a
// wavefront per row took 0.47 ms of 7 M entries, eight times what their bytes do).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void dot_chunk_count(int64_t n, const uint8_t *__restrict__ pair_hit,
                                                       int64_t *__restrict__ chunk_kept)
{
    __shared__ int wave_count[4];
    const int64_t at = (int64_t)blockIdx.x * PAIR_CHUNK + 8 * (int64_t)threadIdx.x;
    int k = 0;
    if (at + 8 <= n)
        k = __popcll(*reinterpret_cast<const unsigned long long *>(pair_hit + at));          // bytes of 0 and 1
    else
        for (int64_t p = at; p < n; ++p)
            k += pair_hit[p];
    k = wave_sum_i32(k);
    if ((threadIdx.x & 63) == 0)
        wave_count[threadIdx.x >> 6] = k;
    __syncthreads();
    if (threadIdx.x == 0)
        chunk_kept[blockIdx.x] = wave_count[0] + wave_count[1] + wave_count[2] + wave_count[3];
}

// The same and where the chunks' pairs go, by one workgroup, four chunks to a wavefront: a launch in place of two.  us of a
// masked product with three launches behind its pairs / two, R-MAT: 500 vertices, edge factor 4 50.3 / 45.9, 2000 and 8 51.6 /
// 50.3, 5000 and 6 67.2 / 65.2; with 128 chunks, the workgroup's loads in two turns, 5000 and 16 89.1 / 90.2, with 256 20000
// and 8 140.6 / 145.7.
constexpr int DOT_PLACES_T = 1024, DOT_PLACES_U = 4, DOT_PLACES_MOST = DOT_PLACES_T / 64 * DOT_PLACES_U;
__global__ __launch_bounds__(DOT_PLACES_T) void dot_chunk_places(int64_t n, const uint8_t *__restrict__ pair_hit,
                                                                 int64_t *__restrict__ chunk_before, int64_t *total)
{
    __shared__ int kept[DOT_PLACES_MOST];
    static_assert(PAIR_CHUNK == 2 * 64 * sizeof(uint4) && DOT_PLACES_MOST == 64, "two loads of a lane to a chunk, a lane to a count");
    const int lane = threadIdx.x & 63, c0 = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)) * DOT_PLACES_U;
    const int full = (int)(n / PAIR_CHUNK), chunks = (int)((n + PAIR_CHUNK - 1) / PAIR_CHUNK);
    const uint4 *quads = reinterpret_cast<const uint4 *>(pair_hit);
    uint4 q[DOT_PLACES_U][2];
#pragma unroll
    for (int u = 0; u < DOT_PLACES_U; ++u)
#pragma unroll
        for (int h = 0; h < 2; ++h)
            q[u][h] = c0 + u < full ? quads[(c0 + u) * 128 + 64 * h + lane] : make_uint4(0, 0, 0, 0);
#pragma unroll
    for (int u = 0; u < DOT_PLACES_U; ++u) {
        int k = 0;
#pragma unroll
        for (int h = 0; h < 2; ++h)
            k += __popc(q[u][h].x) + __popc(q[u][h].y) + __popc(q[u][h].z) + __popc(q[u][h].w);          // bytes of 0 and 1
        if (c0 + u == full)          // what is left behind the last whole chunk
            for (int64_t at = (int64_t)full * PAIR_CHUNK + 8 * lane; at < n; at += 8 * 64)
                if (at + 8 <= n)
                    k += __popcll(*reinterpret_cast<const unsigned long long *>(pair_hit + at));
                else
                    for (int64_t p = at; p < n; ++p)
                        k += pair_hit[p];
        k = wave_sum_i32(k);
        if (lane == 0)
            kept[c0 + u] = k;
    }
    __syncthreads();
    if (c0 == 0) {
        const int k = kept[lane], inc = wave_inclusive_scan(k);
        if (lane < chunks)
            chunk_before[lane] = inc - k;
        if (lane == 63) {
            chunk_before[chunks] = inc;
            if (total)
                *total = inc;
        }
    }
}

// Cpos (or null): where the rows begin.
__global__ __launch_bounds__(256) void dot_chunk_compact(int64_t rb, int64_t re, const int64_t *__restrict__ Mpos,
                                                         const int32_t *__restrict__ Mcrd,
                                                         const double *__restrict__ pair_val,
                                                         const uint8_t *__restrict__ pair_hit,
                                                         const int64_t *__restrict__ chunk_before, int64_t *__restrict__ Cpos,
                                                         int32_t *__restrict__ Ccrd, double *__restrict__ Cval)
{
    constexpr int SEGS = PAIR_CHUNK / 64, PER = SEGS / 4;
    __shared__ unsigned long long bits[SEGS + 1];
    __shared__ int before[SEGS + 1];
    __shared__ int64_t bound[2];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t in0 = Mpos[rb], begin = (int64_t)blockIdx.x * PAIR_CHUNK, n = Mpos[re] - in0;
    const int count = (int)(n - begin < PAIR_CHUNK ? n - begin : PAIR_CHUNK);
    const bool at_end = begin + count == n;
    unsigned hits = 0;
#pragma unroll
    for (int u = 0; u < PER; ++u) {
        const int i = (wave * PER + u) * 64 + lane;
        const bool h = i < count && pair_hit[begin + i];
        hits |= (unsigned)h << u;
        const unsigned long long m = __ballot(h);
        if (lane == 0)
            bits[wave * PER + u] = m;
    }
    if (Cpos && wave < 2) {
        const int64_t x = wave == 1 && at_end ? re : pair_lower_bound(Mpos, rb, re, in0 + begin + (wave ? count : 0), lane);
        if (lane == 0)
            bound[wave] = x;
    }
    __syncthreads();
    if (wave == 0) {
        const int c = lane < SEGS ? __popcll(bits[lane]) : 0, inc = wave_inclusive_scan(c);
        if (lane <= SEGS)
            before[lane] = inc - c;
        if (lane == SEGS)
            bits[SEGS] = 0;
    }
    __syncthreads();
    const int64_t out = chunk_before[blockIdx.x];
    const auto rank = [&](int i) { return before[i >> 6] + __popcll(bits[i >> 6] & ((1ull << (i & 63)) - 1ull)); };
    if (Cpos) {
        for (int64_t x = bound[0] + threadIdx.x; x < bound[1]; x += 256)
            Cpos[x - rb] = out + rank((int)(Mpos[x] - in0 - begin));
        if (at_end && threadIdx.x == 0)
            Cpos[re - rb] = out + rank(count);
    }
#pragma unroll
    for (int u = 0; u < PER; ++u) {
        const int i = (wave * PER + u) * 64 + lane;
        if (hits >> u & 1u) {
            const int64_t o = out + rank(i), p = begin + i;
            Ccrd[o] = Mcrd[in0 + p];
            Cval[o] = pair_val[p];
        }
    }
}

// chunk_before[c]: pairs that met a product in front of chunk c of n; the number of all of them behind the last (and in
// total, a mailbox's word).
static int dot_chunks(int64_t n, const uint8_t *pair_hit, int64_t **chunk_before, int64_t *chunks, int64_t *total = nullptr)
{
    *chunks = ceil_div(n, PAIR_CHUNK);
    COMET_CHK(g_pair_chunk.ensure(sizeof(int64_t) * 2 * (size_t)(*chunks + 1), false));
    int64_t *kept = (int64_t *)g_pair_chunk.ptr;
    *chunk_before = kept + *chunks + 1;
    if (*chunks > 0 && *chunks <= DOT_PLACES_MOST) {
        KernelTimer t("spgemm_symbolic_dot_count");
        dot_chunk_places<<<dim3(1), dim3(DOT_PLACES_T), 0, stream()>>>(n, pair_hit, *chunk_before, total);
        COMET_HIPCHK(hipGetLastError());
        return COMET_HIP_OK;
    }
    if (*chunks > 0) {
        KernelTimer t("spgemm_symbolic_dot_count");
        dot_chunk_count<<<dim3((unsigned)*chunks), dim3(256), 0, stream()>>>(n, pair_hit, kept);
    }
    return exclusive_scan_i64(kept, *chunks, *chunk_before, total);
}
