// Masked products taken pair by pair: what their plans and kernels share, and the summed form (included by
// spgemm.hip, inside namespace comet, after the helpers of the product kernels).
//
// The work of both forms is a set of intersections: row x of one matrix (the "table") with a list, a row of another,
// for every list that x is paired with; an intersection costs the length of the list that is streamed against the
// table of the other.  Every pair is taken from the side whose row is the longer one, so it costs the shorter one's
// length:
//   SUM of C<M> = A*B, B a pattern matrix: sum over stored (i, k) of A of a_ik * b * |B_k and M_i|.  Side 0: table
//   M_i, lists B_k that are not longer; side 1: table B_k, lists M_i that are shorter, over the columns of A.
//   (Triangle count of the scale-20 R-MAT graph: 2.27 G look-ups instead of the 8.07 G of walking every B_k.)
//   C<M> = A*B: the dot product of A_i and column j of B for every stored (i, j) of M.  Side 0: table A_i, lists
//   the columns of B that are not longer; side 1: table column j, lists A_i that are shorter.
// The plan of a side keeps its pairs row by row as (first entry, length) of the list: a look at one array instead of
// two dependent ones, and no lane spent on pairs that belong to the other side.

struct PairEnt {
    uint32_t start, len;         // first entry of the list, number of entries
};
// Entries of a matrix that a PairEnt can name.  (The transposes that the plans are made from number them in 32 bits too,
// and a launch with a lane for each has to stay below 2^32 lanes.)
constexpr int64_t PAIR_NNZ_MAX = (1ll << 32) - (1 << 12);

// One side of a pair problem on the device.
struct PairSide {
    const int64_t *Tpos;
    const int32_t *Tcrd;
    const double *Tval;
    const int64_t *kpos;         // the pairs of row x: [kpos[x], kpos[x + 1])
    const PairEnt *ent;
    const double *weight;        // sum: A's value of the pair (null: one value for all, applied by the caller)
    const uint32_t *place;       // product: where the pair's result goes
    const int32_t *Lcrd;
    const double *Lval;
    uint32_t Lnnz;               // at least 4: a lane reads four columns at a time
    const uint2 *heavy;          // rows a workgroup takes, in parts: row, part | parts << 16
    const uint4 *ranged;         // product: the same as row and pairs [y, z) of the row; or null
    const int32_t *light;        // rows a wavefront takes
    const int64_t *counts;       // [0]: entries of heavy | entries of light << 32
};

// Rows of at most this many table entries are taken by a wavefront, in a bucket table of its own.
constexpr int PAIR_LIGHT_LOG = 8;                 // log2 of the buckets of four columns
constexpr int PAIR_LIGHT_MAX = (1 << PAIR_LIGHT_LOG) * 3 / 4;        // three quarters of a column per bucket
constexpr int PAIR_LIGHT_WORK = 8192;               // and of at most this many look-ups
constexpr int PAIR_LIST_COST = 8;                                    // what taking a list up costs, in look-ups
constexpr int64_t PAIR_ITEM_MIN = 16384;                             // look-ups a part of a row is worth at least
constexpr int64_t PAIR_SHARES = 2048;                                // parts that all the work would make, at most
// Products whose lists, columns and values, take more than this: parts by stretches of the lists.  Smaller lists are in the
// L2s by themselves (30000 vertices, edge factor 16, 10 MB 316 us, by stretches 344; 60000 and 12, 17 MB 467 / 455).  A part is
// worth 200,000 look-ups then, 140,000 where two workgroups share a CU (up to PAIR_RANGED_COLS columns) - a table is built
// and cleared for it -, us at 60,000 / 100,000 / 140,000 / 200,000: 160000 and 8 1091 / 1023 / 976 / 947, 260000 and 8 1309 / 1279
// / 1219 / 1184, 90000 and 16 1080 / 1063 / 1022 / 1041; and a 4096th of all at least (2048th, 8192th: 200003 and 16 3046,
// 3177 against 2935).  Beyond PAIR_RANGED_MOST columns the larger tables of more parts cost what the L2s save, ms without / by
// stretches, edge factor 16: 262144 3.92 / 3.45, 500000 10.6 / 10.1, 700000 35.3 / 34.2, 2^20 39.9 / 40.0; 2^20 and 8 12.2 / 12.3;
// a permuted graph of 2^20 34.2 / 35.6.
constexpr int64_t PAIR_RANGED_MOST = 3 << 18;
constexpr int64_t PAIR_RANGED_LISTS = 14 << 20, PAIR_RANGED_COLS = 1 << 17, PAIR_RANGED_TWO = 140000, PAIR_RANGED_ONE = 200000;
constexpr int64_t PAIR_RANGED_SHARES = 4096;

// strict 0: lists not longer than the table's row, 1: shorter ones, 2: all of them (no second side)
__device__ __forceinline__ bool pair_kept(int strict, int64_t len, int64_t tlen)
{
    return strict == 2 || (strict ? len < tlen : len <= tlen);
}

// The entries of P, rows [first, last), are looked at PAIR_CHUNK at a time wherever the rows end - a column of a power-law
// matrix has a hundred thousand times the entries of the next - and every kept one finds its place by counting those in
// front of it.  (A wavefront per row: 2.2 ms a pass for 15.7 M entries, all but 0.2 of it the longest row's.)
constexpr int PAIR_CHUNK = 2048;

// first x in [lo, hi) with pos[x] >= v, or hi: a wavefront's search, 64 steps at a time
__device__ __forceinline__ int64_t pair_lower_bound(const int64_t *__restrict__ pos, int64_t lo, int64_t hi, int64_t v,
                                                    int lane)
{
    while (hi > lo) {
        const int64_t step = (hi - lo + 63) / 64, x = lo + step * lane;
        // pos ascends: the lanes that see a smaller value are the first ones
        const int below = __popcll(__ballot(x < hi && pos[x] < v));
        if (below == 0)
            break;                                    // pos[lo] >= v
        const int64_t next = lo + step * (below - 1) + 1;
        hi = lo + step * below < hi ? lo + step * below : hi;
        lo = next;
    }
    return lo;
}

// FILL = false: of each chunk, the number of kept pairs and what they cost (look-ups, and PAIR_LIST_COST for every list).
// FILL = true: those are the sums over the chunks before; the kept pairs are written, and for every row where its pairs
// begin (kpos) and what all pairs before it cost (wpos).  With a pair go its weight, P's value times scale (sum), or where
// the result goes: p, or what perm says, less out0 (product).
// A pair is kept when its list is not empty, passes pair_kept, and its other index lies in [xlo, xhi).
template <bool FILL>
__global__ __launch_bounds__(256) void pair_pass(int64_t first, int64_t last, const int64_t *__restrict__ Tpos,
                                                 const int64_t *__restrict__ Ppos, const int32_t *__restrict__ Pcrd,
                                                 const int64_t *__restrict__ Lpos, int strict, int64_t xlo, int64_t xhi,
                                                 int64_t *__restrict__ chunk_kept, int64_t *__restrict__ chunk_work,
                                                 int64_t *__restrict__ kpos, int64_t *__restrict__ wpos,
                                                 PairEnt *__restrict__ ent, const double *__restrict__ Pval, double scale,
                                                 double *__restrict__ weight, const double *__restrict__ perm,
                                                 int64_t out0, uint32_t *__restrict__ place)
{
    constexpr int SEGS = PAIR_CHUNK / 64, PER = SEGS / 4;
    __shared__ int mark[PAIR_CHUNK];
    __shared__ int64_t bound[2];
    __shared__ int seg_row[SEGS], seg_kept[SEGS];
    __shared__ int64_t seg_work[SEGS];
    __shared__ int at_kept[FILL ? PAIR_CHUNK + 1 : 1];
    __shared__ int64_t at_work[FILL ? PAIR_CHUNK + 1 : 1];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t begin = Ppos[first] + (int64_t)blockIdx.x * PAIR_CHUNK, stop = Ppos[last];
    const int count = (int)(stop - begin < PAIR_CHUNK ? stop - begin : PAIR_CHUNK);
    const bool at_end = begin + count == stop;
    for (int i = threadIdx.x; i < PAIR_CHUNK; i += 256)
        mark[i] = 0;
    if (wave < 2) {
        // rows [bound[0], bound[1]) begin in this chunk; those that begin at the very end belong to the last one
        const int64_t x = wave == 1 && at_end ? last : pair_lower_bound(Ppos, first, last, begin + (wave ? count : 0), lane);
        if (lane == 0)
            bound[wave] = x;
    }
    __syncthreads();
    const int64_t rlo = bound[0], rhi = bound[1];
    for (int64_t x = rlo + threadIdx.x; x < rhi; x += 256) {
        const int64_t at = Ppos[x] - begin;
        if (at < count)
            atomicMax(&mark[at], (int)(x - rlo) + 1);          // of rows that begin at one entry the last one has it
    }
    __syncthreads();
    int row[PER];
#pragma unroll
    for (int u = 0; u < PER; ++u) {
        const int seg = wave * PER + u;
        row[u] = wave_inclusive_max(mark[seg * 64 + lane]);
        if (lane == 63)
            seg_row[seg] = row[u];
    }
    __syncthreads();
    int carry = 0;
    for (int s = 0; s < wave * PER; ++s)
        carry = seg_row[s] > carry ? seg_row[s] : carry;
    int64_t start[PER];
    int length[PER];
    int rank[PER];
    unsigned keeps = 0;
#pragma unroll
    for (int u = 0; u < PER; ++u) {
        const int seg = wave * PER + u, i = seg * 64 + lane;
        row[u] = row[u] > carry ? row[u] : carry;
        carry = __shfl(row[u], 63, 64);
        bool keep = false;
        start[u] = 0;
        length[u] = 0;
        if (i < count) {
            const int64_t x = rlo - 1 + row[u];
            const int64_t tlen = Tpos[x + 1] - Tpos[x];
            const int y = Pcrd[begin + i];
            start[u] = Lpos[y];
            const int64_t len = Lpos[y + 1] - start[u];
            length[u] = (int)len;
            keep = len > 0 && pair_kept(strict, len, tlen) && y >= xlo && y < xhi;
        }
        const unsigned long long m = __ballot(keep);
        rank[u] = __popcll(m & ((1ull << lane) - 1ull));
        keeps |= (unsigned)keep << u;
        int64_t w = keep ? (int64_t)length[u] + PAIR_LIST_COST : 0;
        if constexpr (FILL) {
            const int64_t own = w;
            for (int d = 1; d < 64; d <<= 1) {
                const int64_t o = __shfl_up(w, d, 64);
                w += lane >= d ? o : 0;
            }
            at_kept[i] = rank[u];
            at_work[i] = w - own;
            if (lane == 63)
                seg_work[seg] = w;
        } else {
            for (int d = 32; d > 0; d >>= 1)
                w += __shfl_down(w, d, 64);
            if (lane == 0)
                seg_work[seg] = w;
        }
        if (lane == 0)
            seg_kept[seg] = __popcll(m);
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        int k = 0;
        int64_t w = 0;
        for (int s = 0; s < SEGS; ++s) {
            const int ks = seg_kept[s];
            const int64_t ws = seg_work[s];
            seg_kept[s] = k;
            seg_work[s] = w;
            k += ks;
            w += ws;
        }
        if constexpr (FILL) {
            at_kept[PAIR_CHUNK] = k;
            at_work[PAIR_CHUNK] = w;
        } else {
            chunk_kept[blockIdx.x] = k;
            chunk_work[blockIdx.x] = w;
        }
    }
    if constexpr (FILL) {
        __syncthreads();
        const int64_t k0 = chunk_kept[blockIdx.x], w0 = chunk_work[blockIdx.x];
        for (int64_t x = rlo + threadIdx.x; x < rhi; x += 256) {
            const int at = (int)(Ppos[x] - begin);
            const int seg = at >> 6;
            kpos[x - first] = k0 + (at < count ? at_kept[at] + seg_kept[seg] : at_kept[PAIR_CHUNK]);
            wpos[x - first] = w0 + (at < count ? at_work[at] + seg_work[seg] : at_work[PAIR_CHUNK]);
        }
        if (at_end && threadIdx.x == 0) {
            kpos[last - first] = k0 + at_kept[PAIR_CHUNK];
            wpos[last - first] = w0 + at_work[PAIR_CHUNK];
        }
#pragma unroll
        for (int u = 0; u < PER; ++u) {
            const int seg = wave * PER + u;
            if (keeps >> u & 1u) {
                const int64_t o = k0 + seg_kept[seg] + rank[u], p = begin + seg * 64 + lane;
                ent[o] = PairEnt{(uint32_t)start[u], (uint32_t)length[u]};
                if (weight)
                    weight[o] = Pval[p] * scale;
                if (place)
                    place[o] = (uint32_t)((perm ? (int64_t)perm[p] : p) - out0);
            }
        }
    }
}

// The structure of a matrix turned over, the entries of a row in no order: count, scan, then place.
template <bool PLACE>
__global__ __launch_bounds__(256) void pair_turn(int64_t nrows, const int64_t *__restrict__ pos,
                                                 const int32_t *__restrict__ crd, unsigned long long *__restrict__ count,
                                                 int32_t *__restrict__ turned)
{
    const int lane = threadIdx.x & 63;
    const int64_t x = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (x >= nrows)
        return;
    for (int64_t p = pos[x] + lane; p < pos[x + 1]; p += 64) {
        const unsigned long long at = atomicAdd(&count[crd[p]], 1ull);
        if constexpr (PLACE)
            turned[at] = (int32_t)x;
    }
}

// How a row is taken: parts of a heavy row in the low half, 1 for a light one in the high half.  only: 0 by the
// table's length, 1 every row by workgroups, 2 every row by wavefronts.  A short table's row is light up to light_work
// look-ups whatever a part of a heavy one has.
__global__ void pair_parts(int64_t first, int64_t n, const int64_t *__restrict__ Tpos, const int64_t *__restrict__ kpos,
                           const int64_t *__restrict__ wpos, int only, int light_max, int64_t light_work,
                           int64_t shares, int64_t item_min, int64_t *__restrict__ packed)
{
    const int64_t x = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (x >= n)
        return;
    const int64_t kept = kpos[x + 1] - kpos[x], tlen = Tpos[first + x + 1] - Tpos[first + x];
    const int64_t work = wpos[x + 1] - wpos[x];
    int64_t v = 0;
    const int64_t share = wpos[n] / shares, target = share > item_min ? share : item_min;
    // a short table may be paired with a hundred thousand lists: no wavefront gets more than a fraction of a part
    const int64_t fraction = target / 8 < PAIR_LIGHT_WORK ? target / 8 : PAIR_LIGHT_WORK;
    const int64_t most_light = fraction > light_work ? fraction : light_work;
    if (kept > 0 && (only == 2 || (only == 0 && tlen <= light_max && work <= most_light))) {
        v = 1ll << 32;
    } else if (kept > 0) {
        // parts small enough that the last ones even out over the CUs, each of some wavefronts' worth of pairs
        const int64_t most = kept / 32 + 1;
        v = work / target + 1;
        v = v < most ? v : most;
        v = v < 32768 ? v : 32768;
    }
    packed[x] = v;
}

__global__ void pair_items(int64_t first, int64_t n, const int64_t *__restrict__ packed, const int64_t *__restrict__ off,
                           uint2 *__restrict__ heavy, int32_t *__restrict__ light, int64_t *__restrict__ counts)
{
    const int64_t x = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (x == 0)
        counts[0] = off[n];
    if (x >= n)
        return;
    const int64_t v = packed[x], o = off[x];
    if (v >> 32) {
        light[o >> 32] = (int32_t)(first + x);
    } else {
        for (int64_t q = 0; q < v; ++q)
            heavy[(o & 0xffffffff) + q] = make_uint2((unsigned)(first + x), (unsigned)q | (unsigned)(v << 16));
    }
}

// The parts of heavy rows cut where their lists lie: part q of v has the pairs whose lists begin in the q-th v-th of the lists'
// entries.  keys: the middle of that, in 2^20ths; a row in one part goes anywhere.
__global__ void pair_ranges(int64_t first, int64_t n, const int64_t *__restrict__ packed, const int64_t *__restrict__ off,
                            const int64_t *__restrict__ kpos, const PairEnt *__restrict__ ent, uint32_t Lnnz,
                            uint4 *__restrict__ ranged, uint64_t *__restrict__ keys, uint32_t *__restrict__ idx)
{
    const int64_t x = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (x >= n)
        return;
    const int64_t v = packed[x], ks = kpos[x], kn = kpos[x + 1] - ks;
    if (v >> 32)
        return;
    int64_t from = 0;
    for (int64_t q = 0; q < v; ++q) {
        int64_t to = kn;
        if (q + 1 < v) {          // first pair whose list begins at the bound or behind it
            const uint32_t bound = (uint32_t)((uint64_t)Lnnz * (uint64_t)(q + 1) / (uint64_t)v);
            int64_t lo = from;
            while (lo < to) {
                const int64_t mid = (lo + to) >> 1;
                if (ent[ks + mid].start < bound)
                    lo = mid + 1;
                else
                    to = mid;
            }
        }
        const int64_t at = (off[x] & 0xffffffff) + q;
        ranged[at] = make_uint4((unsigned)(first + x), (unsigned)from, (unsigned)to, 0);
        keys[at] = v > 1 ? (uint64_t)((2 * q + 1) * (1ll << 19) / v) : (uint64_t)((uint32_t)x * 0x9E3779B1u >> 12);
        idx[at] = (uint32_t)at;
        from = to;
    }
}

__global__ void pair_ranges_sorted(int64_t n, const uint4 *__restrict__ ranged, const uint32_t *__restrict__ idx,
                                   uint4 *__restrict__ sorted)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n)
        sorted[i] = ranged[idx[i]];
}

// ---------------------------------------------------------------------------
// The walk.  A wavefront holds up to 64 lists, one per lane, and streams them end to end: the lists are cut into quads
// of four columns, quad s of the whole goes to lane s mod 64, and four such rows of 64 quads are a turn.  Every lane
// has work whatever the lengths are - lists of twenty columns fill a load as well as lists of ten thousand - and the
// loads of a turn (4 KiB a wavefront) are issued before the look-ups of the turn before it.  Which list a quad
// belongs to comes from a mark that each list leaves at its first quad.
// ---------------------------------------------------------------------------
template <bool WEIGHTS, int ROWS>
struct QuadTurn {
    sg_i4u q[ROWS];
    int rows;                    // rows of 64 quads in it
    int wlo[WEIGHTS ? ROWS : 1], whi[WEIGHTS ? ROWS : 1];          // the lists' weights
    uint32_t mask[ROWS];            // which of the four columns are the list's
};

constexpr int QUAD_MARKS = 32;           // bytes of LDS a wavefront's marks take at most, zero between walks

// A row of 64 quads whose first lies at0 / 4 quads into the whole (at0: the lane's, four columns a quad): the list it
// belongs to, where to read four columns that hold it - further in front than it begins where the array would end - and
// which of the four are the list's; none where the quads have ended (there one place for all lanes is read).  m: the row's marks; before: lists that begin before
// the row, less one.
__device__ __forceinline__ void quad_place(uint2 m, uint32_t &before, int a0, int end, uint32_t at0, uint32_t most,
                                           int &owner, uint32_t &from, uint32_t &mask)
{
    owner = (int)__builtin_amdgcn_mbcnt_hi(m.y, __builtin_amdgcn_mbcnt_lo(m.x, before));
    before += __popc(m.x) + __popc(m.y);
    const uint32_t at = (uint32_t)lane_value(a0, owner) + at0;
    const int left = (int)((uint32_t)lane_value(end, owner) - at);          // right across 2^31 too
    from = left <= 0 ? 0u : at < most ? at : most;
    const int n = left < 0 ? 0 : left < 4 ? left : 4;
    mask = __builtin_amdgcn_ubfe(0xfu, 0, n) << ((at - from) & 31u);
}

// start, len, w: the lane's list and its weight; lanes without one (len 0) come after those with.  consume(turn) looks the
// columns of a turn up; the last turn stays in `pend`, whose loads are under way when the next walk - of more lists,
// against the same table - issues its own: the caller consumes it when there are no more.
// The list of a quad is the number of lists that begin at or before it, counted by mbcnt from a bit for each beginning.
// (A running maximum of list numbers over the lanes took three times the instructions: 1.67 ms for the long rows of the
// scale-20 graph instead of 1.49.)
template <bool WEIGHTS, int ROWS, typename CONSUME>
__device__ __forceinline__ void quad_walk(QuadTurn<WEIGHTS, ROWS> &pend, uint32_t start, int len, double w,
                                          const int32_t *__restrict__ Lcrd, uint32_t Lnnz, uint32_t *marks, int lane,
                                          CONSUME consume)
{
    const int quads = (len + 3) >> 2;
    const int inc = wave_inclusive_scan(quads), pre = inc - quads;
    const int Q = __builtin_amdgcn_readlane(inc, 63);
    const int a0 = (int)(start - 4u * (uint32_t)pre), end = (int)(start + (uint32_t)len);
    const uint32_t most = Lnnz - 4u;
    uint32_t before = 0;                 // lists that begin before this row of quads, less one
    for (int base = 0; base < Q; base += 64 * ROWS) {
        // a list that begins at quad s > 0 sets bit s - 1: the bits below a quad are the lists up to its own
        const uint32_t bit = (uint32_t)(pre - 1 - base);
        if (len > 0 && bit < 64u * ROWS)
            atomicOr(&marks[bit >> 5], 1u << (bit & 31u));
        wave_lds_order();
        uint2 m[ROWS];
#pragma unroll
        for (int r = 0; r < ROWS; ++r)
            m[r] = reinterpret_cast<const uint2 *>(marks)[r];
        wave_lds_order();
        if (lane < 2 * ROWS)
            marks[lane] = 0;
        QuadTurn<WEIGHTS, ROWS> now;
        now.rows = (Q - base + 63) >> 6 < ROWS ? (Q - base + 63) >> 6 : ROWS;
        const uint32_t at0 = 4u * (uint32_t)(base + lane);
#pragma unroll
        for (int r = 0; r < ROWS; ++r) {
            if (r < now.rows) {
                int owner;
                uint32_t from;
                quad_place(m[r], before, a0, end, at0 + 256u * r, most, owner, from, now.mask[r]);
                if constexpr (WEIGHTS) {
                    now.wlo[r] = lane_value(__double2loint(w), owner);
                    now.whi[r] = lane_value(__double2hiint(w), owner);
                }
                now.q[r] = *reinterpret_cast<const sg_i4u *>(Lcrd + from);
            }
        }
        wave_lds_order();
        consume(pend);
        pend = now;
    }
}

// ---------------------------------------------------------------------------
// The summed form.  hits: lane's number of look-ups that met the table.
// ---------------------------------------------------------------------------
// a bucket read or cleared as one 16-byte access; may_alias, because the same words are also written one at a
// time by atomicCAS through an int pointer, and without it the compiler is free to reorder the two kinds
typedef int si_bucket __attribute__((ext_vector_type(4), may_alias));
struct BucketProbe {
    const int *tab;
    uint32_t mult;
    int shift;               // 32 - log2 of the buckets
    __device__ __forceinline__ static int bucket(int j, uint32_t mult, int shift)
    {
        return (int)((uint32_t)__umul24((uint32_t)j, mult) >> shift);      // __umul24 returns int: shift it as unsigned
    }
    __device__ __forceinline__ uint32_t one(int j) const
    {
        const si_bucket b = *reinterpret_cast<const si_bucket *>(tab + 4 * bucket(j, mult, shift));
        return (b.x == j) | (b.y == j) | (b.z == j) | (b.w == j);
    }
};
struct BisectProbe {
    const int32_t *m;       // the table's row, ascending
    int n;
    __device__ __forceinline__ uint32_t one(int j) const
    {
        int lo = 0, hi = n;
        while (lo < hi) {
            const int mid = (lo + hi) >> 1;
            if (m[mid] < j)
                lo = mid + 1;
            else
                hi = mid;
        }
        return lo < n && m[lo] == j;
    }
};
struct BitmapProbe {                     // the bitmap at address 0 of the LDS: an addition less for a look-up
    __device__ __forceinline__ uint32_t one(int j) const
    {
        const uint32_t word = *reinterpret_cast<const __attribute__((address_space(3))) uint32_t *>((uint32_t)j >> 5 << 2);
        return __builtin_amdgcn_ubfe(word, (uint32_t)j, 1);          // five bits of the offset count
    }
};

// ONE: every pair weighs the same, the hits are counted; else part gains hits * weight, list by list (a list without
// hits adds nothing, whatever its weight: 0 * inf would be NaN).
template <bool ONE, int ROWS, typename PROBE>
__device__ __forceinline__ void sum_turn(const QuadTurn<!ONE, ROWS> &t, const PROBE &probe, uint32_t &hits, double &part)
{
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
        if (r < t.rows) {
            uint32_t met = probe.one(t.q[r].w);
            met = met << 1 | probe.one(t.q[r].z);
            met = met << 1 | probe.one(t.q[r].y);
            met = met << 1 | probe.one(t.q[r].x);
            const uint32_t h = __popc(met & t.mask[r]);
            if constexpr (ONE)
                hits += h;
            else if (h)
                part += (double)h * __hiloint2double(t.whi[r], t.wlo[r]);
        }
    }
}

// What a workgroup is about to take, fetched while the row before it is walked.
struct PairItem {
    int64_t ts, ks;
    int tlen, kn, part, parts, side, index;          // index < 0: nothing left
};
// RANGED: the sides may have their parts by stretches of the lists
template <bool RANGED>
__device__ __forceinline__ PairItem pair_item(const PairSide &s0, const PairSide &s1, uint32_t n0, uint32_t n1,
                                              unsigned long long tk)
{
    PairItem it;
    it.index = -1;
    if (tk < (unsigned long long)n0 + n1) {
        const bool one = tk >= n0;
        const int64_t *Tpos = one ? s1.Tpos : s0.Tpos, *kpos = one ? s1.kpos : s0.kpos;
        const unsigned long long at = one ? tk - n0 : tk;
        const uint4 *ranged = !RANGED ? nullptr : one ? s1.ranged : s0.ranged;
        it.side = one;
        it.index = (int)tk;
        uint32_t x;
        if (ranged) {
            const uint4 h = ranged[at];
            x = h.x;
            it.part = 0;
            it.parts = 1;
            it.ks = kpos[x] + h.y;
            it.kn = (int)(h.z - h.y);
        } else {
            const uint2 h = (one ? s1.heavy : s0.heavy)[at];
            x = h.x;
            it.part = (int)(h.y & 0xffffu);
            it.parts = (int)(h.y >> 16);
            it.ks = kpos[x];
            it.kn = (int)(kpos[x + 1] - it.ks);
        }
        it.ts = Tpos[x];
        it.tlen = (int)(Tpos[x + 1] - it.ts);
    }
    return it;
}
__device__ __forceinline__ PairItem pair_item_read(const PairItem &l)
{
    PairItem it;
    it.ts = uniform_i64_sg(l.ts);
    it.ks = uniform_i64_sg(l.ks);
    it.tlen = __builtin_amdgcn_readfirstlane(l.tlen);
    it.kn = __builtin_amdgcn_readfirstlane(l.kn);
    it.part = __builtin_amdgcn_readfirstlane(l.part);
    it.parts = __builtin_amdgcn_readfirstlane(l.parts);
    it.side = __builtin_amdgcn_readfirstlane(l.side);
    it.index = __builtin_amdgcn_readfirstlane(l.index);
    return it;
}

// The sum of the workgroups' hits, made as they end: each adds its own and an arrival to the word of its eighth, whose last
// adds the eighth's to one more word, whose last has the result and puts the words and the tickets back to zero.  Sums are
// below 2^53, of 2^32 pairs with as many columns as a bitmap in LDS, and 9 bits are left for the workgroups of an eighth, 224
// at most.  (Additions to one word take
// 14 ns each for all XCDs: 70 us for the 5120 wavefronts of the short rows alone, 18 for 1280 workgroups, 2 in eighths.
// A launch behind them that added up what they had written: 1.2 to 2 us a call more, triangle counts of 1000 vertices 18.1
// in place of 16.9, of 60000 72.1 in place of 70.6, of 400000 145.0 in place of 143.0.)
constexpr int PAIR_EIGHTHS = 8, PAIR_WORD_APART = 16;          // a cache line of 128 bytes to a word
constexpr int PAIR_WORDS = 8 + PAIR_WORD_APART * (PAIR_EIGHTHS + 1);
constexpr unsigned long long PAIR_ARRIVAL = 1ull << 55;
struct PairTotal {
    unsigned long long *words;        // 8 tickets, then the eighths' words and the last one; zero between calls
    unsigned blocks, first;           // workgroups of all launches that add, and of those in front of this one
    double each;                      // what a hit is worth
    double *result;
};
__device__ __forceinline__ void pair_block_hits(unsigned long long *wave_hits, unsigned long long hits, int waves,
                                                const PairTotal &t)
{
    for (int d = 32; d > 0; d >>= 1)
        hits += ((unsigned long long)(unsigned)__shfl_down((int)(hits >> 32), d, 64) << 32) +
                (unsigned long long)(unsigned)__shfl_down((int)(hits & 0xffffffffu), d, 64);
    if ((threadIdx.x & 63) == 0)
        wave_hits[threadIdx.x >> 6] = hits;
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long all = 0;
        for (int w = 0; w < waves; ++w)
            all += wave_hits[w];
        const unsigned eighth = (t.first + blockIdx.x) % PAIR_EIGHTHS;
        // adds what arrives to a word; whether it was the last of n, and then the sum
        const auto last = [&](unsigned which, unsigned n) {
            unsigned long long *word = t.words + 8 + PAIR_WORD_APART * which;
            const unsigned long long now = atomicAdd(word, all + PAIR_ARRIVAL) + all + PAIR_ARRIVAL;
            all = now & (PAIR_ARRIVAL - 1);
            if (now / PAIR_ARRIVAL != n)
                return false;
            __hip_atomic_store(word, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            return true;
        };
        if (last(eighth, (t.blocks + PAIR_EIGHTHS - 1 - eighth) / PAIR_EIGHTHS) &&
            last(PAIR_EIGHTHS, t.blocks < PAIR_EIGHTHS ? t.blocks : PAIR_EIGHTHS)) {
            t.words[0] = 0;
            *t.result = all ? (double)all * t.each : 0.0;
        }
    }
}

// tickets[0]: next heavy part; total: of the hits (ONE)
// The rows of long tables: a workgroup per part of a row, the table's row as a bitmap of nwords words in LDS.  The
// pairs of the part are dealt to the wavefronts in batches - as they come when hits are counted, in a fixed order
// when weights are added, so that the sum does not depend on scheduling.
// Bound by the lists' way from the memory-side cache (8.7 GB a call on the scale-20 graph, 5.6 TB/s) and, at two thirds
// of the LDS cycles, by the look-ups' bank conflicts; registers for two wavefronts' workgroups a CU keep both busy.
// Whole call, triangle counts: n = 2^20 4.8 -> 1.7 ms, 200003 1.1 -> 0.38, 20351 2.0 -> 0.13, 1000 0.22 -> 0.04.
struct PairHeavyShared {                 // in LDS behind the bitmap
    PairItem slot[2];
    double wave_part[SG_WAVES];
    unsigned long long wave_hits[SG_WAVES];
    alignas(16) uint32_t marks[SG_WAVES][QUAD_MARKS / 4];
    int batch_next;
};
template <bool ONE>
__global__ __launch_bounds__(SG_T) void pair_sum_heavy_kernel(PairSide s0, PairSide s1, int nwords,
                                                              unsigned long long *tickets, PairTotal total,
                                                              double *__restrict__ out)
{
    uint32_t *bm = sg_dyn_lds;
    PairHeavyShared &sh = *reinterpret_cast<PairHeavyShared *>(sg_dyn_lds + nwords);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    uint32_t *marks = sh.marks[wave];
    for (int w = threadIdx.x; w < nwords + (int)(sizeof sh / 4); w += SG_T)
        sg_dyn_lds[w] = 0;
    __syncthreads();
    const uint32_t n0 = (uint32_t)(s0.counts[0] & 0xffffffff), n1 = (uint32_t)(s1.counts[0] & 0xffffffff);
    if (threadIdx.x == 0)
        sh.slot[0] = pair_item<false>(s0, s1, n0, n1, blockIdx.x);
    __syncthreads();
    PairItem it = pair_item_read(sh.slot[0]);
    int cur = 0;
    uint32_t hits = 0;
    unsigned long long all_hits = 0;
    const BitmapProbe probe;
    while (it.index >= 0) {
        const PairSide s = it.side ? s1 : s0;
        for (int t = threadIdx.x; t < it.tlen; t += SG_T) {
            const uint32_t j = (uint32_t)s.Tcrd[it.ts + t];
            atomicOr(&bm[j >> 5], 1u << (j & 31u));
        }
        if (threadIdx.x == 0)
            sh.batch_next = SG_WAVES;
        lds_barrier();
        if (threadIdx.x == 0)
            sh.slot[cur ^ 1] = pair_item<false>(s0, s1, n0, n1, gridDim.x + atomicAdd(&tickets[0], 1ull));
        // batches of 64 pairs, or fewer where that leaves the wavefronts less than four each
        const int mine = (it.kn + it.parts - 1) / it.parts;          // pairs of a part, about
        int B = mine / (4 * SG_WAVES);
        B = B > 64 ? 64 : B < 2 ? 2 : B;
        const int nb = (it.kn + B - 1) / B;
        double part = 0.0;
        PairEnt e{0, 0};
        double w = 0.0;
        const auto fetch = [&](int j) {
            const int64_t p = (int64_t)(it.part + it.parts * j) * B + lane;
            e.len = 0;
            if (lane < B && p < it.kn) {
                e = s.ent[it.ks + p];
                if constexpr (!ONE)
                    w = s.weight[it.ks + p];
            }
        };
        QuadTurn<!ONE, 4> pend;
        pend.rows = 0;
        int j = wave;
        fetch(j);
        while (it.part + it.parts * j < nb) {
            const uint32_t bs = e.start;
            const int len = (int)e.len;
            const double wj = w;
            if constexpr (ONE) {
                int d = 0;
                if (lane == 0)
                    d = atomicAdd(&sh.batch_next, 1);
                j = __builtin_amdgcn_readfirstlane(d);
            } else {
                j += SG_WAVES;
            }
            fetch(j);          // the next batch's pairs arrive while this one is walked
            quad_walk<!ONE>(pend, bs, len, wj, s.Lcrd, s.Lnnz, marks, lane,
                            [&](const QuadTurn<!ONE, 4> &t) { sum_turn<ONE>(t, probe, hits, part); });
        }
        sum_turn<ONE>(pend, probe, hits, part);
        if constexpr (ONE) {
            all_hits += hits;
            hits = 0;
        } else {
            part = wave_sum_f64(part);
            if (lane == 0)
                sh.wave_part[wave] = part;
        }
        lds_barrier();
        if constexpr (!ONE) {
            if (threadIdx.x == 0) {
                double total = 0.0;
                for (int v = 0; v < SG_WAVES; ++v)
                    total += sh.wave_part[v];
                out[it.index] = total;
            }
        }
        for (int t = threadIdx.x; t < it.tlen; t += SG_T)
            bm[(uint32_t)s.Tcrd[it.ts + t] >> 5] = 0;
        cur ^= 1;
        it = pair_item_read(sh.slot[cur]);
        lds_barrier();
    }
    if constexpr (ONE)
        pair_block_hits(sh.wave_hits, all_hits, SG_WAVES, total);
}

// The rows of short tables: a wavefront per row, the table's row in buckets of four columns in LDS - a look-up is one
// 16-byte read and four compares, without a loop.  A row goes in if no bucket overflows; after three more multipliers
// it is searched by bisection in memory, as are rows longer than the table is meant for.  What takes the time is one
// wavefront's chain - the row's bounds, its columns and pairs, the lists - so the columns and pairs of the next row are
// fetched ahead, and every row's table goes through one LDS access a column.
constexpr int PAIR_LIGHT_ROWS = 2;
constexpr int PAIR_LIGHT_OCC = 5;             // workgroups of four wavefronts on a CU
constexpr int PAIR_LIGHT_WAVES = 4;

template <bool ONE>
__global__ __launch_bounds__(PAIR_LIGHT_WAVES * 64, PAIR_LIGHT_OCC) void pair_sum_light_kernel(
    PairSide s0, PairSide s1, PairTotal total, double *__restrict__ out)
{
    constexpr int NB = 1 << PAIR_LIGHT_LOG;
    __shared__ __align__(16) int table[PAIR_LIGHT_WAVES][NB * 4];
    __shared__ __align__(16) uint32_t all_marks[PAIR_LIGHT_WAVES][QUAD_MARKS / 4];
    __shared__ unsigned long long wave_hits[PAIR_LIGHT_WAVES];
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    int *tab = table[wv];
    uint32_t *marks = all_marks[wv];
    for (int b = lane; b < NB; b += 64)
        reinterpret_cast<si_bucket *>(tab)[b] = si_bucket{-1, -1, -1, -1};
    if (lane < QUAD_MARKS / 4)
        marks[lane] = 0;
    wave_lds_order();
    const uint32_t h0 = (uint32_t)(s0.counts[0] & 0xffffffff), h1 = (uint32_t)(s1.counts[0] & 0xffffffff);
    const uint32_t n0 = (uint32_t)(s0.counts[0] >> 32), n1 = (uint32_t)(s1.counts[0] >> 32);
    const unsigned long long n = (unsigned long long)n0 + n1;
    unsigned long long all_hits = 0;
    // Dealt out in advance, row i to wavefront i mod `waves`, which looks at 64 of its rows at a time.  A shared counter
    // costs more than it evens out: tens of thousands of draws at the 14 ns one of them takes (0.71 ms for the rows of
    // 200003 vertices, edge factor 16, instead of 0.19).
    const unsigned long long waves = (unsigned long long)gridDim.x * PAIR_LIGHT_WAVES;
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
        // the columns and the first 64 pairs of the next row arrive while this one is walked
        constexpr int PER = (PAIR_LIGHT_MAX + 63) / 64;
        int jn[PER];
        PairEnt en{0, 0};
        double wn = 0.0;
        const auto ahead = [&](int r) {
            const PairSide &s = tk + r * waves >= n0 ? s1 : s0;
            const int64_t ts = readlane_i64(l_ts, r), ks = readlane_i64(l_ks, r);
            const int tlen = __builtin_amdgcn_readlane(l_tlen, r), kn = __builtin_amdgcn_readlane(l_kn, r);
#pragma unroll
            for (int u = 0; u < PER; ++u)
                jn[u] = 64 * u + lane < tlen ? s.Tcrd[ts + 64 * u + lane] : -1;
            en.len = 0;
            if (lane < kn) {
                en = s.ent[ks + lane];
                if constexpr (!ONE)
                    wn = s.weight[ks + lane];
            }
        };
        ahead(0);
        for (int r = 0; r < nr; ++r) {
            const PairSide s = tk + r * waves >= n0 ? s1 : s0;
            const int64_t ts = readlane_i64(l_ts, r), ks = readlane_i64(l_ks, r);
            const int tlen = __builtin_amdgcn_readlane(l_tlen, r), kn = __builtin_amdgcn_readlane(l_kn, r);
            PairEnt e = en;
            double w = wn;
            int j[PER];
#pragma unroll
            for (int u = 0; u < PER; ++u)
                j[u] = jn[u];
            if (r + 1 < nr)
                ahead(r + 1);
            const auto fetch = [&](int b) {
                e.len = 0;
                if (b + lane < kn) {
                    e = s.ent[ks + b + lane];
                    if constexpr (!ONE)
                        w = s.weight[ks + b + lane];
                }
            };
            bool hashed = false;
            uint32_t mult = 0;
            // as many buckets as keep them three quarters of a column full, 64 at least
            int log_nb = 6;
            while (log_nb < PAIR_LIGHT_LOG && tlen > (1 << log_nb) * 3 / 4)
                ++log_nb;
            const int shift = 32 - log_nb;
            if (tlen <= PAIR_LIGHT_MAX) {
                for (int attempt = 0; attempt < 4 && !hashed; ++attempt) {
                    mult = attempt == 0 ? 0x9E3779u : attempt == 1 ? 0x85EBCBu : attempt == 2 ? 0xC2B2AFu : 0x27D4EBu;
                    bool placed = true;
#pragma unroll
                    for (int u = 0; u < PER; ++u) {
                        bool in = j[u] < 0;
                        if (!in) {
                            int *bk = tab + 4 * BucketProbe::bucket(j[u], mult, shift);
#pragma unroll
                            for (int x = 0; x < 4; ++x)
                                if (!in) {
                                    const int old = atomicCAS(&bk[x], -1, j[u]);
                                    in = old == -1 || old == j[u];
                                }
                        }
                        placed = placed && in;
                    }
                    hashed = !__any(!placed);
                    if (!hashed)
                        for (int b = lane; b < (1 << log_nb); b += 64)
                            reinterpret_cast<si_bucket *>(tab)[b] = si_bucket{-1, -1, -1, -1};
                }
            }
            double part = 0.0;
            uint32_t hits = 0;
            QuadTurn<!ONE, PAIR_LIGHT_ROWS> pend;
            pend.rows = 0;
            const auto walk = [&](const auto &probe) {
                for (int b = 0; b < kn; b += 64) {
                    const uint32_t bs = e.start;
                    const int len = (int)e.len;
                    const double wj = w;
                    fetch(b + 64);
                    quad_walk<!ONE>(pend, bs, len, wj, s.Lcrd, s.Lnnz, marks, lane,
                                    [&](const QuadTurn<!ONE, PAIR_LIGHT_ROWS> &t) { sum_turn<ONE>(t, probe, hits, part); });
                }
                sum_turn<ONE>(pend, probe, hits, part);
            };
            if (hashed)
                walk(BucketProbe{tab, mult, shift});
            else
                walk(BisectProbe{s.Tcrd + ts, tlen});
            if constexpr (ONE) {
                all_hits += hits;
            } else {
                part = wave_sum_f64(part);
                if (lane == 0)
                    out[h0 + h1 + tk + r * waves] = part;
            }
            if (hashed)
                for (int b = lane; b < (1 << log_nb); b += 64)
                    reinterpret_cast<si_bucket *>(tab)[b] = si_bucket{-1, -1, -1, -1};
            wave_lds_order();
        }
    }
    if constexpr (ONE)
        pair_block_hits(wave_hits, all_hits, PAIR_LIGHT_WAVES, total);
}

// partial[block] = sum of a fixed share of the rows' sums
__global__ __launch_bounds__(256) void pair_sum_partial(PairSide s0, PairSide s1, const double *__restrict__ out,
                                                        double *__restrict__ partial)
{
    __shared__ double lds[256];
    const auto both = [](int64_t c) { return (c & 0xffffffff) + (c >> 32); };
    const int64_t n = both(s0.counts[0]) + both(s1.counts[0]);
    double v = 0.0;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256)
        v += out[i];
    lds[threadIdx.x] = v;
    __syncthreads();
    for (int d = 128; d > 0; d >>= 1) {
        if ((int)threadIdx.x < d)
            lds[threadIdx.x] += lds[threadIdx.x + d];
        __syncthreads();
    }
    if (threadIdx.x == 0)
        partial[blockIdx.x] = lds[0];
}

// The result of 256 sums to the host's word, the ticket back to zero for the next call.
__global__ __launch_bounds__(256) void pair_sum_finish(unsigned long long *__restrict__ tickets,
                                                       const double *__restrict__ partial, double *__restrict__ result)
{
    __shared__ double lds[256];
    lds[threadIdx.x] = partial[threadIdx.x];
    __syncthreads();
    for (int d = 128; d > 0; d >>= 1) {
        if ((int)threadIdx.x < d)
            lds[threadIdx.x] += lds[threadIdx.x + d];
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        *result = lds[0];
        tickets[0] = 0;
    }
}

// ---------------------------------------------------------------------------
// Plans
// ---------------------------------------------------------------------------
static Workspace g_pair_range, g_pair_chunk, g_pair_row, g_pair_turn, g_pair_tickets, g_pair_out, g_pair_partial;

// pos[first] and pos[last] of x
static int pair_ends(const Csr *x, int64_t first, int64_t last, int64_t *word, int64_t *ends)
{
    if (first == 0 && last == x->nrows) {
        ends[0] = 0;
        ends[1] = x->nnz;
        return COMET_HIP_OK;
    }
    COMET_HIPCHK(hipMemcpyAsync(word, x->pos + first, sizeof(int64_t), hipMemcpyDeviceToHost, stream()));
    COMET_CHK(stream_wait());
    ends[0] = *(volatile int64_t *)word;
    COMET_HIPCHK(hipMemcpyAsync(word, x->pos + last, sizeof(int64_t), hipMemcpyDeviceToHost, stream()));
    COMET_CHK(stream_wait());
    ends[1] = *(volatile int64_t *)word;
    return COMET_HIP_OK;
}

constexpr int64_t PAIR_ROOM_UNSEEN = 1 << 18;
// From this number of pairs on the two kernels of a call run side by side: they leave each other room on the CUs, but the
// second stream starts some 40 us late, which only longer walks make up for (sums: 134 us one after the other and 154 side
// by side with 0.14 M pairs, 486 and 376 with 3.5 M, 1821 and 1648 with 15.6 M).
constexpr int64_t PAIR_BESIDE = 1 << 20;

// The plan of one side for rows [first, last) of T and P: built on the GPU.
// val: P's values become weights (times scale), or null; places: the results' places are kept.
static int pair_side_plan(const Csr *T, const Csr *P, const Csr *L, int64_t first, int64_t last, int strict, int64_t xlo,
                          int64_t xhi, int only, int light_max, bool weights, double scale, bool places,
                          const double *perm, int64_t out0, PairSidePlan *plan)
{
    const int64_t n = last - first;
    plan->first = first;
    if (n <= 0 || L->nnz == 0) {
        COMET_HIPCHK(dev_malloc((void **)&plan->counts, sizeof(int64_t)));
        COMET_HIPCHK(hipMemsetAsync(plan->counts, 0, sizeof(int64_t), stream()));
        return COMET_HIP_OK;
    }
    void *word = nullptr;
    COMET_CHK(mailbox(&word));
    int64_t ends[2];
    COMET_CHK(pair_ends(P, first, last, (int64_t *)word, ends));
    const int64_t entries = ends[1] - ends[0];
    if (entries == 0) {
        COMET_HIPCHK(dev_malloc((void **)&plan->counts, sizeof(int64_t)));
        COMET_HIPCHK(hipMemsetAsync(plan->counts, 0, sizeof(int64_t), stream()));
        return COMET_HIP_OK;
    }
    const int64_t chunks = ceil_div(entries, PAIR_CHUNK);
    COMET_CHK(g_pair_chunk.ensure(sizeof(int64_t) * 4 * (size_t)(chunks + 1), false));
    COMET_CHK(g_pair_row.ensure(sizeof(int64_t) * 2 * (size_t)(n + 1), false));
    int64_t *kept = (int64_t *)g_pair_chunk.ptr, *work = kept + chunks + 1, *kept_before = work + chunks + 1,
            *work_before = kept_before + chunks + 1;
    int64_t *wpos = (int64_t *)g_pair_row.ptr, *parts = wpos + n + 1;
    COMET_HIPCHK(dev_malloc((void **)&plan->kpos, sizeof(int64_t) * (size_t)(n + 1)));
    COMET_HIPCHK(dev_malloc((void **)&plan->counts, sizeof(int64_t)));
    const dim3 grid((unsigned)chunks), rows((unsigned)ceil_div(n, 256)), block(256);
    {
        KernelTimer t("spgemm_pair_plan");
        pair_pass<false><<<grid, block, 0, stream()>>>(first, last, T->pos, P->pos, P->crd, L->pos, strict, xlo, xhi, kept,
                                                       work, nullptr, nullptr, nullptr, nullptr, 0.0, nullptr, nullptr, 0,
                                                       nullptr);
    }
    COMET_CHK(exclusive_scan_i64(kept, chunks, kept_before));
    COMET_CHK(exclusive_scan_i64(work, chunks, work_before));
    // room for all entries where that is little; else the host waits for their number
    int64_t npairs = entries;
    if (entries > PAIR_ROOM_UNSEEN) {
        COMET_HIPCHK(hipMemcpyAsync(word, kept_before + chunks, sizeof(int64_t), hipMemcpyDeviceToHost, stream()));
        COMET_CHK(stream_wait());
        npairs = *(volatile int64_t *)word;
    }
    plan->pairs = npairs;
    COMET_HIPCHK(dev_malloc((void **)&plan->ent, sizeof(PairEnt) * (size_t)(npairs > 0 ? npairs : 1)));
    if (weights)
        COMET_HIPCHK(dev_malloc((void **)&plan->weight, sizeof(double) * (size_t)(npairs > 0 ? npairs : 1)));
    if (places)
        COMET_HIPCHK(dev_malloc((void **)&plan->place, sizeof(uint32_t) * (size_t)(npairs > 0 ? npairs : 1)));
    pair_pass<true><<<grid, block, 0, stream()>>>(first, last, T->pos, P->pos, P->crd, L->pos, strict, xlo, xhi, kept_before,
                                                  work_before, plan->kpos, wpos, (PairEnt *)plan->ent, P->val, scale,
                                                  plan->weight, perm, out0, plan->place);
    const bool ranged = places && T->ncols <= PAIR_RANGED_MOST && L->nnz * (int64_t)(sizeof(int32_t) + sizeof(double)) > PAIR_RANGED_LISTS;
    const int64_t item_min = !ranged ? PAIR_ITEM_MIN : T->ncols <= PAIR_RANGED_COLS ? PAIR_RANGED_TWO : PAIR_RANGED_ONE;
    pair_parts<<<rows, block, 0, stream()>>>(first, n, T->pos, plan->kpos, wpos, only, light_max, 0,
                                             ranged ? PAIR_RANGED_SHARES : PAIR_SHARES, item_min, parts);
    COMET_CHK(exclusive_scan_i64(parts, n, wpos));
    COMET_HIPCHK(hipMemcpyAsync(word, wpos + n, sizeof(int64_t), hipMemcpyDeviceToHost, stream()));
    if (npairs == entries)          // what was room is a number
        COMET_HIPCHK(hipMemcpyAsync((int64_t *)word + 1, kept_before + chunks, sizeof(int64_t), hipMemcpyDeviceToHost, stream()));
    COMET_CHK(stream_wait());
    const int64_t packed = *(volatile int64_t *)word;
    if (npairs == entries)
        plan->pairs = *((volatile int64_t *)word + 1);
    plan->nheavy = packed & 0xffffffff;
    plan->nlight = packed >> 32;
    COMET_HIPCHK(dev_malloc((void **)&plan->heavy, sizeof(uint2) * (size_t)(plan->nheavy > 0 ? plan->nheavy : 1)));
    COMET_HIPCHK(dev_malloc((void **)&plan->light, sizeof(int32_t) * (size_t)(plan->nlight > 0 ? plan->nlight : 1)));
    pair_items<<<rows, block, 0, stream()>>>(first, n, parts, wpos, (uint2 *)plan->heavy, plan->light, plan->counts);
    COMET_HIPCHK(hipGetLastError());
    if (ranged && plan->nheavy > 0) {          // without memory for them the parts stay as pair_items has them
        const auto ranges = [&]() -> int {
            const size_t items = (size_t)plan->nheavy;
            COMET_CHK(g_pair_range.ensure((sizeof(uint4) + 2 * sizeof(uint64_t) + 2 * sizeof(uint32_t)) * items, false));
            COMET_HIPCHK(dev_malloc((void **)&plan->ranged, sizeof(uint4) * items));
            uint4 *list = (uint4 *)g_pair_range.ptr;
            uint64_t *keys = (uint64_t *)(list + items);
            uint32_t *idx = (uint32_t *)(keys + 2 * items);
            pair_ranges<<<rows, block, 0, stream()>>>(first, n, parts, wpos, plan->kpos, (const PairEnt *)plan->ent, (uint32_t)L->nnz,
                                                      list, keys, idx);
            COMET_CHK(sort_pairs_u64_u32(keys, keys + items, idx, idx + items, plan->nheavy, 20));
            pair_ranges_sorted<<<dim3((unsigned)ceil_div(plan->nheavy, 256)), block, 0, stream()>>>(
                plan->nheavy, list, idx + items, (uint4 *)plan->ranged);
            return COMET_HIP_OK;
        };
        if (!plan_made(ranges)) {
            (void)dev_free(plan->ranged);
            plan->ranged = nullptr;
        }
    }
    if (L->nnz < 4) {          // a lane reads four columns at a time
        constexpr size_t room = 4 * (sizeof(double) + sizeof(int32_t));
        COMET_HIPCHK(dev_malloc((void **)&plan->padded, room));
        COMET_HIPCHK(hipMemsetAsync(plan->padded, 0, room, stream()));
        COMET_HIPCHK(hipMemcpyAsync(plan->padded, L->val, sizeof(double) * (size_t)L->nnz, hipMemcpyDeviceToDevice, stream()));
        COMET_HIPCHK(hipMemcpyAsync(plan->padded + 4, L->crd, sizeof(int32_t) * (size_t)L->nnz, hipMemcpyDeviceToDevice,
                                    stream()));
    }
    COMET_HIPCHK(hipGetLastError());
    return COMET_HIP_OK;
}

static PairSide pair_side(const PairSidePlan &p, const Csr *T, const Csr *L)
{
    PairSide s;
    s.Tpos = T->pos;
    s.Tcrd = T->crd;
    s.Tval = T->val;
    s.kpos = p.kpos ? p.kpos - p.first : nullptr;
    s.ent = (const PairEnt *)p.ent;
    s.weight = p.weight;
    s.place = p.place;
    s.Lcrd = p.padded ? reinterpret_cast<const int32_t *>(p.padded + 4) : L->crd;
    s.Lval = p.padded ? p.padded : L->val;
    s.Lnnz = p.padded ? 4u : (uint32_t)L->nnz;
    s.heavy = (const uint2 *)p.heavy;
    s.ranged = (const uint4 *)p.ranged;
    s.light = p.light;
    s.counts = p.counts;
    return s;
}

// The plan kept in A's handle for these matrices, range and mode, or room for a new one (its sides empty).
constexpr size_t PAIR_PLANS_KEPT = 4;
static PairPlan *pair_plan_slot(Csr *a, const PairPlan &key, bool *found)
{
    for (PairPlan &p : a->pair_plans)
        if (p.b_uid == key.b_uid && p.mask_uid == key.mask_uid && p.kind == key.kind && p.first == key.first &&
            p.last == key.last) {
            *found = true;
            return &p;
        }
    *found = false;
    if (a->pair_plans.size() >= PAIR_PLANS_KEPT) {
        pair_plan_free(a->pair_plans.front());
        a->pair_plans.erase(a->pair_plans.begin());
    }
    a->pair_plans.push_back(key);
    return &a->pair_plans.back();
}

static int pair_tickets(unsigned long long **tickets)
{
    COMET_CHK(g_pair_tickets.ensure(PAIR_WORDS * sizeof(unsigned long long), true));          // a call's last workgroup or kernel clears them
    *tickets = (unsigned long long *)g_pair_tickets.ptr;
    return COMET_HIP_OK;
}

// After the launches of a call: one that failed leaves the tickets that the others drew, or their hits, behind (null: it has
// drawn none).
static int pair_launched(unsigned long long *tickets)
{
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess && tickets)
        (void)hipMemsetAsync(tickets, 0, PAIR_WORDS * sizeof *tickets, stream());
    COMET_HIPCHK(e);
    return COMET_HIP_OK;
}

// Whether the matrices can be walked pair by pair: entries are named in 32 bits, and so is the length of 64 lists end to
// end (lists without duplicates are not longer than the bitmap is wide).
static int pair_form_fits(const Csr *a, const Csr *b, const Csr *m, bool *fits)
{
    const int64_t most = std::max(a->nnz, std::max(b->nnz, m->nnz));
    bool ok_b = true, ok_m = true;
    if (most > (1ll << 26) && most <= PAIR_NNZ_MAX) {
        COMET_CHK(dot_no_duplicates(b, &ok_b));
        COMET_CHK(dot_no_duplicates(m, &ok_m));
    }
    *fits = most <= PAIR_NNZ_MAX && ok_b && ok_m;
    return COMET_HIP_OK;
}

// pos and crd of A turned over, in workspaces.
static int pair_turned(const Csr *a, Csr *turned)
{
    const size_t n = (size_t)a->ncols + 1;
    COMET_CHK(g_pair_turn.ensure(sizeof(int64_t) * 2 * n + sizeof(int32_t) * (size_t)(a->nnz + 1), false));
    int64_t *pos = (int64_t *)g_pair_turn.ptr, *count = pos + n;
    int32_t *crd = (int32_t *)(count + n);
    COMET_HIPCHK(hipMemsetAsync(count, 0, sizeof(int64_t) * n, stream()));
    const dim3 grid((unsigned)ceil_div(a->nrows, 4)), block(256);
    pair_turn<false><<<grid, block, 0, stream()>>>(a->nrows, a->pos, a->crd, (unsigned long long *)count, crd);
    COMET_CHK(exclusive_scan_i64(count, a->ncols, pos));
    COMET_HIPCHK(hipMemcpyAsync(count, pos, sizeof(int64_t) * n, hipMemcpyDeviceToDevice, stream()));
    pair_turn<true><<<grid, block, 0, stream()>>>(a->nrows, a->pos, a->crd, (unsigned long long *)count, crd);
    COMET_HIPCHK(hipGetLastError());
    turned->nrows = a->ncols;
    turned->ncols = a->nrows;
    turned->nnz = a->nnz;
    turned->pos = pos;
    turned->crd = crd;
    return COMET_HIP_OK;
}

// Whether every row is sent one way: 1 to workgroups, 2 to wavefronts (the tests send each class of rows through both).
static int pair_only()
{
    const char *env = getenv("COMET_HIP_MASKED_SUM_ONLY");
    return !env ? 0 : strcmp(env, "workgroup") == 0 ? 1 : strcmp(env, "wavefront") == 0 ? 2 : 0;
}

// Workgroups of the two kernels of a sum, and the LDS of those of the long rows.
struct PairGrids {
    unsigned heavy, light;
    int nwords;
    size_t lds;
};
static PairGrids pair_grids(int64_t nheavy, int64_t nlight, int64_t ncols)
{
    PairGrids g;
    g.nwords = (int)ceil_div(ceil_div(ncols, 32), 4) * 4;
    g.lds = sizeof(uint32_t) * (size_t)g.nwords + sizeof(PairHeavyShared);
    const int per_cu = (int)std::max<size_t>(1, std::min<size_t>(2, (size_t)(150 * 1024) / g.lds));
    g.heavy = (unsigned)std::min<int64_t>(nheavy, (int64_t)num_cus() * per_cu);
    g.light = (unsigned)std::min<int64_t>(ceil_div(nlight, PAIR_LIGHT_WAVES), (int64_t)num_cus() * PAIR_LIGHT_OCC);
    return g;
}

// SUM of C<M> = A*B for a pattern matrix B (every value is b->iso_value).
static int pair_masked_sum(Csr *a, Csr *b, Csr *m, double *result)
{
    const int only = pair_only();
    bool one = false;
    COMET_CHK(csr_is_iso(a, &one));
    PairPlan key;
    key.b_uid = b->uid;
    key.mask_uid = m->uid;
    key.kind = 1 + only;
    key.first = 0;
    key.last = a->nrows;
    bool found = false;
    PairPlan *plan = pair_plan_slot(a, key, &found);
    if (!found) {
        const auto build = [&]() -> int {
            // a column stored twice counts twice as a product's and once as the mask's: no swapping sides then
            bool ok_b = false, ok_m = false;
            COMET_CHK(dot_no_duplicates(b, &ok_b));
            COMET_CHK(dot_no_duplicates(m, &ok_m));
            const bool both = ok_b && ok_m;
            const int64_t all = 1ll << 62;
            COMET_CHK(pair_side_plan(m, a, b, 0, a->nrows, both ? 0 : 2, 0, all, only, PAIR_LIGHT_MAX, !one, b->iso_value,
                                     false, nullptr, 0, &plan->side[0]));
            if (both) {
                // Which row of A an entry of a column comes from is all that counting hits asks for: in any order, and
                // that takes 6 launches instead of a sort's 25 (a first call on 1000 rows 0.42 -> 0.30 ms).  A long
                // column's atomics would wait for each other.
                Csr *at = nullptr, turned;
                if (one && a->nnz <= PAIR_ROOM_UNSEEN) {
                    COMET_CHK(pair_turned(a, &turned));
                    at = &turned;
                } else {
                    COMET_CHK(dot_transposed(a, &at));
                }
                COMET_CHK(pair_side_plan(b, at, m, 0, at->nrows, 1, 0, all, only, PAIR_LIGHT_MAX, !one, b->iso_value,
                                         false, nullptr, 0, &plan->side[1]));
            } else {
                COMET_CHK(pair_side_plan(b, a, m, 0, 0, 1, 0, all, only, PAIR_LIGHT_MAX, false, 1.0, false, nullptr, 0,
                                         &plan->side[1]));
            }
            return COMET_HIP_OK;
        };
        const int rc = build();
        if (rc != COMET_HIP_OK) {
            pair_plan_free(a->pair_plans.back());
            a->pair_plans.pop_back();
            return rc;
        }
    }
    const PairSide s0 = pair_side(plan->side[0], m, b), s1 = pair_side(plan->side[1], b, m);
    const int64_t nheavy = plan->side[0].nheavy + plan->side[1].nheavy, nlight = plan->side[0].nlight + plan->side[1].nlight;
    unsigned long long *tickets = nullptr;
    double *out = nullptr, *partial = nullptr, *word = nullptr;
    COMET_CHK(pair_tickets(&tickets));
    COMET_CHK(mailbox((void **)&word));
    if (!one) {
        COMET_CHK(g_pair_out.ensure(sizeof(double) * (size_t)(nheavy + nlight + 1), false));
        COMET_CHK(g_pair_partial.ensure(sizeof(double) * 256, false));
        out = (double *)g_pair_out.ptr;
        partial = (double *)g_pair_partial.ptr;
    }
    const bool beside = nheavy > 0 && nlight > 0 && plan->side[0].pairs + plan->side[1].pairs >= PAIR_BESIDE;
    const PairGrids grids = pair_grids(nheavy, nlight, b->ncols);
    PairTotal total{tickets, grids.heavy + grids.light, 0, a->iso_value * b->iso_value, word};
    if (one && total.blocks == 0) {
        *result = 0.0;
        return COMET_HIP_OK;
    }
    if (beside)
        COMET_CHK(aux_fork());
    if (nheavy > 0) {
        const int nwords = grids.nwords;
        const size_t lds = grids.lds;
        const dim3 grid(grids.heavy), block(SG_T);
        KernelTimer t("spgemm_masked_sum");
        if (one) {
            COMET_CHK(sg_allow_lds(pair_sum_heavy_kernel<true>, lds));
            pair_sum_heavy_kernel<true><<<grid, block, lds, stream()>>>(s0, s1, nwords, tickets, total, out);
        } else {
            COMET_CHK(sg_allow_lds(pair_sum_heavy_kernel<false>, lds));
            pair_sum_heavy_kernel<false><<<grid, block, lds, stream()>>>(s0, s1, nwords, tickets, total, out);
        }
    }
    if (nlight > 0) {
        const dim3 grid(grids.light), block(PAIR_LIGHT_WAVES * 64);
        const hipStream_t on = beside ? aux_stream() : stream();
        KernelTimer t("spgemm_masked_sum_small", on);
        total.first = grids.heavy;
        if (one)
            pair_sum_light_kernel<true><<<grid, block, 0, on>>>(s0, s1, total, out);
        else
            pair_sum_light_kernel<false><<<grid, block, 0, on>>>(s0, s1, total, out);
    }
    if (beside)
        COMET_CHK(aux_join());
    if (!one) {
        KernelTimer t("spgemm_masked_sum_reduce");
        pair_sum_partial<<<dim3(256), dim3(256), 0, stream()>>>(s0, s1, out, partial);
    }
    if (!one)
        pair_sum_finish<<<dim3(1), dim3(256), 0, stream()>>>(tickets, partial, word);
    COMET_CHK(pair_launched(tickets));
    COMET_CHK(stream_wait());
    *result = *(volatile double *)word;
    return COMET_HIP_OK;
}
