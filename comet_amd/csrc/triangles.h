// Triangle counts: SUM of C<L> = L*L for one strictly triangular matrix L of equal values (included by spgemm.hip after
// masked_pairs.h).  What is counted are the triangles of the graph with an edge for every entry, and their number does not
// depend on how the vertices are called.  So they get new numbers, most edges first, and every vertex a row: its neighbours
// with smaller numbers.  Nobody has many of those - 672 at most for the R-MAT graph of 2^20 vertices, where rows of L have
// up to 20698 entries -, and they are close together, because a few thousand vertices are most of all neighbours.
// Rows are therefore kept as words: the number of a group of sixteen vertices and a bit for each of them.  A triangle is
// an edge and a vertex that both ends' rows hold; an edge costs the words of the shorter row, looked up in a table of the
// longer one, and a word is a look-up for all its vertices: 1.1 G look-ups of 4 bytes instead of 2.3 G.
// A graph whose rows of L are about equally long keeps its numbers: there are no hubs to bring together, its rows are as
// short as they would be, and neighbours that lie next to each other stay there.
// The plan is made at the first count, in the place of the plan of L's pairs, which costs as much or more: us of a first
// count / of each one after it, this form | the pairs of L as it is, R-MAT with 16 edges a vertex: n = 2^20 4140 / 792 | 4430 /
// 1555, 200003 1120 / 161 | 1165 / 324, 60000 605 / 72 | 685 / 161, 20351 440 / 46 | 500 / 81, 1000 190 / 18 | 205 / 40; rows
// about equally long, uniform edges, 300000 vertices and 16 a vertex 865 / 166 | 1290 / 208, 30000 and 3 153 / 26 | 230 / 28,
// 5000 and 40 158 / 38 | 235 / 45, 1000 and 10 114 / 18 | 170 / 18, a triangulated mesh of 10^6 1000 / 428 | 1230 / 420, a
// band of 32 diagonals, 300000 1330 / 148 | 2800 / 1185.
// Bound by the rows' way from the memory-side cache for large graphs (5 TB/s), by the chain of a wavefront - bounds of a
// row, its table, its lists - for small ones.

constexpr int TRI_GROUP_LOG = 4;                         // vertices of a word: bits 0-15; bits 16-31: which sixteen
constexpr int64_t TRI_MOST = 1ll << (16 + TRI_GROUP_LOG);       // vertices that can be named

// The lanes of a wavefront that have the same k: how many, which of them is the first, and how many are before this one.
struct TriAlike {
    int all, first, before;
};
__device__ __forceinline__ TriAlike tri_alike(int k, int lane)
{
    TriAlike t{0, 0, 0};
    uint64_t left = ~0ull;
    while (left) {
        const int first = __builtin_ctzll(left);
        const uint64_t same = __ballot(k == __builtin_amdgcn_readlane(k, first));
        if (same >> lane & 1)
            t = TriAlike{(int)__popcll(same), first, (int)__popcll(same & ((1ull << lane) - 1ull))};
        left &= ~same;
    }
    return t;
}

// Up to this many edges the plan counts - the entries of every column, the pairs of every end - where it sorts longer
// arrays: a sort of so few entries takes twenty launches.  A first count, us, counting / sorting: 5000 vertices and 79
// thousand edges 309 / 382, 20351 and 0.35 M 498 / 652, 60000 and 0.9 M 678 / 856; 200003 and 1.8 M 958 / 846, 3.5 M 1357 /
// 1277, 2^20 and 15.7 M 5260 / 4180 (all with the vertices sorted by their edges, 50 to 200 us more than now).
constexpr int64_t TRI_COUNTED = 1 << 20;

// counts[c][v]: entries of column v that the workgroups c, c + copies, ... come to; copies is a power of two.  (Atomics on
// one word wait for each other, 14 ns each.)
__global__ __launch_bounds__(256) void tri_columns(int64_t n, int64_t nnz, const int32_t *__restrict__ crd, unsigned copies,
                                                   unsigned *__restrict__ counts)
{
    const int lane = threadIdx.x & 63;
    const int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int v = p < nnz ? crd[p] : -1;
    const TriAlike t = tri_alike(v, lane);
    if (v >= 0 && t.first == lane)
        atomicAdd(&counts[(blockIdx.x & (copies - 1)) * n + v], (unsigned)t.all);
}

__global__ __launch_bounds__(256) void tri_column_keys(int64_t nnz, const int32_t *__restrict__ crd, uint64_t *__restrict__ keys)
{
    const int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (p < nnz)
        keys[p] = (uint64_t)crd[p];
}

// The vertices by their edges, most first, of equally many those first that were: places for each by counting, TRI_UNIT
// vertices to a wavefront.  Up to 511 edges every number is a class of its own, above there are 32 to a factor of two.  (A
// sort of so few keys takes up to 24 launches, 230 us for 2^20 vertices; this takes five.)
constexpr int TRI_UNIT = 1024, TRI_CLASSES = 1024;
__device__ __forceinline__ int tri_class(unsigned edges)
{
    const int log = 31 - __clz((int)edges);
    return TRI_CLASSES - 1 - (edges < 512 ? (int)edges : 512 + (log - 9) * 32 + (int)(edges >> (log - 5) & 31u));
}

// An edge is an entry of the vertex' row or of its column: starts (if given) says how many the columns before each have,
// otherwise counts does, copy by copy.  classes[v], and held[c * units + unit]: vertices of class c.
constexpr unsigned TRI_COPIES = 16;          // at most
__global__ __launch_bounds__(256) void tri_degrees(int64_t n, const int64_t *__restrict__ pos, unsigned copies,
                                                   const unsigned *__restrict__ counts, const int64_t *__restrict__ starts,
                                                   uint32_t *__restrict__ classes, int64_t *__restrict__ held)
{
    __shared__ unsigned here[TRI_CLASSES];
    for (int c = threadIdx.x; c < TRI_CLASSES; c += 256)
        here[c] = 0;
    __syncthreads();
#pragma unroll
    for (int t = 0; t < TRI_UNIT; t += 256) {
        const int64_t v = (int64_t)blockIdx.x * TRI_UNIT + t + threadIdx.x;
        if (v < n) {
            unsigned edges = (unsigned)(pos[v + 1] - pos[v]);
            if (starts) {
                edges += (unsigned)(starts[v + 1] - starts[v]);
            } else {
#pragma unroll
                for (unsigned c = 0; c < TRI_COPIES; ++c) {          // all loads at once
                    const unsigned held_there = counts[(c < copies ? c : 0u) * n + v];
                    edges += c < copies ? held_there : 0u;
                }
            }
            const int k = tri_class(edges);
            classes[v] = (uint32_t)k;
            atomicAdd(&here[k], 1u);
        }
    }
    __syncthreads();
    for (int c = threadIdx.x; c < TRI_CLASSES; c += 256)
        held[(int64_t)c * gridDim.x + blockIdx.x] = here[c];
}

// rank[v]: v's new number; before[c * units + unit]: vertices of the classes before c, and of c in the units before
__global__ __launch_bounds__(64) void tri_ranks(int64_t n, const uint32_t *__restrict__ classes,
                                                const int64_t *__restrict__ before, uint32_t *__restrict__ rank)
{
    __shared__ unsigned next[TRI_CLASSES];
    for (int c = threadIdx.x; c < TRI_CLASSES; c += 64)
        next[c] = (unsigned)before[(int64_t)c * gridDim.x + blockIdx.x];
    __syncthreads();
    const int lane = threadIdx.x;
    const int64_t first = (int64_t)blockIdx.x * TRI_UNIT + lane;
    int ks[TRI_UNIT / 64];
#pragma unroll
    for (int t = 0; t < TRI_UNIT / 64; ++t)
        ks[t] = first + 64 * t < n ? (int)classes[first + 64 * t] : -1;
#pragma unroll
    for (int t = 0; t < TRI_UNIT / 64; ++t) {
        const int k = ks[t];
        const TriAlike a = tri_alike(k, lane);
        if (k >= 0)
            rank[first + 64 * t] = next[k] + (unsigned)a.before;
        __syncthreads();
        if (k >= 0 && a.first == lane)
            next[k] += (unsigned)a.all;
        __syncthreads();
    }
}

// keys[p] = larger new number << bits | smaller one, whatever rows the entries are of (a wavefront per row: 0.49 ms for
// 15.7 M entries, most of it the longest row's).  Without rank the numbers stay, or for an upper triangle are counted from
// the last vertex, and the keys are in order.
__global__ __launch_bounds__(256) void tri_edge_keys(int64_t n, int64_t nnz, const int64_t *__restrict__ pos,
                                                     const int32_t *__restrict__ crd, const uint32_t *__restrict__ rank,
                                                     bool upper, int bits, uint64_t *__restrict__ keys)
{
    const int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t first = uniform_i64_sg(p - (threadIdx.x & 63));
    if (first >= nnz)
        return;
    // the last row that begins at or before an entry: the wavefront's first one, then each lane's from there on
    const auto row_of = [&](int64_t q, int64_t lo, int64_t hi) {
        while (lo < hi) {
            const int64_t mid = (lo + hi + 1) >> 1;
            if (pos[mid] <= q)
                lo = mid;
            else
                hi = mid - 1;
        }
        return lo;
    };
    const int64_t last = first + 63 < nnz ? first + 63 : nnz - 1;
    const int64_t lo = row_of(first, 0, n - 1), hi = row_of(last, lo, n - 1);
    if (p >= nnz)
        return;
    const int64_t row = row_of(p, lo, hi);
    if (rank) {
        const uint64_t a = rank[row], b = rank[crd[p]];
        keys[p] = a > b ? a << bits | b : b << bits | a;
    } else if (upper) {
        keys[nnz - 1 - p] = (uint64_t)(n - 1 - row) << bits | (uint64_t)(n - 1 - crd[p]);
    } else {
        keys[p] = (uint64_t)row << bits | (uint64_t)crd[p];
    }
}

// opens[p] = 1 where sorted key p begins a word
__global__ __launch_bounds__(256) void tri_opens(int64_t nnz, const uint64_t *__restrict__ keys, int64_t *__restrict__ opens)
{
    const int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (p < nnz)
        opens[p] = p == 0 || keys[p - 1] >> TRI_GROUP_LOG != keys[p] >> TRI_GROUP_LOG;
}

// at[r] = first p with keys[p] >> bits >= r, for r in [0, n]
__global__ __launch_bounds__(256) void tri_row_starts(int64_t n, int64_t nnz, const uint64_t *__restrict__ keys, int bits,
                                                      int64_t *__restrict__ at)
{
    const int64_t r = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (r > n)
        return;
    int64_t lo = 0, hi = nnz;
    while (lo < hi) {
        const int64_t mid = (lo + hi) >> 1;
        if ((int64_t)(keys[mid] >> bits) < r)
            lo = mid + 1;
        else
            hi = mid;
    }
    at[r] = lo;
}

// quads[r]: four words each, of row r; word_at[p]: words that begin before key p
__global__ __launch_bounds__(256) void tri_row_quads(int64_t n, const int64_t *__restrict__ row_at,
                                                     const int64_t *__restrict__ word_at, int64_t *__restrict__ quads)
{
    const int64_t r = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (r < n)
        quads[r] = (word_at[row_at[r + 1]] - word_at[row_at[r]] + 3) >> 2;
}

// tpos[r] = first word of row r; the quad in front of all rows is empty
__global__ __launch_bounds__(256) void tri_word_starts(int64_t n, const int64_t *__restrict__ quads_before,
                                                       int64_t *__restrict__ tpos)
{
    const int64_t r = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (r <= n)
        tpos[r] = 4 * (quads_before[r] + 1);
}

__global__ __launch_bounds__(256) void tri_words(int64_t nnz, const uint64_t *__restrict__ keys, int bits,
                                                 const int64_t *__restrict__ row_at, const int64_t *__restrict__ word_at,
                                                 const int64_t *__restrict__ tpos, uint32_t *__restrict__ words)
{
    const int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (p >= nnz || word_at[p] == word_at[p + 1])
        return;
    const uint64_t group = keys[p] >> TRI_GROUP_LOG;
    const int64_t r = (int64_t)(keys[p] >> bits);
    uint32_t in = 0;
    for (int64_t q = p; q < nnz && keys[q] >> TRI_GROUP_LOG == group; ++q)
        in |= 1u << ((uint32_t)keys[q] & ((1u << TRI_GROUP_LOG) - 1u));
    const uint32_t which = (uint32_t)(group & ((1ull << (bits - TRI_GROUP_LOG)) - 1ull));
    words[tpos[r] + word_at[p] - word_at[row_at[r]]] = which << 16 | in;
}

// An edge is looked at from the end with the longer row: keys = that end (n: the other has no row, nothing to do),
// lists = the other end.  count, where there is one: pairs of every end.
__global__ __launch_bounds__(256) void tri_pairs(int64_t n, int64_t nnz, const uint64_t *__restrict__ edges, int bits,
                                                 const int64_t *__restrict__ tpos, uint64_t *__restrict__ keys,
                                                 uint32_t *__restrict__ lists, unsigned long long *__restrict__ count)
{
    const int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x;
    int64_t end = n;
    if (p < nnz) {
        const int64_t a = (int64_t)(edges[p] >> bits), b = (int64_t)(edges[p] & ((1ull << bits) - 1ull));
        const int64_t la = tpos[a + 1] - tpos[a], lb = tpos[b + 1] - tpos[b];
        end = lb == 0 ? n : la > lb ? a : b;
        keys[p] = (uint64_t)end;
        lists[p] = (uint32_t)(la > lb ? b : a);
    }
    if (count) {
        const int lane = threadIdx.x & 63;
        const TriAlike t = tri_alike((int)end, lane);
        if (end < n && t.first == lane)
            atomicAdd(&count[end], (unsigned long long)t.all);
    }
}

// The pairs of an end next to each other, in any order: left[x] of those of x have no place yet.  (A place behind the last
// one's is never read: the pairs of all ends may be fewer than the edges.)
__global__ __launch_bounds__(256) void tri_place(int64_t n, int64_t nnz, const uint64_t *__restrict__ keys,
                                                 const uint32_t *__restrict__ lists, const int64_t *__restrict__ tpos,
                                                 const int64_t *__restrict__ kpos, unsigned long long *__restrict__ left,
                                                 PairEnt *__restrict__ ent, int64_t *__restrict__ work)
{
    const int lane = threadIdx.x & 63;
    const int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int end = p < nnz ? (int)keys[p] : (int)n;
    const TriAlike t = tri_alike(end, lane);
    int before = 0;
    if (end < n && t.first == lane)
        before = (int)atomicAdd(&left[end], 0ull - (unsigned long long)t.all) - t.all;
    before = __shfl(before, t.first, 64);
    if (end < n) {
        const int64_t l = lists[p], s = tpos[l], len = tpos[l + 1] - s, at = kpos[end] + before + t.before;
        ent[at] = PairEnt{(uint32_t)(s >> 2), (uint32_t)(len >> 2)};
        work[at] = len + PAIR_LIST_COST;
    }
}

__global__ __launch_bounds__(256) void tri_entries(int64_t n, int64_t nnz, const uint64_t *__restrict__ keys,
                                                   const uint32_t *__restrict__ lists, const int64_t *__restrict__ tpos,
                                                   PairEnt *__restrict__ ent, int64_t *__restrict__ work)
{
    const int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (p >= nnz)
        return;
    const int64_t l = lists[p], s = tpos[l], len = tpos[l + 1] - s;
    const bool in = (int64_t)keys[p] < n;
    ent[p] = PairEnt{(uint32_t)(s >> 2), in ? (uint32_t)(len >> 2) : 0u};
    work[p] = in ? len + PAIR_LIST_COST : 0;
}

__global__ __launch_bounds__(256) void tri_row_work(int64_t n, const int64_t *__restrict__ kpos,
                                                    const int64_t *__restrict__ work_before, int64_t *__restrict__ wpos)
{
    const int64_t r = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (r <= n)
        wpos[r] = work_before[kpos[r]];
}

// ---------------------------------------------------------------------------
// The walk of masked_pairs.h on rows that are whole quads: no lane needs a mask, one that has no quad takes the empty one.
// ---------------------------------------------------------------------------
template <int ROWS>
struct TriTurn {
    uint4 q[ROWS];
    int rows;
};

template <int ROWS, typename CONSUME>
__device__ __forceinline__ void tri_walk(TriTurn<ROWS> &pend, uint32_t start, int quads, const uint4 *__restrict__ rows,
                                         uint32_t *marks, int lane, CONSUME consume)
{
    const int inc = wave_inclusive_scan(quads), pre = inc - quads;
    const int Q = __builtin_amdgcn_readlane(inc, 63);
    const int a0 = (int)(start - (uint32_t)pre), end = (int)(start + (uint32_t)quads);
    uint32_t before = 0;                 // lists that begin before this row of quads, less one
    for (int base = 0; base < Q; base += 64 * ROWS) {
        const uint32_t bit = (uint32_t)(pre - 1 - base);
        if (quads > 0 && bit < 64u * ROWS)
            atomicOr(&marks[bit >> 5], 1u << (bit & 31u));
        wave_lds_order();
        uint2 m[ROWS];
#pragma unroll
        for (int r = 0; r < ROWS; ++r)
            m[r] = reinterpret_cast<const uint2 *>(marks)[r];
        wave_lds_order();
        if (lane < 2 * ROWS)
            marks[lane] = 0;
        TriTurn<ROWS> now;
        now.rows = (Q - base + 63) >> 6 < ROWS ? (Q - base + 63) >> 6 : ROWS;
#pragma unroll
        for (int r = 0; r < ROWS; ++r) {
            if (r < now.rows) {
                const int owner = (int)__builtin_amdgcn_mbcnt_hi(m[r].y, __builtin_amdgcn_mbcnt_lo(m[r].x, before));
                before += __popc(m[r].x) + __popc(m[r].y);
                const uint32_t at = (uint32_t)lane_value(a0, owner) + (uint32_t)(base + 64 * r + lane);
                now.q[r] = rows[at < (uint32_t)lane_value(end, owner) ? at : 0u];
            }
        }
        wave_lds_order();
        consume(pend);
        pend = now;
    }
}

// the table of a long row: its sixteen bits of every group, at address 0 of the LDS
struct TriBitsProbe {
    __device__ __forceinline__ uint32_t common(uint32_t w) const
    {
        return *reinterpret_cast<const __attribute__((address_space(3))) uint16_t *>(w >> 15 & 0x1fffeu) & w;
    }
};
// of a short one: its words in buckets of four
// (The bucket of a word's group: the upper of the low 24 bits of its product with 0.618 x 2^24, or what is tried after that,
// so that groups next to each other, as most are, come far apart.  The upper of 32 bits, as for the pairs of columns, put
// six neighbours into one bucket of four and such rows were looked up by bisection: us a count, that way / this, R-MAT with
// 16 edges a vertex, n = 200003 253 / 158, 60000 100 / 76, 20351 64 / 49, 5000 40 / 27, 1000 22 / 18; uniform edges, 5000 and
// 40 a vertex 60 / 43, 3000 and 30 46 / 28, 1000 and 40 45 / 27.)
constexpr int TRI_TRIES = 4;
__host__ __device__ __forceinline__ uint32_t tri_multiplier(int attempt)
{
    return attempt == 0 ? 0x9E3779u : attempt == 1 ? 0x85EBCBu : attempt == 2 ? 0xC2B2AFu : 0x27D4EBu;
}
__host__ __device__ __forceinline__ int tri_bucket(uint32_t w, uint32_t mult, int log_nb)
{
#ifdef __HIP_DEVICE_COMPILE__
    return (int)__builtin_amdgcn_ubfe(__umul24(w >> 16, mult), 24 - log_nb, log_nb);
#else
    return (int)(((uint64_t)(w >> 16) * mult & 0xffffffu) >> (24 - log_nb));
#endif
}
struct TriBucketProbe {
    const int *tab;
    uint32_t mult;
    int log_nb;              // log2 of the buckets
    __device__ __forceinline__ uint32_t common(uint32_t w) const
    {
        const si_bucket b = *reinterpret_cast<const si_bucket *>(tab + 4 * tri_bucket(w, mult, log_nb));
        const uint32_t x[4] = {(uint32_t)b.x ^ w, (uint32_t)b.y ^ w, (uint32_t)b.z ^ w, (uint32_t)b.w ^ w};
        uint32_t same = 0;           // where the group is the same: the bits that differ, turned over
#pragma unroll
        for (int c = 0; c < 4; ++c)
            same |= x[c] < 0x10000u ? ~x[c] : 0u;
        return same & w & 0xffffu;
    }
};
struct TriBisectProbe {
    const uint32_t *row;    // the table's words, ascending, behind them empty ones
    int n;
    __device__ __forceinline__ uint32_t common(uint32_t w) const
    {
        int lo = 0, hi = n;
        while (lo < hi) {
            const int mid = (lo + hi) >> 1;
            const uint32_t v = row[mid];
            if (v != 0 && v >> 16 < w >> 16)
                lo = mid + 1;
            else
                hi = mid;
        }
        return lo < n && row[lo] >> 16 == w >> 16 ? row[lo] & w & 0xffffu : 0u;
    }
};

template <int ROWS, typename PROBE>
__device__ __forceinline__ void tri_sum(const TriTurn<ROWS> &t, const PROBE &probe, uint32_t &hits)
{
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
        if (r < t.rows) {
            const uint32_t a = probe.common(t.q[r].x), b = probe.common(t.q[r].y), c = probe.common(t.q[r].z),
                           d = probe.common(t.q[r].w);
            hits += __popc(a | b << 16) + __popc(c | d << 16);
        }
    }
}

// As pair_sum_heavy_kernel.  nwords: 32-bit words of the table.
__global__ __launch_bounds__(SG_T) void tri_heavy_kernel(PairSide s, int nwords, unsigned long long *tickets,
                                                         PairTotal total)
{
    uint16_t *bits = reinterpret_cast<uint16_t *>(sg_dyn_lds);
    PairHeavyShared &sh = *reinterpret_cast<PairHeavyShared *>(sg_dyn_lds + nwords);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    uint32_t *marks = sh.marks[wave];
    const uint32_t *words = reinterpret_cast<const uint32_t *>(s.Tcrd);
    const uint4 *rows = reinterpret_cast<const uint4 *>(s.Lcrd);
    for (int w = threadIdx.x; w < nwords + (int)(sizeof sh / 4); w += SG_T)
        sg_dyn_lds[w] = 0;
    __syncthreads();
    const uint32_t n = (uint32_t)(s.counts[0] & 0xffffffff);
    if (threadIdx.x == 0)
        sh.slot[0] = pair_item<false>(s, s, n, 0, blockIdx.x);
    __syncthreads();
    PairItem it = pair_item_read(sh.slot[0]);
    int cur = 0;
    unsigned long long all_hits = 0;
    const TriBitsProbe probe;
    while (it.index >= 0) {
        for (int t = threadIdx.x; t < it.tlen; t += SG_T) {
            const uint32_t w = words[it.ts + t];
            if (w)
                bits[w >> 16] = (uint16_t)w;
        }
        if (threadIdx.x == 0)
            sh.batch_next = SG_WAVES;
        lds_barrier();
        if (threadIdx.x == 0)
            sh.slot[cur ^ 1] = pair_item<false>(s, s, n, 0, gridDim.x + atomicAdd(&tickets[0], 1ull));
        const int mine = (it.kn + it.parts - 1) / it.parts;          // pairs of a part, about
        int B = mine / (4 * SG_WAVES);
        B = B > 64 ? 64 : B < 2 ? 2 : B;
        const int nb = (it.kn + B - 1) / B;
        PairEnt e{0, 0};
        const auto fetch = [&](int j) {
            const int64_t p = (int64_t)(it.part + it.parts * j) * B + lane;
            e.len = 0;
            if (lane < B && p < it.kn)
                e = s.ent[it.ks + p];
        };
        TriTurn<4> pend;
        pend.rows = 0;
        uint32_t hits = 0;
        int j = wave;
        fetch(j);
        while (it.part + it.parts * j < nb) {
            const PairEnt now = e;
            int d = 0;
            if (lane == 0)
                d = atomicAdd(&sh.batch_next, 1);
            j = __builtin_amdgcn_readfirstlane(d);
            fetch(j);          // the next batch's pairs arrive while this one is walked
            tri_walk(pend, now.start, (int)now.len, rows, marks, lane,
                     [&](const TriTurn<4> &t) { tri_sum(t, probe, hits); });
        }
        tri_sum(pend, probe, hits);
        all_hits += hits;
        lds_barrier();
        for (int t = threadIdx.x; t < it.tlen; t += SG_T)
            bits[words[it.ts + t] >> 16] = 0;
        cur ^= 1;
        it = pair_item_read(sh.slot[cur]);
        lds_barrier();
    }
    pair_block_hits(sh.wave_hits, all_hits, SG_WAVES, total);
}

// As pair_sum_light_kernel.
__global__ __launch_bounds__(PAIR_LIGHT_WAVES * 64, PAIR_LIGHT_OCC) void tri_light_kernel(
    PairSide s, PairTotal total)
{
    constexpr int NB = 1 << PAIR_LIGHT_LOG;
    __shared__ __align__(16) int table[PAIR_LIGHT_WAVES][NB * 4];
    __shared__ __align__(16) uint32_t all_marks[PAIR_LIGHT_WAVES][QUAD_MARKS / 4];
    __shared__ unsigned long long wave_hits[PAIR_LIGHT_WAVES];
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    int *tab = table[wv];
    uint32_t *marks = all_marks[wv];
    const uint32_t *words = reinterpret_cast<const uint32_t *>(s.Tcrd);
    const uint4 *rows = reinterpret_cast<const uint4 *>(s.Lcrd);
    const auto clear = [&](int buckets) {
        for (int b = lane; b < buckets; b += 64)
            reinterpret_cast<si_bucket *>(tab)[b] = si_bucket{0, 0, 0, 0};
    };
    clear(NB);
    if (lane < QUAD_MARKS / 4)
        marks[lane] = 0;
    wave_lds_order();
    const unsigned long long n = (unsigned long long)s.counts[0] >> 32;
    unsigned long long all_hits = 0;
    const unsigned long long waves = (unsigned long long)gridDim.x * PAIR_LIGHT_WAVES;
    const unsigned long long wave_id = blockIdx.x + (unsigned long long)gridDim.x * wv;
    for (unsigned long long tk = wave_id; tk < n; tk += 64 * waves) {
        const unsigned long long left = (n - 1 - tk) / waves + 1;
        const int nr = (int)(left < 64 ? left : 64);
        int64_t l_ts = 0, l_ks = 0;
        int l_tlen = 0, l_kn = 0;
        if (lane < nr) {
            const int x = s.light[tk + lane * waves];
            l_ts = s.Tpos[x];
            l_tlen = (int)(s.Tpos[x + 1] - l_ts);
            l_ks = s.kpos[x];
            l_kn = (int)(s.kpos[x + 1] - l_ks);
        }
        // the words and the first 64 pairs of the next row arrive while this one is walked
        constexpr int PER = (PAIR_LIGHT_MAX + 63) / 64;
        uint32_t wn[PER];
        PairEnt en{0, 0};
        const auto ahead = [&](int r) {
            const int64_t ts = readlane_i64(l_ts, r), ks = readlane_i64(l_ks, r);
            const int tlen = __builtin_amdgcn_readlane(l_tlen, r), kn = __builtin_amdgcn_readlane(l_kn, r);
#pragma unroll
            for (int u = 0; u < PER; ++u)
                wn[u] = 64 * u + lane < tlen ? words[ts + 64 * u + lane] : 0u;
            en.len = 0;
            if (lane < kn)
                en = s.ent[ks + lane];
        };
        ahead(0);
        for (int r = 0; r < nr; ++r) {
            const int64_t ts = readlane_i64(l_ts, r), ks = readlane_i64(l_ks, r);
            const int tlen = __builtin_amdgcn_readlane(l_tlen, r), kn = __builtin_amdgcn_readlane(l_kn, r);
            PairEnt e = en;
            uint32_t w[PER];
#pragma unroll
            for (int u = 0; u < PER; ++u)
                w[u] = wn[u];
            if (r + 1 < nr)
                ahead(r + 1);
            const auto fetch = [&](int b) {
                e.len = 0;
                if (b + lane < kn)
                    e = s.ent[ks + b + lane];
            };
            bool hashed = false;
            uint32_t mult = 0;
            // as many buckets as keep them three quarters of a word full, 64 at least
            int log_nb = 6;
            while (log_nb < PAIR_LIGHT_LOG && tlen > (1 << log_nb) * 3 / 4)
                ++log_nb;
            if (tlen <= PAIR_LIGHT_MAX) {
                for (int attempt = 0; attempt < TRI_TRIES && !hashed; ++attempt) {
                    mult = tri_multiplier(attempt);
                    bool placed = true;
#pragma unroll
                    for (int u = 0; u < PER; ++u) {
                        bool in = w[u] == 0;
                        if (!in) {
                            int *bk = tab + 4 * tri_bucket(w[u], mult, log_nb);
#pragma unroll
                            for (int x = 0; x < 4; ++x)
                                if (!in)
                                    in = atomicCAS(&bk[x], 0, (int)w[u]) == 0;
                        }
                        placed = placed && in;
                    }
                    hashed = !__any(!placed);
                    if (!hashed)
                        clear(1 << log_nb);
                }
            }
            wave_lds_order();
            uint32_t hits = 0;
            TriTurn<PAIR_LIGHT_ROWS> pend;
            pend.rows = 0;
            const auto walk = [&](const auto &probe) {
                for (int b = 0; b < kn; b += 64) {
                    const PairEnt now = e;
                    fetch(b + 64);
                    tri_walk(pend, now.start, (int)now.len, rows, marks, lane,
                             [&](const TriTurn<PAIR_LIGHT_ROWS> &t) { tri_sum(t, probe, hits); });
                }
                tri_sum(pend, probe, hits);
            };
            if (hashed)
                walk(TriBucketProbe{tab, mult, log_nb});
            else
                walk(TriBisectProbe{words + ts, tlen});
            all_hits += hits;
            wave_lds_order();
            if (hashed)
                clear(1 << log_nb);
            wave_lds_order();
        }
    }
    pair_block_hits(wave_hits, all_hits, PAIR_LIGHT_WAVES, total);
}

// A wavefront's row may have this many look-ups in a small graph too, whose parts of PAIR_ITEM_MIN would make it 2048: rows
// of a hundred words are too little for a workgroup.  us a count, 2048 / 3072: uniform edges, 20000 vertices and 30 each
// 61 / 43, 10000 and 40 64 / 48, 5000 and 40 43 / 38; R-MAT, 16 a vertex, 60000 76 / 71, 20351 49 / 46.  (4096 and more
// are faster still for these, but take every row of some graphs from the workgroups.)
constexpr int TRI_LIGHT_WORK = 3072;

// ---------------------------------------------------------------------------
// The plan, kept in the handle as tri (its side holds the pairs) with tri_state 2; 1: the matrix is not of the kind, or the
// plan could not be made, and the pairs of L as it is serve all its counts.
// ---------------------------------------------------------------------------
static int tri_plan(Csr *a, int only)
{
    a->tri_state = 1;
    const int64_t n = a->nrows, nnz = a->nnz;
    if (n != a->ncols || n > TRI_MOST || nnz == 0 || nnz >= (1ll << 31))
        return COMET_HIP_OK;
    bool alone = false;
    COMET_CHK(dot_no_duplicates(a, &alone));
    if (!alone || a->sides == 3)                 // 3: neither strictly lower nor strictly upper
        return COMET_HIP_OK;
    int64_t *word = nullptr;
    COMET_CHK(mailbox((void **)&word));
    const dim3 block(256), per_row((unsigned)ceil_div(n + 1, 256)), per_entry((unsigned)ceil_div(nnz, 256));
    int bits = TRI_GROUP_LOG;                    // of a vertex
    while ((1ll << bits) < n)
        ++bits;
    TriPlan &plan = a->tri;
    PairSidePlan &side = plan.side;
    // Scratch: three arrays of a 64-bit and two of a 32-bit word for every entry, two of a 64-bit word for every row, in one
    // allocation (each costs about as much as a small count).
    char *scratch = nullptr;
    const size_t entries = ((size_t)std::max(nnz, n + TRI_UNIT) + 64) & ~(size_t)63, rows = ((size_t)n + 65) & ~(size_t)63;
    const int64_t quads_most = nnz / 4 + n + 2;
    const bool room =
        dev_malloc((void **)&scratch, 32 * entries + 16 * rows) == hipSuccess &&
        dev_malloc((void **)&plan.words, 16 * (size_t)quads_most) == hipSuccess &&
        dev_malloc((void **)&plan.tpos, 8 * rows) == hipSuccess && dev_malloc((void **)&side.kpos, 8 * rows) == hipSuccess &&
        dev_malloc((void **)&side.counts, 8) == hipSuccess && dev_malloc(&side.ent, sizeof(PairEnt) * (size_t)nnz) == hipSuccess;
    uint64_t *k0 = (uint64_t *)scratch, *k1 = k0 + entries;
    int64_t *w0 = (int64_t *)(k1 + entries), *r0 = w0 + entries, *r1 = r0 + rows;
    uint32_t *i0 = (uint32_t *)(r1 + rows), *i1 = i0 + entries;
    const auto run = [&]() -> int {
        KernelTimer t("triangle_plan");
        uint32_t *rank = i0, *classes = i1;
        // ---- the edges in order of their rows, the vertices by their number of edges where that pays
        if (a->uneven) {
            unsigned copies = 0, *counts = nullptr;
            int64_t *starts = nullptr;
            if (nnz <= TRI_COUNTED) {
                copies = TRI_COPIES, counts = (unsigned *)k1;
                while (sizeof(unsigned) * copies * (size_t)n > 8 * entries)
                    copies /= 2;
                COMET_HIPCHK(hipMemsetAsync(counts, 0, sizeof(unsigned) * copies * (size_t)n, stream()));
                tri_columns<<<per_entry, block, 0, stream()>>>(n, nnz, a->crd, copies, counts);
            } else {
                starts = r0;
                tri_column_keys<<<per_entry, block, 0, stream()>>>(nnz, a->crd, k0);
                COMET_CHK(sort_pairs_u64_u32(k0, k1, i0, i1, nnz, bits));          // (of the keys alone, see below)
                tri_row_starts<<<per_row, block, 0, stream()>>>(n, nnz, k1, 0, starts);
            }
            const unsigned units = (unsigned)ceil_div(n, TRI_UNIT);
            tri_degrees<<<dim3(units), block, 0, stream()>>>(n, a->pos, copies, counts, starts, classes, w0);
            COMET_CHK(exclusive_scan_i64(w0, (int64_t)units * TRI_CLASSES, (int64_t *)k0));
            tri_ranks<<<dim3(units), dim3(64), 0, stream()>>>(n, classes, (const int64_t *)k0, rank);
            tri_edge_keys<<<per_entry, block, 0, stream()>>>(n, nnz, a->pos, a->crd, rank, false, bits, k0);
            // As far as the group of the smaller number: the order of the entries of a word does not matter.  What goes along is
            // read by nobody; a sort of keys alone is a fifth quicker (3880 us for the first count of 2^20 vertices, this way
            // 4240), but its code takes 4 ms to come to the device, once for every program that counts triangles.
            COMET_CHK(sort_pairs_u64_u32(k0, k1, i0, i1, nnz, 2 * bits, TRI_GROUP_LOG));
        } else {
            tri_edge_keys<<<per_entry, block, 0, stream()>>>(n, nnz, a->pos, a->crd, nullptr, a->sides == 1, bits, k1);
        }
        // ---- the rows
        int64_t *opens = (int64_t *)k0;
        tri_opens<<<per_entry, block, 0, stream()>>>(nnz, k1, opens);
        COMET_CHK(exclusive_scan_i64(opens, nnz, w0));
        tri_row_starts<<<per_row, block, 0, stream()>>>(n, nnz, k1, bits, r0);
        tri_row_quads<<<per_row, block, 0, stream()>>>(n, r0, w0, r1);
        COMET_CHK(exclusive_scan_i64(r1, n, side.kpos));
        tri_word_starts<<<per_row, block, 0, stream()>>>(n, side.kpos, plan.tpos);
        COMET_HIPCHK(hipMemsetAsync(plan.words, 0, 16 * (size_t)quads_most, stream()));
        tri_words<<<per_entry, block, 0, stream()>>>(nnz, k1, bits, r0, w0, plan.tpos, plan.words);
        // ---- the edges by the end they are looked at from
        int64_t *work = (int64_t *)k0;
        if (nnz <= TRI_COUNTED) {
            unsigned long long *count = (unsigned long long *)r1;
            COMET_HIPCHK(hipMemsetAsync(count, 0, 8 * (size_t)n, stream()));
            tri_pairs<<<per_entry, block, 0, stream()>>>(n, nnz, k1, bits, plan.tpos, k0, i0, count);
            COMET_CHK(exclusive_scan_i64(r1, n, side.kpos));
            work = (int64_t *)k1;
            tri_place<<<per_entry, block, 0, stream()>>>(n, nnz, k0, i0, plan.tpos, side.kpos, count, (PairEnt *)side.ent, work);
        } else {
            tri_pairs<<<per_entry, block, 0, stream()>>>(n, nnz, k1, bits, plan.tpos, k0, i0, nullptr);
            COMET_CHK(sort_pairs_u64_u32(k0, k1, i0, i1, nnz, bits + 1));          // n is among the keys
            tri_row_starts<<<per_row, block, 0, stream()>>>(n, nnz, k1, 0, side.kpos);
            tri_entries<<<per_entry, block, 0, stream()>>>(n, nnz, k1, i1, plan.tpos, (PairEnt *)side.ent, work);
        }
        COMET_CHK(exclusive_scan_i64(work, nnz, w0));
        tri_row_work<<<per_row, block, 0, stream()>>>(n, side.kpos, w0, r0);
        pair_parts<<<per_row, block, 0, stream()>>>(0, n, plan.tpos, side.kpos, r0, only, PAIR_LIGHT_MAX, TRI_LIGHT_WORK, PAIR_SHARES,
                                                    PAIR_ITEM_MIN, r1);
        COMET_CHK(exclusive_scan_i64(r1, n, r0, word));
        COMET_CHK(stream_wait());
        const int64_t packed = *(volatile int64_t *)word;
        side.nheavy = packed & 0xffffffff;
        side.nlight = packed >> 32;
        side.pairs = nnz;
        COMET_HIPCHK(dev_malloc(&side.heavy, sizeof(uint2) * (size_t)(side.nheavy > 0 ? side.nheavy : 1)));
        COMET_HIPCHK(dev_malloc((void **)&side.light, sizeof(int32_t) * (size_t)(side.nlight > 0 ? side.nlight : 1)));
        pair_items<<<per_row, block, 0, stream()>>>(0, n, r1, r0, (uint2 *)side.heavy, side.light, side.counts);
        COMET_HIPCHK(hipGetLastError());
        a->tri_state = 2;
        return COMET_HIP_OK;
    };
    const int rc = room ? run() : COMET_HIP_ERR_HIP;
    (void)dev_free(scratch);
    if (a->tri_state != 2)
        tri_plan_free(plan);
    return rc;
}

// (The two kernels side by side: 889 us instead of 875 for n = 2^20, 260 / 255 for 200003, 92 / 70 for 20351.)
static int tri_count(Csr *a, double *result)
{
    PairSide s = pair_side(a->tri.side, a, a);
    s.Tpos = a->tri.tpos;
    s.Tcrd = s.Lcrd = reinterpret_cast<const int32_t *>(a->tri.words);
    const int64_t nheavy = a->tri.side.nheavy, nlight = a->tri.side.nlight;
    unsigned long long *tickets = nullptr;
    double *word = nullptr;
    COMET_CHK(pair_tickets(&tickets));
    COMET_CHK(mailbox((void **)&word));
    const PairGrids grids = pair_grids(nheavy, nlight, a->ncols);
    PairTotal total{tickets, grids.heavy + grids.light, 0, a->iso_value * a->iso_value, word};
    if (total.blocks == 0) {
        *result = 0.0;
        return COMET_HIP_OK;
    }
    if (nheavy > 0) {
        COMET_CHK(sg_allow_lds(tri_heavy_kernel, grids.lds));
        KernelTimer t("spgemm_masked_sum");
        tri_heavy_kernel<<<dim3(grids.heavy), dim3(SG_T), grids.lds, stream()>>>(s, grids.nwords, tickets, total);
    }
    if (nlight > 0) {
        KernelTimer t("spgemm_masked_sum_small");
        total.first = grids.heavy;
        tri_light_kernel<<<dim3(grids.light), dim3(PAIR_LIGHT_WAVES * 64), 0, stream()>>>(s, total);
    }
    COMET_CHK(pair_launched(tickets));
    COMET_CHK(stream_wait());
    *result = *(volatile double *)word;
    return COMET_HIP_OK;
}
