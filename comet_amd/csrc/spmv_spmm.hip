// CSR SpMV and CSR SpMM for gfx950.
//
// Both kernels add products in ascending nonzero order with an unfused
// multiply then add, the order and arithmetic of the loop nests the reference
// generates (lib/Conversion/IndexTreeToSCF/IndexTreeToSCF.cpp:529-621 row
// loop, :667-700 nonzero loop, :476-489 dense inner loop, :1247-1284
// lhs = lhs + a*b), so a row handled by one wavefront reproduces the CPU
// result bit for bit.  This file is compiled with -ffp-contract=off.
#include <stdlib.h>

#include <algorithm>
#include <memory>
#include <queue>
#include <utility>
#include <vector>

#include "common.h"

namespace comet {

// ============================================================================
// SpMV: 256 rows per workgroup, one lane per row.  The workgroup streams the
// contiguous nonzero range of its rows through LDS in passes of SPMV_PASS
// products: all lanes compute val*x[crd] with coalesced loads of crd/val,
// then each lane adds the slice of the pass that belongs to its row, in
// order.  HBM traffic is the compulsory one (crd, val, pos once; x gathered).
// A slice of 128 products and more is added by the whole workgroup instead.
// ============================================================================
#ifndef COMET_SPMV_T
#define COMET_SPMV_T 256
#endif
#ifndef COMET_SPMV_PASS
#define COMET_SPMV_PASS 2048
#endif
constexpr int SPMV_T = COMET_SPMV_T;         // rows (= lanes) per workgroup
constexpr int SPMV_PASS = COMET_SPMV_PASS;   // products staged in LDS per pass

constexpr int SPMV_LONG = 128;               // a row's share of a pass from which the workgroup adds it together

__device__ inline int64_t uniform_i64(int64_t v)
{
    return ((int64_t)__builtin_amdgcn_readfirstlane((int)(v >> 32)) << 32) |
           (uint32_t)__builtin_amdgcn_readfirstlane((int)(v & 0xffffffff));
}

// The LDS a workgroup streams products through.
struct SpmvStage {
    double prod[SPMV_PASS];
    double part[SPMV_T / 64];
    int64_t long_lo[SPMV_PASS / SPMV_LONG + 1], long_hi[SPMV_PASS / SPMV_LONG + 1];
    int long_owner[SPMV_PASS / SPMV_LONG + 1], nlong;
};

// The rows [r0, rlast) of one tile, rlast - r0 <= SPMV_T, lane tid owning row r0 + tid: returns acc + the lane's row
// times x, added in the order of the row's nonzeros.  Every lane of the workgroup calls it (it holds barriers).
// P: the row pointers' type - int64 for a matrix as uploaded, int32 for the column blocks of the plan, whose row
// pointers are read again by every pass
template <typename P>
__device__ __forceinline__ double spmv_tile(SpmvStage &st, const P *__restrict__ pos, const int32_t *__restrict__ crd,
                                            const double *__restrict__ val, const double *__restrict__ x, int64_t r0,
                                            int64_t rlast, double acc)
{
    const int tid = threadIdx.x;
    const int64_t r = r0 + tid;
    const int64_t ps = (int64_t)pos[r < rlast ? r : rlast];
    const int64_t pe = (int64_t)pos[r + 1 < rlast ? r + 1 : rlast];
    const int64_t bs = uniform_i64((int64_t)pos[r0]), be = uniform_i64((int64_t)pos[rlast]);
    for (int64_t cs = bs; cs < be; cs += SPMV_PASS) {
        const int64_t ce = cs + SPMV_PASS < be ? cs + SPMV_PASS : be;
        // a pass with fewer products than SPMV_LONG holds no long share: it skips the bookkeeping and its barriers
        const bool may_be_long = ce - cs >= SPMV_LONG;
        if (may_be_long && tid == 0)
            st.nlong = 0;
        for (int64_t i = cs + tid; i < ce; i += SPMV_T)
            st.prod[i - cs] = val[i] * x[crd[i]];
        __syncthreads();
        const int64_t lo = ps > cs ? ps : cs, hi = pe < ce ? pe : ce;
        if (hi - lo < SPMV_LONG) {           // the usual case: the lane adds its row's share in order
            for (int64_t p = lo; p < hi; ++p)
                acc = acc + st.prod[p - cs];
        } else {                             // at most SPMV_PASS / SPMV_LONG lanes per pass come here
            const int slot = atomicAdd(&st.nlong, 1);
            st.long_owner[slot] = tid;
            st.long_lo[slot] = lo;
            st.long_hi[slot] = hi;
        }
        if (may_be_long) {
            // Shares of SPMV_LONG products and more are added by the whole workgroup: lane t takes products
            // t, t + 256, ..., the partial sums are added along each wavefront and then across wavefronts.
            // A fixed order, though not the row's own: such a row agrees with the sequential sum to rounding,
            // not to the bit.  The shares are of different rows, so the order in which they are taken is free.
            __syncthreads();
            const int n = __builtin_amdgcn_readfirstlane(st.nlong);
            for (int k = 0; k < n; ++k) {
                const int owner = __builtin_amdgcn_readfirstlane(st.long_owner[k]);
                const int64_t l = uniform_i64(st.long_lo[k]), h = uniform_i64(st.long_hi[k]);
                double s = 0.0;
                for (int64_t p = l + tid; p < h; p += SPMV_T)
                    s = s + st.prod[p - cs];
                for (int d = 32; d > 0; d >>= 1)
                    s = s + __shfl_down(s, d, 64);
                if ((tid & 63) == 0)
                    st.part[tid >> 6] = s;
                __syncthreads();
                if (tid == owner) {
                    double t = st.part[0];
                    for (int w = 1; w < SPMV_T / 64; ++w)
                        t = t + st.part[w];
                    acc = acc + t;
                }
                __syncthreads();
            }
        }
        __syncthreads();
    }
    return acc;
}

template <bool ACC, typename P>
__global__ __launch_bounds__(SPMV_T) void spmv_csr_stream(const P *__restrict__ pos,
                                                          const int32_t *__restrict__ crd,
                                                          const double *__restrict__ val,
                                                          const double *__restrict__ x,
                                                          double *__restrict__ y, int64_t nrows)
{
    __shared__ SpmvStage st;
    const int64_t r0 = (int64_t)blockIdx.x * SPMV_T;
    const int64_t r = r0 + threadIdx.x;
    const int64_t rlast = r0 + SPMV_T < nrows ? r0 + SPMV_T : nrows;
    double acc = 0.0;
    if (ACC && r < nrows)
        acc = y[r];
    acc = spmv_tile(st, pos, crd, val, x, r0, rlast, acc);
    if (r < nrows)
        y[r] = acc;
}

// All column blocks of the plan in one launch.  A workgroup owns `tiles` tiles of `tile_rows` rows (tile k of
// workgroup w is tile k * gridDim.x + w) and goes through the blocks in order, all its tiles in each; the row sums
// stay in LDS from block to block instead of going through y.  The grid is what the GPU holds at once, so all
// workgroups are in the same block at about the same time and gather from the same slice of x - nothing waits for
// that, it only keeps the slice in the L2.  A row's products are still added in the order of its nonzeros.
// (Measured on the benchmark matrix, 10^6 rows of 10 nonzeros: 0.061 ms against 0.076 ms for a launch per block.
// One visit per block and workgroup instead - its rows consecutive, two or three to a lane, the sums in registers -
// took 0.072 ms, 0.066 with the products staged 512 at a time: the workgroups then load together and add together,
// and the memory side idles while they add.)
constexpr int SPMV_MAX_BLOCKS = 16;
struct SpmvBases { int64_t v[SPMV_MAX_BLOCKS]; };
extern __shared__ double spmv_row_sums[];

template <typename P>
__global__ __launch_bounds__(SPMV_T) void spmv_csr_blocks(const P *__restrict__ bpos, const int32_t *__restrict__ bcrd,
                                                          const double *__restrict__ bval, SpmvBases base, int nb,
                                                          const double *__restrict__ x, double *__restrict__ y,
                                                          int64_t nrows, int tile_rows, int tiles, int accumulate)
{
    __shared__ SpmvStage st;
    const int tid = threadIdx.x;
    for (int k = 0; k < tiles; ++k) {
        const int64_t r = ((int64_t)k * gridDim.x + blockIdx.x) * tile_rows + tid;
        spmv_row_sums[k * SPMV_T + tid] = accumulate && tid < tile_rows && r < nrows ? y[r] : 0.0;
    }
    for (int b = 0; b < nb; ++b) {
        const P *pos = bpos + (int64_t)b * (nrows + 1);
        const int32_t *crd = bcrd + base.v[b];
        const double *val = bval + base.v[b];
        for (int k = 0; k < tiles; ++k) {
            const int64_t r0 = ((int64_t)k * gridDim.x + blockIdx.x) * tile_rows;
            if (r0 >= nrows)
                break;
            const int64_t rlast = r0 + tile_rows < nrows ? r0 + tile_rows : nrows;
            spmv_row_sums[k * SPMV_T + tid] = spmv_tile(st, pos, crd, val, x, r0, rlast, spmv_row_sums[k * SPMV_T + tid]);
        }
    }
    for (int k = 0; k < tiles; ++k) {
        const int64_t r = ((int64_t)k * gridDim.x + blockIdx.x) * tile_rows + tid;
        if (tid < tile_rows && r < nrows)
            y[r] = spmv_row_sums[k * SPMV_T + tid];
    }
}

// ----------------------------------------------------------------------------
// Column-blocked plan for SpMV.  The gather of x has no locality: with x larger
// than an L2 (4 MiB per XCD) every nonzero moves a cache line across the
// fabric.  The plan re-stores A as NB column blocks whose slice of x (<= 2 MiB)
// stays in L2, and SpMV runs one pass per block.  Pass b starts each row's
// accumulator from the y that pass b-1 left, and columns ascend inside a row,
// so the additions happen in exactly the original nonzero order: the result is
// still bit-identical to the sequential loop nest.
// ----------------------------------------------------------------------------
// Measured on the 10^6 x 10^6 Poisson(10) matrix (x = 8 MB), ms per SpMV: one pass 0.115, slices of
// 4 MiB (2 passes) 0.075, 2 MiB (4 passes) 0.077, 1 MiB (8) 0.099, 512 KiB (16) 0.140.
#ifndef COMET_SPMV_SLICE_KB
#define COMET_SPMV_SLICE_KB 2048
#endif
constexpr int64_t SPMV_SLICE_BYTES = (int64_t)COMET_SPMV_SLICE_KB << 10;

__device__ inline int64_t lower_bound_col(const int32_t *__restrict__ crd, int64_t lo, int64_t hi, int64_t col)
{
    while (lo < hi) {
        const int64_t mid = (lo + hi) >> 1;
        if (crd[mid] < col)
            lo = mid + 1;
        else
            hi = mid;
    }
    return lo;
}

// cnt[b * nrows + r] = nonzeros of row r with column in block b
__global__ void spmv_narrow_pos(const int64_t *__restrict__ in, int32_t *__restrict__ out, int64_t n)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n)
        out[i] = (int32_t)in[i];
}

__global__ void spmv_split_count(const int64_t *__restrict__ pos, const int32_t *__restrict__ crd, int64_t nrows,
                                 int nb, int64_t block_cols, int64_t *__restrict__ cnt)
{
    const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= nrows)
        return;
    const int64_t s = pos[r], e = pos[r + 1];
    int64_t prev = s;
    for (int b = 0; b < nb; ++b) {
        const int64_t next = b + 1 < nb ? lower_bound_col(crd, prev, e, (int64_t)(b + 1) * block_cols) : e;
        cnt[(int64_t)b * nrows + r] = next - prev;
        prev = next;
    }
}

__global__ void spmv_split_scatter(const int64_t *__restrict__ pos, const int32_t *__restrict__ crd,
                                   const double *__restrict__ val, int64_t nrows, int nb, int64_t block_cols,
                                   const int64_t *__restrict__ bpos, SpmvBases base, int32_t *__restrict__ bcrd,
                                   double *__restrict__ bval)
{
    const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= nrows)
        return;
    int64_t p = pos[r];
    for (int b = 0; b < nb; ++b) {
        const int64_t *bp = bpos + (int64_t)b * (nrows + 1);
        const int64_t o = base.v[b] + bp[r], n = bp[r + 1] - bp[r];
        for (int64_t t = 0; t < n; ++t) {
            bcrd[o + t] = crd[p + t];
            bval[o + t] = val[p + t];
        }
        p += n;
    }
}

static Workspace g_spmv_cnt;

static int spmv_plan(Csr *a)
{
    if (a->spmv_nb > 0)
        return COMET_HIP_OK;
    int nb = 1;
    const int64_t slice_bytes = SPMV_SLICE_BYTES;
    if (a->ncols * 8 > slice_bytes + slice_bytes / 2 && a->nnz >= (1 << 20)) {
        nb = (int)std::min<int64_t>(SPMV_MAX_BLOCKS, ceil_div(a->ncols * 8, slice_bytes));
    }
    if (nb <= 1) {
        a->spmv_nb = 1;
        return COMET_HIP_OK;
    }
    const int64_t n = a->nrows, block_cols = ceil_div(a->ncols, nb);
    COMET_CHK(g_spmv_cnt.ensure(sizeof(int64_t) * (size_t)nb * (size_t)n, false));
    int64_t *cnt = (int64_t *)g_spmv_cnt.ptr;
    int64_t *bpos = nullptr;
    int32_t *bcrd = nullptr;
    double *bval = nullptr;
    COMET_HIPCHK(dev_malloc((void **)&bpos, sizeof(int64_t) * (size_t)nb * (size_t)(n + 1)));
    auto cleanup = [&]() {
        (void)dev_free(bpos);
        (void)dev_free(bcrd);
        (void)dev_free(bval);
    };
    const dim3 grid((unsigned)ceil_div(n, 256)), block(256);
    {
        KernelTimer t("spmv_split_count");
        spmv_split_count<<<grid, block, 0, stream()>>>(a->pos, a->crd, n, nb, block_cols, cnt);
    }
    SpmvBases base;
    std::vector<int64_t> totals(nb);
    for (int b = 0; b < nb; ++b) {
        int rc = exclusive_scan_i64(cnt + (int64_t)b * n, n, bpos + (int64_t)b * (n + 1));
        if (rc != COMET_HIP_OK) {
            cleanup();
            return rc;
        }
    }
    for (int b = 0; b < nb; ++b) {
        if (hipMemcpyAsync(&totals[b], bpos + (int64_t)b * (n + 1) + n, sizeof(int64_t), hipMemcpyDeviceToHost,
                           stream()) != hipSuccess) {
            cleanup();
            return set_error(COMET_HIP_ERR_HIP, "reading block sizes failed");
        }
    }
    if (hipStreamSynchronize(stream()) != hipSuccess) {
        cleanup();
        return set_error(COMET_HIP_ERR_HIP, "SpMV plan synchronisation failed");
    }
    int64_t run = 0;
    a->spmv_base.assign(nb, 0);
    for (int b = 0; b < nb; ++b) {
        base.v[b] = run;
        a->spmv_base[b] = run;
        run += totals[b];
    }
    // the blocks cut every row into consecutive segments, so they always hold all nonzeros, in order
    if (dev_malloc((void **)&bcrd, sizeof(int32_t) * (size_t)a->nnz) != hipSuccess ||
        dev_malloc((void **)&bval, sizeof(double) * (size_t)a->nnz) != hipSuccess) {
        cleanup();
        return set_error(COMET_HIP_ERR_HIP, "allocating the column-blocked copy failed");
    }
    {
        KernelTimer t("spmv_split_scatter");
        spmv_split_scatter<<<grid, block, 0, stream()>>>(a->pos, a->crd, a->val, n, nb, block_cols, bpos, base, bcrd,
                                                         bval);
    }
    if (hipGetLastError() != hipSuccess) {
        cleanup();
        return set_error(COMET_HIP_ERR_HIP, "SpMV plan kernel launch failed");
    }
    // the blocks' row pointers are read by every pass: 32 bits are enough for them unless a block holds 2^31 nonzeros
    bool narrow = true;
    for (int b = 0; b < nb; ++b)
        narrow = narrow && totals[b] < (1ll << 31);
    if (narrow) {
        int32_t *bpos32 = nullptr;
        const int64_t count = (int64_t)nb * (n + 1);
        if (dev_malloc((void **)&bpos32, sizeof(int32_t) * (size_t)count) == hipSuccess) {
            spmv_narrow_pos<<<dim3((unsigned)ceil_div(count, 256)), dim3(256), 0, stream()>>>(bpos, bpos32, count);
            if (hipStreamSynchronize(stream()) == hipSuccess) {
                a->spmv_bpos32 = bpos32;
                (void)dev_free(bpos);
                bpos = nullptr;
            } else {
                (void)dev_free(bpos32);
            }
        } else {
            (void)hipGetLastError();        // an allocation that may fail: the 64-bit pointers stay in use
        }
    }
    a->spmv_bpos = bpos;
    a->spmv_bcrd = bcrd;
    a->spmv_bval = bval;
    a->spmv_nb = nb;
    return COMET_HIP_OK;
}

// ============================================================================
// SpMM, nonzero-split: the nonzeros of A are cut into chunks of SPMM_CH (a half
// or a quarter of that where there are not many) and one wavefront owns each
// chunk, whatever rows it covers, so Zipf-distributed row lengths cost nothing
// in balance.  A lane owns two dense columns, 16 bytes of a row of B, so that a
// tile of kt columns takes kt / 2 lanes and a wavefront holds 64 / (kt / 2)
// groups of them, each with a run of the chunk's nonzeros of its own, SPMM_U
// gathers of B deep.  Which row a nonzero is of is worked out once per chunk in
// LDS.  A row of fewer than SPMM_WHOLE nonzeros, or one that lies inside one
// block of SPMM_CH, is summed in nonzero order: where a boundary of a chunk would
// cut it, it goes to the one it begins in.  The other rows are cut wherever that
// happens; the pieces of a chunk are added in LDS, and what the chunk has of them
// goes to `carry` (two slots of a tile's columns per chunk: [0] a piece whose row
// began in an earlier chunk, [1] a piece whose row goes on into the next), from
// where the wavefront that leaves the last piece of a row (`arrived` counts them,
// by the chunk the row begins in, from zero) adds them in chunk order.
// The groups' runs end with rows, so one run may be much longer than the others:
// then every group gathers the same number of nonzeros, and the sum of a row goes
// from group to group.  Until that was so, one group went through a row of up to
// 255 nonzeros by itself, 22 of the 24 us that a matrix of 2000 rows took (zipf, 12
// nonzeros a row; 14 now); 20000 rows and K = 8 30 -> 20, 500000 and K = 3 175 -> 152.
// Empty rows are cleared by all wavefronts, an equal share of the matrix's rows to each, whichever chunk they lie in: the
// last rows of a graph are nearly all empty, and one wavefront's chunk had a thousand of them (us, R-MAT scale 16, 8 edges a
// vertex K = 3 66 -> 29, K = 33 80 -> 45, scale 18 and 16 K = 8 180 -> 110, scale 19 and 16 K = 33 614 -> 499; 300000 rows, nine
// of ten empty, K = 3 56 -> 13; the loads for it cost 100000 rows of 9 in a band 0.3 of 14).
// Bound by the latency of that where the matrix is small, by the gathers' way from
// the memory-side cache where B is larger than an L2.
// ============================================================================
#ifndef COMET_SPMM_U
#define COMET_SPMM_U 8
#endif
constexpr int SPMM_CH = 256;                  // nonzeros per wavefront, at most, but for the end of a row that is not cut
constexpr int SPMM_WHOLE = 128;               // a row of fewer nonzeros is never cut
constexpr int SPMM_HELD = SPMM_CH + SPMM_WHOLE;
constexpr int SPMM_GRAIN = 64;                // the row of every so many'th nonzero is kept
constexpr int SPMM_U = COMET_SPMM_U;          // B-row loads in flight per lane
constexpr int SPMM_WAVES = 4;                 // wavefronts per workgroup
constexpr int SPMM_TURNS = 4;                 // sums handed from group to group in the time of a round of gathers

// chunk_row[c] = the row r with pos[r] <= c*grain < pos[r+1]; arrived[0 .. counts) = 0 (counts 0: not asked for)
__global__ void spmm_chunk_rows(const int64_t *__restrict__ pos, int64_t nrows, int64_t nchunks, int grain,
                                int32_t *__restrict__ chunk_row, unsigned *__restrict__ arrived, int64_t counts)
{
    int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= nchunks)
        return;
    for (int64_t i = c; i < counts; i += nchunks)
        arrived[i] = 0;
    const int64_t target = c * grain;
    int64_t lo = 0, hi = nrows;   // first index in pos[0..nrows] with pos > target lies in [1, nrows]
    while (lo < hi) {
        int64_t mid = (lo + hi) >> 1;
        if (pos[mid + 1] > target)
            hi = mid;
        else
            lo = mid + 1;
    }
    chunk_row[c] = (int32_t)lo;
}

typedef double spmm_pair __attribute__((ext_vector_type(2), aligned(8)));

struct SpmmChunkLds {
    union {
        struct {
            double val[SPMM_HELD];
            int32_t crd[SPMM_HELD];
        };
        double piece[2][128];            // of every group: its head and its tail, over the entries
    };
    int32_t row[SPMM_HELD + 4];            // the last one: whose row goes on past the chunk
};

// W: columns of a lane, 2 unless K is 1.  SMALL: B is within 4 GiB.
template <bool ACC, int W, bool SMALL>
__global__ __launch_bounds__(SPMM_WAVES * 64, ACC ? 4 : 6) void spmm_csr_nnzsplit(
    const int64_t *__restrict__ pos, const int32_t *__restrict__ crd, const double *__restrict__ val,
    int64_t nnz, int64_t nrows, const int32_t *__restrict__ chunk_row, int grain, int chunk_len, int64_t nchunks, const uint32_t *__restrict__ order,
    const double *__restrict__ B, int64_t ldb, double *__restrict__ C, int64_t ldc, int K, int tile_cols, int rows_each,
    double *__restrict__ carry, unsigned *__restrict__ arrived, const int32_t *__restrict__ rowmap)
{
    __shared__ __align__(16) SpmmChunkLds all[SPMM_WAVES];
    // rowmap: the matrix lists only some rows of C (row r of pos is row rowmap[r] of C); nullptr: all of them
    auto crow = [&](int64_t r) -> int64_t { return rowmap ? (int64_t)rowmap[r] : r; };
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    // the order's eighths, one to an XCD (workgroup w runs on XCD w % 8, and the grid is a multiple of eight wide)
    int64_t chunk = (int64_t)(order ? blockIdx.x >> 3 : blockIdx.x) * SPMM_WAVES + wave;
    if (order) {
        const int64_t eighth = (nchunks + 7) / 8, at = (blockIdx.x & 7) * eighth + chunk;
        chunk = chunk < eighth && at < nchunks ? (int64_t)__builtin_amdgcn_readfirstlane((int)order[at]) : nchunks;
    }
    if (chunk >= nchunks)
        return;
    SpmmChunkLds &sh = all[wave];
    const int64_t tile = (int64_t)blockIdx.y * tile_cols;
    const int kt = (int)(K - tile < tile_cols ? K - tile : tile_cols);
    const int L = (kt + W - 1) / W, G = 64 / L;               // lanes of a group, groups
    const int g = lane / L, sub = lane - g * L;
    // the last lane of an odd tile has one column, and reads the one before it as well
    const bool half = W == 2 && sub == L - 1 && (kt & 1);
    const int64_t col = tile + W * sub, from = col - (half ? 1 : 0);
    // rows of which the empty ones are this wavefront's to clear: where the first of them begin is loaded here
    const int64_t z0 = chunk * rows_each, z1 = z0 + rows_each < nrows ? z0 + rows_each : nrows;
    int64_t zp = 0;
    if (!ACC && z0 + lane <= z1)
        zp = pos[z0 + lane];
    // ---- the nonzeros [s, e) of the chunk, moved to the ends of rows that are not to be cut, and the rows they are of
    const int64_t s_cut = chunk * chunk_len, e_cut = s_cut + chunk_len < nnz ? s_cut + chunk_len : nnz;
    const int64_t block = s_cut / SPMM_CH * SPMM_CH;
    const int64_t r0 = __builtin_amdgcn_readfirstlane(chunk_row[s_cut / grain]);
    const int64_t rn = e_cut < nnz ? (int64_t)__builtin_amdgcn_readfirstlane(chunk_row[e_cut / grain]) : nrows;
    int64_t s = s_cut, e = e_cut;
    const int64_t p0 = pos[r0], q0 = pos[r0 + 1];
    const auto whole = [&](int64_t p, int64_t q) { return q - p < SPMM_WHOLE || (p >= block && q <= block + SPMM_CH); };
    const bool head = p0 < s_cut && !whole(p0, q0);          // the first row is a piece of one
    if (p0 < s_cut && !head)                             // an earlier chunk's
        s = q0;
    bool tail = false;                                   // the last row goes on into the next block
    if (rn < nrows) {
        const int64_t pn = pos[rn], qn = pos[rn + 1];
        if (pn < e_cut) {
            tail = !whole(pn, qn);
            e = tail ? e_cut : qn;
        }
    }
    const int n = e > s ? (int)(e - s) : 0;
    for (int t = lane; t < n; t += 64) {      // A is streamed once: keep it from displacing B in the caches
        sh.crd[t] = __builtin_nontemporal_load(crd + s + t);
        sh.val[t] = __builtin_nontemporal_load(val + s + t);
    }
    for (int t = lane; t < n; t += 64)
        sh.row[t] = 0;
    if constexpr (!ACC)          // accumulating leaves empty rows untouched
        for (int64_t base = z0; base < z1; base += 63) {
            if (base > z0 && base + lane <= z1)
                zp = pos[base + lane];
            const int64_t zq = __shfl_down(zp, 1, 64);
            unsigned long long empty = __ballot(lane < 63 && base + lane < z1 && zp == zq);
            while (empty) {          // as many next to each other as there are groups
                const int first = __builtin_ctzll(empty), r = first + g;
                if (g < G && r < 64 && (empty >> r & 1)) {
                    double *to = C + crow(base + r) * ldc + col;
                    if (W == 2 && !half) {
                        spmm_pair v;
                        v.x = v.y = 0.0;
                        *reinterpret_cast<spmm_pair *>(to) = v;
                    } else {
                        *to = 0.0;
                    }
                }
                empty = first + G < 64 ? empty >> (first + G) << (first + G) : 0;
            }
        }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
    for (int64_t base = r0 + 1; base <= rn && base < nrows; base += 64) {
        const int64_t r = base + lane;
        int64_t p = 0, q = 0;
        const bool in = r <= rn && r < nrows;
        if (in) {
            p = pos[r];
            q = pos[r + 1];
        }
        if (in && p < q && p < e)
            sh.row[p - s] = (int32_t)(r - r0);
    }
    if (n == 0)
        return;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
    int last = 0;
    for (int t = 0; t < n; t += 64) {
        int m = wave_inclusive_max(t + lane < n ? sh.row[t + lane] : 0);
        m = m > last ? m : last;
        if (t + lane < n)
            sh.row[t + lane] = m;
        last = __builtin_amdgcn_readlane(m, 63);
    }
    if (lane == 0)
        sh.row[n] = tail ? last : -1;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");

    // ---- every group its run
    const int run = (n + G - 1) / G;
    auto cut = [&](int32_t r) { return (head && r == 0) || (tail && r == last); };
    auto begin = [&](int x) -> int {
        const int t = x * run < n ? x * run : n;
        if (t == 0 || t == n)
            return t;
        const int32_t r = sh.row[t];
        return sh.row[t - 1] != r || cut(r) ? t : (int)(pos[r0 + r + 1] - s);
    };
    const int a = begin(g), z = g < G ? begin(g + 1) : n;
    int longest = g < G ? z - a : 0, until = z;
    double ax = 0.0, ay = 0.0, hx = 0.0, hy = 0.0;          // hx, hy: the piece of a row that began before
    auto store = [&](int32_t r, double x, double y) {
        double *to = C + crow(r0 + r) * ldc + col;
        if (W == 2 && !half) {           // C is written once and not read again by this kernel
            spmm_pair v;
            v.x = x;
            v.y = y;
            __builtin_nontemporal_store(v, reinterpret_cast<spmm_pair *>(to));
        } else {
            __builtin_nontemporal_store(x, to);
        }
    };
    // rounds of gathers with every group on its run, and with the nonzeros dealt evenly
    const int even = (run + SPMM_U - 1) / SPMM_U;
    bool in_turn = __any(longest > SPMM_U * (even + 1));
    if (in_turn) {
        const int most = __builtin_amdgcn_readlane(wave_inclusive_max(longest), 63);
        const int next = SPMM_U * (lane + 1), at = next < n ? next : 1;
        in_turn = ((most + SPMM_U - 1) / SPMM_U - even) * SPMM_TURNS > __popcll(__ballot(next < n && sh.row[at - 1] == sh.row[at]));
    }
    if (!in_turn) {
        for (int t0 = 0; __any(t0 < longest); t0 += SPMM_U) {
            spmm_pair b[SPMM_U], c[ACC ? SPMM_U : 1];
            double v[SPMM_U];
            // bit u: the row of the batch's nonzero u ends with it (all of this read before the first is used: the adds of a
            // long row are one chain, and a look into LDS in it costs more than the rest)
            unsigned ends = 0;
            int32_t r = sh.row[a + t0 < n ? a + t0 : n - 1];
            const bool fresh = t0 == 0 || sh.row[a + t0 - 1 < n ? a + t0 - 1 : n - 1] != r;
    #pragma unroll
            for (int u = 0; u < SPMM_U; ++u) {
                const int t = a + t0 + u < n ? a + t0 + u : n - 1;
                const uint32_t j = (uint32_t)sh.crd[t];
                v[u] = sh.val[t];
                const double *at = SMALL ? reinterpret_cast<const double *>(reinterpret_cast<const char *>(B) +
                                                                            (j * (uint32_t)ldb + (uint32_t)from) * 8u)
                                         : B + (int64_t)j * ldb + from;
                if constexpr (W == 2)
                    b[u] = *reinterpret_cast<const spmm_pair *>(at);
                else
                    b[u].x = *at;
                const int32_t next = sh.row[t + 1];
                if constexpr (ACC) {         // where a row begins; the value of a row in pieces is added with them
                    if (t0 + u < longest && (u == 0 ? fresh : (ends >> (u - 1) & 1u) != 0) && !cut(r)) {
                        const double *to = C + crow(r0 + r) * ldc + from;
                        if constexpr (W == 2)
                            c[u] = *reinterpret_cast<const spmm_pair *>(to);
                        else
                            c[u].x = *to;
                    }
                }
                ends |= (unsigned)(next != r && t0 + u < longest) << u;
                r = next;
            }
            bool begins = fresh;
    #pragma unroll
            for (int u = 0; u < SPMM_U; ++u) {
                if constexpr (ACC)
                    if (begins && t0 + u < longest && !cut(sh.row[a + t0 + u])) {
                        ax = half ? c[u].y : c[u].x;
                        ay = W == 2 ? c[u].y : 0.0;
                    }
                const double x = ax + v[u] * (half ? b[u].y : b[u].x), y = W == 2 ? ay + v[u] * b[u].y : 0.0;
                ax = t0 + u < longest ? x : ax;
                ay = t0 + u < longest ? y : ay;
                begins = (ends >> u & 1u) != 0;
                if (begins) {
                    const int32_t mine = sh.row[a + t0 + u];
                    if (head && mine == 0) {
                        hx = ax;
                        hy = ay;
                    } else {
                        store(mine, ax, ay);
                    }
                    ax = ay = 0.0;
                }
            }
        }
    } else {
        // all groups gather, SPMM_U nonzeros each.  Rows that begin in a group's nonzeros are summed there; the sum of one
        // that goes on is handed from group to group, each adding its products in order.
        double ox = 0.0, oy = 0.0;           // what is open at the end of a batch
        const auto ended = [&](int32_t row, double x, double y) {
            if (head && row == 0) {
                hx = x;
                hy = y;
            } else {
                store(row, x, y);
            }
        };
        for (int t0 = 0; t0 < n; t0 += G * SPMM_U) {
            spmm_pair p[SPMM_U], c[ACC ? SPMM_U : 1];
            const int first = t0 + g * SPMM_U, mine = g < G ? n - first : 0;          // of the batch's nonzeros, the first mine
            unsigned ends = 0;
            int32_t r = sh.row[first < n ? first : n - 1];
            const bool fresh = first == 0 || sh.row[first - 1 < n ? first - 1 : n - 1] != r;
#pragma unroll
            for (int u = 0; u < SPMM_U; ++u) {
                const int t = first + u < n ? first + u : n - 1;
                const uint32_t j = (uint32_t)sh.crd[t];
                const double *at = SMALL ? reinterpret_cast<const double *>(reinterpret_cast<const char *>(B) +
                                                                            (j * (uint32_t)ldb + (uint32_t)from) * 8u)
                                         : B + (int64_t)j * ldb + from;
                if constexpr (W == 2)
                    p[u] = *reinterpret_cast<const spmm_pair *>(at);
                else
                    p[u].x = *at;
                const int32_t next = sh.row[t + 1];
                if constexpr (ACC) {
                    if (u < mine && (u == 0 ? fresh : (ends >> (u - 1) & 1u) != 0) && !cut(r)) {
                        const double *to = C + crow(r0 + r) * ldc + from;
                        if constexpr (W == 2)
                            c[u] = *reinterpret_cast<const spmm_pair *>(to);
                        else
                            c[u].x = *to;
                    }
                }
                ends |= (unsigned)(next != r && u < mine) << u;
                r = next;
            }
            // the first `lead` go on with a row of the nonzeros before
            const int own = mine < SPMM_U ? (mine > 0 ? mine : 0) : SPMM_U;
            const int lead = fresh ? 0 : ends != 0 && __builtin_ctz(ends) < own ? __builtin_ctz(ends) + 1 : own;
            bool begins = true;
            ax = ay = 0.0;
#pragma unroll
            for (int u = 0; u < SPMM_U; ++u) {
                const double v = sh.val[first + u < n ? first + u : n - 1];
                p[u].x = v * (half ? p[u].y : p[u].x);
                p[u].y = W == 2 ? v * p[u].y : 0.0;
                if (u >= lead && u < own) {
                    if constexpr (ACC)
                        if (begins && !cut(sh.row[first + u])) {
                            ax = half ? c[u].y : c[u].x;
                            ay = W == 2 ? c[u].y : 0.0;
                        }
                    ax += p[u].x;
                    ay += p[u].y;
                    begins = (ends >> u & 1u) != 0;
                    if (begins) {
                        ended(sh.row[first + u], ax, ay);
                        ax = ay = 0.0;
                    }
                }
            }
            unsigned long long on = __ballot(lead > 0 && sub == 0);
            while (on) {
                const int at = __builtin_ctzll(on);          // the first lane of group x
                on &= on - 1;
                const int before = (at > 0 ? at - L : (G - 1) * L) + sub;
                double sx = __shfl(at > 0 ? ax : ox, before & 63, 64), sy = W == 2 ? __shfl(at > 0 ? ay : oy, before & 63, 64) : 0.0;
                if (lane - sub == at) {
#pragma unroll
                    for (int u = 0; u < SPMM_U; ++u) {
                        sx = u < lead ? sx + p[u].x : sx;
                        sy = u < lead ? sy + p[u].y : sy;
                    }
                    if (ends >> (lead - 1) & 1u) {
                        ended(sh.row[first + lead - 1], sx, sy);
                    } else {
                        ax = sx;
                        ay = sy;
                    }
                }
            }
            ox = ax;
            oy = ay;
            if (t0 + G * SPMM_U >= n && g != (n - 1 - t0) / SPMM_U)          // the rest has been handed on
                ax = ay = 0.0;
        }
        longest = until = n;
    }
    if (!head && !tail)
        return;
    // ---- the pieces, a lane per column; what a group's run ends inside of is a piece of the first row or of the last
    if (longest > 0 && head && sh.row[until - 1] == 0 && sh.row[until] == 0) {
        hx = ax;
        hy = ay;
        ax = ay = 0.0;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
    if (g < G) {
        if (W == 2 && !half) {
            sh.piece[0][g * kt + 2 * sub] = hx;
            sh.piece[0][g * kt + 2 * sub + 1] = hy;
            sh.piece[1][g * kt + 2 * sub] = ax;
            sh.piece[1][g * kt + 2 * sub + 1] = ay;
        } else {
            sh.piece[0][g * kt + W * sub] = hx;
            sh.piece[1][g * kt + W * sub] = ax;
        }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
    if (lane >= kt)
        return;
    const int slot = 2 * tile_cols;
    double *slots = carry + (int64_t)blockIdx.y * nchunks * slot + lane;
    double began = 0.0, goes_on = 0.0;
    for (int x = 0; x < G; ++x) {
        began += sh.piece[0][x * kt + lane];
        goes_on += sh.piece[1][x * kt + lane];
    }
    const bool both = head && tail && last == 0;          // one row, through the chunk
    if (head)
        __hip_atomic_store(slots + chunk * slot, began, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (tail && !both)
        __hip_atomic_store(slots + chunk * slot + tile_cols, goes_on, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    // Whoever leaves the last piece of a row adds all of them, in order.  The pieces are written and read past the L2s
    // (agent scope), and this wavefront's have arrived before it counts itself in.
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    auto finish = [&](int64_t r) {
        const int64_t c0 = pos[r] / chunk_len, c1 = (pos[r + 1] - 1) / chunk_len;
        unsigned *count = arrived + (int64_t)blockIdx.y * nchunks + c0;
        unsigned before = 0;
        if (lane == 0)
            before = __hip_atomic_fetch_add(count, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if ((int64_t)(unsigned)__builtin_amdgcn_readfirstlane((int)before) != c1 - c0)
            return;
        if (lane == 0)
            __hip_atomic_store(count, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);          // for the next call on the workspace
        double *to = C + crow(r) * ldc + tile + lane;
        double sum = __hip_atomic_load(slots + c0 * slot + tile_cols, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (ACC)
            sum = *to + sum;
#pragma unroll 8
        for (int64_t c = c0 + 1; c <= c1; ++c)
            sum += __hip_atomic_load(slots + c * slot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        *to = sum;
    };
    if (head)
        finish(r0);
    if (tail && !both)
        finish(rn);
}

// ============================================================================
// SpMM, long rows: column sweep with the row sums in registers.
// ============================================================================
constexpr int SPMM_HW = 16;      // wavefronts per workgroup of the sweep
#ifndef COMET_SPMM_HR_BITS
#define COMET_SPMM_HR_BITS 3
#endif
#ifndef COMET_SPMM_HEAVY_MIN
#define COMET_SPMM_HEAVY_MIN 128
#endif
constexpr int SPMM_HRB = COMET_SPMM_HR_BITS;         // bits of a list entry that name the owned row
constexpr int SPMM_HR = 1 << SPMM_HRB;               // rows a wavefront can own
constexpr int SPMM_HCOLB = 20;                       // bits of a list entry for the column, counted from the first column of its XCD's range
// Workgroups of the sweep per XCD, one to a CU: all 32 CUs of an XCD when the sweep has the GPU to itself; fewer
// when the rows that are neither long nor single hold enough of the matrix to be worth running beside it - the
// chunk kernel that takes them waits on HBM, the sweep on the path from the L2 to the CU, and on the CUs the
// sweep leaves free the chunk kernel is not starved by it (inside a CU the older wavefronts of the sweep win every
// arbitration).  Measured on the benchmark matrix (ms per product): 32 and the kernels one after the other 0.329;
// side by side with 28 workgroups per XCD 0.336, 26 0.348, 25 0.355, 24 0.311, 23 0.319, 22 0.325.
constexpr int SPMM_HG_ALONE = 32, SPMM_HG_SHARED = 24;
constexpr int spmm_hbins(int g) { return g * SPMM_HW; }               // wavefronts (= row bins) per XCD
constexpr int spmm_hslots(int g) { return spmm_hbins(g) * SPMM_HR; }  // slots for partial sums per XCD
constexpr int spmm_hrows(int g) { return g * (SPMM_HW - 1) * SPMM_HR; }    // long rows the plan can hold
// Rows of middling length - too short for a register of their own over the whole sweep, long enough that eight
// partial sums cost less than fetching their rows of B from beyond the L2 - keep their sums in the LDS of the
// sweep's workgroups, 64 doubles per row and workgroup, and their entries ride in the lists of the wavefronts that
// own long rows, so they move through the columns at the sweep's pace and find their rows of B in the L2.
#ifndef COMET_SPMM_MED_MIN
#define COMET_SPMM_MED_MIN 32
#endif
constexpr int SPMM_MED_MIN_LEN = COMET_SPMM_MED_MIN;   // such a row has at least this many nonzeros
constexpr int SPMM_MSLOTS = 287;                        // sums a workgroup keeps in LDS, beside the entries of its lists (SWEEP_LDS)
constexpr int SPMM_HEAVY_MIN_LEN = COMET_SPMM_HEAVY_MIN;              // a long row has at least this many nonzeros
constexpr int64_t SPMM_UNEVEN_SWEEP = 24 << 20;         // bytes of B from which on rows of any alignment are swept
constexpr int SPMM_HCB = 32;                         // column blocks a wavefront's list is cut into

// One workgroup per (XCD x, row group g); workgroup w runs on XCD w % 8.  XCD x
// sweeps its eighth of the column range in ascending order, so a row of B is
// pulled into that XCD's L2 once and hit by every long row that uses it.  A
// wavefront owns up to SPMM_HR rows and keeps their sums in registers.  Its list
// is cut into 32 column blocks; inside a block the entries of one row follow
// each other, columns ascending, so a row is still summed in ascending column
// order, and a run of entries of one row is added into one plain register: the
// register file is indexed dynamically only where a run begins.
//
// Rows with a single nonzero ride along: the last wavefront of every workgroup
// owns no long rows; its list holds such rows, ordered by column, and it stores
// each product straight to that row of C.  It moves through the columns with
// the others, so its rows of B come out of the L2 window the long rows keep
// warm instead of being fetched from HBM one row each.  (Stores inside the
// lists of the long rows would stall them: loads and stores share one in-order
// counter, so every wait for a gather behind a store waits for that store too.)
//
// A lane owns two adjacent dense columns and a half-wavefront one row of B, so
// one load instruction fetches two rows, 16 bytes per lane: a CU takes 8-byte
// gathers out of the L2 at 23 bytes per clock however few rows are in play,
// 16-byte ones at 42 (measured with a gather-only kernel on a table of 0.3 to
// 4 MB per XCD).  The two halves take the even and the odd entries of the same
// run - runs are padded to even length by the plan, the pad carries no value -
// and their sums are added once, at the end.
//
// A wavefront holds 64 entries of its list at a time in LDS, where a half reads
// its entry with one 16-byte access; the next 64 are fetched while these are
// used.  (Entries one per lane, handed out by shuffles, and a branch for the pad
// of every pair took 23 instructions a pair, these 14.)  The
// gathers go out in batches of 8 pairs (16 rows of B) and the batch is added
// before the next one is issued: with sixteen wavefronts per CU the memory path
// is kept busy by the other wavefronts (batches of 4 or 16 pairs, before the
// wavefronts were kept together: 0.25 ms for the long rows alone instead of
// 0.19).  What bounds it is not settled: 29 M lines a product of 500000 rows and
// K = 64, 60 of them under way a CU, back in 257 clocks on average - 1.5 times
// as long as where every line comes from the L2; but the chunk kernel beside it
// keeps 140 to 160 under way.
// Entry = column - first column of the XCD's range (the low 24 bits, so that the byte offset of the row of B is one
// 24-bit multiply-add on the entry as it is) | real, first-of-run, kept-in-LDS | owned row << SPMM_E_ROW | partner-is-a-pad.  The slot of
// a row kept in LDS is the entry's second word.
constexpr int SPMM_HP = 8;       // pairs of entries per batch of gathers
constexpr int SPMM_E_REAL = 1 << 24;           // not a pad
constexpr int SPMM_E_FIRST = 1 << 25;          // the entry opens a run of one owned row
constexpr int SPMM_E_MED = 1 << 26;            // the entry adds into a sum kept in LDS, in the slot its second word names
constexpr int SPMM_E_ROW = 27;                 // where the owned row sits
constexpr int SPMM_E_LONE = 1 << (SPMM_E_ROW + SPMM_HRB);          // the odd entry of the pair is a pad
constexpr unsigned SPMM_E_COLMASK = 0xffffffu;
static_assert(SPMM_HCOLB <= 24 && SPMM_E_ROW + SPMM_HRB < 31, "an entry is 32 bits");
constexpr int SPMM_HWL = SPMM_HW - 1;          // wavefronts of a workgroup that own long rows

// SMALL: B spans less than 4 GiB and has fewer than 2^24 rows of fewer than 2^24 bytes, so the byte offset of a
// gather is one 24-bit multiply and one add in 32 bits on top of a scalar base, instead of a 64-bit multiply.
typedef int spmm_v4i __attribute__((ext_vector_type(4)));
typedef double spmm_v2d __attribute__((ext_vector_type(2)));

// A batch: the entries of SPMM_HP pairs, each half its own, and the rows of B they name.
struct HeavyBatch {
    spmm_v4i q[SPMM_HP];
    spmm_pair b[SPMM_HP];
};

// ring_half: the wavefront's 64 entries in LDS, from the half's first one on
template <bool SMALL>
__device__ inline void heavy_issue(HeavyBatch &x, const spmm_v4i *ring_half, int t0, int npairs,
                                   const double *__restrict__ B, int64_t ldb, int64_t col)
{
#pragma unroll
    for (int u = 0; u < SPMM_HP; ++u) {
        const int t = t0 + u < npairs ? t0 + u : npairs - 1;     // past the end: reload the last one, never used
        x.q[u] = ring_half[2 * t];
    }
#pragma unroll
    for (int u = 0; u < SPMM_HP; ++u) {
        const unsigned mine = (unsigned)x.q[u].x;
        if constexpr (SMALL) {
            const unsigned off = __umul24(mine, (unsigned)ldb * 8u) + (unsigned)col * 8u;
            x.b[u] = *reinterpret_cast<const spmm_pair *>(reinterpret_cast<const char *>(B) + off);
        } else {
            const int64_t j = (int64_t)(mine & SPMM_E_COLMASK);
            x.b[u] = *reinterpret_cast<const spmm_pair *>(B + j * ldb + col);
        }
    }
}

extern __shared__ double spmm_medium_sums[];
__device__ inline void heavy_add(double (&accx)[SPMM_HR], double (&accy)[SPMM_HR], double2 &run, int &run_slot,
                                 const HeavyBatch &x, int t0, int npairs, int at, bool active)
{
#pragma unroll
    for (int u = 0; u < SPMM_HP; ++u) {
        if (t0 + u < npairs) {
            const int e0 = __builtin_amdgcn_readfirstlane(x.q[u].x);
            if (e0 & SPMM_E_FIRST) {             // a run starts on an even entry
                accx[run_slot] = run.x;
                accy[run_slot] = run.y;
                run_slot = ((unsigned)e0 >> SPMM_E_ROW) & (SPMM_HR - 1);
                run.x = accx[run_slot];
                run.y = accy[run_slot];
            }
            const double v = __hiloint2double(x.q[u].w, x.q[u].z);
            if (!(e0 & (SPMM_E_MED | SPMM_E_LONE))) {
                run.x = __builtin_fma(v, x.b[u].x, run.x);
                run.y = __builtin_fma(v, x.b[u].y, run.y);
            } else if (e0 & SPMM_E_MED) {        // both entries of a pair are of the same kind
                const double px = v * x.b[u].x, py = v * x.b[u].y;
                // a row of middling length: its sum lives in LDS.  An add that returns nothing is issued and
                // forgotten; all entries of such a row are in this wavefront's list, in column order, and the adds
                // of one wavefront to one address are carried out in the order it issued them.
                if ((x.q[u].x & SPMM_E_REAL) && active) {
                    double *sum = spmm_medium_sums + x.q[u].y * 64 + at;
                    if (!(at & 1))                   // (an odd one is the neighbour's second column)
                        __hip_atomic_fetch_add(sum, px, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                    __hip_atomic_fetch_add(sum + 1, py, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                }
            } else if (x.q[u].x & SPMM_E_REAL) {         // a pad carries no value, not even zero times a row of B
                run.x = __builtin_fma(v, x.b[u].x, run.x);
                run.y = __builtin_fma(v, x.b[u].y, run.y);
            }
        }
    }
}

// The list of rows with one nonzero: a stream of pairs of entries, one entry per half-wavefront; each is one
// gather of B and one store to C.  Loads and stores share one in-order counter, so the loop is built to have
// the same number of each on every path: 32 entries at a time go through a 64-entry ring in LDS that only
// this wavefront touches (fetched one turn ahead, so no wait ever reaches back past a store), every lane always
// stores - pads, idle lanes and the turns past the end of the list store to a dump row - and nothing is
// branched around.  A wait for a batch of gathers then never includes the stores issued behind it.
// NB = pairs per batch; KB = where the turn's 32 entries start in the ring.
template <bool SMALL, bool ACC, int NB, int KB>
__device__ inline void single_issue(spmm_pair (&b)[NB], spmm_pair (&c)[NB], const spmm_v4i *ring_half, int t,
                                    const double *__restrict__ B, int64_t ldb, const double *__restrict__ C,
                                    int64_t ldc, int64_t col)
{
#pragma unroll
    for (int u = 0; u < NB; ++u) {
        const spmm_v4i q = ring_half[(KB + 2 * (t + u)) & 63];
        const unsigned mine = (unsigned)q.x;
        if constexpr (SMALL) {
            const unsigned off = __umul24(mine, (unsigned)ldb * 8u) + (unsigned)col * 8u;
            b[u] = *reinterpret_cast<const spmm_pair *>(reinterpret_cast<const char *>(B) + off);
        } else {
            const int64_t j = (int64_t)(mine & SPMM_E_COLMASK);
            b[u] = *reinterpret_cast<const spmm_pair *>(B + j * ldb + col);
        }
        if constexpr (ACC)
            c[u] = *reinterpret_cast<const spmm_pair *>(C + (int64_t)q.y * ldc + col);
    }
    __builtin_amdgcn_sched_barrier(0);       // the gathers stay in front of the stores of the other batch
}

template <bool ACC, int NB, int KB>
__device__ inline void single_store(const spmm_pair (&b)[NB], const spmm_pair (&c)[NB], const spmm_v4i *ring_half, int t,
                                    int64_t pair0, int64_t npairs, double *__restrict__ C, int64_t ldc, int64_t col,
                                    bool active, double *__restrict__ dump)
{
#pragma unroll
    for (int u = 0; u < NB; ++u) {
        const spmm_v4i q = ring_half[(KB + 2 * (t + u)) & 63];
        const double v = __hiloint2double(q.w, q.z);
        spmm_pair o;
        o.x = (ACC ? c[u].x : 0.0) + v * b[u].x;
        o.y = (ACC ? c[u].y : 0.0) + v * b[u].y;
        const bool ok = pair0 + t + u < npairs && active && (q.x & SPMM_E_REAL);
        double *dst = ok ? C + (int64_t)q.y * ldc + col : dump;
        __builtin_nontemporal_store(o, reinterpret_cast<spmm_pair *>(dst));       // C is written once, not read again
        if (u & 1)
            __builtin_amdgcn_sched_barrier(0);       // two pairs at a time: keeps the entries read ahead few
    }
}

// Where the wavefronts of a workgroup are in their lists, in steps of 1024 columns: one that is more than `slack` steps
// ahead of the last one waits for it.  The last one waits for nobody.  Left alone the four wavefronts of a SIMD drift
// apart - the older one wins every arbitration - and rows of B leave the L2 before the slow ones come to them (500000
// rows, K = 64: 11 M lines from beyond the L2s instead of 5, 374 us instead of 311).  us by columns that a wavefront may
// be ahead, 2048 / 3072 / 4096 / 8192: K = 64 311 / 313 / 318 / 341, 48 269 / 269 / 273 / 284, 32 231 / 223 / 225 / 232,
// 16 215 / 205 / 206 / 211.  sweep_slack says how far that may be.
constexpr int SPMM_PACE_LOG = 10;
struct SweepPace {
    int *at;                 // of every wavefront, in LDS
    int slack, wave, mine;
    __device__ inline void reach(int ent)
    {
        const int here = (int)((unsigned)__builtin_amdgcn_readfirstlane(ent) & SPMM_E_COLMASK) >> SPMM_PACE_LOG;
        if (here == mine)
            return;
        mine = here;
        const int lane = threadIdx.x & 63;
        if (lane == 0)
            __hip_atomic_store(&at[wave], here, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        const int l = lane & (SPMM_HW - 1);
        while (__any(__hip_atomic_load(&at[l], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) < here - slack))
            __builtin_amdgcn_s_sleep(1);
    }
    __device__ inline void done()
    {
        if ((threadIdx.x & 63) == 0)
            __hip_atomic_store(&at[wave], 1 << 30, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
};

template <bool SMALL, bool ACC>
__device__ inline void single_rows(const spmm_v4i *__restrict__ list, int64_t n, int lane, int half,
                                   const double *__restrict__ B, int64_t ldb, double *__restrict__ C, int64_t ldc,
                                   int64_t col, bool active, spmm_v4i *ring, double *__restrict__ dump, SweepPace &pace)
{
    constexpr int NB = ACC ? 4 : 8;
    spmm_pair b0[NB], b1[NB], c0[NB], c1[NB];
    const int64_t npairs = n >> 1;           // the list has an even number of entries
    const int l32 = lane & 31;
    auto fetch = [&](int64_t turn) {         // the 32 entries of a turn, one per lane of each half
        const int64_t i = turn * 32 + l32;
        return __builtin_nontemporal_load(list + (i < n ? i : n - 1));
    };
    const spmm_v4i *ring_half = ring + half;
    ring[l32] = fetch(0);
    spmm_v4i next = fetch(1);
    single_issue<SMALL, ACC, NB, 0>(b0, c0, ring_half, 0, B, ldb, C, ldc, col);
    // a turn = 16 pairs: its entries, and those of the next turn for the gathers issued ahead, are in the ring
    auto turn = [&](auto kb, int64_t k) {
        constexpr int KB = decltype(kb)::value;
        pace.reach(next.x);
        ring[((KB + 32) & 63) + l32] = next;            // turn k + 1, over the entries of turn k - 1
        next = fetch(k + 2);
        for (int t = 0; t < 16; t += 2 * NB) {
            single_issue<SMALL, ACC, NB, KB>(b1, c1, ring_half, t + NB, B, ldb, C, ldc, col);
            single_store<ACC, NB, KB>(b0, c0, ring_half, t, k * 16, npairs, C, ldc, col, active, dump);
            single_issue<SMALL, ACC, NB, KB>(b0, c0, ring_half, t + 2 * NB, B, ldb, C, ldc, col);
            single_store<ACC, NB, KB>(b1, c1, ring_half, t + NB, k * 16, npairs, C, ldc, col, active, dump);
        }
    };
    for (int64_t k = 0; k * 16 < npairs; k += 2) {
        turn(std::integral_constant<int, 0>(), k);
        turn(std::integral_constant<int, 32>(), k + 1);
    }
}

// the sweep's LDS without the sums of the rows of middling length: 64 entries and a place of every wavefront
constexpr size_t SWEEP_LDS = SPMM_HW * (64 * sizeof(spmm_v4i) + sizeof(int));
static_assert(SWEEP_LDS + SPMM_MSLOTS * 64 * sizeof(double) <= 160 * 1024, "as many sums as a plan hands out fit a CU's LDS");

template <bool SMALL, bool ACC>
__global__ __launch_bounds__(SPMM_HW * 64) void spmm_heavy_sweep(
    const int64_t *__restrict__ seg, const HeavyEnt *__restrict__ hent, const double *__restrict__ B, int64_t ldb,
    int64_t K, double *__restrict__ partial, double *__restrict__ C, int64_t ldc, int G, int64_t xcols, int nslots,
    double *__restrict__ partial_medium, int slack)
{
    const int lane = threadIdx.x & 63, half = lane >> 5, sub = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int x = blockIdx.x & 7, g = blockIdx.x >> 3;
    B += (int64_t)x * xcols * ldb;          // the entries count columns from the first one of this XCD's range
    // A lane's two columns.  Where K is odd, the last lane has the last two: the first of them is its neighbour's second,
    // and both lanes add it and store it alike.  Idle lanes gather a valid address and store nothing.
    int64_t col = (int64_t)blockIdx.y * 64 + 2 * sub;
    const bool active = col < K;
    if (col > K - 2)
        col = K - 2;
    const int at = (int)(col - (int64_t)blockIdx.y * 64);          // in the tile (of an active lane)
    const int64_t bin = ((int64_t)x * G + g) * SPMM_HW + wave;
    const int64_t s = seg[bin], e = seg[bin + 1];          // both even
    const spmm_v4i *list = reinterpret_cast<const spmm_v4i *>(hent);
    __shared__ spmm_v4i rings[SPMM_HW][64];          // entries of every wavefront's list
    __shared__ int reached[SPMM_HW];
    if (lane == 0)
        reached[wave] = s < e ? 0 : 1 << 30;
    __syncthreads();
    SweepPace pace{reached, slack, wave, 0};
    if (wave == SPMM_HWL) {                   // the wavefront of the rows with one nonzero
        if (s < e)             // this wavefront's slots of `partial` hold no row: the dump
            single_rows<SMALL, ACC>(list + s, e - s, lane, half, B, ldb, C, ldc, col, active, rings[wave],
                                    partial + bin * SPMM_HR * K + col, pace);
        pace.done();
        return;
    }
    double accx[SPMM_HR], accy[SPMM_HR];      // two plain arrays: each is indexed through M0, a double2 array is not
#pragma unroll
    for (int r = 0; r < SPMM_HR; ++r)
        accx[r] = accy[r] = 0.0;
    // the sums in LDS whose entries this wavefront's list holds: slot mod SPMM_HWL = wavefront
    for (int sl = wave; sl < nslots; sl += SPMM_HWL)
        spmm_medium_sums[sl * 64 + lane] = 0.0;
    if (s < e) {
        HeavyBatch x;
        double2 run = make_double2(0.0, 0.0);
        int run_slot = 0;
        spmm_v4i *ring = rings[wave];
        const spmm_v4i *ring_half = ring + half;
        const auto fetch = [&](int64_t at) {         // behind the list's last entry: that one
            const int64_t i = at + lane;
            return __builtin_nontemporal_load(list + (i < e ? i : e - 1));
        };
        const auto put = [&](spmm_v4i q) {           // the wavefront's own reads of the ring are issued before
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
            ring[lane] = q;
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
        };
        put(fetch(s));
        spmm_v4i next = fetch(s + 64);
        int64_t base = s;
        // 32 pairs at a time, the first batch of the next 32 in flight over the loop's back edge
        heavy_issue<SMALL>(x, ring_half, 0, (int)((e - s < 64 ? e - s : 64) >> 1), B, ldb, col);
        while (e - base >= 64) {
#pragma unroll
            for (int t0 = 0; t0 < 32; t0 += SPMM_HP) {
                heavy_add(accx, accy, run, run_slot, x, 0, SPMM_HP, at, active);
                if (t0 + SPMM_HP < 32)
                    heavy_issue<SMALL>(x, ring_half, t0 + SPMM_HP, 32, B, ldb, col);
            }
            base += 64;
            if (base < e) {
                pace.reach(next.x);
                put(next);
                next = fetch(base + 64);
                heavy_issue<SMALL>(x, ring_half, 0, (int)((e - base < 64 ? e - base : 64) >> 1), B, ldb, col);
            }
        }
        const int np = (int)((e - base) >> 1);
        for (int t0 = 0; t0 < np; t0 += SPMM_HP) {
            heavy_add(accx, accy, run, run_slot, x, t0, np, at, active);
            if (t0 + SPMM_HP < np)
                heavy_issue<SMALL>(x, ring_half, t0 + SPMM_HP, np, B, ldb, col);
        }
        accx[run_slot] = run.x;
        accy[run_slot] = run.y;
        pace.done();
    }
    {   // this wavefront's sums in LDS: one partial sum per row and XCD, like the long rows'
        const int64_t c1 = (int64_t)blockIdx.y * 64 + lane;
        double *mout = partial_medium + ((int64_t)x * G + g) * nslots * K;
        for (int sl = wave; sl < nslots; sl += SPMM_HWL)
            if (c1 < K)
                mout[(int64_t)sl * K + c1] = spmm_medium_sums[sl * 64 + lane];
    }
    // even entries + odd entries, then the lower half writes both columns
    double *out = partial + (((int64_t)x * G + g) * SPMM_HW + wave) * SPMM_HR * K;
#pragma unroll
    for (int r = 0; r < SPMM_HR; ++r) {
        const double ox = __shfl_down(accx[r], 32, 64), oy = __shfl_down(accy[r], 32, 64);
        if (active && half == 0) {
            out[(int64_t)r * K + col] = accx[r] + ox;
            out[(int64_t)r * K + col + 1] = accy[r] + oy;
        }
    }
}

// Steps that a wavefront of the sweep may be ahead of the last one.  Within a block of columns a list goes from row to row,
// each time from the block's first column to its last: both ends of a block have to be close enough, or wavefronts wait for
// others that are in the same block.  2 or 3 steps hold a block of up to 2048 or 3072 columns, 524288 or 786432 in all; us
// with 2, 3 steps | with what the block takes | without waiting, K = 64: 10^6 columns 765 | 4: 744 | 1004, 500000 rows of
// 4 M columns 825 | 16: 587 | 713, 250000 of 8 M 803 | 31: 408 | 415; K = 16: 10^6 373 | 4: 368 | 383.
static int sweep_slack(int64_t xcols, int64_t K)
{
    const int64_t block = ceil_div(xcols, SPMM_HCB);
    return (int)std::max<int64_t>(K >= 48 ? 2 : 3, ((block - 1) >> SPMM_PACE_LOG) + 1);
}

// C[rows[i]][0..K) = 0
__global__ void zero_listed_rows_f64(double *__restrict__ C, const int32_t *__restrict__ rows, int64_t nlisted,
                                     int64_t K, int64_t ldc)
{
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t total = nlisted * K, step = (int64_t)gridDim.x * blockDim.x;
    for (; i < total; i += step)
        C[(int64_t)rows[i / K] * ldc + (i % K)] = 0.0;
}

__global__ void fill_rows_f64(double *__restrict__ C, int64_t nrows, int64_t K, int64_t ldc, double v)
{
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    int64_t total = nrows * K;
    int64_t step = (int64_t)gridDim.x * blockDim.x;
    for (; i < total; i += step)
        C[(i / K) * ldc + (i % K)] = v;
}

static Workspace g_spmm_carry, g_spmm_arrived;

// Nonzeros of a chunk: a half or a quarter of SPMM_CH where that makes 8192 wavefronts at most, 32 for every CU.  (The
// number is also what the scratch of the form without allocations holds, which cuts rows in the same places.)
constexpr int64_t SPMM_SHORT_CHUNKS = 8192;
// Tiles narrower than 64 columns where that makes 4096 wavefronts at most: more groups for the same nonzeros.  Only for a B
// that an L2 holds, since a tile's part of a row of B is lines of its own.  us with tiles of 64 / narrow ones, zipf, 16
// nonzeros a row: 2000 rows K = 64 22.4 / 15.6, 4000 rows K = 48 23.7 / 15.5, 8000 rows K = 64 28.6 / 22.3; with 8192
// wavefronts at most 16000 rows and K = 17 took 24.9 in place of 20.7; 120000 rows and K = 33, B 32 MB, 102 in place of 87.
constexpr int64_t SPMM_NARROW_B = 4 << 20, SPMM_NARROW_WAVES = 4096;
static int spmm_chunk_len(int64_t nnz, int64_t tiles)
{
    for (int len = SPMM_CH / 4; len < SPMM_CH; len *= 2)
        if (tiles * ceil_div(nnz, len) <= SPMM_SHORT_CHUNKS)
            return len;
    return SPMM_CH;
}

// How a product is cut: chunks of len nonzeros, tiles of `cols` columns.
struct SpmmShape {
    int len, cols;
    int64_t chunks, tiles;
};
static SpmmShape spmm_shape(const Csr *a, int64_t K)
{
    SpmmShape h;
    h.cols = 64;
    if (a->ncols * K * 8 <= SPMM_NARROW_B)
        for (int w = 16; w < 64; w += 8) {
            const int64_t tiles = ceil_div(K, w);
            if (tiles * ceil_div(a->nnz, SPMM_CH / 4) <= SPMM_NARROW_WAVES) {
                h.cols = 2 * (int)ceil_div(K, 2 * tiles);
                break;
            }
        }
    h.tiles = ceil_div(K, h.cols);
    h.len = spmm_chunk_len(a->nnz, h.tiles);
    h.chunks = ceil_div(a->nnz, h.len);
    return h;
}

static int spmm_chunk_scratch(const SpmmShape &h)
{
    COMET_CHK(g_spmm_carry.ensure(sizeof(double) * 2 * (size_t)h.cols * (size_t)(h.tiles * h.chunks), false));
    return g_spmm_arrived.ensure(sizeof(unsigned) * (size_t)(h.tiles * h.chunks), true);
}

// ---------------------------------------------------------------------------
// Chunks by columns.  A chunk of a row of many chunks has its columns in a short
// range, and taken in the order of the matrix every chunk's rows of B come from
// somewhere else.  So, from a matrix's second product on, the chunks are taken in
// the order of their columns, an eighth of them by every XCD: an L2 then sees an
// eighth of B, ascending, in place of all of it (workgroup w runs on XCD w % 8).
// Pieces of rows are added in the order of the chunks' numbers, so the sums are what they are as stored, unless the chunks are
// shorter (below): a long row is cut in more places then, and its rounding may differ from that of the first product.
// It pays where rows of four chunks and more hold half of the matrix and few columns do not (SPMM_CROWDED): graphs
// whose columns are as uneven as their rows have the rows of B that count in every L2 as it is.
// us, zipf, 16 nonzeros a row, as stored / by columns: 30000 rows K = 64 51 / 38, 60001 rows K = 33 61 / 45, 250000 rows
// K = 15 146 / 99, 500000 rows K = 3 153 / 121, K = 15 298 / 182, 1000000 rows K = 8 343 / 249.
// Chunks of half the length keep a window of a larger B in the L2: 120000 rows K = 33 83 / 75, 250000 rows K = 32 131 / 105;
// below 28 MiB of B, or 48 with 16 columns and less, they only cost (120000 rows K = 8 38 / 39, 500000 rows K = 8 119 / 128).
// The sweep takes over where B is larger than 56 MiB, or 80 with 32 columns and less; by columns / sweep: 150000 rows K = 48
// 93 / 95, K = 56 114 / 104, 250000 rows K = 32 105 / 127, 500000 rows K = 17 206 / 225, K = 21 245 / 229.
// ---------------------------------------------------------------------------
constexpr int64_t SPMM_ORDER_B = 1 << 20;               // bytes of B from which on chunks go by columns

// keys[c]: where chunk c has its columns, in 65536ths of the matrix; a chunk of several rows, which has them everywhere, goes
// where its number puts it
__global__ __launch_bounds__(256) void spmm_order_keys(const int32_t *__restrict__ crd, int64_t nnz, int64_t ncols,
                                                       const int32_t *__restrict__ chunk_row, int chunk_len, int64_t nchunks, uint64_t *__restrict__ keys, uint32_t *__restrict__ idx)
{
    const int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (c >= nchunks)
        return;
    const int64_t s = c * chunk_len, e = s + chunk_len;
    uint64_t key = (uint64_t)(c * 65536 / nchunks);
    if (e < nnz && chunk_row[s / SPMM_GRAIN] == chunk_row[e / SPMM_GRAIN])
        key = (uint64_t)((int64_t)crd[s + chunk_len / 2] * 65536 / ncols);
    keys[c] = key;
    idx[c] = (uint32_t)c;
}

static Workspace g_spmm_order, g_long_entries;
static int spmm_plan(Csr *a);

static int spmm_order(Csr *a, const SpmmShape &h)
{
    uint32_t *&kept = a->spmm_order[h.len / SPMM_GRAIN / 2];
    if (kept)
        return COMET_HIP_OK;
    COMET_CHK(spmm_plan(a));
    COMET_CHK(g_spmm_order.ensure((2 * sizeof(uint64_t) + sizeof(uint32_t)) * (size_t)h.chunks, false));
    uint64_t *keys = (uint64_t *)g_spmm_order.ptr, *sorted = keys + h.chunks;
    uint32_t *idx = (uint32_t *)(sorted + h.chunks), *order = nullptr;
    COMET_HIPCHK(dev_malloc((void **)&order, sizeof(uint32_t) * (size_t)h.chunks));
    spmm_order_keys<<<dim3((unsigned)ceil_div(h.chunks, 256)), dim3(256), 0, stream()>>>(
        a->crd, a->nnz, a->ncols, a->spmm_chunk_row, h.len, h.chunks, keys, idx);
    const int rc = sort_pairs_u64_u32(keys, sorted, idx, order, h.chunks, 16);
    if (rc != COMET_HIP_OK) {
        (void)dev_free(order);
        return rc;
    }
    kept = order;
    return COMET_HIP_OK;
}

// held[i] += entries of the rows of 128 << i entries and more
__global__ __launch_bounds__(256) void spmm_long_entries(int64_t nrows, const int64_t *__restrict__ pos,
                                                         unsigned long long *__restrict__ held)
{
    int64_t mine[SPMM_LONG_KINDS] = {};
    for (int64_t r = (int64_t)blockIdx.x * 256 + threadIdx.x; r < nrows; r += (int64_t)gridDim.x * 256) {
        const int64_t len = pos[r + 1] - pos[r];
#pragma unroll
        for (int i = 0; i < SPMM_LONG_KINDS; ++i)
            mine[i] += len >= (SPMM_HEAVY_MIN_LEN << i) ? len : 0;
    }
#pragma unroll
    for (int i = 0; i < SPMM_LONG_KINDS; ++i) {
        for (int d = 32; d > 0; d >>= 1)
            mine[i] += ((int64_t)__shfl_down((int)(mine[i] >> 32), d, 64) << 32) + (int64_t)(uint32_t)__shfl_down((int)mine[i], d, 64);
        if ((threadIdx.x & 63) == 0 && mine[i] > 0)
            atomicAdd(&held[i], (unsigned long long)mine[i]);
    }
}

// a->long_nnz: asked of the device once, 20 us
static int spmm_long_rows(Csr *a)
{
    if (a->long_nnz[0] >= 0)
        return COMET_HIP_OK;
    unsigned long long *held = nullptr;
    const size_t bytes = SPMM_LONG_KINDS * sizeof *held;
    COMET_CHK(mailbox((void **)&held));
    COMET_CHK(g_long_entries.ensure(bytes, false));
    COMET_HIPCHK(hipMemsetAsync(g_long_entries.ptr, 0, bytes, stream()));
    spmm_long_entries<<<dim3((unsigned)std::min<int64_t>(ceil_div(a->nrows, 256), 2 * (int64_t)num_cus())), dim3(256), 0, stream()>>>(
        a->nrows, a->pos, (unsigned long long *)g_long_entries.ptr);
    COMET_HIPCHK(hipGetLastError());
    COMET_HIPCHK(hipMemcpyAsync(held, g_long_entries.ptr, bytes, hipMemcpyDeviceToHost, stream()));
    COMET_CHK(stream_wait());
    for (int i = 0; i < SPMM_LONG_KINDS; ++i)
        a->long_nnz[i] = (int64_t)((volatile unsigned long long *)held)[i];
    a->heavy_nnz = a->long_nnz[0];
    return COMET_HIP_OK;
}

// Columns that hold four times what they would if all held the same.  Where such columns hold this share of the entries, chunks
// stay as they are stored.  Share, and us as stored / by columns: columns n * u^p of a random u, rows as zipf, 60000 rows K = 33
// p = 2 (0.10) 54.8 / 44.7, p = 4 (0.30) 44.0 / 39.5, p = 6 (0.38) 37.9 / 37.2, the same columns at random places 38.9 / 35.1,
// 250000 rows K = 21 p = 6 (0.42) 113.9 / 91.2; R-MAT scale 13, 32 edges a vertex (0.50) K = 17 21.6 / 22.1, K = 32 23.6 / 23.9,
// 18 and 16 (0.73) K = 17 156 / 196, K = 31 194 / 223, 17 and 32 (0.75) K = 31 162 / 196, K = 48 201 / 232, its vertices at random
// places K = 33 185 / 200.  The sweep is no way out for these either: 18 and 16 K = 24 156 / 518 swept, 17 and 32 K = 32 145 / 457.
constexpr double SPMM_CROWDED = 0.46;
constexpr int64_t SPMM_COLUMN_SAMPLE = 1 << 19;           // entries that are looked at, about

// count[j] += samples in column j: one at a random place of every `every` entries (at the same place of each it might be of
// every row the first)
__global__ __launch_bounds__(256) void spmm_column_counts(int64_t samples, int64_t every, int64_t nnz, const int32_t *__restrict__ crd,
                                                          uint32_t *__restrict__ count)
{
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= samples)
        return;
    const int64_t p = i * every + (int64_t)((uint32_t)i * 0x9E3779B1u >> 8) % every;
    atomicAdd(&count[crd[p < nnz ? p : nnz - 1]], 1u);
}

// *held += samples in columns of `least` and more
__global__ __launch_bounds__(256) void spmm_column_share(int64_t ncols, const uint32_t *__restrict__ count, uint32_t least,
                                                         unsigned long long *__restrict__ held)
{
    int mine = 0;          // all samples fit
    for (int64_t j = (int64_t)blockIdx.x * 256 + threadIdx.x; j < ncols; j += (int64_t)gridDim.x * 256)
        mine += count[j] >= least ? (int)count[j] : 0;
    for (int d = 32; d > 0; d >>= 1)
        mine += __shfl_down(mine, d, 64);
    if ((threadIdx.x & 63) == 0 && mine > 0)
        atomicAdd(held, (unsigned long long)mine);
}

// a->crowded_columns: asked of the device once
static int spmm_crowded(Csr *a)
{
    const int64_t every = ceil_div(a->nnz, SPMM_COLUMN_SAMPLE), samples = ceil_div(a->nnz, every);
    const size_t bytes = sizeof(unsigned long long) + sizeof(uint32_t) * (size_t)a->ncols;
    unsigned long long *word = nullptr, *held = nullptr;
    COMET_CHK(mailbox((void **)&word));
    COMET_HIPCHK(dev_malloc((void **)&held, bytes));          // given back: 4 bytes a column may be much
    const auto run = [&]() -> int {
        uint32_t *count = (uint32_t *)(held + 1);
        COMET_HIPCHK(hipMemsetAsync(held, 0, bytes, stream()));
        spmm_column_counts<<<dim3((unsigned)ceil_div(samples, 256)), dim3(256), 0, stream()>>>(samples, every, a->nnz, a->crd, count);
        // (a column that happens to be seen a few times is not a crowded one)
        const uint32_t least = (uint32_t)std::max<int64_t>(8, ceil_div(4 * samples, a->ncols));
        spmm_column_share<<<dim3((unsigned)std::min<int64_t>(ceil_div(a->ncols, 256), 2 * (int64_t)num_cus())), dim3(256), 0, stream()>>>(
            a->ncols, count, least, held);
        COMET_HIPCHK(hipGetLastError());
        COMET_HIPCHK(hipMemcpyAsync(word, held, sizeof *word, hipMemcpyDeviceToHost, stream()));
        return stream_wait();
    };
    const int rc = run();
    (void)dev_free(held);
    COMET_CHK(rc);
    a->crowded_columns = (double)*(volatile unsigned long long *)word > SPMM_CROWDED * (double)samples;
    return COMET_HIP_OK;
}

// Whether a product of a matrix that has been multiplied before goes through its chunks by columns, *h as it is cut then.
// *stored: it does not, because of its columns, and is not to be swept.
static bool spmm_by_columns(Csr *a, int64_t K, SpmmShape *h, bool *stored)
{
    *stored = false;
    const int64_t bytes = a->ncols * K * 8, most = K < 16 ? INT64_MAX : (K > 32 ? 56 : 80) << 20;
    if (a->nnz == 0 || bytes < SPMM_ORDER_B || bytes > most || a->rowmap || getenv("COMET_HIP_SPMM_NO_COLUMNS") ||
        getenv("COMET_HIP_SPMM_GROUPS") || getenv("COMET_HIP_SPMM_MEDIUM"))
        return false;           // the last two shape the sweep, and ask for it
    SpmmShape cut = *h;
    if (cut.len == SPMM_CH && bytes > (K > 16 ? 28 << 20 : 48 << 20)) {
        cut.len = SPMM_CH / 2;
        cut.chunks = ceil_div(a->nnz, cut.len);
    }
    if (cut.chunks >= 1ll << 31 || (a->long_nnz[0] < 0 && !plan_made([&] { return spmm_long_rows(a); })))
        return false;
    if (a->long_nnz[1 + cut.len / SPMM_GRAIN / 2] * 2 < a->nnz || (a->crowded_columns < 0 && !plan_made([&] { return spmm_crowded(a); })))
        return false;
    *stored = a->crowded_columns == 1;
    if (*stored || !plan_made([&] { return spmm_order(a, cut); }))
        return false;
    *h = cut;
    return true;
}

static int spmm_plan(Csr *a)
{
    const int64_t nchunks = ceil_div(a->nnz, SPMM_GRAIN);
    if (a->spmm_chunk_row && a->spmm_nchunks == nchunks)
        return COMET_HIP_OK;
    if (a->spmm_chunk_row) {
        COMET_HIPCHK(dev_free(a->spmm_chunk_row));
        a->spmm_chunk_row = nullptr;
    }
    COMET_HIPCHK(dev_malloc((void **)&a->spmm_chunk_row, sizeof(int32_t) * (size_t)(nchunks > 0 ? nchunks : 1)));
    a->spmm_nchunks = nchunks;
    if (nchunks > 0) {
        KernelTimer t("spmm_chunk_rows");
        spmm_chunk_rows<<<dim3((unsigned)ceil_div(nchunks, 256)), dim3(256), 0, stream()>>>(
            a->pos, a->nrows, nchunks, SPMM_GRAIN, a->spmm_chunk_row, nullptr, 0);
    }
    COMET_HIPCHK(hipGetLastError());
    return COMET_HIP_OK;
}


// ---------------------------------------------------------------------------
// Plan for the sweep: pick the long rows, deal them to the 512 wavefronts of an
// XCD so that every wavefront gets the same number of nonzeros, and re-store
// their nonzeros as one list per (XCD, wavefront), ordered by column.
// ---------------------------------------------------------------------------
// cnt[h * 8 + x] = nonzeros of long row h whose column lies in the range XCD x sweeps
__global__ void heavy_count(int64_t nheavy, const int32_t *__restrict__ hrow, const int64_t *__restrict__ pos,
                            const int32_t *__restrict__ crd, int64_t xcols, int32_t *__restrict__ cnt)
{
    const int64_t h = (int64_t)blockIdx.x * (blockDim.x >> 3) + (threadIdx.x >> 3);
    const int x = threadIdx.x & 7;
    if (h >= nheavy)
        return;
    const int64_t s = pos[hrow[h]], e = pos[hrow[h] + 1];
    auto first_at_least = [&](int64_t c) {
        int64_t lo = s, hi = e;
        while (lo < hi) {
            const int64_t mid = (lo + hi) >> 1;
            if (crd[mid] < c)
                lo = mid + 1;
            else
                hi = mid;
        }
        return lo;
    };
    cnt[h * 8 + x] = (int32_t)(first_at_least((int64_t)(x + 1) * xcols) - first_at_least((int64_t)x * xcols));
}

__global__ void heavy_make_keys(int64_t nheavy, const int32_t *__restrict__ hrow, const int32_t *__restrict__ hcode,
                                const int64_t *__restrict__ hstart, const int64_t *__restrict__ pos,
                                const int32_t *__restrict__ crd, int64_t xcols, int hbins,
                                uint64_t *__restrict__ keys, uint32_t *__restrict__ idx)
{
    const int64_t h = blockIdx.x;
    if (h >= nheavy)
        return;
    const int64_t ps = pos[hrow[h]], len = pos[hrow[h] + 1] - ps, o = hstart[h];
    for (int64_t t = threadIdx.x; t < len; t += blockDim.x) {
        const uint64_t c = (uint64_t)(uint32_t)crd[ps + t];
        const uint64_t x = c / (uint64_t)xcols;
        const uint64_t cb = (c - x * (uint64_t)xcols) * SPMM_HCB / (uint64_t)xcols;   // column block inside the range
        const uint64_t code = (uint64_t)hcode[x * nheavy + h];       // wavefront * SPMM_HR + slot on that XCD
        keys[o + t] = ((((x * hbins + (code >> SPMM_HRB)) * SPMM_HCB + cb) * (2 * SPMM_HR) +
                        (code & (SPMM_HR - 1))) << 28) | c;
        idx[o + t] = (uint32_t)(ps + t);
    }
}

// The rows with one nonzero, dealt round-robin to the last wavefronts of the workgroups of the XCD that sweeps
// their column; these wavefronts own no long rows, so their lists are simply ordered by column.
__global__ void single_make_keys(int64_t nsingle, const int32_t *__restrict__ srow, const int64_t *__restrict__ pos,
                                 const int32_t *__restrict__ crd, int64_t xcols, int groups,
                                 uint64_t *__restrict__ keys, uint32_t *__restrict__ idx)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nsingle)
        return;
    const uint64_t c = (uint64_t)(uint32_t)crd[pos[srow[i]]];
    const uint64_t x = c / (uint64_t)xcols;
    const uint64_t cb = (c - x * (uint64_t)xcols) * SPMM_HCB / (uint64_t)xcols;
    const uint64_t bin = (uint64_t)(i % groups) * SPMM_HW + SPMM_HWL;
    keys[i] = ((((x * (uint64_t)spmm_hbins(groups) + bin) * SPMM_HCB + cb) * (2 * SPMM_HR) + SPMM_HR) << 28) | c;
    idx[i] = (uint32_t)i;
}

// The rows of middling length: row m of their list is kept by workgroup m % groups of every XCD, in slot
// j = m / groups, and its entries go into the list of wavefront j % SPMM_HWL of that workgroup, behind the runs of
// the wavefront's long rows in every column block.  idx = the entry's place among all such entries.
__global__ void medium_make_keys(int64_t nmedium, const int32_t *__restrict__ mrow, const int64_t *__restrict__ mstart,
                                 const int64_t *__restrict__ pos, const int32_t *__restrict__ crd, int64_t xcols,
                                 int groups, uint64_t *__restrict__ keys, uint32_t *__restrict__ idx)
{
    const int64_t m = blockIdx.x;
    if (m >= nmedium)
        return;
    const int64_t ps = pos[mrow[m]], len = pos[mrow[m] + 1] - ps, o = mstart[m];
    const uint64_t bin = (uint64_t)(m % groups) * SPMM_HW + (uint64_t)((m / groups) % SPMM_HWL);
    for (int64_t t = threadIdx.x; t < len; t += blockDim.x) {
        const uint64_t c = (uint64_t)(uint32_t)crd[ps + t];
        const uint64_t x = c / (uint64_t)xcols;
        const uint64_t cb = (c - x * (uint64_t)xcols) * SPMM_HCB / (uint64_t)xcols;
        keys[o + t] = ((((x * (uint64_t)spmm_hbins(groups) + bin) * SPMM_HCB + cb) * (2 * SPMM_HR) + SPMM_HR + 1) << 28) | c;
        idx[o + t] = (uint32_t)(o + t);
    }
}

// first[e] = 1 where entry e of the ordered list opens a run (another row, column block or wavefront)
__global__ void heavy_mark_runs(int64_t n, const uint64_t *__restrict__ keys, int64_t *__restrict__ first)
{
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e < n)
        first[e] = (e == 0 || (keys[e - 1] >> 28) != (keys[e] >> 28)) ? 1 : 0;
}

// start[r] = first entry of run r (runs[e] = runs opened before e); start[nruns] = n
__global__ void heavy_run_starts(int64_t n, const int64_t *__restrict__ first, const int64_t *__restrict__ runs,
                                 int64_t *__restrict__ start)
{
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e < n && first[e])
        start[runs[e]] = e;
    if (e == n)
        start[runs[n]] = n;
}

__global__ void heavy_run_odd(int64_t nruns, const int64_t *__restrict__ start, int64_t *__restrict__ odd)
{
    const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (r < nruns)
        odd[r] = (start[r + 1] - start[r]) & 1;
}

// Writes the list with every run padded to even length: entry e of run r lands at e + (pads in front of r).
// idx is a position in val for a long row's entry, a position in srow for a row with one nonzero, and a place
// among the entries of the rows of middling length for one of those.
__global__ void heavy_fill(int64_t n, const uint64_t *__restrict__ keys, const uint32_t *__restrict__ idx,
                           const double *__restrict__ val, const int64_t *__restrict__ pos,
                           const int32_t *__restrict__ srow, int64_t nmedium, const int32_t *__restrict__ mrow,
                           const int64_t *__restrict__ mstart, int groups, const int64_t *__restrict__ first,
                           const int64_t *__restrict__ runs, const int64_t *__restrict__ start,
                           const int64_t *__restrict__ pads, int64_t xcols, HeavyEnt *__restrict__ hent)
{
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= n)
        return;
    const uint64_t k = keys[e];
    const int64_t r = runs[e] + first[e] - 1;
    const int64_t p = e + pads[r];
    const bool direct = ((k >> 28) & SPMM_HR) != 0;
    const uint64_t c = k & 0xfffffffull;
    const uint32_t col = (uint32_t)(c - (c / (uint64_t)xcols) * (uint64_t)xcols);     // inside its XCD's range
    HeavyEnt out;
    if (direct && ((k >> 28) & 1)) {          // a row of middling length: which one, from the entry's place
        const int64_t at = idx[e];
        int64_t lo = 0, hi = nmedium - 1;      // the last m with mstart[m] <= at
        while (lo < hi) {
            const int64_t mid = (lo + hi + 1) >> 1;
            if (mstart[mid] <= at)
                lo = mid;
            else
                hi = mid - 1;
        }
        out.ent = (int32_t)(col | SPMM_E_REAL | SPMM_E_MED);
        out.row = (int32_t)(lo / groups);
        out.val = val[pos[mrow[lo]] + (at - mstart[lo])];
    } else if (direct) {
        out.ent = (int32_t)(col | SPMM_E_REAL);
        out.row = srow[idx[e]];
        out.val = val[pos[out.row]];
    } else {
        out.ent = (int32_t)(col | SPMM_E_REAL | (first[e] ? (uint32_t)SPMM_E_FIRST : 0u) |
                            ((uint32_t)((k >> 28) & (SPMM_HR - 1)) << SPMM_E_ROW));
        out.row = 0;
        out.val = val[idx[e]];
    }
    const bool lone = e + 1 == start[r + 1] && ((start[r + 1] - start[r]) & 1);          // last entry of a run of odd length
    if (lone)
        out.ent |= SPMM_E_LONE;
    hent[p] = out;
    if (lone) {
        out.ent &= ~(SPMM_E_REAL | SPMM_E_FIRST);      // same column (a valid address), no value
        out.val = 0.0;
        hent[p + 1] = out;
    }
}

// seg[b] = position in the padded list of the first entry whose (XCD, wavefront) number is >= b
__global__ void heavy_segments(int64_t n, const uint64_t *__restrict__ keys, const int64_t *__restrict__ runs,
                               const int64_t *__restrict__ pads, int hbins, int64_t *__restrict__ seg)
{
    const int64_t b = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (b > 8 * hbins)
        return;
    int64_t lo = 0, hi = n;
    while (lo < hi) {
        const int64_t mid = (lo + hi) >> 1;
        if ((int64_t)(keys[mid] >> 28) / (SPMM_HCB * 2 * SPMM_HR) < b)
            lo = mid + 1;
        else
            hi = mid;
    }
    seg[b] = lo + pads[runs[lo]];      // lo opens a run (or is n): runs[lo] is that run's number
}

__global__ void light_lengths(int64_t nlight, const int32_t *__restrict__ rowmap, const int64_t *__restrict__ pos,
                              int64_t *__restrict__ len)
{
    const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (r < nlight)
        len[r] = pos[rowmap[r] + 1] - pos[rowmap[r]];
}

__global__ void light_copy(int64_t nlight, const int32_t *__restrict__ rowmap, const int64_t *__restrict__ pos,
                           const int32_t *__restrict__ crd, const double *__restrict__ val,
                           const int64_t *__restrict__ lpos, int32_t *__restrict__ lcrd, double *__restrict__ lval)
{
    // one 16-lane group per row: the rows copied here are short
    const int64_t r = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 4;
    const int sub = threadIdx.x & 15;
    if (r >= nlight)
        return;
    const int64_t n = lpos[r + 1] - lpos[r], src = pos[rowmap[r]], dst = lpos[r];
    for (int64_t t = sub; t < n; t += 16) {
        lcrd[dst + t] = crd[src + t];
        lval[dst + t] = val[src + t];
    }
}

// C[row] (+)= the eight per-XCD sums of a long row, in XCD (= column) order
template <bool ACC>
__global__ __launch_bounds__(256) void spmm_heavy_combine(int64_t nheavy, const int32_t *__restrict__ hrow,
                                                          const int32_t *__restrict__ hcode,
                                                          const double *__restrict__ partial, int hslots,
                                                          int64_t nmedium, const int32_t *__restrict__ mrow, int groups,
                                                          int nslots, const double *__restrict__ partial_medium,
                                                          double *__restrict__ C, int64_t ldc, int64_t K)
{
    const int lane = threadIdx.x & 63;
    const int64_t h = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    const int64_t col = (int64_t)blockIdx.y * 64 + lane;
    if (h >= nheavy + nmedium || col >= K)
        return;
    if (h >= nheavy) {          // a row of middling length: slot m / groups of workgroup m % groups of every XCD
        const int64_t m = h - nheavy, row = mrow[m];
        double acc = ACC ? C[row * ldc + col] : 0.0;
        for (int x = 0; x < 8; ++x)
            acc = acc + partial_medium[((((int64_t)x * groups + m % groups) * nslots) + m / groups) * K + col];
        C[row * ldc + col] = acc;
        return;
    }
    const int64_t row = hrow[h];
    double acc = ACC ? C[row * ldc + col] : 0.0;
    for (int x = 0; x < 8; ++x)
        acc = acc + partial[((int64_t)x * hslots + hcode[x * nheavy + h]) * K + col];
    C[row * ldc + col] = acc;
}

static Workspace g_heavy_partial, g_medium_partial;

// Launches the sweep with `lds` bytes of dynamic LDS, asking for more than the 64 KiB a kernel gets by default.
template <typename Kern, typename... Args>
static int sweep_launch(Kern kernel, dim3 grid, dim3 block, size_t lds, Args... args)
{
    if (lds > 64 * 1024)
        COMET_HIPCHK(hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                         (int)lds));
    kernel<<<grid, block, lds, stream()>>>(args...);
    return COMET_HIP_OK;
}

// Whether rows of B and C that are no multiple of 16 bytes are swept: most of the matrix has to be in the long rows, and a
// row of B in several of them.  us, chunks as stored / sweep at K = 17, 33, 63, and of the entries the share in long rows and how many
// of them there are a column: zipf, 200000 rows of 4 (0.69, 2.7) 62 / 124, 77 / 131, 113 / 113, of 8 (0.81, 6.5) 87 / 100, 115 /
// 107, 177 / 106, 100000 of 16 (0.86, 14) K = 33 101 / 78, 63 159 / 83; R-MAT scale 17, 4 edges a vertex (0.37, 2.8) K = 33
// 50 / 145, 16 (0.54, 15) 115 / 332.
static bool sweep_uneven(const Csr *a, int64_t K)
{
    return a->heavy_nnz * 4 >= a->nnz * 3 && a->heavy_nnz >= (K < 32 ? 8 : 4) * a->ncols;
}

// even: the call's rows are multiples of 16 bytes; if not, the plan is made only if the sweep is worth it for such, and is
// left to a call with even ones otherwise
static int spmm_heavy_plan(Csr *a, bool even, int64_t K)
{
    if (a->heavy_state != 0)
        return COMET_HIP_OK;
    a->heavy_state = 1;
    if (a->nnz < (1 << 19) || a->nnz >= (1ll << 32) || ceil_div(a->ncols, 8) >= (1ll << SPMM_HCOLB))
        return COMET_HIP_OK;        // a list entry has SPMM_HCOLB bits for the column inside an XCD's eighth
    const int64_t n = a->nrows;
    // The long rows may hold too little for the sweep: looked at before the row pointers are fetched and gone through here
    // (300000 rows: 540 us).  Those that are long may be more than the sweep holds.
    COMET_CHK(spmm_long_rows(a));
    if (!even && !sweep_uneven(a, K)) {
        a->heavy_state = 0;
        return COMET_HIP_OK;
    }
    if (a->heavy_nnz == 0 || a->heavy_nnz * 4 < a->nnz)
        return COMET_HIP_OK;
    std::vector<int64_t> pos((size_t)n + 1);
    COMET_HIPCHK(hipMemcpyAsync(pos.data(), a->pos, sizeof(int64_t) * (size_t)(n + 1), hipMemcpyDeviceToHost,
                                stream()));
    COMET_HIPCHK(hipStreamSynchronize(stream()));
    std::vector<std::pair<int64_t, int32_t>> cand;       // (-length, row): sorts longest first, ties by row
    std::vector<std::pair<int64_t, int32_t>> mcand;      // the same for the rows of middling length
    // Off unless COMET_HIP_SPMM_MEDIUM is set: on the benchmark matrix it takes 0.4 GB off the traffic past the L2
    // (the rows of B these rows gather are hits) and costs time - an entry of such a row takes the sweep 11 ns of a
    // CU, the chunk kernel beside the sweep 16, but the sweep is the longer of the two: 0.343 against 0.312 ms.
    const bool medium_on = getenv("COMET_HIP_SPMM_MEDIUM") != nullptr;
    for (int64_t r = 0; r < n; ++r) {
        const int64_t len = pos[(size_t)r + 1] - pos[(size_t)r];
        if (len >= SPMM_HEAVY_MIN_LEN)
            cand.emplace_back(-len, (int32_t)r);
        else if (medium_on && len >= SPMM_MED_MIN_LEN)
            mcand.emplace_back(-len, (int32_t)r);
    }
    std::sort(cand.begin(), cand.end());
    std::sort(mcand.begin(), mcand.end());
    // How many CUs of an XCD the sweep takes: all of them, unless the rows that are neither long nor single (with
    // the sweep at full size) hold at least a sixteenth of the matrix; COMET_HIP_SPMM_GROUPS overrides.
    int G = SPMM_HG_ALONE;
    {
        int64_t long_nnz = 0, single = 0;
        for (size_t k = 0; k < cand.size() && (int64_t)k < spmm_hrows(SPMM_HG_ALONE); ++k)
            long_nnz -= cand[k].first;
        for (int64_t r = 0; r < n; ++r)
            single += pos[(size_t)r + 1] - pos[(size_t)r] == 1;
        if ((a->nnz - long_nnz - single) * 16 >= a->nnz)
            G = SPMM_HG_SHARED;
        if (const char *e = getenv("COMET_HIP_SPMM_GROUPS")) {
            const int g = atoi(e);
            if (g >= 1 && g <= SPMM_HG_ALONE)
                G = g;
        }
    }
    const int hbins = spmm_hbins(G);
    // rows of middling length: the long rows the sweep has no register for, then the rows below them, longest
    // first, as many as the workgroups have slots in LDS
    std::vector<int32_t> mrow;
    std::vector<int64_t> mstart(1, 0);
    if (medium_on) {
        for (size_t k = (size_t)spmm_hrows(G); k < cand.size() && (int64_t)mrow.size() < (int64_t)G * SPMM_MSLOTS; ++k) {
            mrow.push_back(cand[k].second);
            mstart.push_back(mstart.back() - cand[k].first);
        }
        for (size_t k = 0; k < mcand.size() && (int64_t)mrow.size() < (int64_t)G * SPMM_MSLOTS; ++k) {
            mrow.push_back(mcand[k].second);
            mstart.push_back(mstart.back() - mcand[k].first);
        }
    }
    const int64_t M = (int64_t)mrow.size(), mnnz = mstart.back();
    if ((int64_t)cand.size() > spmm_hrows(G))
        cand.resize((size_t)spmm_hrows(G));
    const int64_t H = (int64_t)cand.size();
    int64_t hnnz = 0;
    for (auto &c : cand)
        hnnz -= c.first;
    a->heavy_nnz = hnnz;          // of those the sweep holds
    if (!even && !sweep_uneven(a, K)) {
        a->heavy_state = 0;
        return COMET_HIP_OK;
    }
    if (H == 0 || hnnz * 4 < a->nnz)
        return COMET_HIP_OK;        // the long rows hold too little of the matrix to pay for a second kernel
    std::vector<int32_t> hrow((size_t)H), hcode((size_t)(8 * H)), cnt((size_t)(8 * H));
    std::vector<int64_t> hstart((size_t)H + 1, 0);
    std::vector<char> is_long((size_t)n, 0);         // 1: long, 2: of middling length
    for (int64_t m = 0; m < M; ++m)
        is_long[(size_t)mrow[(size_t)m]] = 2;
    for (int64_t k = 0; k < H; ++k) {
        hrow[(size_t)k] = cand[(size_t)k].second;
        is_long[(size_t)hrow[(size_t)k]] = 1;
        hstart[(size_t)k + 1] = hstart[(size_t)k] - cand[(size_t)k].first;
    }
    // the other rows: one nonzero -> an entry of the sweep's lists; none -> cleared; the rest -> `light`
    std::vector<int32_t> srow, erow, lrow;
    for (int64_t r = 0; r < n; ++r) {
        const int64_t len = pos[(size_t)r + 1] - pos[(size_t)r];
        if (is_long[(size_t)r])
            continue;
        (len == 0 ? erow : len == 1 ? srow : lrow).push_back((int32_t)r);
    }
    const int64_t S = (int64_t)srow.size(), E = (int64_t)erow.size(), L = (int64_t)lrow.size();
    const int64_t nent = hnnz + S + mnnz;          // entries of the lists before padding
    int32_t *d_cnt = nullptr, *d_srow = nullptr;
    int64_t *d_hstart = nullptr, *d_len = nullptr, *d_mstart = nullptr;
    int64_t *d_first = nullptr, *d_runs = nullptr, *d_start = nullptr, *d_odd = nullptr, *d_pads = nullptr;
    uint64_t *k_in = nullptr, *k_out = nullptr;
    uint32_t *i_in = nullptr, *i_out = nullptr;
    Csr *light = new Csr();
    char *scratch = nullptr;        // everything that does not outlive the planning, in one allocation
    auto cleanup = [&](bool failed) {
        (void)dev_free(scratch);
        if (failed) {
            (void)dev_free(a->heavy_seg);
            (void)dev_free(a->heavy_ent);
            (void)dev_free(a->heavy_row);
            (void)dev_free(a->heavy_code);
            (void)dev_free(a->medium_row);
            a->medium_row = nullptr;
            (void)dev_free(a->empty_rows);
            a->heavy_seg = nullptr;
            a->heavy_ent = nullptr;
            a->heavy_row = a->heavy_code = a->empty_rows = nullptr;
            a->nempty = 0;
            light->owns = true;
            csr_release(light);
        }
    };
#define HEAVY_TRY(call)                                                                                       \
    do {                                                                                                      \
        if ((call) != hipSuccess) {                                                                           \
            cleanup(true);                                                                                    \
            return set_error(COMET_HIP_ERR_HIP, "%s failed while planning the long rows", #call);             \
        }                                                                                                     \
    } while (0)
    auto at_least_one = [](int64_t v) { return (size_t)(v > 0 ? v : 1); };
    {
        // (an allocation and its release cost about as much as a product each: fourteen arrays, one of each)
        size_t total = 0;
        const auto room = [&](size_t bytes) {
            const size_t at = total;
            total += (bytes + 255) & ~(size_t)255;
            return at;
        };
        const size_t o_cnt = room(4 * (size_t)(8 * H)), o_srow = room(4 * at_least_one(S)),
                     o_hstart = room(8 * (size_t)(H + 1)), o_mstart = room(8 * (size_t)(M + 1)),
                     o_len = room(8 * at_least_one(L)), o_kin = room(8 * (size_t)nent), o_kout = room(8 * (size_t)nent),
                     o_iin = room(4 * (size_t)nent), o_iout = room(4 * (size_t)nent), o_first = room(8 * (size_t)nent),
                     o_runs = room(8 * (size_t)(nent + 1)), o_start = room(8 * (size_t)(nent + 1)),
                     o_odd = room(8 * (size_t)nent), o_pads = room(8 * (size_t)(nent + 1));
        HEAVY_TRY(dev_malloc((void **)&scratch, total));
        d_cnt = (int32_t *)(scratch + o_cnt);
        d_srow = (int32_t *)(scratch + o_srow);
        d_hstart = (int64_t *)(scratch + o_hstart);
        d_mstart = (int64_t *)(scratch + o_mstart);
        d_len = (int64_t *)(scratch + o_len);
        k_in = (uint64_t *)(scratch + o_kin);
        k_out = (uint64_t *)(scratch + o_kout);
        i_in = (uint32_t *)(scratch + o_iin);
        i_out = (uint32_t *)(scratch + o_iout);
        d_first = (int64_t *)(scratch + o_first);
        d_runs = (int64_t *)(scratch + o_runs);
        d_start = (int64_t *)(scratch + o_start);
        d_odd = (int64_t *)(scratch + o_odd);
        d_pads = (int64_t *)(scratch + o_pads);
    }
    HEAVY_TRY(dev_malloc((void **)&a->medium_row, 4 * at_least_one(M)));
    if (M > 0)
        HEAVY_TRY(hipMemcpyAsync(a->medium_row, mrow.data(), 4 * (size_t)M, hipMemcpyHostToDevice, stream()));
    HEAVY_TRY(hipMemcpyAsync(d_mstart, mstart.data(), 8 * (size_t)(M + 1), hipMemcpyHostToDevice, stream()));
    HEAVY_TRY(dev_malloc((void **)&a->heavy_seg, 8 * (size_t)(8 * hbins + 1)));
    HEAVY_TRY(dev_malloc((void **)&a->heavy_row, 4 * (size_t)H));
    HEAVY_TRY(dev_malloc((void **)&a->heavy_code, 4 * (size_t)(8 * H)));
    HEAVY_TRY(dev_malloc((void **)&a->empty_rows, 4 * at_least_one(E)));
    HEAVY_TRY(dev_malloc((void **)&light->rowmap, 4 * at_least_one(L)));
    HEAVY_TRY(hipMemcpyAsync(a->heavy_row, hrow.data(), 4 * (size_t)H, hipMemcpyHostToDevice, stream()));
    if (S > 0)
        HEAVY_TRY(hipMemcpyAsync(d_srow, srow.data(), 4 * (size_t)S, hipMemcpyHostToDevice, stream()));
    if (E > 0)
        HEAVY_TRY(hipMemcpyAsync(a->empty_rows, erow.data(), 4 * (size_t)E, hipMemcpyHostToDevice, stream()));
    if (L > 0)
        HEAVY_TRY(hipMemcpyAsync(light->rowmap, lrow.data(), 4 * (size_t)L, hipMemcpyHostToDevice, stream()));
    HEAVY_TRY(hipMemcpyAsync(d_hstart, hstart.data(), 8 * (size_t)(H + 1), hipMemcpyHostToDevice, stream()));
    const int64_t xcols = ceil_div(a->ncols, 8);
    // Every XCD gets its own assignment of rows to wavefronts, by what the row holds in that XCD's column
    // range: longest first, each to the least loaded wavefront that still has a free slot.  Wavefronts with
    // equal lists move through the columns at the same pace, which is what keeps the rows of B they share
    // inside the L2 between uses.
    heavy_count<<<dim3((unsigned)ceil_div(H, 32)), dim3(256), 0, stream()>>>(H, a->heavy_row, a->pos, a->crd, xcols,
                                                                             d_cnt);
    HEAVY_TRY(hipMemcpyAsync(cnt.data(), d_cnt, 4 * (size_t)(8 * H), hipMemcpyDeviceToHost, stream()));
    HEAVY_TRY(hipStreamSynchronize(stream()));
    for (int x = 0; x < 8; ++x) {
        std::vector<std::pair<int32_t, int32_t>> order((size_t)H);       // (-count, row index)
        for (int64_t k = 0; k < H; ++k)
            order[(size_t)k] = {-cnt[(size_t)(k * 8 + x)], (int32_t)k};
        std::sort(order.begin(), order.end());
        // (time the wavefront needs for its list so far, wavefront).  The four wavefronts of a SIMD do not
        // run at the same speed: the older one wins every arbitration, and the measured entry rates of
        // wavefronts 0-3, 4-7, 8-11, 12-15 of a workgroup are as 1.12 : 1.05 : 0.96 : 0.87.
        static const double pace[4] = {1.0 / 1.12, 1.0 / 1.05, 1.0 / 0.96, 1.0 / 0.87};
        std::priority_queue<std::pair<double, int32_t>, std::vector<std::pair<double, int32_t>>,
                            std::greater<std::pair<double, int32_t>>> bins;
        std::vector<int32_t> used((size_t)hbins, 0);
        for (int32_t b = 0; b < hbins; ++b)
            if (b % SPMM_HW != SPMM_HWL)        // the last wavefront of a workgroup takes the rows with one nonzero
                bins.push({0.0, b});
        for (auto &o : order) {
            auto top = bins.top();
            bins.pop();
            const int32_t b = top.second;
            hcode[(size_t)(x * H + o.second)] = b * SPMM_HR + used[(size_t)b];
            if (++used[(size_t)b] < SPMM_HR)
                bins.push({top.first - o.first * pace[(b % SPMM_HW) / 4], b});
        }
    }
    HEAVY_TRY(hipMemcpyAsync(a->heavy_code, hcode.data(), 4 * (size_t)(8 * H), hipMemcpyHostToDevice, stream()));
    {
        KernelTimer t("heavy_make_keys");
        heavy_make_keys<<<dim3((unsigned)H), dim3(256), 0, stream()>>>(H, a->heavy_row, a->heavy_code, d_hstart,
                                                                       a->pos, a->crd, xcols, hbins, k_in, i_in);
        if (S > 0)
            single_make_keys<<<dim3((unsigned)ceil_div(S, 256)), dim3(256), 0, stream()>>>(
                S, d_srow, a->pos, a->crd, xcols, G, k_in + hnnz, i_in + hnnz);
        if (M > 0)
            medium_make_keys<<<dim3((unsigned)M), dim3(64), 0, stream()>>>(M, a->medium_row, d_mstart, a->pos, a->crd,
                                                                          xcols, G, k_in + hnnz + S, i_in + hnnz + S);
    }
    if (sort_pairs_u64_u32(k_in, k_out, i_in, i_out, nent, 28 + (SPMM_HRB + 1) + 5 + 12) != COMET_HIP_OK) {
        cleanup(true);
        return COMET_HIP_ERR_HIP;
    }
    // runs (entries of one row inside one column block of one wavefront's list) are padded to even length
    const dim3 per_entry((unsigned)ceil_div(nent + 1, 256));
    heavy_mark_runs<<<per_entry, dim3(256), 0, stream()>>>(nent, k_out, d_first);
    if (exclusive_scan_i64(d_first, nent, d_runs) != COMET_HIP_OK) {
        cleanup(true);
        return COMET_HIP_ERR_HIP;
    }
    int64_t nruns = 0, npads = 0;
    HEAVY_TRY(hipMemcpyAsync(&nruns, d_runs + nent, 8, hipMemcpyDeviceToHost, stream()));
    HEAVY_TRY(hipStreamSynchronize(stream()));
    heavy_run_starts<<<per_entry, dim3(256), 0, stream()>>>(nent, d_first, d_runs, d_start);
    heavy_run_odd<<<dim3((unsigned)ceil_div(nruns, 256)), dim3(256), 0, stream()>>>(nruns, d_start, d_odd);
    if (exclusive_scan_i64(d_odd, nruns, d_pads) != COMET_HIP_OK) {
        cleanup(true);
        return COMET_HIP_ERR_HIP;
    }
    HEAVY_TRY(hipMemcpyAsync(&npads, d_pads + nruns, 8, hipMemcpyDeviceToHost, stream()));
    HEAVY_TRY(hipStreamSynchronize(stream()));
    HEAVY_TRY(dev_malloc((void **)&a->heavy_ent, sizeof(HeavyEnt) * (size_t)(nent + npads)));
    {
        KernelTimer t("heavy_fill");
        heavy_fill<<<dim3((unsigned)ceil_div(nent, 256)), dim3(256), 0, stream()>>>(
            nent, k_out, i_out, a->val, a->pos, d_srow, M, a->medium_row, d_mstart, G, d_first, d_runs, d_start, d_pads,
            xcols, a->heavy_ent);
        heavy_segments<<<dim3((unsigned)ceil_div(8 * hbins + 1, 256)), dim3(256), 0, stream()>>>(
            nent, k_out, d_runs, d_pads, hbins, a->heavy_seg);
    }
    // the rows of two and more nonzeros that are not long, as a matrix of their own
    light->nrows = L;
    light->ncols = a->ncols;
    light->nnz = a->nnz - hnnz - S - mnnz;
    light->owns = true;
    HEAVY_TRY(dev_malloc((void **)&light->pos, 8 * (size_t)(L + 1)));
    HEAVY_TRY(dev_malloc((void **)&light->crd, 4 * at_least_one(light->nnz)));
    HEAVY_TRY(dev_malloc((void **)&light->val, 8 * at_least_one(light->nnz)));
    if (L > 0) {
        light_lengths<<<dim3((unsigned)ceil_div(L, 256)), dim3(256), 0, stream()>>>(L, light->rowmap, a->pos, d_len);
        if (exclusive_scan_i64(d_len, L, light->pos) != COMET_HIP_OK) {
            cleanup(true);
            return COMET_HIP_ERR_HIP;
        }
        KernelTimer t("light_copy");
        light_copy<<<dim3((unsigned)ceil_div(L * 16, 256)), dim3(256), 0, stream()>>>(
            L, light->rowmap, a->pos, a->crd, a->val, light->pos, light->crd, light->val);
    } else {
        HEAVY_TRY(hipMemsetAsync(light->pos, 0, 8, stream()));
    }
    if (light->nnz > 0 && spmm_plan(light) != COMET_HIP_OK) {          // its chunk table
        cleanup(true);
        return COMET_HIP_ERR_HIP;
    }
    HEAVY_TRY(hipGetLastError());
    HEAVY_TRY(hipStreamSynchronize(stream()));
#undef HEAVY_TRY
    cleanup(false);
    light->heavy_state = 1;
    a->light = light;
    a->heavy_rows = H;
    a->heavy_groups = G;
    a->medium_rows = M;
    a->nempty = E;
    a->heavy_state = 2;
    return COMET_HIP_OK;
}

}  // namespace comet

using namespace comet;

static int spmm_chunks(Csr *a, int64_t K, const double *B, int64_t ldb, double *C, int64_t ldc, int accumulate, const SpmmShape &h,
                       bool ordered = false, hipStream_t on = nullptr);
static int spmv_run(Csr *a, int64_t x_dptr, int64_t y_dptr, int accumulate);
static int spmm_run(Csr *a, int64_t K, int64_t b_dptr, int64_t ldb, int64_t c_dptr, int64_t ldc, int accumulate);

extern "C" int comet_hip_spmv_csr_f64(int64_t csr, int64_t x_dptr, int64_t y_dptr, int accumulate)
{
    COMET_CHK(ensure_init());
    Csr *a = csr_from_handle(csr);
    if (!a)
        return COMET_HIP_ERR_HANDLE;
    return spmv_run(a, x_dptr, y_dptr, accumulate);
}

// The launch of spmv_csr_blocks for a matrix of nrows rows: the fewest tiles per workgroup with which the
// workgroups resident at once cover all rows, and tiles of equal size (a lane per row, at most SPMV_T).  False when
// the rows do not fit the LDS of one grid: then every block is a launch of its own.
constexpr int SPMV_MAX_TILES = 16;
static bool spmv_blocks_shape(int64_t nrows, int *grid, int *tile_rows, int *tiles)
{
    static int per_cu[SPMV_MAX_TILES + 1];       // resident workgroups per CU by tiles per workgroup; 0: not asked yet
    for (int t = 1; t <= SPMV_MAX_TILES; ++t) {
        if (per_cu[t] == 0) {
            int n = 0;
            if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, spmv_csr_blocks<int32_t>, SPMV_T,
                                                             sizeof(double) * SPMV_T * (size_t)t) != hipSuccess || n <= 0)
                n = -1;
            per_cu[t] = n;
        }
        if (per_cu[t] < 0)
            return false;
        const int64_t resident = (int64_t)per_cu[t] * (num_cus() > 0 ? num_cus() : 256);
        if (resident * t * SPMV_T < nrows)
            continue;
        const int64_t g = std::min<int64_t>(resident, ceil_div(nrows, (int64_t)t * 64));
        *grid = (int)g;
        *tiles = t;
        *tile_rows = (int)ceil_div(nrows, g * t);
        return true;
    }
    return false;
}

static int spmv_run(Csr *a, int64_t x_dptr, int64_t y_dptr, int accumulate)
{
    if ((a->ncols > 0 && !x_dptr) || (a->nrows > 0 && !y_dptr))
        return set_error(COMET_HIP_ERR_ARG, "null vector passed to a sparse matrix-vector product");
    if (a->nrows == 0)
        return COMET_HIP_OK;
    // The column-blocked copy costs some twenty products: a matrix multiplied once runs on its own arrays, the copy
    // is made when it is multiplied again.
    const bool plan_now = a->spmv_uses > 0 || plan_at_once();
    a->spmv_uses = a->spmv_uses < 2 ? a->spmv_uses + 1 : 2;
    if (plan_now && a->spmv_nb == 0 && !plan_made([&] { return spmv_plan(a); }))
        a->spmv_nb = 1;
    const int nb = a->spmv_nb > 0 ? a->spmv_nb : 1;
    const unsigned blocks = (unsigned)ceil_div(a->nrows, SPMV_T);
    const double *x = (const double *)x_dptr;
    double *y = (double *)y_dptr;
    if (nb > 1 && a->spmv_bpos32 && getenv("COMET_HIP_SPMV_LAUNCH_PER_BLOCK") == nullptr) {
        // all column blocks in one launch, the row sums staying on chip - when the workgroups the GPU holds at once
        // have room for all rows
        int grid = 0, tile_rows = 0, tiles = 0;
        if (spmv_blocks_shape(a->nrows, &grid, &tile_rows, &tiles)) {
            SpmvBases base;
            for (int b = 0; b < nb; ++b)
                base.v[b] = a->spmv_base[b];
            KernelTimer t("spmv_csr_blocks");
            spmv_csr_blocks<int32_t><<<dim3((unsigned)grid), dim3(SPMV_T), sizeof(double) * SPMV_T * (size_t)tiles,
                                       stream()>>>(a->spmv_bpos32, a->spmv_bcrd, a->spmv_bval, base, nb, x, y,
                                                   a->nrows, tile_rows, tiles, accumulate);
            COMET_HIPCHK(hipGetLastError());
            return COMET_HIP_OK;
        }
    }
    for (int b = 0; b < nb; ++b) {
        const int32_t *crd = nb == 1 ? a->crd : a->spmv_bcrd + a->spmv_base[b];
        const double *val = nb == 1 ? a->val : a->spmv_bval + a->spmv_base[b];
        const bool acc = accumulate || b > 0;   // later passes continue the row sums the earlier ones left in y
        KernelTimer t("spmv_csr_stream");
        if (nb > 1 && a->spmv_bpos32) {
            const int32_t *pos = a->spmv_bpos32 + (int64_t)b * (a->nrows + 1);
            if (acc)
                spmv_csr_stream<true, int32_t><<<dim3(blocks), dim3(SPMV_T), 0, stream()>>>(pos, crd, val, x, y, a->nrows);
            else
                spmv_csr_stream<false, int32_t><<<dim3(blocks), dim3(SPMV_T), 0, stream()>>>(pos, crd, val, x, y, a->nrows);
        } else {
            const int64_t *pos = nb == 1 ? a->pos : a->spmv_bpos + (int64_t)b * (a->nrows + 1);
            if (acc)
                spmv_csr_stream<true, int64_t><<<dim3(blocks), dim3(SPMV_T), 0, stream()>>>(pos, crd, val, x, y, a->nrows);
            else
                spmv_csr_stream<false, int64_t><<<dim3(blocks), dim3(SPMV_T), 0, stream()>>>(pos, crd, val, x, y, a->nrows);
        }
    }
    COMET_HIPCHK(hipGetLastError());
    return COMET_HIP_OK;
}

extern "C" int comet_hip_debug_sweep_slack(int64_t ncols, int64_t K)
{
    return sweep_slack(ceil_div(ncols, 8), K);
}

extern "C" int comet_hip_spmm_csr_f64(int64_t csr, int64_t K, int64_t b_dptr, int64_t ldb, int64_t c_dptr,
                                      int64_t ldc, int accumulate)
{
    COMET_CHK(ensure_init());
    Csr *a = csr_from_handle(csr);
    if (!a)
        return COMET_HIP_ERR_HANDLE;
    return spmm_run(a, K, b_dptr, ldb, c_dptr, ldc, accumulate);
}

static int spmm_run(Csr *a, int64_t K, int64_t b_dptr, int64_t ldb, int64_t c_dptr, int64_t ldc, int accumulate)
{
    if (K < 0 || ldb < K || ldc < K)
        return set_error(COMET_HIP_ERR_ARG, "bad K/ldb/ldc (%lld, %lld, %lld)", (long long)K, (long long)ldb,
                         (long long)ldc);
    if (K == 0 || a->nrows == 0)
        return COMET_HIP_OK;
    if (!c_dptr || (a->nnz > 0 && !b_dptr))
        return set_error(COMET_HIP_ERR_ARG, "null matrix passed to a sparse-dense matrix product");
    double *C = (double *)c_dptr;
    const double *B = (const double *)b_dptr;
    if (ceil_div(K, 64) > 65535)
        return set_error(COMET_HIP_ERR_SIZE, "K = %lld needs more than 65535 column tiles", (long long)K);
    // long rows: column sweep with the sums on chip; everything else: one wavefront per 256 nonzeros
    // Rows of B and C that are no multiple of 16 bytes are swept where B is so large that its gathers come from far away
    // (chunks as stored / sweep, us: K = 33 40000 rows 51 / 65, 60001 69 / 68, 120000 121 / 87, 250000 242 / 153, 500000 477 / 277;
    // K = 63 40000 71 / 74, 60001 102 / 77, 500000 758 / 358; K = 17 60001 52 / 60, 500000 348 / 230: zipf, 16 entries a row),
    // where the matrix is right for it (sweep_uneven), and where no tile of columns holds a single one.
    const bool even = (K & 1) == 0 && (ldb & 1) == 0 && (b_dptr & 15) == 0 && (ldc & 1) == 0 && (c_dptr & 15) == 0;
    const bool uneven_pays = K % 64 != 1 && a->ncols * ldb * 8 >= SPMM_UNEVEN_SWEEP && (a->heavy_nnz < 0 || sweep_uneven(a, K));
    const bool sweep_fits = K >= 16 && K <= 2048 && (even || uneven_pays) && getenv("COMET_SPMM_NO_SWEEP") == nullptr;
    // The plan (the long rows as per-XCD lists, the rest re-packed) costs some forty products: a matrix multiplied
    // once goes through the chunk kernel whole, the plan is made when it is multiplied again.
    const bool plan_now = a->spmm_uses > 0 || plan_at_once();
    a->spmm_uses = a->spmm_uses < 2 ? a->spmm_uses + 1 : 2;
    SpmmShape h = spmm_shape(a, K);
    bool stored = false;
    const bool by_columns = plan_now && spmm_by_columns(a, K, &h, &stored);
    if (by_columns || stored)
        return spmm_chunks(a, K, B, ldb, C, ldc, accumulate, h, by_columns);
    if (sweep_fits && plan_now && a->heavy_state == 0)
        (void)plan_made([&] { return spmm_heavy_plan(a, even, K); });          // or the chunk kernel goes on taking all rows
    if (a->heavy_state != 2 || !sweep_fits)
        return spmm_chunks(a, K, B, ldb, C, ldc, accumulate, h);
    const int G = a->heavy_groups;
    // rows of middling length: ceil(rows / G) sums of 64 doubles in the LDS of every workgroup
    const int nslots = (int)ceil_div(a->medium_rows, G);
    const size_t medium_lds = sizeof(double) * 64 * (size_t)nslots;
    // what the kernels leave sums in; without room for it the chunk kernel takes all rows
    const SpmmShape light = spmm_shape(a->light, K);
    const auto scratch = [&]() -> int {
        COMET_CHK(g_heavy_partial.ensure(sizeof(double) * 8 * (size_t)spmm_hslots(G) * (size_t)K, false));
        COMET_CHK(g_medium_partial.ensure(sizeof(double) * 8 * (size_t)G * (size_t)(nslots > 0 ? nslots : 1) * (size_t)K, false));
        return a->light->nnz > 0 ? spmm_chunk_scratch(light) : COMET_HIP_OK;
    };
    if (!plan_made(scratch))
        return spmm_chunks(a, K, B, ldb, C, ldc, accumulate, h);
    double *partial = (double *)g_heavy_partial.ptr, *partial_medium = (double *)g_medium_partial.ptr;
    // rows of two and more nonzeros that are not long: one wavefront per 256 nonzeros
    // with CUs left free by the sweep, the chunk kernel of the rows in between runs beside it on a second stream
    const bool overlap = a->light->nnz > 0 && G < SPMM_HG_ALONE;
    if (overlap) {
        // (what it needs from stream() - its chunk table, its scratch - is in place before the fork)
        COMET_CHK(aux_fork());
    } else if (a->light->nnz > 0)
        COMET_CHK(spmm_chunks(a->light, K, B, ldb, C, ldc, accumulate, light));
    const unsigned tiles = (unsigned)ceil_div(K, 64);
    if (!accumulate && a->nempty > 0) {
        KernelTimer t("zero_listed_rows_f64");
        const unsigned blocks = (unsigned)std::min<int64_t>(ceil_div(a->nempty * K, 256), 65536);
        zero_listed_rows_f64<<<dim3(blocks), dim3(256), 0, stream()>>>(C, a->empty_rows, a->nempty, K, ldc);
    }
    // long rows (sums on chip, left in `partial`) and rows of one nonzero (stored to C)
    {
        KernelTimer t("spmm_heavy_sweep");
        const bool small_b = a->ncols < (1 << 24) && ldb * 8 < (1 << 24) && a->ncols * ldb * 8 < (1ll << 32);
        const dim3 grid(8 * G, tiles), block(SPMM_HW * 64);
        const int slack = sweep_slack(ceil_div(a->ncols, 8), K);
        const auto launch = [&](auto kernel) {
            return sweep_launch(kernel, grid, block, medium_lds, a->heavy_seg, a->heavy_ent, B, ldb, K, partial, C, ldc, G,
                                ceil_div(a->ncols, 8), nslots, partial_medium, slack);
        };
        if (small_b)
            COMET_CHK(accumulate ? launch(spmm_heavy_sweep<true, true>) : launch(spmm_heavy_sweep<true, false>));
        else
            COMET_CHK(accumulate ? launch(spmm_heavy_sweep<false, true>) : launch(spmm_heavy_sweep<false, false>));
    }
    if (overlap) {      // the rows in between, on the CUs the sweep leaves free
        COMET_CHK(spmm_chunks(a->light, K, B, ldb, C, ldc, accumulate, light, false, aux_stream()));
        COMET_CHK(aux_join());
    }
    {
        KernelTimer t("spmm_heavy_combine");
        const dim3 grid((unsigned)ceil_div(a->heavy_rows + a->medium_rows, 4), tiles);
        if (accumulate)
            spmm_heavy_combine<true><<<grid, dim3(256), 0, stream()>>>(a->heavy_rows, a->heavy_row, a->heavy_code,
                                                                       partial, spmm_hslots(G), a->medium_rows,
                                                                       a->medium_row, G, nslots, partial_medium, C, ldc, K);
        else
            spmm_heavy_combine<false><<<grid, dim3(256), 0, stream()>>>(a->heavy_rows, a->heavy_row, a->heavy_code,
                                                                        partial, spmm_hslots(G), a->medium_rows,
                                                                       a->medium_row, G, nslots, partial_medium, C, ldc, K);
    }
    COMET_HIPCHK(hipGetLastError());
    return COMET_HIP_OK;
}

// The chunk kernel: the row of every grain'th nonzero in chunk_row, chunks of h.len nonzeros (a multiple of grain), two
// slots for each of them and column tile in carry and a zero in arrived; order: the chunks in the order they are taken in, or
// null.  timed: events may be recorded (not where the stream is being captured).
static void spmm_chunk_launch(const Csr *a, int64_t K, const double *B, int64_t ldb, double *C, int64_t ldc, int accumulate,
                              const int32_t *chunk_row, int grain, const SpmmShape &h, const uint32_t *order, double *carry,
                              unsigned *arrived, hipStream_t on, bool timed)
{
    const int64_t wide = order ? 8 * ceil_div(ceil_div(h.chunks, 8), SPMM_WAVES) : ceil_div(h.chunks, SPMM_WAVES);
    const dim3 grid((unsigned)wide, (unsigned)h.tiles), block(SPMM_WAVES * 64);
    const auto split = [&](auto kernel) {
        std::unique_ptr<KernelTimer> t(timed ? new KernelTimer("spmm_csr_nnzsplit", on) : nullptr);
        kernel<<<grid, block, 0, on>>>(a->pos, a->crd, a->val, a->nnz, a->nrows, chunk_row, grain, h.len, h.chunks, order, B, ldb, C,
                                       ldc, (int)K, h.cols, (int)ceil_div(a->nrows, h.chunks), carry, arrived, a->rowmap);
    };
    const bool small_b = K > 1 && a->ncols * ldb * 8 < (1ll << 32);
    if (K == 1)
        accumulate ? split(spmm_csr_nnzsplit<true, 1, false>) : split(spmm_csr_nnzsplit<false, 1, false>);
    else if (small_b)
        accumulate ? split(spmm_csr_nnzsplit<true, 2, true>) : split(spmm_csr_nnzsplit<false, 2, true>);
    else
        accumulate ? split(spmm_csr_nnzsplit<true, 2, false>) : split(spmm_csr_nnzsplit<false, 2, false>);
}

// ordered: h is how spmm_by_columns cut the product
static int spmm_chunks(Csr *a, int64_t K, const double *B, int64_t ldb, double *C, int64_t ldc, int accumulate, const SpmmShape &h,
                       bool ordered, hipStream_t on)
{
    if (!on)
        on = stream();
    if (a->nnz == 0) {
        if (!accumulate) {
            KernelTimer t("fill_rows_f64", on);
            unsigned blocks = (unsigned)std::min<int64_t>(ceil_div(a->nrows * K, 256), 65536);
            fill_rows_f64<<<dim3(blocks), dim3(256), 0, on>>>(C, a->nrows, K, ldc, 0.0);
            COMET_HIPCHK(hipGetLastError());
        }
        return COMET_HIP_OK;
    }
    COMET_CHK(spmm_plan(a));
    COMET_CHK(spmm_chunk_scratch(h));
    spmm_chunk_launch(a, K, B, ldb, C, ldc, accumulate, a->spmm_chunk_row, SPMM_GRAIN, h,
                      ordered ? a->spmm_order[h.len / SPMM_GRAIN / 2] : nullptr, (double *)g_spmm_carry.ptr,
                      (unsigned *)g_spmm_arrived.ptr, on, true);
    COMET_HIPCHK(hipGetLastError());
    return COMET_HIP_OK;
}

// ---------------------------------------------------------------------------
// Yardstick for the sweep: how fast the CUs can take rows of a dense operand out of the L2 when nothing else is
// done with them.  Every wavefront walks a list of row numbers; a half-wavefront fetches one row of 64 doubles,
// 16 bytes per lane (the sweep's load shape), sixteen loads in flight, and only sums what arrives.  Workgroup w
// (on XCD w mod 8) draws its rows from the w-mod-8-th eighth of the table, so with a table of at most 4 MiB per
// XCD every gather after the first touch is an L2 hit.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(1024) void gather_rows_bench_kernel(const int32_t *__restrict__ idx, int64_t per_wave,
                                                                 const double *__restrict__ table,
                                                                 double *__restrict__ out)
{
    const int lane = threadIdx.x & 63, half = lane >> 5, sub = lane & 31;
    const int64_t wave = (int64_t)blockIdx.x * 16 + (threadIdx.x >> 6);
    const int32_t *my = idx + wave * per_wave;
    double2 acc = make_double2(0.0, 0.0);
    for (int64_t i = 0; i < per_wave; i += 32) {
        double2 b[16];
#pragma unroll
        for (int u = 0; u < 16; ++u) {
            const int64_t j = my[i + 2 * u + half];
            b[u] = *reinterpret_cast<const double2 *>(table + j * 64 + sub * 2);
        }
#pragma unroll
        for (int u = 0; u < 16; ++u) {
            acc.x += b[u].x;
            acc.y += b[u].y;
        }
    }
    out[wave * 64 + lane] = acc.x + acc.y;
}

// idx[w * per_wave + i]: row of `table` (rows of 64 doubles) that wavefront w fetches i-th; 16 wavefronts per
// workgroup, `workgroups` workgroups; per_wave a multiple of 32; out holds workgroups * 1024 doubles.
extern "C" int comet_hip_gather_rows_bench(int64_t workgroups, int64_t per_wave, int64_t idx_dptr, int64_t table_dptr,
                                           int64_t table_rows, int64_t out_dptr)
{
    COMET_CHK(ensure_init());
    if (workgroups <= 0 || workgroups > 65535 || per_wave <= 0 || (per_wave & 31) || !idx_dptr || !table_dptr ||
        table_rows <= 0 || !out_dptr)
        return set_error(COMET_HIP_ERR_ARG, "bad arguments to comet_hip_gather_rows_bench");
    {
        KernelTimer t("gather_rows_bench");
        gather_rows_bench_kernel<<<dim3((unsigned)workgroups), dim3(1024), 0, stream()>>>(
            (const int32_t *)idx_dptr, per_wave, (const double *)table_dptr, (double *)out_dptr);
    }
    COMET_HIPCHK(hipGetLastError());
    return COMET_HIP_OK;
}

// ---------------------------------------------------------------------------
// SpMM for callers that cannot allocate (code under graph capture, serving loops that forbid hipMalloc): the
// chunk kernel with its scratch - the chunk -> row table, the carry slots of rows cut by a chunk boundary and the
// counts of their pieces - in one array that lives in the library's image instead of in allocated workspaces.  Every
// device holds its own copy at its own address; the address is looked up once per device, when the library is
// initialised there, and host code uses that pointer, never the array's name.
// ---------------------------------------------------------------------------
constexpr int64_t SPMM_STATIC_SLOTS = SPMM_SHORT_CHUNKS;      // (64-column tiles of K) x (chunks of 256 nonzeros) the array has room for
constexpr size_t SPMM_STATIC_TABLE_BYTES = sizeof(int32_t) * (size_t)SPMM_STATIC_SLOTS;
constexpr size_t SPMM_STATIC_CARRY_BYTES = sizeof(double) * 2 * 64 * (size_t)SPMM_STATIC_SLOTS;
static __device__ __align__(256) unsigned char spmm_static_scratch[2 * SPMM_STATIC_TABLE_BYTES + SPMM_STATIC_CARRY_BYTES];
constexpr int SPMM_STATIC_MAX_DEVICES = 64;
static unsigned char *g_spmm_static_ptr[SPMM_STATIC_MAX_DEVICES];     // device address of the array, per device

namespace comet {
int spmm_static_setup(int device)
{
    if (device < 0 || device >= SPMM_STATIC_MAX_DEVICES)
        return set_error(COMET_HIP_ERR_ARG, "device %d has no slot for the static SpMM scratch", device);
    unsigned char *ptr = nullptr;
    COMET_HIPCHK(hipGetSymbolAddress((void **)&ptr, HIP_SYMBOL(spmm_static_scratch)));
    g_spmm_static_ptr[device] = ptr;
    return COMET_HIP_OK;
}
}  // namespace comet

extern "C" int64_t comet_hip_debug_noalloc_scratch(int64_t *bytes)
{
    int device = -1;
    if (bytes)
        *bytes = (int64_t)sizeof spmm_static_scratch;
    if (!is_initialised() || hipGetDevice(&device) != hipSuccess || device < 0 || device >= SPMM_STATIC_MAX_DEVICES)
        return 0;
    return reinterpret_cast<int64_t>(g_spmm_static_ptr[device]);
}

extern "C" int comet_hip_spmm_csr_f64_noalloc(int64_t csr, int64_t K, int64_t b_dptr, int64_t ldb, int64_t c_dptr,
                                              int64_t ldc, int accumulate, int64_t on_stream)
{
    // on_stream: the hipStream_t the caller wants the kernels on (a stream under graph capture, a serving loop's own
    // stream), as an integer; 0 = the library's stream, like every other entry point
    const hipStream_t on = on_stream ? (hipStream_t)on_stream : stream();
    if (!is_initialised())       // bringing the device up creates streams: the caller does that beforehand
        return set_error(COMET_HIP_ERR_ARG, "comet_hip_spmm_csr_f64_noalloc: call comet_hip_init first");
    Csr *a = csr_from_handle(csr);
    if (!a)
        return COMET_HIP_ERR_HANDLE;
    if (K < 0 || ldb < K || ldc < K)
        return set_error(COMET_HIP_ERR_ARG, "bad K/ldb/ldc (%lld, %lld, %lld)", (long long)K, (long long)ldb,
                         (long long)ldc);
    if (K == 0 || a->nrows == 0)
        return COMET_HIP_OK;
    if (!c_dptr || (a->nnz > 0 && !b_dptr))
        return set_error(COMET_HIP_ERR_ARG, "null matrix passed to a sparse-dense matrix product");
    const int64_t tiles = ceil_div(K, 64);
    const int64_t nchunks = ceil_div(a->nnz, SPMM_CH);
    if (tiles > 65535 || tiles * nchunks > SPMM_STATIC_SLOTS)
        return set_error(COMET_HIP_ERR_SIZE,
                         "comet_hip_spmm_csr_f64_noalloc: ceil(K/64) * ceil(nnz/%d) = %lld exceeds the %lld slots of the "
                         "static scratch (nnz up to %lld at K <= 64); use comet_hip_spmm_csr_f64",
                         SPMM_CH, (long long)(tiles * nchunks), (long long)SPMM_STATIC_SLOTS,
                         (long long)(SPMM_STATIC_SLOTS * SPMM_CH));
    int device = -1;
    COMET_HIPCHK(hipGetDevice(&device));
    unsigned char *scratch = device >= 0 && device < SPMM_STATIC_MAX_DEVICES ? g_spmm_static_ptr[device] : nullptr;
    if (!scratch)
        return set_error(COMET_HIP_ERR_ARG, "the static SpMM scratch was not set up on device %d", device);
    double *C = (double *)c_dptr;
    if (a->nnz == 0) {
        if (!accumulate) {
            const unsigned blocks = (unsigned)std::min<int64_t>(ceil_div(a->nrows * K, 256), 65536);
            fill_rows_f64<<<dim3(blocks), dim3(256), 0, on>>>(C, a->nrows, K, ldc, 0.0);
            COMET_HIPCHK(hipGetLastError());
        }
        return COMET_HIP_OK;
    }
    // Every word the kernels read from the array is written earlier in the same call: the table in full and a zero in
    // every count by the first kernel, a carry slot by the chunk that leaves a piece of a row in it.  So what the array
    // holds when a call begins - calls that overlapped may leave anything - does not matter.
    int32_t *chunk_row = reinterpret_cast<int32_t *>(scratch);
    double *carry = reinterpret_cast<double *>(scratch + SPMM_STATIC_TABLE_BYTES);
    const SpmmShape h = spmm_shape(a, K);
    unsigned *arrived = reinterpret_cast<unsigned *>(scratch + SPMM_STATIC_TABLE_BYTES + SPMM_STATIC_CARRY_BYTES);
    spmm_chunk_rows<<<dim3((unsigned)ceil_div(h.chunks, 256)), dim3(256), 0, on>>>(a->pos, a->nrows, h.chunks, h.len, chunk_row, arrived,
                                                                                   h.tiles * h.chunks);
    spmm_chunk_launch(a, K, (const double *)b_dptr, ldb, C, ldc, accumulate, chunk_row, h.len, h, nullptr, carry, arrived, on, false);
    COMET_HIPCHK(hipGetLastError());
    return COMET_HIP_OK;
}

// ---------------------------------------------------------------------------
// Dense operand on the left: y[j] (+)= sum_i x[i] * B[i,j] and
// C[a,c] (+)= sum_b A[a,b] * B[b,c] with B in CSR.  The reference's nests run
// over the dense index outermost and scatter into the output
// (test/integration/ops/mult_DenseVecxCSR.ta, mult_DenseMatxCSR.ta through
// lib/Conversion/IndexTreeToSCF/IndexTreeToSCF.cpp:529-700,1247-1284), so an
// output element receives its products in ascending order of the contracted
// index.  That is the order in which the transpose of B holds them, so both
// products run as SpMV / SpMM over the transpose (built once, kept in the
// handle) and round like the reference; the dense matrix operands are turned
// by a tiled transpose on the way in and out.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void transpose2d_tile(const double *__restrict__ in, int64_t ld_in, int64_t rows,
                                                        int64_t cols, double *__restrict__ out, int64_t ld_out)
{
    __shared__ double tile[32][33];
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;       // 32 x 8 threads
    const int64_t r0 = (int64_t)blockIdx.y * 32, c0 = (int64_t)blockIdx.x * 32;
    for (int k = ty; k < 32; k += 8)
        if (r0 + k < rows && c0 + tx < cols)
            tile[k][tx] = in[(r0 + k) * ld_in + c0 + tx];
    __syncthreads();
    for (int k = ty; k < 32; k += 8)
        if (c0 + k < cols && r0 + tx < rows)
            out[(c0 + k) * ld_out + r0 + tx] = tile[tx][k];
}

static int transpose2d(const double *in, int64_t ld_in, int64_t rows, int64_t cols, double *out, int64_t ld_out)
{
    if (rows == 0 || cols == 0)
        return COMET_HIP_OK;
    if (ceil_div(rows, 32) > 65535)
        return set_error(COMET_HIP_ERR_SIZE, "dense operand with %lld rows is too tall to turn", (long long)rows);
    KernelTimer t("transpose2d_tile");
    transpose2d_tile<<<dim3((unsigned)ceil_div(cols, 32), (unsigned)ceil_div(rows, 32)), dim3(256), 0, stream()>>>(
        in, ld_in, rows, cols, out, ld_out);
    COMET_HIPCHK(hipGetLastError());
    return COMET_HIP_OK;
}

static int transposed_of(Csr *b, Csr **out)
{
    if (!b->transposed) {
        b->transposed = csr_transposed_copy(b);
        if (!b->transposed)
            return COMET_HIP_ERR_HIP;
    }
    *out = b->transposed;
    return COMET_HIP_OK;
}

extern "C" int comet_hip_vecmat_csr_f64(int64_t csr, int64_t x_dptr, int64_t y_dptr, int accumulate)
{
    COMET_CHK(ensure_init());
    Csr *b = csr_from_handle(csr);
    if (!b)
        return COMET_HIP_ERR_HANDLE;
    Csr *t = nullptr;
    COMET_CHK(transposed_of(b, &t));
    return spmv_run(t, x_dptr, y_dptr, accumulate);
}

static Workspace g_left_a, g_left_c;

extern "C" int comet_hip_densemat_csr_f64(int64_t csr, int64_t M, int64_t a_dptr, int64_t lda, int64_t c_dptr,
                                          int64_t ldc, int accumulate)
{
    COMET_CHK(ensure_init());
    Csr *b = csr_from_handle(csr);
    if (!b)
        return COMET_HIP_ERR_HANDLE;
    if (M < 0 || lda < b->nrows || ldc < b->ncols)
        return set_error(COMET_HIP_ERR_ARG, "bad M/lda/ldc (%lld, %lld, %lld)", (long long)M, (long long)lda,
                         (long long)ldc);
    if (M == 0 || b->ncols == 0)
        return COMET_HIP_OK;
    if (!c_dptr || (b->nrows > 0 && !a_dptr))
        return set_error(COMET_HIP_ERR_ARG, "null matrix passed to comet_hip_densemat_csr_f64");
    Csr *t = nullptr;
    COMET_CHK(transposed_of(b, &t));
    COMET_CHK(g_left_a.ensure(sizeof(double) * (size_t)(b->nrows > 0 ? b->nrows : 1) * (size_t)M, false));
    COMET_CHK(g_left_c.ensure(sizeof(double) * (size_t)b->ncols * (size_t)M, false));
    double *at = (double *)g_left_a.ptr, *ct = (double *)g_left_c.ptr;
    COMET_CHK(transpose2d((const double *)a_dptr, lda, M, b->nrows, at, M));
    if (accumulate)
        COMET_CHK(transpose2d((const double *)c_dptr, ldc, M, b->ncols, ct, M));
    COMET_CHK(spmm_run(t, M, (int64_t)at, M, (int64_t)ct, M, accumulate));
    return transpose2d(ct, M, b->ncols, M, (double *)c_dptr, ldc);
}

// ============================================================================
// SDDMM: A = B .* (C x D), B and A sparse with one structure, C and D dense.
// The reference computes this as T = C x D followed by B .* T, and with
// --opt-fusion keeps only the entries of T that B samples
// (lib/Dialect/IndexTree/Transforms/KernelFusion.cpp:1049-1220; the test is
// test/integration/kernels/sddmm.ta).  Either way a stored entry (i, j) gets
// val * sum_k C[i,k] * D[k,j], the sum unfused and in ascending k.
// A wavefront takes 64 stored entries, KT = 16 columns of C and of the transposed D at a time: a group of eight lanes has
// eight entries next to each other, and loads 128 bytes of each one's row of D, 16 a lane - the row of C only where it
// is not that of the entry before, and entries of one row lie together.  The products go to LDS, and lane e adds those
// of entry e in ascending k while the next 16 columns are on their way.  (Other numbers of entries and columns at a time: where
// they are chosen.)  (Sixteen entries and 64 columns at a time read C
// for every entry and left three quarters of the lanes idle in the sums: whole call, zipf, 16 entries a row, 250000 rows K = 64
// 304 -> 228 us, 48 270 -> 179, 33 259 -> 195, 17 124 -> 109, 9 83 -> 67, 5 66 -> 58; 500000 rows K = 15 216 -> 166, 3 121 ->
// 98.)  Bound by the
// way of D's rows from the L2s: 16 of the 18.6 M lines that the CUs ask for at K = 64, 80 of them under way a CU, a third
// of them beyond the L2.  D is transposed first, so that its "row" for a
// column j is contiguous; the row of every entry comes from a list kept in B's handle (searching pos per entry cost
// 80 % of the time).
// ============================================================================
constexpr int SDDMM_W = 4;               // wavefronts per workgroup

// order (or null: as stored): the places of the entries in B, XCD x's from start.v[x] on; rows, cols: theirs, in that order
// SMALL: an address is a 24-bit multiply and an add
struct SddmmStart { int64_t v[9]; };
template <bool SMALL>
struct SddmmAt {
    using Off = std::conditional_t<SMALL, uint32_t, int64_t>;
    __device__ static Off row(int r, int64_t ld, int64_t col)
    {
        if constexpr (SMALL)
            return __umul24((unsigned)r, (unsigned)ld * 8u) + (unsigned)col * 8u;
        else
            return ((int64_t)r * ld + col) * 8;
    }
    __device__ static const double *at(const double *base, Off o)
    {
        return reinterpret_cast<const double *>(reinterpret_cast<const char *>(base) + o);
    }
};
// KT: columns of a row that are products at a time; R: entries of KT / 2 lanes
template <bool SMALL, int KT, int R>
__global__ __launch_bounds__(SDDMM_W * 64, 4) void sddmm_kernel(int64_t nnz, const int32_t *__restrict__ order,
                                                             SddmmStart start, const int32_t *__restrict__ rows,
                                                             const int32_t *__restrict__ cols,
                                                             const double *__restrict__ val,
                                                             const double *__restrict__ C, int64_t ldc,
                                                             const double *__restrict__ Dt, int64_t ldt, int64_t K,
                                                             double *__restrict__ out)
{
    using At = SddmmAt<SMALL>;
    constexpr int LANES = KT / 2, E = 64 / LANES * R;
    // a row of products in LDS: 16-byte accesses of consecutive lanes, one row apart, fall into different banks
    constexpr int LD = KT + 2;
    __shared__ __align__(16) double tiles[SDDMM_W][E * LD];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    double *tile = tiles[wave];
    const int64_t first = order ? start.v[blockIdx.x & 7] : 0, end = order ? start.v[(blockIdx.x & 7) + 1] : nnz;
    const int64_t base = first + ((int64_t)(order ? blockIdx.x >> 3 : blockIdx.x) * SDDMM_W + wave) * E;
    if (base >= end)
        return;
    const int cnt = (int)(end - base < E ? end - base : E);
    // lane e owns entry base + e; behind the last one, that one again
    const int64_t at = base + (lane < cnt ? lane : cnt - 1);
    const int my_col = cols[at], my_row = rows[at];
    const int64_t p = order ? order[at] : at;
    const double v = val[p];
    const int prev = __shfl_up(my_row, 1, 64);
    const unsigned long long again = __ballot(lane > 0 && my_row == prev);      // entries in the row of the one before
    double t = 0.0;
    const auto sum = [&](int n) {
        const double2 *mine = reinterpret_cast<const double2 *>(tile + (lane & (E - 1)) * LD);
        int q = 0;
#pragma unroll 8
        for (; q < n / 2; ++q) {
            const double2 w = mine[q];
            t = t + w.x;
            t = t + w.y;
        }
        if (n & 1)
            t = t + mine[q].x;
    };
    // Pieces of KT columns, a last one of more than half as many like them, the lanes behind its end idle; a shorter rest
    // takes as many lanes to an entry as it has columns for, two a lane.  The next piece is on its way while one is added (the
    // rest too took more registers than there are).
    const int64_t whole = K / KT;
    const int rest = (int)(K - whole * KT);
    const int64_t pieces = whole + (rest > KT / 2 ? 1 : 0);
    const int rn = pieces > whole ? 0 : rest;
    spmm_pair c[R], d[R];
    if (pieces > 0) {
        const int g = lane / LANES, sub = lane % LANES;
        const unsigned kept = (unsigned)(again >> (R * g)) & ~1u;      // bit u: the row of C is there already
        // in a last piece: one column back where the lane has one only, to the first where it has none
        const bool half = rest - 1 == 2 * sub;
        const int back = half ? 1 : 2 * sub < rest ? 0 : 2 * sub;
        typename At::Off co[R], dO[R];
#pragma unroll
        for (int u = 0; u < R; ++u) {
            co[u] = At::row(__shfl(my_row, R * g + u, 64), ldc, 2 * sub);
            dO[u] = At::row(__shfl(my_col, R * g + u, 64), ldt, 2 * sub);
        }
        const auto load = [&](int64_t i) {
            const double *Ck = C + i * KT, *Dk = Dt + i * KT;
            const typename At::Off less = i == whole ? (typename At::Off)back * 8 : 0;
#pragma unroll
            for (int u = 0; u < R; ++u) {
                if (!(kept >> u & 1u))
                    c[u] = *reinterpret_cast<const spmm_pair *>(At::at(Ck, co[u] - less));
                d[u] = *reinterpret_cast<const spmm_pair *>(At::at(Dk, dO[u] - less));
            }
        };
        load(0);
        for (int64_t i = 0; i < pieces; ++i) {
            const bool one = half && i == whole;
            spmm_pair cur = c[0];
#pragma unroll
            for (int u = 0; u < R; ++u) {
                cur.x = kept >> u & 1u ? cur.x : c[u].x;
                cur.y = kept >> u & 1u ? cur.y : c[u].y;
                double2 q = make_double2(cur.x * d[u].x, cur.y * d[u].y);
                if (one)
                    q.x = q.y;
                *reinterpret_cast<double2 *>(tile + (R * g + u) * LD + 2 * sub) = q;
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
            if (i + 1 < pieces)
                load(i + 1);
            sum(i < whole ? KT : rest);
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
        }
    }
    if (rn > 0) {
        const int rL = (rn + 1) / 2, rG = 64 / rL, rounds = (E + rG - 1) / rG;
        const int rg = lane / rL, rsub = lane - rg * rL, e0 = rg * rounds;
        // the last lane of an odd number has one column, and reads the one before it as well, if there is one
        const bool rhalf = rsub == rL - 1 && (rn & 1);
        const unsigned rkept = (unsigned)(again >> (e0 & 63)) & ~1u;
        const int64_t from = K - rn + 2 * rsub, at = from - (rhalf && from > 0 ? 1 : 0);
#pragma unroll
        for (int u = 0; u < R; ++u) {
            if (u < rounds) {
                const int e = e0 + u < E ? e0 + u : E - 1;
                const int r = __shfl(my_row, e, 64), j = __shfl(my_col, e, 64);
                const double *cp = At::at(C, At::row(r, ldc, at)), *dp = At::at(Dt, At::row(j, ldt, at));
                if (K > 1) {
                    if (!(rkept >> u & 1u))
                        c[u] = *reinterpret_cast<const spmm_pair *>(cp);
                    d[u] = *reinterpret_cast<const spmm_pair *>(dp);
                } else {
                    c[u].x = c[u].y = *cp;
                    d[u].x = d[u].y = *dp;
                }
            }
        }
        spmm_pair cur = c[0];
#pragma unroll
        for (int u = 0; u < R; ++u) {
            const int e = e0 + u;
            if (u < rounds && rg < rG && e < E) {
                cur.x = K > 1 && (rkept >> u & 1u) ? cur.x : c[u].x;
                cur.y = K > 1 && (rkept >> u & 1u) ? cur.y : c[u].y;
                double2 q = make_double2(cur.x * d[u].x, cur.y * d[u].y);
                if (rhalf)
                    q.x = q.y;
                *reinterpret_cast<double2 *>(tile + e * LD + 2 * rsub) = q;
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
        sum(rn);
    }
    if (lane < cnt)
        out[p] = v * t;
}

// ---------------------------------------------------------------------------
// The order of the entries that keeps D in the L2s.  Every gather of a row of D
// is a trip to the memory-side cache when D is larger than an L2 and columns come
// as they please.  But in a matrix with long rows most entries are theirs, and
// the rows of C they need are few: those entries are taken by blocks of columns,
// every block by one XCD (the blocks dealt so that the XCDs have equal shares),
// and within a block as stored.  The other entries go behind them as stored.
// The sizes are what fits an L2 at K = 64.  They are kept for every K: wider rows are taken 64 columns at a time, and a
// slice that only half fits still saves most of its trips.  Whole call as stored / in order, us: 200000 rows, 3.7 M
// entries, K = 3 51 / 51, 9 91 / 65, 24 135 / 89, 48 204 / 140, 64 271 / 178, 128 533 / 361, 256 1077 / 831; 1000000 rows,
// 15 M entries, K = 3 340 / 287, 24 719 / 572, 48 1039 / 817, 64 1383 / 1068, 128 2929 / 2137.
// ---------------------------------------------------------------------------
constexpr int64_t SDDMM_SLICE = 4608;               // columns of a block, at least: 2.25 MiB of D at K = 64
constexpr int SDDMM_BLOCKS_MOST = 4096;
constexpr int64_t SDDMM_LONG_ROWS = 4096;           // long rows at most: 2 MiB of C at K = 64
constexpr int64_t SDDMM_ORDER_NNZ = 1 << 19;        // fewer entries are not worth ordering
constexpr int64_t SDDMM_ORDER_D = 8 << 20;          // bytes of D: less stays in the L2s by itself

// rows[b], entries[b]: rows of [2^b, 2^(b + 1)) entries, and the entries in them
__global__ __launch_bounds__(256) void sddmm_row_lengths(const int64_t *__restrict__ pos, int64_t nrows,
                                                         unsigned long long *__restrict__ rows,
                                                         unsigned long long *__restrict__ entries)
{
    __shared__ unsigned long long n[64], s[64];
    if (threadIdx.x < 64)
        n[threadIdx.x] = s[threadIdx.x] = 0;
    __syncthreads();
    for (int64_t r = (int64_t)blockIdx.x * 256 + threadIdx.x; r < nrows; r += (int64_t)gridDim.x * 256) {
        const unsigned long long len = (unsigned long long)(pos[r + 1] - pos[r]);
        if (len) {
            const int b = 63 - __clzll((long long)len);
            atomicAdd(&n[b], 1ull);
            atomicAdd(&s[b], len);
        }
    }
    __syncthreads();
    if (threadIdx.x < 64 && n[threadIdx.x]) {
        atomicAdd(&rows[threadIdx.x], n[threadIdx.x]);
        atomicAdd(&entries[threadIdx.x], s[threadIdx.x]);
    }
}

// count[c / slice]: entries of long rows in the block
__global__ __launch_bounds__(256) void sddmm_block_counts(int64_t nnz, const int32_t *__restrict__ entry_row,
                                                          const int32_t *__restrict__ crd, const int64_t *__restrict__ pos,
                                                          int64_t min_len, int64_t slice, int nblocks,
                                                          unsigned *__restrict__ count)
{
    __shared__ unsigned n[SDDMM_BLOCKS_MOST];
    for (int b = threadIdx.x; b < nblocks; b += 256)
        n[b] = 0;
    __syncthreads();
    for (int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x; p < nnz; p += (int64_t)gridDim.x * 256) {
        const int64_t r = entry_row[p];
        if (pos[r + 1] - pos[r] >= min_len)
            atomicAdd(&n[crd[p] / slice], 1u);
    }
    __syncthreads();
    for (int b = threadIdx.x; b < nblocks; b += 256)
        if (n[b])
            atomicAdd(&count[b], n[b]);
}

// where[first[b] + share]: the place of a share of block b in the order; short_ends[x]: the entries of short rows up to
// this one are XCD x's, and come behind its blocks, at short_place[x]
struct SddmmShort { int64_t ends[8]; int32_t place[8]; };
__global__ __launch_bounds__(256) void sddmm_keys(int64_t nnz, const int32_t *__restrict__ entry_row,
                                                  const int32_t *__restrict__ crd, const int64_t *__restrict__ pos,
                                                  int64_t min_len, int64_t slice, const int32_t *__restrict__ first,
                                                  const int32_t *__restrict__ where, SddmmShort shorts,
                                                  uint64_t *__restrict__ keys, uint32_t *__restrict__ idx)
{
    const int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (p >= nnz)
        return;
    const int64_t r = entry_row[p];
    int key;
    if (pos[r + 1] - pos[r] >= min_len) {
        const int b = (int)(crd[p] / slice);
        const int shares = first[b + 1] - first[b];
        key = where[first[b] + (shares > 1 ? (int)(p * shares / nnz) : 0)];
    } else {
        int x = 0;
        while (x < 7 && p >= shorts.ends[x])
            ++x;
        key = shorts.place[x];
    }
    keys[p] = (uint64_t)key;
    idx[p] = (uint32_t)p;
}

// the entries' rows and columns in the order of their places
__global__ __launch_bounds__(256) void sddmm_gather(int64_t nnz, const int32_t *__restrict__ order,
                                                    const int32_t *__restrict__ entry_row, const int32_t *__restrict__ crd,
                                                    int32_t *__restrict__ rows, int32_t *__restrict__ cols)
{
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= nnz)
        return;
    const int p = order[i];
    rows[i] = entry_row[p];
    cols[i] = crd[p];
}

// start[x] = first entry whose key is limit[x] or more
__global__ void sddmm_starts(int64_t nnz, const uint64_t *__restrict__ keys, SddmmStart limit, int64_t *__restrict__ start)
{
    if (threadIdx.x >= 9)
        return;
    int64_t lo = 0, hi = nnz;
    while (lo < hi) {
        const int64_t mid = (lo + hi) >> 1;
        if ((int64_t)keys[mid] < limit.v[threadIdx.x])
            lo = mid + 1;
        else
            hi = mid;
    }
    start[threadIdx.x] = lo;
}

static Workspace g_sddmm_plan;

static int sddmm_order(Csr *b, const int32_t *rows)
{
    b->sddmm_state = 1;
    if (b->nnz >= (1ll << 31))
        return COMET_HIP_OK;
    // ---- which rows are long
    COMET_CHK(g_sddmm_plan.ensure(sizeof(uint64_t) * 128 + sizeof(int32_t) * 2 * (SDDMM_BLOCKS_MOST + 1) + 9 * sizeof(int64_t), false));
    unsigned long long *hist = (unsigned long long *)g_sddmm_plan.ptr, lengths[128];
    COMET_HIPCHK(hipMemsetAsync(hist, 0, sizeof lengths, stream()));
    sddmm_row_lengths<<<dim3((unsigned)std::min<int64_t>(ceil_div(b->nrows, 256), 1024)), dim3(256), 0, stream()>>>(
        b->pos, b->nrows, hist, hist + 64);
    COMET_HIPCHK(hipMemcpyAsync(lengths, hist, sizeof lengths, hipMemcpyDeviceToHost, stream()));
    COMET_CHK(stream_wait());
    int bits = 63;
    int64_t nlong = 0, in_long = 0;
    while (bits >= 5 && nlong + (int64_t)lengths[bits] <= SDDMM_LONG_ROWS) {
        nlong += (int64_t)lengths[bits];
        in_long += (int64_t)lengths[64 + bits];
        --bits;
    }
    const int64_t min_len = 1ll << (bits + 1);
    if (in_long * 3 < b->nnz)          // less than a third of the entries: not worth a plan
        return COMET_HIP_OK;
    // ---- the blocks of columns, and which XCD takes which
    const int64_t slice = std::max<int64_t>(SDDMM_SLICE, ceil_div(b->ncols, SDDMM_BLOCKS_MOST));
    const int nblocks = (int)ceil_div(b->ncols, slice);
    unsigned *count = (unsigned *)(hist + 128);
    COMET_HIPCHK(hipMemsetAsync(count, 0, sizeof(unsigned) * (size_t)nblocks, stream()));
    sddmm_block_counts<<<dim3((unsigned)std::min<int64_t>(ceil_div(b->nnz, 1024), 2048)), dim3(256), 0, stream()>>>(
        b->nnz, rows, b->crd, b->pos, min_len, slice, nblocks, count);
    std::vector<unsigned> counts((size_t)nblocks);
    COMET_HIPCHK(hipMemcpyAsync(counts.data(), count, sizeof(unsigned) * (size_t)nblocks, hipMemcpyDeviceToHost, stream()));
    COMET_CHK(stream_wait());
    // a block with more than a 32nd of the entries is shared out
    struct Share { int64_t size; int id; };
    std::vector<int32_t> first((size_t)nblocks + 1, 0);
    std::vector<Share> shares;
    for (int c = 0; c < nblocks; ++c) {
        const int n = (int)std::max<int64_t>(1, ceil_div((int64_t)counts[(size_t)c] * 32, in_long));
        for (int k = 0; k < n; ++k)
            shares.push_back({counts[(size_t)c] / n, first[(size_t)c] + k});
        first[(size_t)c + 1] = first[(size_t)c] + n;
    }
    std::stable_sort(shares.begin(), shares.end(), [](const Share &a, const Share &c) { return a.size > c.size; });
    int64_t load[8] = {};
    std::vector<std::vector<int>> of(8);
    for (const Share &s : shares) {
        const int x = (int)(std::min_element(load, load + 8) - load);
        load[x] += s.size;
        of[(size_t)x].push_back(s.id);
    }
    // the short rows fill up to equal shares
    SddmmShort shorts;
    SddmmStart limit;
    std::vector<int32_t> where((size_t)first[(size_t)nblocks]);
    const double each = (double)b->nnz / 8, in_short = (double)(b->nnz - in_long);
    double given = 0.0;
    int32_t place = 0;
    for (int x = 0; x < 8; ++x) {
        limit.v[x] = place;
        std::sort(of[(size_t)x].begin(), of[(size_t)x].end());
        for (int id : of[(size_t)x])
            where[(size_t)id] = place++;
        given += std::max(0.0, each - (double)load[x]);
        shorts.ends[x] = in_short > 0 ? (int64_t)((double)b->nnz * std::min(1.0, given / in_short)) : b->nnz;
        shorts.place[x] = place++;
    }
    limit.v[8] = place;
    int end_bit = 1;
    while ((1ll << end_bit) <= place)
        ++end_bit;
    // ---- the order
    int32_t *d_first = (int32_t *)count, *d_where = nullptr;
    uint64_t *keys = nullptr;
    uint32_t *idx = nullptr, *order = nullptr;
    int64_t *d_start = (int64_t *)(hist + 128) + SDDMM_BLOCKS_MOST + 1;
    const size_t n = (size_t)b->nnz;
    int rc = COMET_HIP_OK;
    if (dev_malloc((void **)&keys, 16 * n) != hipSuccess || dev_malloc((void **)&idx, 4 * n) != hipSuccess ||
        dev_malloc((void **)&order, 12 * n) != hipSuccess ||
        dev_malloc((void **)&d_where, sizeof(int32_t) * where.size()) != hipSuccess) {
        (void)hipGetLastError();          // without the room the entries are taken as stored
        (void)dev_free(order);
        order = nullptr;
    } else {
        const auto run = [&]() -> int {
            COMET_HIPCHK(hipMemcpyAsync(d_first, first.data(), sizeof(int32_t) * first.size(), hipMemcpyHostToDevice, stream()));
            COMET_HIPCHK(hipMemcpyAsync(d_where, where.data(), sizeof(int32_t) * where.size(), hipMemcpyHostToDevice, stream()));
            sddmm_keys<<<dim3((unsigned)ceil_div(b->nnz, 256)), dim3(256), 0, stream()>>>(
                b->nnz, rows, b->crd, b->pos, min_len, slice, d_first, d_where, shorts, keys, idx);
            COMET_CHK(sort_pairs_u64_u32(keys, keys + n, idx, order, b->nnz, end_bit));
            sddmm_gather<<<dim3((unsigned)ceil_div(b->nnz, 256)), dim3(256), 0, stream()>>>(
                b->nnz, (const int32_t *)order, rows, b->crd, (int32_t *)order + n, (int32_t *)order + 2 * n);
            sddmm_starts<<<dim3(1), dim3(64), 0, stream()>>>(b->nnz, keys + n, limit, d_start);
            COMET_HIPCHK(hipMemcpyAsync(b->sddmm_start, d_start, sizeof b->sddmm_start, hipMemcpyDeviceToHost, stream()));
            return stream_wait();
        };
        rc = run();
    }
    (void)dev_free(keys);
    (void)dev_free(idx);
    (void)dev_free(d_where);
    if (rc != COMET_HIP_OK) {
        (void)dev_free(order);
        return rc;
    }
    if (order) {
        b->sddmm_order = (int32_t *)order;
        b->sddmm_state = 2;
    }
    return COMET_HIP_OK;
}

// ---------------------------------------------------------------------------
// Entries by tiles of columns, D as it is: a workgroup has a tile of up to 512
// columns and the entries in it, by rows, up to ten a lane; sixteen rows of the
// tile of D are in LDS while the next sixteen are on their way, a lane reads its
// column there and its row of C from memory, sixteen bytes at a time, and adds in
// ascending k in a register.  D is read once, and neither turned over nor gathered;
// no product goes through LDS.  What is left is the lines of C: one for every run
// of entries of one row in a tile, looked up eight times, since a lane takes
// sixteen bytes of it - the reason why runs have to be long (sddmm_tiles).  250000
// rows K = 64: the CUs' path for what loads return is busy in 91 % of the cycles,
// their address units in 73 (gathering D 83 and 73, in 237 us with D's transposition against 210).  Rows of C staged in LDS, loaded
// a line at a time, were slower (250000 rows K = 64 279 us against 234).
// ---------------------------------------------------------------------------
constexpr int SDDMM_TILE_T = 1024, SDDMM_TILE_COLS = 512, SDDMM_TILE_K = 16, SDDMM_TILE_BATCHES = 10;
constexpr int SDDMM_TILE_ENTRIES = SDDMM_TILE_T * SDDMM_TILE_BATCHES;          // what the registers hold of a tile
constexpr size_t SDDMM_TILE_LDS = sizeof(double) * 2 * SDDMM_TILE_K * SDDMM_TILE_COLS;
static_assert(SDDMM_TILE_K == SDDMM_TILE_T / 64, "a wavefront fetches a row of the tile");

// begin, count: entries in the order; col: first column of the tile
struct SddmmItem { int64_t begin; int32_t count, col; };

extern __shared__ __align__(16) double sddmm_lds[];

template <bool SMALL>
__global__ __launch_bounds__(SDDMM_TILE_T) void sddmm_tile_kernel(const SddmmItem *__restrict__ items, const int32_t *__restrict__ order,
                                                                const int32_t *__restrict__ rows, const int32_t *__restrict__ cols,
                                                                const double *__restrict__ val, const double *__restrict__ C,
                                                                int64_t ldc, const double *__restrict__ D, int64_t ldd,
                                                                int64_t ncols, int64_t K, int width, double *__restrict__ out)
{
    using At = SddmmAt<SMALL>;
    constexpr int KT = SDDMM_TILE_K, NB = SDDMM_TILE_BATCHES, ROW = SDDMM_TILE_COLS;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const SddmmItem it = items[blockIdx.x];
    const int count = it.count, nb = (count + SDDMM_TILE_T - 1) / SDDMM_TILE_T;
    const int w = (int)(ncols - it.col < width ? ncols - it.col : width);
    typename At::Off row[NB];
    int col[NB];
    double t[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        const int e = b * SDDMM_TILE_T + (int)threadIdx.x;
        const int64_t at = it.begin + (e < count ? e : count - 1);
        row[b] = At::row(rows[at], ldc, 0);
        col[b] = b < nb ? cols[at] - it.col : 0;
        t[b] = 0.0;
    }
    double next[ROW / 64];
    const auto fetch = [&](int64_t i) {
        const int64_t k = i * KT + wave;
#pragma unroll
        for (int q = 0; q < ROW / 64; ++q)
            if (k < K && 64 * q + lane < w)
                next[q] = D[k * ldd + it.col + 64 * q + lane];
    };
    const auto put = [&](double *buf) {
#pragma unroll
        for (int q = 0; q < ROW / 64; ++q)
            if (64 * q + lane < w)
                buf[wave * ROW + 64 * q + lane] = next[q];
    };
    const int64_t pieces = K / KT;
    const int rest = (int)(K - pieces * KT);
    fetch(0);
    put(sddmm_lds);
    __syncthreads();
    // Sixteen columns from Ck on, or a last piece of kp: half of a batch's are on their way while the other half is added.
    // MANY: of more than four columns; no load and no sum on a condition then, which would make every sum wait for all loads,
    // but the last two columns in the place of those behind them, and sums that are dropped.
    enum { ALL, MANY, FEW };
    const auto piece = [&](const double *buf, const double *Ck, auto kind, int kp) {
        constexpr int KIND = decltype(kind)::value;
        spmm_pair c[2][KT / 4];
        const auto load = [&](int h, typename At::Off r) {
#pragma unroll
            for (int q = 0; q < KT / 4; ++q) {
                const int k = h * (KT / 2) + 2 * q;
                if (KIND == ALL || (KIND == FEW && k + 1 < kp))
                    c[h][q] = *reinterpret_cast<const spmm_pair *>(At::at(Ck + k, r));
                else if (KIND == MANY)
                    c[h][q] = *reinterpret_cast<const spmm_pair *>(At::at(Ck + (k + 1 < kp ? k : kp - 2), r));
                else if (k < kp)
                    c[h][q].x = *At::at(Ck + k, r);
            }
        };
        const auto add = [&](int h, double &t, const double *d) {
#pragma unroll
            for (int q = 0; q < KT / 4; ++q) {
                const int k = h * (KT / 2) + 2 * q;
                if constexpr (KIND == MANY) {
                    const double x = t + (k + 1 < kp ? c[h][q].x : c[h][q].y) * d[k * ROW];
                    t = k < kp ? x : t;
                    const double y = t + c[h][q].y * d[(k + 1) * ROW];
                    t = k + 1 < kp ? y : t;
                } else {
                    if (KIND == ALL || k < kp)
                        t = t + c[h][q].x * d[k * ROW];
                    if (KIND == ALL || k + 1 < kp)
                        t = t + c[h][q].y * d[(k + 1) * ROW];
                }
            }
        };
        const bool both = KIND == ALL || (KIND == MANY && kp > KT / 2);
        load(0, row[0]);
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            if (b < nb) {
                const double *d = buf + col[b];
                if (both)
                    load(1, row[b]);
                add(0, t[b], d);
                if (b + 1 < NB)
                    load(0, row[b + 1 < NB ? b + 1 : b]);
                if (both)
                    add(1, t[b], d);
            }
        }
    };
    for (int64_t i = 0; i < pieces; ++i) {
        fetch(i + 1);
        piece(sddmm_lds + (i & 1) * KT * ROW, C + i * KT, std::integral_constant<int, ALL>(), KT);
        put(sddmm_lds + ((i + 1) & 1) * KT * ROW);
        __syncthreads();
    }
    if (rest > 4)
        piece(sddmm_lds + (pieces & 1) * KT * ROW, C + pieces * KT, std::integral_constant<int, MANY>(), rest);
    else if (rest > 0)
        piece(sddmm_lds + (pieces & 1) * KT * ROW, C + pieces * KT, std::integral_constant<int, FEW>(), rest);
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        const int e = b * SDDMM_TILE_T + (int)threadIdx.x;
        if (e < count) {
            const int64_t p = order[it.begin + e];
            out[p] = val[p] * t[b];
        }
    }
}

// keys[p]: the tile of entry p
__global__ __launch_bounds__(256) void sddmm_tile_keys(int64_t nnz, const int32_t *__restrict__ crd, int width,
                                                       uint64_t *__restrict__ keys, uint32_t *__restrict__ idx)
{
    const int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (p >= nnz)
        return;
    keys[p] = (uint64_t)(crd[p] / width);
    idx[p] = (uint32_t)p;
}

// start[x] = first entry of tile x or a later one, x = 0 .. ntiles
__global__ __launch_bounds__(256) void sddmm_tile_starts(int64_t nnz, const uint64_t *__restrict__ keys, int64_t ntiles,
                                                         int64_t *__restrict__ start)
{
    const int64_t x = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (x > ntiles)
        return;
    int64_t lo = 0, hi = nnz;
    while (lo < hi) {
        const int64_t mid = (lo + hi) >> 1;
        if ((int64_t)keys[mid] < x)
            lo = mid + 1;
        else
            hi = mid;
    }
    start[x] = lo;
}

// *runs += entries that are not of the row and tile of the one before
__global__ __launch_bounds__(256) void sddmm_tile_runs(int64_t nnz, const int32_t *__restrict__ rows, const int32_t *__restrict__ crd,
                                                       int width, unsigned long long *__restrict__ runs)
{
    unsigned long long mine = 0;
    for (int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x; p < nnz; p += (int64_t)gridDim.x * 256)
        mine += p == 0 || rows[p] != rows[p - 1] || crd[p] / width != crd[p - 1] / width;
    for (int d = 32; d > 0; d >>= 1)
        mine += (unsigned long long)__shfl_down((int)mine, d, 64);
    if ((threadIdx.x & 63) == 0)
        atomicAdd(runs, mine);
}

// How a matrix is cut into tiles: every CU the same number of them (rounds), of as few columns as the entries allow.  (One
// workgroup is on a CU at a time: 250000 columns, K = 64, in 489 tiles 214 us, in 559 275.)
static int64_t sddmm_tile_width(const Csr *b, int64_t *rounds)
{
    const double most = 0.9 * SDDMM_TILE_ENTRIES * (double)b->ncols / (double)b->nnz;
    const int64_t width = most < SDDMM_TILE_COLS ? std::max<int64_t>(1, (int64_t)most) : SDDMM_TILE_COLS;
    *rounds = ceil_div(b->ncols, num_cus() * width);
    return std::max<int64_t>(16, ceil_div(b->ncols, num_cus() * *rounds));
}

// The plan: worth it where a run of entries of one row in one tile is two and a half entries long.  us, whole call, gathered / by
// tiles, and entries a run: zipf 20000 rows of 15 (3.7) K = 33 23.2 / 14.5, 250000 of 16 (2.7) 196 / 149, band of 15 in 100000 rows (15) K = 64 78.8 / 60.6;
// R-MAT scale 15 (2.2) K = 33 38.8 / 44.1, scale 17 (2.1) K = 64 129 / 151; 100000 rows of 16 uniform entries (1.03) K = 64
// 140 / 158, 60000 of 40 K = 16 46 / 102.
constexpr double SDDMM_TILE_RUN = 2.5;
static int sddmm_tiles(Csr *b, const int32_t *rows)
{
    b->sddmm_tile_state = 1;
    int64_t rounds = 0;
    const int64_t width = sddmm_tile_width(b, &rounds);
    {
        unsigned long long *held = nullptr;
        COMET_CHK(mailbox((void **)&held));
        COMET_CHK(g_sddmm_plan.ensure(sizeof *held, false));
        COMET_HIPCHK(hipMemsetAsync(g_sddmm_plan.ptr, 0, sizeof *held, stream()));
        sddmm_tile_runs<<<dim3((unsigned)std::min<int64_t>(ceil_div(b->nnz, 256), 4 * (int64_t)num_cus())), dim3(256), 0, stream()>>>(
            b->nnz, rows, b->crd, (int)width, (unsigned long long *)g_sddmm_plan.ptr);
        COMET_HIPCHK(hipGetLastError());
        COMET_HIPCHK(hipMemcpyAsync(held, g_sddmm_plan.ptr, sizeof *held, hipMemcpyDeviceToHost, stream()));
        COMET_CHK(stream_wait());
        const int64_t runs = (int64_t)*(volatile unsigned long long *)held;
        if ((double)b->nnz < SDDMM_TILE_RUN * (double)runs)
            return COMET_HIP_OK;
    }
    // a tile of more entries than its share is taken in parts
    const int64_t share = ceil_div(5 * b->nnz, 4 * num_cus() * rounds);
    const int64_t most = std::min<int64_t>(SDDMM_TILE_ENTRIES, ceil_div(share, SDDMM_TILE_T) * SDDMM_TILE_T);
    const int64_t ntiles = ceil_div(b->ncols, width);
    int end_bit = 1;
    while ((1ll << end_bit) <= ntiles)
        ++end_bit;
    const size_t n = (size_t)b->nnz;
    uint64_t *keys = nullptr;
    uint32_t *idx = nullptr, *order = nullptr;
    int64_t *d_start = nullptr;
    SddmmItem *d_items = nullptr;
    std::vector<SddmmItem> items;
    const auto run = [&]() -> int {
        COMET_HIPCHK(dev_malloc((void **)&keys, 16 * n));
        COMET_HIPCHK(dev_malloc((void **)&idx, 4 * n));
        COMET_HIPCHK(dev_malloc((void **)&order, 12 * n));
        COMET_HIPCHK(dev_malloc((void **)&d_start, sizeof(int64_t) * (size_t)(ntiles + 1)));
        const dim3 grid((unsigned)ceil_div(b->nnz, 256)), block(256);
        sddmm_tile_keys<<<grid, block, 0, stream()>>>(b->nnz, b->crd, (int)width, keys, idx);
        COMET_CHK(sort_pairs_u64_u32(keys, keys + n, idx, order, b->nnz, end_bit));
        sddmm_gather<<<grid, block, 0, stream()>>>(b->nnz, (const int32_t *)order, rows, b->crd, (int32_t *)order + n,
                                                   (int32_t *)order + 2 * n);
        sddmm_tile_starts<<<dim3((unsigned)ceil_div(ntiles + 1, 256)), block, 0, stream()>>>(b->nnz, keys + n, ntiles, d_start);
        std::vector<int64_t> start((size_t)ntiles + 1);
        COMET_HIPCHK(hipMemcpyAsync(start.data(), d_start, sizeof(int64_t) * start.size(), hipMemcpyDeviceToHost, stream()));
        COMET_CHK(stream_wait());
        for (int64_t x = 0; x < ntiles; ++x) {
            const int64_t held = start[(size_t)x + 1] - start[(size_t)x], parts = ceil_div(held, most);
            for (int64_t q = 0; q < parts; ++q) {
                const int64_t from = start[(size_t)x] + held * q / parts, to = start[(size_t)x] + held * (q + 1) / parts;
                items.push_back({from, (int32_t)(to - from), (int32_t)(x * width)});
            }
        }
        std::stable_sort(items.begin(), items.end(), [](const SddmmItem &a, const SddmmItem &c) { return a.count > c.count; });
        COMET_HIPCHK(dev_malloc((void **)&d_items, sizeof(SddmmItem) * items.size()));
        COMET_HIPCHK(hipMemcpyAsync(d_items, items.data(), sizeof(SddmmItem) * items.size(), hipMemcpyHostToDevice, stream()));
        return stream_wait();
    };
    const int rc = run();
    (void)dev_free(keys);
    (void)dev_free(idx);
    (void)dev_free(d_start);
    if (rc != COMET_HIP_OK) {
        (void)dev_free(order);
        (void)dev_free(d_items);
        return rc;
    }
    b->sddmm_tile_order = (int32_t *)order;
    b->sddmm_items = d_items;
    b->sddmm_nitems = (int64_t)items.size();
    b->sddmm_width = (int)width;
    b->sddmm_tile_state = 2;
    return COMET_HIP_OK;
}

static Workspace g_sddmm_dt;

// Whether a matrix that is sampled at again is to go by tiles for these K columns.  us, zipf, 16 entries a row, gathered /
// by tiles: one tile a CU 10000 rows K = 9 10.6 / 7.6, K = 64 17.4 / 14.6, 35000 K = 24 26 / 16.5, 60000 K = 17 39 / 20, 100000
// K = 3 22.5 / 21.2, K = 33 79 / 52, K = 64 96 / 78 - but 5000 rows K = 64 11.8 / 13.0, a chain of four loads and barriers -;
// two tiles a CU, one after the other, 160000 K = 15 56 / 69, K = 24 81 / 73, 250000 K = 33 196 / 149, K = 64 228 / 207,
// 260000 K = 47 189 / 191 (a last piece of 15 columns costs more than a whole one); three
// 350000 K = 24 176 / 186, K = 64 326 / 329.
static bool sddmm_tiled(const Csr *b, int64_t K)
{
    if (K < 1 || b->nnz < (K > 40 ? 1 << 17 : 1 << 15) || b->nnz >= 1ll << 31)
        return false;
    int64_t rounds = 0;
    (void)sddmm_tile_width(b, &rounds);
    return rounds == 1 || (rounds == 2 && K > 16 && K % 16 <= 12);
}

static int sddmm_values(Csr *b, int64_t K, int64_t c_dptr, int64_t ldc, int64_t d_dptr, int64_t ldd, double *out)
{
    if (K < 0 || ldc < K || ldd < b->ncols || (b->nnz > 0 && (!out || (K > 0 && (!c_dptr || !d_dptr)))))
        return set_error(COMET_HIP_ERR_ARG, "bad operands passed to the sddmm entry point (K %lld, ldc %lld, ldd %lld)",
                         (long long)K, (long long)ldc, (long long)ldd);
    if (b->nnz == 0)
        return COMET_HIP_OK;
    const int32_t *rows = nullptr;
    // ordering the entries costs some five products: made when the matrix is sampled at again
    const bool plan_now = b->sddmm_uses > 0 || plan_at_once();
    b->sddmm_uses = 1;
    if (plan_now && sddmm_tiled(b, K)) {
        COMET_CHK(csr_entry_rows(b, &rows));
        if (b->sddmm_tile_state == 0)
            (void)plan_made([&] { return sddmm_tiles(b, rows); });
        if (b->sddmm_tile_state == 2) {
            KernelTimer t("sddmm_tile_kernel");
            const bool small = b->nrows <= 1 << 24 && ldc * 8 < 1 << 24 && b->nrows * ldc * 8 < (1ll << 32);
            const int32_t *order = b->sddmm_tile_order;
            const auto launch = [&](auto kernel) -> int {
                COMET_HIPCHK(hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                                 (int)SDDMM_TILE_LDS));
                kernel<<<dim3((unsigned)b->sddmm_nitems), dim3(SDDMM_TILE_T), SDDMM_TILE_LDS, stream()>>>(
                    (const SddmmItem *)b->sddmm_items, order, order + b->nnz, order + 2 * b->nnz, b->val, (const double *)c_dptr, ldc,
                    (const double *)d_dptr, ldd, b->ncols, K, b->sddmm_width, out);
                COMET_HIPCHK(hipGetLastError());
                return COMET_HIP_OK;
            };
            return small ? launch(sddmm_tile_kernel<true>) : launch(sddmm_tile_kernel<false>);
        }
    }
    // Rows of D begin at a line of 128 bytes, 16 columns are one line then, unless that makes them nearly twice as long
    // (200000 rows, 3.7 M entries, us, packed / so: K = 3 50 / 71, 9 69 / 65, 15 80 / 73, 17 86 / 91, 18 85 / 79, 28 117 /
    // 105, 50 219 / 179, 61 253 / 197, 100 390 / 317), D very large, or no room for it.
    const int64_t whole = ceil_div(K, 16) * 16;
    int64_t ldt = K > 0 && whole * 5 <= K * 9 && b->ncols <= (1ll << 32) / 8 / whole ? whole : K;
    if (K > 0) {
        const auto room = [&] { return g_sddmm_dt.ensure(sizeof(double) * (size_t)b->ncols * (size_t)ldt, false); };
        if (ldt > K && !plan_made(room))
            ldt = K;
        COMET_CHK(room());
        COMET_CHK(transpose2d((const double *)d_dptr, ldd, K, b->ncols, (double *)g_sddmm_dt.ptr, ldt));
    }
    COMET_CHK(csr_entry_rows(b, &rows));
    const bool large = b->nnz >= SDDMM_ORDER_NNZ && b->ncols * K * 8 >= SDDMM_ORDER_D;
    if (large && plan_now && b->sddmm_state == 0)
        (void)plan_made([&] { return sddmm_order(b, rows); });
    const int32_t *order = large && b->sddmm_state == 2 ? b->sddmm_order : nullptr;
    {
        KernelTimer t("sddmm_kernel");
        SddmmStart start{};
        int64_t longest = 0;
        for (int x = 0; x < 9 && order; ++x) {
            start.v[x] = b->sddmm_start[x];
            longest = x > 0 ? std::max(longest, start.v[x] - start.v[x - 1]) : 0;
        }
        // 64 entries to a wavefront, 32 where there are too few to keep every CU in wavefronts that way (us, 64 / 32: 3.9 M
        // entries K = 64 228 / 231; 0.64 M K = 33 32.9 / 32.7; 0.32 M K = 50 30.6 / 28.5; 0.43 M K = 9 10.9 / 11.8, 16 10.9 /
        // 11.7).
        // Where rows of D come from beyond the L2s, these give two lines next to each other quicker than one now and one later:
        // 32 entries with 32 columns at a time (3.7 M entries as stored, 16 / 32 columns: K = 32 142 / 137, 48 214 / 204, 64
        // 285 / 271, 128 570 / 533, 256 1161 / 1077; in order K = 48 140 / 170, 64 178 / 184), and 32 entries where a row is one
        // line and a rest (64 / 32, 300000 rows of 4 uniform entries K = 17 76 / 67, 24 77 / 74, 150000 of 30 173 / 155, 178 / 172).
        // Up to 8 columns, 8 at a time: more workgroups fit a CU (16 / 8 columns: 100000 rows of a band of 27 K = 1 28 / 23, 5
        // 35 / 26, 8 35 / 28, 300000 of 4 uniform ones 25.0 / 23.0, 40.4 / 39.7, 38.7 / 37.8).
        const bool far = !order && large, narrow = K <= 8, wide = far && K >= 32;
        const bool most = K <= 16 || (b->nnz >= SDDMM_ORDER_NNZ && !far);
        const int per_group = SDDMM_W * (most ? 64 : 32);
        const dim3 grid((unsigned)(order ? 8 * ceil_div(longest, per_group) : ceil_div(b->nnz, per_group)));
        const dim3 block(SDDMM_W * 64);
        const int32_t *by_row = order ? order + b->nnz : rows, *by_col = order ? order + 2 * b->nnz : b->crd;
        const double *C = (const double *)c_dptr, *Dt = (const double *)g_sddmm_dt.ptr;
        // rows named in 24 bits, C and D within 4 GiB: an address is a 24-bit multiply and an add
        const bool small = b->nrows <= 1 << 24 && b->ncols <= 1 << 24 && ldc * 8 < 1 << 24 && ldt * 8 < 1 << 24 &&
                           b->nrows * ldc * 8 < (1ll << 32) && b->ncols * ldt * 8 < (1ll << 32);
        const auto launch = [&](auto kernel) {
            kernel<<<grid, block, 0, stream()>>>(b->nnz, order, start, by_row, by_col, b->val, C, ldc, Dt, ldt, K, out);
        };
        if (narrow)
            small ? launch(sddmm_kernel<true, 8, 4>) : launch(sddmm_kernel<false, 8, 4>);
        else if (wide)
            small ? launch(sddmm_kernel<true, 32, 8>) : launch(sddmm_kernel<false, 32, 8>);
        else if (most)
            small ? launch(sddmm_kernel<true, 16, 8>) : launch(sddmm_kernel<false, 16, 8>);
        else
            small ? launch(sddmm_kernel<true, 16, 4>) : launch(sddmm_kernel<false, 16, 4>);
    }
    COMET_HIPCHK(hipGetLastError());
    return COMET_HIP_OK;
}

extern "C" int comet_hip_sddmm_csr_values_f64(int64_t bh, int64_t K, int64_t c_dptr, int64_t ldc, int64_t d_dptr,
                                              int64_t ldd, int64_t out_val_dptr)
{
    COMET_CHK(ensure_init());
    Csr *b = csr_from_handle(bh);
    if (!b)
        return COMET_HIP_ERR_HANDLE;
    return sddmm_values(b, K, c_dptr, ldc, d_dptr, ldd, (double *)out_val_dptr);
}

extern "C" int64_t comet_hip_sddmm_csr_f64(int64_t bh, int64_t K, int64_t c_dptr, int64_t ldc, int64_t d_dptr,
                                           int64_t ldd)
{
    if (ensure_init() != COMET_HIP_OK)
        return 0;
    Csr *b = csr_from_handle(bh);
    if (!b)
        return 0;
    Csr *a = new Csr();
    if (csr_alloc(a, b->nrows, b->ncols, b->nnz) != COMET_HIP_OK) {
        delete a;
        return 0;
    }
    bool ok = hipMemcpyAsync(a->pos, b->pos, sizeof(int64_t) * (size_t)(b->nrows + 1), hipMemcpyDeviceToDevice,
                             stream()) == hipSuccess;
    if (ok && b->nnz > 0)
        ok = hipMemcpyAsync(a->crd, b->crd, sizeof(int32_t) * (size_t)b->nnz, hipMemcpyDeviceToDevice, stream()) ==
             hipSuccess;
    if (!ok)
        set_error(COMET_HIP_ERR_HIP, "copying the structure of the sampled matrix failed");
    if (!ok || sddmm_values(b, K, c_dptr, ldc, d_dptr, ldd, a->val) != COMET_HIP_OK) {
        csr_release(a);
        return 0;
    }
    return csr_register(a);
}
