// TTGT dense contraction for gfx950: the permutation plan, tensor transposes
// staged through LDS, and an fp64 MFMA GEMM.
//
// Plan = index classification, candidate enumeration, cost rule and selection
// of include/comet/Dialect/Utils/Utils.h:586-946 and
// lib/Dialect/TensorAlgebra/Transforms/TCtoTTGTDyn.cpp:240-272 in pnnl/COMET.
// Execution = the transpose -> collapse -> matmul -> expand -> transpose chain
// of TCtoTTGTDyn.cpp:280-672, with the matmul
// (linalg.matmul -> loops, frontends/comet_dsl/comet.cpp:594-595, or the BLIS
// micro-kernel of lib/ExecutionEngine/blis_interface.cpp:143-181) replaced by
// v_mfma_f64_16x16x4_f64 tiles.
#include <stdio.h>
#include <stdlib.h>

#include <algorithm>
#include <cstring>

#include "common.h"
#include "gett_index.h"

namespace comet {

// ============================================================================
// Transposes.  out dim i = in dim perm[i]; both tensors contiguous row-major.
// Dimensions that stay adjacent are merged first.  If the innermost dimension
// is kept, rows are copied (coalesced on both sides).  Otherwise the innermost
// input dimension (b) and the innermost output dimension (a) form 2-D tiles
// that go through LDS, so that reads run along b and writes run along a.
// ============================================================================
constexpr int TR_MAXRANK = 8;
constexpr int TR_TILE = 32;

struct TrDims {
    int rank;
    int64_t out_shape[TR_MAXRANK];
    int64_t src_stride[TR_MAXRANK];   // input stride of output dim i
    int64_t out_stride[TR_MAXRANK];
};

__global__ __launch_bounds__(256) void transpose_rows_kernel(TrDims d, int64_t total, const double *__restrict__ in,
                                                             double *__restrict__ out)
{
    int64_t o = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t step = (int64_t)gridDim.x * blockDim.x;
    for (; o < total; o += step) {
        int64_t rem = o, src = 0;
        for (int i = d.rank - 1; i >= 0; --i) {
            const int64_t c = rem % d.out_shape[i];
            rem /= d.out_shape[i];
            src += c * d.src_stride[i];
        }
        out[o] = in[src];
    }
}

// Tile over (a = output-innermost dim, b = input-innermost dim).  Batch index =
// all other output dims, flattened in output order.
struct TrTile {
    int nbatch_dims;
    int64_t batch_shape[TR_MAXRANK];
    int64_t batch_src_stride[TR_MAXRANK];
    int64_t batch_out_stride[TR_MAXRANK];
    int64_t na, nb;                // extents of a and b
    int64_t a_src_stride;          // input stride of a  (input stride of b is 1)
    int64_t b_out_stride;          // output stride of b (output stride of a is 1)
};

__global__ __launch_bounds__(256) void transpose_tile_kernel(TrTile d, const double *__restrict__ in,
                                                             double *__restrict__ out)
{
    __shared__ double tile[TR_TILE][TR_TILE + 1];
    int64_t rem = blockIdx.z;
    int64_t src = 0, dst = 0;
    for (int i = d.nbatch_dims - 1; i >= 0; --i) {
        const int64_t c = rem % d.batch_shape[i];
        rem /= d.batch_shape[i];
        src += c * d.batch_src_stride[i];
        dst += c * d.batch_out_stride[i];
    }
    const int64_t a0 = (int64_t)blockIdx.x * TR_TILE, b0 = (int64_t)blockIdx.y * TR_TILE;
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;   // 32 x 8
    for (int r = ty; r < TR_TILE; r += 8) {
        const int64_t a = a0 + r, b = b0 + tx;
        if (a < d.na && b < d.nb)
            tile[r][tx] = in[src + a * d.a_src_stride + b];
    }
    __syncthreads();
    for (int r = ty; r < TR_TILE; r += 8) {
        const int64_t b = b0 + r, a = a0 + tx;
        if (a < d.na && b < d.nb)
            out[dst + b * d.b_out_stride + a] = tile[tx][r];
    }
}

static int transpose_device(int rank, const int64_t *in_shape, const int32_t *perm, const double *in, double *out)
{
    if (rank < 1 || rank > TR_MAXRANK)
        return set_error(COMET_HIP_ERR_ARG, "transpose rank %d outside [1,%d]", rank, TR_MAXRANK);
    bool seen[TR_MAXRANK] = {false};
    int64_t total = 1;
    for (int i = 0; i < rank; ++i) {
        if (perm[i] < 0 || perm[i] >= rank || seen[perm[i]])
            return set_error(COMET_HIP_ERR_ARG, "perm is not a permutation of 0..%d", rank - 1);
        seen[perm[i]] = true;
        if (in_shape[i] < 0)
            return set_error(COMET_HIP_ERR_ARG, "negative extent");
        total *= in_shape[i];
    }
    if (total == 0)
        return COMET_HIP_OK;
    int64_t in_stride[TR_MAXRANK];
    {
        int64_t s = 1;
        for (int i = rank - 1; i >= 0; --i) {
            in_stride[i] = s;
            s *= in_shape[i];
        }
    }
    // output dims with merging of runs that are adjacent in the input too; extent-1 dims dropped
    int n = 0;
    int64_t shp[TR_MAXRANK], sst[TR_MAXRANK];
    int last_in = -2;
    for (int i = 0; i < rank; ++i) {
        const int p = perm[i];
        if (in_shape[p] == 1)
            continue;
        if (n > 0 && p == last_in + 1) {
            shp[n - 1] *= in_shape[p];
            sst[n - 1] = in_stride[p];
        } else {
            shp[n] = in_shape[p];
            sst[n] = in_stride[p];
            ++n;
        }
        last_in = p;
    }
    if (n == 0) {   // single element
        COMET_HIPCHK(hipMemcpyAsync(out, in, sizeof(double), hipMemcpyDeviceToDevice, stream()));
        return COMET_HIP_OK;
    }
    int64_t ost[TR_MAXRANK];
    {
        int64_t s = 1;
        for (int i = n - 1; i >= 0; --i) {
            ost[i] = s;
            s *= shp[i];
        }
    }
    if (n == 1) {
        COMET_HIPCHK(hipMemcpyAsync(out, in, sizeof(double) * (size_t)total, hipMemcpyDeviceToDevice, stream()));
        return COMET_HIP_OK;
    }
    if (sst[n - 1] == 1) {   // innermost kept
        TrDims d;
        d.rank = n;
        for (int i = 0; i < n; ++i) {
            d.out_shape[i] = shp[i];
            d.src_stride[i] = sst[i];
            d.out_stride[i] = ost[i];
        }
        const unsigned blocks = (unsigned)std::min<int64_t>(ceil_div(total, 256), (int64_t)num_cus() * 64);
        KernelTimer t("transpose_rows_kernel");
        transpose_rows_kernel<<<dim3(blocks), dim3(256), 0, stream()>>>(d, total, in, out);
        COMET_HIPCHK(hipGetLastError());
        return COMET_HIP_OK;
    }
    // find the output dim that is innermost in the input
    int bdim = -1;
    for (int i = 0; i < n; ++i)
        if (sst[i] == 1)
            bdim = i;
    if (bdim < 0)
        return set_error(COMET_HIP_ERR_ARG, "internal: no unit-stride dimension");
    TrTile d;
    d.nbatch_dims = 0;
    int64_t nbatch = 1;
    for (int i = 0; i < n - 1; ++i) {
        if (i == bdim)
            continue;
        d.batch_shape[d.nbatch_dims] = shp[i];
        d.batch_src_stride[d.nbatch_dims] = sst[i];
        d.batch_out_stride[d.nbatch_dims] = ost[i];
        ++d.nbatch_dims;
        nbatch *= shp[i];
    }
    d.na = shp[n - 1];
    d.nb = shp[bdim];
    d.a_src_stride = sst[n - 1];
    d.b_out_stride = ost[bdim];
    const int64_t ga = ceil_div(d.na, TR_TILE), gb = ceil_div(d.nb, TR_TILE);
    if (gb > 65535 || nbatch > 65535) {
        // fall back to the gather kernel when the grid would not fit
        TrDims g;
        g.rank = n;
        for (int i = 0; i < n; ++i) {
            g.out_shape[i] = shp[i];
            g.src_stride[i] = sst[i];
            g.out_stride[i] = ost[i];
        }
        const unsigned blocks = (unsigned)std::min<int64_t>(ceil_div(total, 256), (int64_t)num_cus() * 64);
        KernelTimer t("transpose_rows_kernel");
        transpose_rows_kernel<<<dim3(blocks), dim3(256), 0, stream()>>>(g, total, in, out);
        COMET_HIPCHK(hipGetLastError());
        return COMET_HIP_OK;
    }
    KernelTimer t("transpose_tile_kernel");
    transpose_tile_kernel<<<dim3((unsigned)ga, (unsigned)gb, (unsigned)nbatch), dim3(256), 0, stream()>>>(d, in, out);
    COMET_HIPCHK(hipGetLastError());
    return COMET_HIP_OK;
}

// ============================================================================
// Contraction on strided operands: C[m,n] (+)= sum_k A[m,k] * B[k,n], where m, n
// and k are multi-indices and the address of an element is the sum of an offset
// that depends on m (or n) alone and one that depends on k alone.  A tensor in
// any index order is such a matrix, so nothing is transposed: the loads that
// bring a tile to LDS follow the tensor's own layout.  DGEMM is the case of one
// index each.
//
// A workgroup (four wavefronts) makes a BM x BN tile of C, each wavefront
// TM x TN MFMA tiles of 16 x 16.  K advances 16 at a time through
// double-buffered LDS, both operands stored k-major (a 16 x 4 operand is one
// ds_read_b64 per lane).  Offsets of the rows and columns are worked out once
// per tile of C, those of the k of some turns at a time, one to a lane.
// A thread takes its elements along whichever index is contiguous in memory
// (A_M / B_N: the outer one, else along k).  Operand layout of
// v_mfma_f64_16x16x4_f64: lane l supplies A[l%16][l/16] and B[l/16][l%16] and
// receives D[4*v + l/16][l%16], v = 0..3 (measured with one-hot operands).
//
// Rows and columns beyond the matrix repeat the last one and are not stored; k
// beyond the end reads the last k and counts as zero.
//
// The sum over k may be shared out over gridDim.y workgroups per tile, which
// leave partial tiles that gett_reduce adds in order: a contraction with few
// outputs and a long sum otherwise runs on a handful of CUs (30 x 61 outputs
// over 54,900 products: 8.7 ms on the one workgroup that a 128 x 128 tile gave it).
// ============================================================================
#ifndef COMET_GM_OCC
#define COMET_GM_OCC 2
#endif
constexpr int GM_BK = 16, GM_PAD = 4;

typedef double double4_t __attribute__((ext_vector_type(4)));

// The same as the kernel takes it.
struct GettDims {
    int nd;
    uint32_t ext[GETT_MAXRANK];
    int64_t s0[GETT_MAXRANK], s1[GETT_MAXRANK];
};
struct GettArgs {
    GettDims m, n, k;            // m: A, C   n: B, C   k: A, B
    uint32_t M, N, K;
    uint32_t turns;              // turns of 16 k per split
};

// an element by its byte offset from a pointer that is the same for the whole wavefront
__device__ __forceinline__ double gett_load(const double *base, uint32_t bytes)
{
    return *reinterpret_cast<const double *>(reinterpret_cast<const char *>(base) + bytes);
}

// The same with the wavefront's part of the offset in a scalar register: a buffer load, whose address needs no vector
// arithmetic (the compiler turns pointer + offset into a 64-bit add per load inside the loop).
typedef double double2_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ __amdgpu_buffer_rsrc_t gett_buffer(const double *p)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<double *>(p), 0, -1, 0x00027000);
}
__device__ __forceinline__ double gett_fetch(__amdgpu_buffer_rsrc_t p, uint32_t bytes, uint32_t scalar_bytes)
{
    return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(p, bytes, scalar_bytes, 0));
}
__device__ __forceinline__ double2_t gett_fetch2(__amdgpu_buffer_rsrc_t p, uint32_t bytes, uint32_t scalar_bytes)
{
    return __builtin_bit_cast(double2_t, __builtin_amdgcn_raw_buffer_load_b128(p, bytes, scalar_bytes, 0));
}

template <typename OFF>
__device__ __forceinline__ void gett_offsets(const GettDims &g, uint32_t i, OFF *o0, OFF *o1)
{
    OFF a = 0, b = 0;
    for (int d = g.nd - 1; d > 0; --d) {
        const uint32_t q = i / g.ext[d], r = i - q * g.ext[d];
        a += (OFF)r * (OFF)g.s0[d];
        b += (OFF)r * (OFF)g.s1[d];
        i = q;
    }
    *o0 = a + (OFF)i * (OFF)g.s0[0];
    *o1 = b + (OFF)i * (OFF)g.s1[0];
}

// Which tile and share of k a workgroup takes.  Workgroup i runs on XCD i mod 8: an XCD takes an eighth of the list of tiles,
// band by band of GETT_BAND rows of tiles, down the columns of a band, so that the workgroups of its CUs share few rows and
// columns of the operands in its L2.  (Tile i to workgroup i spreads the tiles of a row over the XCDs unless a row has a
// multiple of eight.)  us, tile i to workgroup i / in bands of 4 / 8 / 16 / 32, aebf,dfce->abcd: 77 x 1665 outputs of 532
// products 31.5 / 22.2 / 22.2 / 22.2 / 22.2, 20^6 18.5 / 17.6 / 17.3 / 17.1 / 17.1, 24^6 25.9 / 27.6 / 27.4 / 26.8 / 26.9, 26^6
// 32.1 / 34.5 / 34.1 / 33.8 / 33.7, 28^6 41.8 / 40.8 / 40.7 / 40.0 / 39.9, 36^6 128.2 / 124.0 / 124.5 / 124.5 / 124.3, 61^6
// 1996 / 1912 / 1914 / 1930 / 1974, 62^6 2187 / 2114 / 2118 / 2137 / 2177, 64^6 1980 / 1974 / 1979 / 1982 / 1985.
constexpr uint32_t GETT_XCDS = 8, GETT_BAND = 16;
struct GettPlace {
    uint32_t m, n, share;
};
__device__ __forceinline__ GettPlace gett_place(uint32_t tiles_m, uint32_t tiles_n)
{
    const uint32_t all = gridDim.x * gridDim.y, id = blockIdx.y * gridDim.x + blockIdx.x;
    const uint32_t xcd = id % GETT_XCDS, each = all / GETT_XCDS, more = all % GETT_XCDS;
    const uint32_t i = xcd * each + (xcd < more ? xcd : more) + id / GETT_XCDS;
    GettPlace p;
    p.share = i / gridDim.x;
    const uint32_t t = i - p.share * gridDim.x, band = t / (GETT_BAND * tiles_n), first = band * GETT_BAND;
    const uint32_t rows = tiles_m - first < GETT_BAND ? tiles_m - first : GETT_BAND, in = t - first * tiles_n;
    p.n = in / rows;
    p.m = first + (in - p.n * rows);
    return p;
}

// Of how many turns the offsets of irregular k are worked out at a time: sixteen, but one where sixteen would take the fourth
// workgroup its LDS (3844 sums of 3844 products 37.4 us, with one 33.8); and the LDS of a workgroup.
constexpr int gett_kt(int bn) { return bn == 16 ? 1 : 16; }
constexpr size_t gett_lds(int bm, int bn, bool reg)
{
    return sizeof(double) * 2 * GM_BK * (size_t)(bm + bn + 2 * GM_PAD) + (sizeof(uint32_t) + sizeof(int64_t)) * (size_t)(bm + bn) +
           (reg ? 0 : sizeof(uint32_t) * 4 * GM_BK * (size_t)gett_kt(bn));
}

template <int BM, int BN, int WM, int OCC, bool A_M, bool B_N, bool REG, bool RUN>
__global__ __launch_bounds__(256, OCC) void gett_mfma_kernel(GettArgs g, const double *__restrict__ A,
                                                             const double *__restrict__ B, double *__restrict__ C,
                                                             double *__restrict__ partial, int use_c)
{
    constexpr int WN = 4 / WM, TM = BM / WM / 16, TN = BN / WN / 16;
    constexpr int EA = BM / 16, EB = BN / 16;               // elements a thread stages per turn
    constexpr int LDA = BM + GM_PAD, LDB = BN + GM_PAD;
    constexpr int KSA = 256 / BM, KSB = 256 / BN;
    __shared__ double As[2][GM_BK][LDA];
    __shared__ double Bs[2][GM_BK][LDB];
    // offsets in bytes of the rows (A), the columns (B) and, unless they are regular, of the k of KT turns, twice
    constexpr int KT = gett_kt(BN), KN = REG ? 1 : KT * GM_BK;
    __shared__ uint32_t rowA[BM], colB[BN], kA[REG ? 1 : 2][KN], kB[REG ? 1 : 2][KN];
    __shared__ int64_t rowC[BM], colC[BN];
    static_assert(sizeof As + sizeof Bs + sizeof rowA + sizeof colB + sizeof rowC + sizeof colC + (REG ? 0 : sizeof kA + sizeof kB) ==
                      gett_lds(BM, BN, REG), "what a CU holds is reckoned with it");
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave / WN, wn = wave % WN;
    const GettPlace place = gett_place((g.M + BM - 1) / BM, (g.N + BN - 1) / BN);
    const uint32_t m0 = place.m * BM, n0 = place.n * BN;
    const uint32_t k_begin = place.share * g.turns * GM_BK;
    const uint32_t k_end = k_begin + g.turns * GM_BK < g.K ? k_begin + g.turns * GM_BK : g.K;
    const int nt = (int)((k_end - k_begin + GM_BK - 1) / GM_BK);

    // the offsets of the k of KT turns, one to a lane (by sixteen lanes a turn they were the longest chain of every turn)
    const auto k_offsets = [&](int chunk) {
        if (!REG && tid < KN) {
            const uint32_t k = k_begin + (uint32_t)(KN * chunk) + tid;
            uint32_t a, b;
            gett_offsets(g.k, k < k_end ? k : k_end - 1, &a, &b);
            kA[chunk & 1][tid] = a * 8;
            kB[chunk & 1][tid] = b * 8;
        }
    };
    for (int r = tid; r < BM; r += 256) {
        int64_t a, c;
        gett_offsets(g.m, m0 + r < g.M ? m0 + r : g.M - 1, &a, &c);
        rowA[r] = (uint32_t)(a * 8);
        rowC[r] = c;
    }
    for (int c = tid; c < BN; c += 256) {
        int64_t b, d;
        gett_offsets(g.n, n0 + c < g.N ? n0 + c : g.N - 1, &b, &d);
        colB[c] = (uint32_t)(b * 8);
        colC[c] = d;
    }
    k_offsets(0);
    if (KT == 1 && nt > 1)
        k_offsets(1);
    __syncthreads();

    // thread -> elements of a turn's tiles: along the outer index (one row, E values of k) or along k (one k, E rows).
    // REG: sixteen k of a turn are always equally spaced, so an element's offset from the turn's first k never
    // changes: it stays in a register, the turn's part is added to the pointer by the scalar unit, and a turn costs
    // no vector arithmetic at all - it would be taken from the matrix cores' time (4096^3: 2318 us with an add and a
    // 64-bit shift per element, see the figures at GETT_SHAPES).
    // RUN: a thread's elements follow each other along the contiguous index: one address, sixteen bytes a load.
    const int a_k = RUN ? (A_M ? tid / 16 : tid * EA % 16) : A_M ? tid / BM : tid & 15;
    const int a_r = RUN ? (A_M ? tid % 16 * EA : tid * EA / 16) : A_M ? tid % BM : tid >> 4;
    const int b_k = RUN ? (B_N ? tid / 16 : tid * EB % 16) : B_N ? tid / BN : tid & 15;
    const int b_c = RUN ? (B_N ? tid % 16 * EB : tid * EB / 16) : B_N ? tid % BN : tid >> 4;
    const int last = g.k.nd - 1;
    const int64_t sa = g.k.s0[last], sb = g.k.s1[last];          // strides of the innermost k
    constexpr int NA = RUN || (A_M && !REG) ? 1 : EA, NB = RUN || (B_N && !REG) ? 1 : EB;
    uint32_t ao[NA], bo[NB];
    if constexpr (RUN) {           // a run beyond the last row is the last one (their number is a multiple of EA then)
        ao[0] = rowA[A_M && m0 + a_r >= g.M ? g.M - EA - m0 : a_r] + (uint32_t)(a_k * sa * 8);
        bo[0] = colB[B_N && n0 + b_c >= g.N ? g.N - EB - n0 : b_c] + (uint32_t)(b_k * sb * 8);
    } else {
#pragma unroll
        for (int e = 0; e < NA; ++e)
            ao[e] = A_M ? rowA[a_r] + (REG ? (uint32_t)((a_k + KSA * e) * sa * 8) : 0)
                        : rowA[a_r + 16 * e] + (REG ? (uint32_t)(a_k * sa * 8) : 0);
#pragma unroll
        for (int e = 0; e < NB; ++e)
            bo[e] = B_N ? colB[b_c] + (REG ? (uint32_t)((b_k + KSB * e) * sb * 8) : 0)
                        : colB[b_c + 16 * e] + (REG ? (uint32_t)(b_k * sb * 8) : 0);
    }
    double ra[EA], rb[EB];
    // REG: where the turn to load next begins, and how many turns are left in the innermost dimension
    const __amdgpu_buffer_rsrc_t Ab = gett_buffer(A), Bb = gett_buffer(B);
    uint32_t At = 0, Bt = 0, k_next = k_begin, run = 0, outer = 0;

    const auto load_tiles = [&](int t) {
        const uint32_t left = k_end - k_begin - (uint32_t)t * GM_BK;
        if constexpr (REG) {
            if (run == 0) {
                if (t > 0 && last == 1) {          // two dimensions: the next of the outer one, no divisions
                    outer += 1;
                    At = outer * (uint32_t)(g.k.s0[0] * 8);
                    Bt = outer * (uint32_t)(g.k.s1[0] * 8);
                    run = g.k.ext[1] / GM_BK;
                } else {
                    int64_t oa, ob;
                    gett_offsets(g.k, k_next, &oa, &ob);
                    At = (uint32_t)(oa * 8);
                    Bt = (uint32_t)(ob * 8);
                    outer = k_next / g.k.ext[last];
                    run = last > 0 ? (g.k.ext[last] - k_next % g.k.ext[last]) / GM_BK : ~0u;
                }
            }
            if constexpr (RUN) {          // whole turns only
#pragma unroll
                for (int e = 0; e < EA; e += 2) {
                    const double2_t v = gett_fetch2(Ab, ao[0] + e * 8, At);
                    ra[e] = v.x;
                    ra[e + 1] = v.y;
                }
#pragma unroll
                for (int e = 0; e < EB; e += 2) {
                    const double2_t v = gett_fetch2(Bb, bo[0] + e * 8, Bt);
                    rb[e] = v.x;
                    rb[e + 1] = v.y;
                }
            } else if (left >= GM_BK) {
#pragma unroll
                for (int e = 0; e < EA; ++e)
                    ra[e] = gett_fetch(Ab, ao[e], At);
#pragma unroll
                for (int e = 0; e < EB; ++e)
                    rb[e] = gett_fetch(Bb, bo[e], Bt);
            } else {          // the last turn: k beyond the end read the last k and count as zero
#pragma unroll
                for (int e = 0; e < EA; ++e) {
                    const int k = A_M ? a_k + KSA * e : a_k, over = k < (int)left ? 0 : k - (int)left + 1;
                    ra[e] = gett_fetch(Ab, ao[e] - (uint32_t)(over * sa * 8), At);
                    ra[e] = over ? 0.0 : ra[e];
                }
#pragma unroll
                for (int e = 0; e < EB; ++e) {
                    const int k = B_N ? b_k + KSB * e : b_k, over = k < (int)left ? 0 : k - (int)left + 1;
                    rb[e] = gett_fetch(Bb, bo[e] - (uint32_t)(over * sb * 8), Bt);
                    rb[e] = over ? 0.0 : rb[e];
                }
            }
            At += (uint32_t)(GM_BK * 8 * sa);
            Bt += (uint32_t)(GM_BK * 8 * sb);
            k_next += GM_BK;
            --run;
        } else {
            const uint32_t *ka = kA[t / KT & 1] + t % KT * GM_BK, *kb = kB[t / KT & 1] + t % KT * GM_BK;
#pragma unroll
            for (int e = 0; e < EA; ++e)
                ra[e] = gett_load(A, A_M ? ao[0] + ka[a_k + KSA * e] : ao[A_M ? 0 : e] + ka[a_k]);
#pragma unroll
            for (int e = 0; e < EB; ++e)
                rb[e] = gett_load(B, B_N ? bo[0] + kb[b_k + KSB * e] : bo[B_N ? 0 : e] + kb[b_k]);
            if (left < GM_BK) {
#pragma unroll
                for (int e = 0; e < EA; ++e)
                    ra[e] = (uint32_t)(A_M ? a_k + KSA * e : a_k) < left ? ra[e] : 0.0;
#pragma unroll
                for (int e = 0; e < EB; ++e)
                    rb[e] = (uint32_t)(B_N ? b_k + KSB * e : b_k) < left ? rb[e] : 0.0;
            }
        }
    };
    const auto store_tiles = [&](int buf) {
        if constexpr (RUN) {
#pragma unroll
            for (int e = 0; e < EA; ++e)
                As[buf][A_M ? a_k : a_k + e][A_M ? a_r + e : a_r] = ra[e];
#pragma unroll
            for (int e = 0; e < EB; ++e)
                Bs[buf][B_N ? b_k : b_k + e][B_N ? b_c + e : b_c] = rb[e];
        } else {
#pragma unroll
            for (int e = 0; e < EA; ++e)
                As[buf][A_M ? a_k + KSA * e : a_k][A_M ? a_r : a_r + 16 * e] = ra[e];
#pragma unroll
            for (int e = 0; e < EB; ++e)
                Bs[buf][B_N ? b_k + KSB * e : b_k][B_N ? b_c : b_c + 16 * e] = rb[e];
        }
    };

    double4_t acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
            acc[i][j] = (double4_t){0.0, 0.0, 0.0, 0.0};

    load_tiles(0);
    store_tiles(0);
    __syncthreads();
    const int fr = lane & 15, fk = lane >> 4;
    for (int t = 0; t < nt; ++t) {
        const int cur = t & 1;
        double af[2][TM], bf[2][TN];
        const auto fragments = [&](int ks) {          // the operands of the MFMAs of k ks .. ks + 3
#pragma unroll
            for (int i = 0; i < TM; ++i)
                af[ks / 4 & 1][i] = As[cur][ks + fk][wm * (TM * 16) + i * 16 + fr];
#pragma unroll
            for (int j = 0; j < TN; ++j)
                bf[ks / 4 & 1][j] = Bs[cur][ks + fk][wn * (TN * 16) + j * 16 + fr];
        };
        fragments(0);
        if (t + 1 < nt)
            load_tiles(t + 1);
        if (!REG && (t + 2) % KT == 0 && t + 2 < nt)
            k_offsets((t + 2) / KT);           // for the loads of the next turn
#pragma unroll
        for (int ks = 0; ks < GM_BK; ks += 4) {
            if (ks + 4 < GM_BK)
                fragments(ks + 4);
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(af[ks / 4 & 1][i], bf[ks / 4 & 1][j], acc[i][j], 0, 0, 0);
        }
        if (t + 1 < nt)
            store_tiles(cur ^ 1);
        __syncthreads();
    }

    const bool whole = gridDim.y == 1, inside = m0 + BM <= g.M && n0 + BN <= g.N;
    double *out = whole ? C : partial + (uint64_t)place.share * g.M * g.N;
    int64_t cols[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j) {
        const int c = wn * (TN * 16) + j * 16 + fr;
        cols[j] = whole ? colC[c] : (int64_t)(n0 + c);
    }
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int r = wm * (TM * 16) + i * 16 + 4 * v + fk;
            double *row = out + (whole ? rowC[r] : (int64_t)(m0 + r) * g.N);
            if (inside) {
#pragma unroll
                for (int j = 0; j < TN; ++j)
                    row[cols[j]] = whole && use_c ? row[cols[j]] + acc[i][j][v] : acc[i][j][v];
            } else if (m0 + r < g.M) {
#pragma unroll
                for (int j = 0; j < TN; ++j)
                    if (n0 + wn * (TN * 16) + j * 16 + fr < g.N)
                        row[cols[j]] = whole && use_c ? row[cols[j]] + acc[i][j][v] : acc[i][j][v];
            }
        }
}

// C[m,n] (+)= the partial tiles.  `group` threads of a workgroup share an output: each adds every group-th partial in order of
// k, up to eight of them on their way at once, then those sums are added by halves, a step of a fixed tree at a time.
// Bound by the trips to memory one after the other: 491 shares of 1830 outputs, 31 to a thread and four at once, took 6.5 us,
// now 5.7, 3 of them the launch.
constexpr int GETT_REDUCE_T = 1024, GETT_REDUCE_U = 8;
__global__ __launch_bounds__(GETT_REDUCE_T) void gett_reduce(GettArgs g, int splits, int group, const double *__restrict__ partial,
                                                             double *__restrict__ C, int use_c)
{
    __shared__ double lds[GETT_REDUCE_T];
    const int per = GETT_REDUCE_T / group, o = threadIdx.x % per, share = threadIdx.x / per;
    const uint64_t total = (uint64_t)g.M * g.N, i = (uint64_t)blockIdx.x * per + o;
    double s = 0.0;
    if (i < total) {
        const double *at = partial + i;
        for (int z = share; z < splits; z += GETT_REDUCE_U * group) {
            double p[GETT_REDUCE_U];
#pragma unroll
            for (int u = 0; u < GETT_REDUCE_U; ++u)
                p[u] = z + u * group < splits ? at[(uint64_t)(z + u * group) * total] : 0.0;
#pragma unroll
            for (int u = 0; u < GETT_REDUCE_U; ++u)
                s = z + u * group < splits ? s + p[u] : s;
        }
    }
    for (int half = group / 2; half > 0; half /= 2) {
        if (share >= half && share < 2 * half)
            lds[threadIdx.x - half * per] = s;
        __syncthreads();
        if (share < half)
            s = s + lds[threadIdx.x];
        __syncthreads();
    }
    if (share != 0 || i >= total)
        return;
    int64_t ma, mc, nb, nc;
    gett_offsets(g.m, (uint32_t)(i / g.N), &ma, &mc);
    gett_offsets(g.n, (uint32_t)(i % g.N), &nb, &nc);
    C[mc + nc] = use_c ? C[mc + nc] + s : s;
}

// The tile shapes: workgroups a CU holds, the time of a turn of 16 k divided by them on a full CU, and the time of a
// turn of a workgroup that has its CU to itself (measured, us; 4096^3 takes 1908 / 2125 / 2440 / 3109 us with the four
// shapes, the first at 92 % of the matrix cores' rate).  The launch takes the shape and the number of shares of k that
// these figures make cheapest, a last round that fills no more than some of the workgroups' places by what it leaves to a
// CU: small tiles and many shares where the outputs are few, the large tile where they are
// not, and the narrow ones where one side of C is short.
struct GettShape {
    int bm, bn, resident;
    double turn_us, alone_us;
};
constexpr GettShape GETT_SHAPES[] = {{128, 128, 2, 1.86, 2.65}, {64, 64, 4, 0.52, 1.2}, {64, 32, 5, 0.30, 0.71}, {128, 16, 4, 0.38, 0.83}};
// What adding the shares up costs besides reading them, a launch: 10 x 60 x 12 x 40 over 120 products take 13.7 us in eight
// shares, 10.9 in one.
constexpr double GETT_REDUCE_US = 5.0;
// bytes a us that partial tiles are written and read at: few and large, many and small (62 x 62 outputs 97 shares 12.3 us, 194
// 14.4; 300 x 650 over 225 products one share 18.4, four 16.5)
constexpr double GETT_REDUCE_FEW = 6.0e6, GETT_REDUCE_MANY = 3.0e6;
// The large tile loses more where the k have to be looked up: 52^6 in the large tile 790, in the next 812, 62^6 2170 and 2190 to
// 2275, which without this come out as 632 / 708 and 1798 / 1890 (and 64^6, regular, as 1910 / 2130).
constexpr double GETT_IRREGULAR = 1.06;
constexpr int GETT_NSHAPES = sizeof(GETT_SHAPES) / sizeof(GETT_SHAPES[0]);

static Workspace g_gett_partial;

template <int BM, int BN, int WM, int OCC, bool REG, bool RUN>
static void gett_launch(bool a_m, bool b_n, dim3 grid, const GettArgs &g, const double *A, const double *B, double *C,
                        double *partial, int use_c)
{
    const dim3 block(256);
    if (a_m && b_n)
        gett_mfma_kernel<BM, BN, WM, OCC, true, true, REG, RUN><<<grid, block, 0, stream()>>>(g, A, B, C, partial, use_c);
    else if (a_m)
        gett_mfma_kernel<BM, BN, WM, OCC, true, false, REG, RUN><<<grid, block, 0, stream()>>>(g, A, B, C, partial, use_c);
    else if (b_n)
        gett_mfma_kernel<BM, BN, WM, OCC, false, true, REG, RUN><<<grid, block, 0, stream()>>>(g, A, B, C, partial, use_c);
    else
        gett_mfma_kernel<BM, BN, WM, OCC, false, false, REG, RUN><<<grid, block, 0, stream()>>>(g, A, B, C, partial, use_c);
}

// C (+)= A * B over the three indices, none of them empty, A and B within the reach of 32-bit byte offsets.
static int gett_run(GettIndex m, GettIndex n, GettIndex k, int64_t M, int64_t N, int64_t K, const double *A,
                    const double *B, double *C, double beta)
{
    const auto unit_in_c = [](const GettIndex &g) {
        for (int d = 0; d < g.nd; ++d)
            if (g.s1[d] == 1)
                return true;
        return false;
    };
    // Which operand gives the columns: the shorter side when it is short enough for a narrow tile, else the one whose
    // index is contiguous in C, so that sixteen lanes store sixteen neighbours.
    const int64_t shorter = M < N ? M : N;
    const bool swap = shorter <= 32 ? M < N : unit_in_c(m) && !unit_in_c(n);
    if (swap) {
        std::swap(m, n);
        std::swap(M, N);
        std::swap(A, B);
        std::swap(k.s0, k.s1);
    }
    GettArgs g;
    const bool a_m = gett_order(&m, 0);
    const bool b_n = gett_order(&n, 0);
    if (!a_m)
        (void)gett_order(&m, 1);
    if (!b_n)
        (void)gett_order(&n, 1);
    (void)gett_order(&k, a_m ? 1 : 0);
    for (GettIndex *x : {&m, &n, &k})
        if (x->nd == 0) {          // an index of one element
            x->nd = 1;
            x->ext[0] = 1;
            x->s0[0] = x->s1[0] = 0;
        }
    const auto dims = [](const GettIndex &x, GettDims *out) {
        out->nd = x.nd;
        for (int d = 0; d < x.nd; ++d) {
            out->ext[d] = (uint32_t)x.ext[d];
            out->s0[d] = x.s0[d];
            out->s1[d] = x.s1[d];
        }
    };
    dims(m, &g.m);
    dims(n, &g.n);
    dims(k, &g.k);
    g.M = (uint32_t)M;
    g.N = (uint32_t)N;
    g.K = (uint32_t)K;
    const int64_t nk = ceil_div(K, GM_BK);
    const bool reg = k.nd == 1 || k.ext[k.nd - 1] % GM_BK == 0;
    const int64_t cus = num_cus() > 0 ? num_cus() : 256;
    int best = 0;
    int64_t splits = 1;
    double best_us = 0.0;
    for (int c = 0; c < GETT_NSHAPES; ++c) {
        const GettShape &sh = GETT_SHAPES[c];
        const int64_t tiles = ceil_div(M, sh.bm) * ceil_div(N, sh.bn);
        // (shares by powers of two only: 48^6 490 us, now in three 437; 60^6 1900, now 1805; 28^6 45.4, 41.8)
        for (int64_t s = 1; s <= nk && s <= 1024; s += s < 8 ? 1 : s) {
            const int64_t turns = ceil_div(nk, s), groups = tiles * ceil_div(nk, turns);
            const int64_t full = groups / (cus * sh.resident), rest = groups % (cus * sh.resident);
            const double slower = c == 0 && !reg ? GETT_IRREGULAR : 1.0;
            const auto round_us = [&](int64_t a_cu) {
                return (double)turns * std::max(sh.alone_us, (double)a_cu * sh.turn_us) * slower + 2.5;
            };
            const double us = (double)full * round_us(sh.resident) + (rest > 0 ? round_us(ceil_div(rest, cus)) : 0.0) +
                              (s > 1 ? GETT_REDUCE_US + (double)ceil_div(nk, turns) * (double)(M * N) * 16.0 /
                                                            (s <= 4 ? GETT_REDUCE_FEW : GETT_REDUCE_MANY)
                                     : 0.0);
            if (best_us == 0.0 || us < best_us) {
                best_us = us;
                best = c;
                splits = ceil_div(nk, turns);
                g.turns = (uint32_t)turns;
            }
        }
    }
    // COMET_HIP_GETT="shape,shares of k" overrides the choice (every shape is right for every product: the tests send
    // the same one through all of them)
    if (const char *e = getenv("COMET_HIP_GETT")) {
        long long c = 0, s = 1;
        if (sscanf(e, "%lld,%lld", &c, &s) == 2 && c >= 0 && c < GETT_NSHAPES && s >= 1 && s <= nk && s < 65536) {
            best = (int)c;
            g.turns = (uint32_t)ceil_div(nk, s);
            splits = ceil_div(nk, (int64_t)g.turns);
        }
    }
    const GettShape &sh = GETT_SHAPES[best];
    const int64_t tiles = ceil_div(M, sh.bm) * ceil_div(N, sh.bn);
    if (tiles > INT32_MAX)
        return set_error(COMET_HIP_ERR_SIZE, "contraction of %lld x %lld outputs exceeds the launch grid", (long long)M,
                         (long long)N);
    double *partial = nullptr;
    if (splits > 1) {
        COMET_CHK(g_gett_partial.ensure(sizeof(double) * (size_t)splits * (size_t)M * (size_t)N, false));
        partial = (double *)g_gett_partial.ptr;
    }
    const dim3 grid((unsigned)tiles, (unsigned)splits);
    const int use_c = beta != 0.0;
    {
        KernelTimer t("gett_mfma_kernel");
        // sixteen bytes at a time: a thread's run along the contiguous index is unbroken and aligned
        const auto runs = [](const GettIndex &x, const int64_t *s, bool along, int run) {
            for (int d = 0; d < x.nd; ++d)
                if (along && d == x.nd - 1 ? x.ext[d] % run != 0 || s[d] != 1 : s[d] % 2 != 0)
                    return false;
            return true;
        };
        const int ra = a_m ? sh.bm / 16 : 2, rb = b_n ? sh.bn / 16 : 2;
        const bool unbroken = reg && K % GM_BK == 0 && sh.bn >= 64 && (((uintptr_t)A | (uintptr_t)B) & 15) == 0 &&
                           runs(m, m.s0, a_m, ra) && runs(k, k.s0, !a_m, 2) && runs(n, n.s0, b_n, rb) &&
                           runs(k, k.s1, !b_n, 2);
        const auto launch = [&](auto kernel_shape, auto wave_rows, auto occ) {
            constexpr GettShape S = GETT_SHAPES[decltype(kernel_shape)::value];
            constexpr int WM = decltype(wave_rows)::value, OCC = decltype(occ)::value;
            static_assert(S.resident * gett_lds(S.bm, S.bn, false) <= 160 * 1024, "a CU has room for them");
            if constexpr (S.bn >= 64)
                if (unbroken)
                    return gett_launch<S.bm, S.bn, WM, OCC, true, true>(a_m, b_n, grid, g, A, B, C, partial, use_c);
            if (reg)
                gett_launch<S.bm, S.bn, WM, OCC, true, false>(a_m, b_n, grid, g, A, B, C, partial, use_c);
            else
                gett_launch<S.bm, S.bn, WM, OCC, false, false>(a_m, b_n, grid, g, A, B, C, partial, use_c);
        };
        using std::integral_constant;
        if (best == 0)
            launch(integral_constant<int, 0>(), integral_constant<int, 2>(), integral_constant<int, COMET_GM_OCC>());
        else if (best == 1)
            launch(integral_constant<int, 1>(), integral_constant<int, 2>(), integral_constant<int, 4>());
        else if (best == 2)
            launch(integral_constant<int, 2>(), integral_constant<int, 2>(), integral_constant<int, 4>());
        else
            launch(integral_constant<int, 3>(), integral_constant<int, 4>(), integral_constant<int, 4>());
    }
    if (splits > 1) {
        int group = 1;
        while (group < GETT_REDUCE_T / 16 && group * 4 < splits)
            group *= 2;
        KernelTimer t("gett_reduce");
        gett_reduce<<<dim3((unsigned)ceil_div(M * N, GETT_REDUCE_T / group)), dim3(GETT_REDUCE_T), 0, stream()>>>(
            g, (int)splits, group, partial, C, use_c);
    }
    COMET_HIPCHK(hipGetLastError());
    return COMET_HIP_OK;
}

// Elements an operand may have to be read through 32-bit byte offsets (its last byte is one that a buffer may hold).
constexpr int64_t GETT_SPAN = (1ll << 29) - 1;

static int gett_pieces(const GettIndex &m, const GettIndex &n, const GettIndex &k, int64_t limit, int64_t M, int64_t N,
                       int64_t K, const double *A, const double *B, double *C, double beta)
{
    const GettCut cut = gett_cut(m, n, k, limit);
    if (cut.which < 0)
        return gett_run(m, n, k, M, N, K, A, B, C, beta);
    const GettIndex &x = cut.which == 0 ? m : cut.which == 1 ? n : k;
    const int64_t ext = x.ext[cut.d];
    const int64_t o0 = x.s0[cut.d] * cut.first, o1 = x.s1[cut.d] * cut.first;
    for (int half = 0; half < 2; ++half) {
        const int64_t part = half == 0 ? cut.first : ext - cut.first;
        const GettIndex p = gett_part(x, cut.d, part);
        if (cut.which == 0)
            COMET_CHK(gett_pieces(p, n, k, limit, M / ext * part, N, K, A + (half ? o0 : 0), B, C + (half ? o1 : 0), beta));
        else if (cut.which == 1)
            COMET_CHK(gett_pieces(m, p, k, limit, M, N / ext * part, K, A, B + (half ? o0 : 0), C + (half ? o1 : 0), beta));
        else          // the second half of the sum adds to the first
            COMET_CHK(gett_pieces(m, n, p, limit, M, N, K / ext * part, A + (half ? o0 : 0), B + (half ? o1 : 0), C,
                                  half ? 1.0 : beta));
    }
    return COMET_HIP_OK;
}

// C (+)= A * B over the three indices.
static int gett_device(const GettIndex &m, const GettIndex &n, const GettIndex &k, int64_t M, int64_t N, int64_t K,
                       const double *A, const double *B, double *C, double beta)
{
    if (M == 0 || N == 0)
        return COMET_HIP_OK;
    if (K == 0) {               // empty sums; C is whole and contiguous
        if (beta == 0.0)
            COMET_HIPCHK(hipMemsetAsync(C, 0, sizeof(double) * (size_t)(M * N), stream()));
        return COMET_HIP_OK;
    }
    // COMET_HIP_GETT_SPAN=elements cuts smaller operands (the pieces make the same result: the tests cut small ones)
    int64_t limit = GETT_SPAN;
    if (const char *e = getenv("COMET_HIP_GETT_SPAN"))
        if (const long long asked = atoll(e); asked > 0 && asked < limit)
            limit = asked;
    return gett_pieces(m, n, k, limit, M, N, K, A, B, C, beta);
}

// Row-major C[M,N] = beta*C + A[M,K]*B[K,N].
static int dgemm_device(int64_t M, int64_t N, int64_t K, const double *A, const double *B, double *C, double beta)
{
    if (M < 0 || N < 0 || K < 0)
        return set_error(COMET_HIP_ERR_ARG, "negative GEMM size");
    if (beta != 0.0 && beta != 1.0)
        return set_error(COMET_HIP_ERR_ARG, "beta must be 0 or 1 (got %g)", beta);
    GettIndex m{}, n{}, k{};
    gett_add_dim(&m, M, K, N);
    gett_add_dim(&n, N, 1, 1);
    gett_add_dim(&k, K, 1, N);
    return gett_device(m, n, k, M, N, K, A, B, C, beta);
}

// ============================================================================
// Plan
// ============================================================================
static bool contains(const int32_t *v, int n, int32_t x)
{
    for (int i = 0; i < n; ++i)
        if (v[i] == x)
            return true;
    return false;
}

// position in `in` of each element of `out` (Utils.h:722-733)
static void positions_of(const int32_t *in, const int32_t *out, int n, int32_t *perm)
{
    for (int i = 0; i < n; ++i)
        perm[i] = (int32_t)(std::find(in, in + n, out[i]) - in);
}

static int make_plan(int32_t rankA, const int32_t *a_lab, int32_t rankB, const int32_t *b_lab, int32_t rankC,
                     const int32_t *c_lab, const int64_t *extent, int32_t which, comet_ttgt_plan *plan)
{
    if (rankA < 1 || rankB < 1 || rankC < 1 || rankA > 8 || rankB > 8 || rankC > 8)
        return set_error(COMET_HIP_ERR_ARG, "tensor rank outside [1,8]");
    std::vector<int32_t> m, n, k;
    for (int i = 0; i < rankA; ++i) {
        if (contains(c_lab, rankC, a_lab[i])) {
            if (contains(b_lab, rankB, a_lab[i]))
                return set_error(COMET_HIP_ERR_ARG, "label %d appears in A, B and C: not a TTGT contraction", a_lab[i]);
            m.push_back(a_lab[i]);
        } else {
            k.push_back(a_lab[i]);
        }
    }
    for (int i = 0; i < rankB; ++i) {
        if (contains(c_lab, rankC, b_lab[i]))
            n.push_back(b_lab[i]);
        else if (!contains(a_lab, rankA, b_lab[i]))
            return set_error(COMET_HIP_ERR_ARG, "label %d of B is neither contracted with A nor kept in C", b_lab[i]);
    }
    for (int32_t x : k)
        if (!contains(b_lab, rankB, x))
            return set_error(COMET_HIP_ERR_ARG, "label %d of A is neither contracted with B nor kept in C", x);
    if ((int)(m.size() + k.size()) != rankA || (int)(n.size() + k.size()) != rankB ||
        (int)(m.size() + n.size()) != rankC)
        return set_error(COMET_HIP_ERR_ARG, "index sets do not form a GEMM (repeated or missing labels)");
    std::sort(m.begin(), m.end());
    std::sort(n.begin(), n.end());
    std::sort(k.begin(), k.end());
    int64_t M = 1, N = 1, K = 1;
    for (int32_t x : m) M *= extent[x];
    for (int32_t x : n) N *= extent[x];
    for (int32_t x : k) K *= extent[x];
    const double a_size = (double)(K * M), b_size = (double)(N * K), c_size = (double)(M * N);
    auto cost_of = [](double size, const int32_t *perm) { return perm[0] != 0 ? size / 0.71 : size; };

    int32_t cand = 0;
    bool have = false;
    double best = 0.0;
    do {
        do {
            do {
                for (int sw = 0; sw < 2; ++sw) {
                    comet_ttgt_plan cur;
                    std::memset(&cur, 0, sizeof cur);
                    cur.rankA = rankA;
                    cur.rankB = rankB;
                    cur.rankC = rankC;
                    // (written in place: a candidate's three lists in vectors were most of what a plan takes)
                    const auto join = [](const std::vector<int32_t> &x, const std::vector<int32_t> &y, int32_t *to) {
                        std::copy(y.begin(), y.end(), std::copy(x.begin(), x.end(), to));
                    };
                    join(sw ? k : m, sw ? m : k, cur.a_idx);
                    join(sw ? n : k, sw ? k : n, cur.b_idx);
                    join(sw ? n : m, sw ? m : n, cur.c_idx);
                    positions_of(a_lab, cur.a_idx, rankA, cur.permA);
                    positions_of(b_lab, cur.b_idx, rankB, cur.permB);
                    positions_of(c_lab, cur.c_idx, rankC, cur.permC);
                    cur.transA = !std::equal(cur.a_idx, cur.a_idx + rankA, a_lab);
                    cur.transB = !std::equal(cur.b_idx, cur.b_idx + rankB, b_lab);
                    cur.transC = !std::equal(cur.c_idx, cur.c_idx + rankC, c_lab);
                    cur.swapAB = sw;
                    cur.M = M;
                    cur.N = N;
                    cur.K = K;
                    double t = 0.0;
                    if (cur.transA) t = t + cost_of(a_size, cur.permA);
                    if (cur.transB) t = t + cost_of(b_size, cur.permB);
                    if (cur.transC) t = t + cost_of(c_size, cur.permC);
                    cur.cost = t;
                    cur.candidate = cand;
                    const bool take = which >= 0 ? cand == which : (!have || t < best);
                    if (take) {
                        *plan = cur;
                        best = t;
                        have = true;
                    }
                    ++cand;
                }
            } while (std::next_permutation(k.begin(), k.end()));
        } while (std::next_permutation(n.begin(), n.end()));
    } while (std::next_permutation(m.begin(), m.end()));
    if (which >= cand || !have)
        return set_error(COMET_HIP_ERR_ARG, "candidate %d does not exist (%d candidates)", which, cand);
    plan->ncandidates = cand;
    return COMET_HIP_OK;
}

static Workspace g_tt_a, g_tt_b, g_tt_c;

// The dimension of a tensor that the plan puts at position i of its matrix form.
static int plan_dim(int32_t trans, const int32_t *perm, int i) { return trans ? perm[i] : i; }

// Position of the first m, n and k dimension in the plan's forms of A, B and C (swapAB: A = [k m], B = [n k], C = [n m],
// else A = [m k], B = [k n], C = [m n]), and whether the forms agree dimension by dimension.
struct PlanDims {
    int nm, nn, nk;
    int am, ak, bn, bk, cm, cn;
};
static PlanDims plan_dims(const comet_ttgt_plan &p)
{
    PlanDims d;
    d.nk = (p.rankA + p.rankB - p.rankC) / 2;
    d.nm = p.rankA - d.nk;
    d.nn = p.rankB - d.nk;
    d.am = p.swapAB ? d.nk : 0;
    d.ak = p.swapAB ? 0 : d.nm;
    d.bn = p.swapAB ? 0 : d.nk;
    d.bk = p.swapAB ? d.nn : 0;
    d.cm = p.swapAB ? d.nn : 0;
    d.cn = p.swapAB ? 0 : d.nm;
    return d;
}

static bool gett_fits(const comet_ttgt_plan &p, const int64_t *a_shape, const int64_t *b_shape, const int64_t *c_shape)
{
    if ((p.rankA + p.rankB - p.rankC) % 2 != 0)
        return false;
    const PlanDims d = plan_dims(p);
    if (d.nk < 0 || d.nm < 0 || d.nn < 0 || d.nm + d.nn != p.rankC)
        return false;
    const auto a = [&](int i) { return a_shape[plan_dim(p.transA, p.permA, i)]; };
    const auto b = [&](int i) { return b_shape[plan_dim(p.transB, p.permB, i)]; };
    const auto c = [&](int i) { return c_shape[plan_dim(p.transC, p.permC, i)]; };
    int64_t M = 1, N = 1, K = 1;
    for (int i = 0; i < d.nm; ++i) {
        if (a(d.am + i) != c(d.cm + i))
            return false;
        M *= a(d.am + i);
    }
    for (int i = 0; i < d.nn; ++i) {
        if (b(d.bn + i) != c(d.cn + i))
            return false;
        N *= b(d.bn + i);
    }
    for (int i = 0; i < d.nk; ++i) {
        if (a(d.ak + i) != b(d.bk + i))
            return false;
        K *= a(d.ak + i);
    }
    return M == p.M && N == p.N && K == p.K;
}

constexpr double GETT_TURN_MIN = 1.28e8;

static int contract_strided(const comet_ttgt_plan &p, const int64_t *a_shape, const int64_t *b_shape,
                            const int64_t *c_shape, const double *A, const double *B, double *C, double beta)
{
    const auto strides = [](const int64_t *shape, int rank, int64_t *out) {
        int64_t s = 1;
        for (int i = rank - 1; i >= 0; --i) {
            out[i] = s;
            s *= shape[i];
        }
    };
    int64_t sa[8], sb[8], sc[8];
    strides(a_shape, p.rankA, sa);
    strides(b_shape, p.rankB, sb);
    strides(c_shape, p.rankC, sc);
    const PlanDims d = plan_dims(p);
    GettIndex m{}, n{}, k{};
    const auto da = [&](int i) { return plan_dim(p.transA, p.permA, i); };
    const auto db = [&](int i) { return plan_dim(p.transB, p.permB, i); };
    const auto dc = [&](int i) { return plan_dim(p.transC, p.permC, i); };
    for (int i = 0; i < d.nm; ++i)
        gett_add_dim(&m, a_shape[da(d.am + i)], sa[da(d.am + i)], sc[dc(d.cm + i)]);
    for (int i = 0; i < d.nn; ++i)
        gett_add_dim(&n, b_shape[db(d.bn + i)], sb[db(d.bn + i)], sc[dc(d.cn + i)]);
    for (int i = 0; i < d.nk; ++i)
        gett_add_dim(&k, a_shape[da(d.ak + i)], sa[da(d.ak + i)], sb[db(d.bk + i)]);
    // Both operands contiguous along k, but along different dimensions of it: whatever order k is taken in, one of
    // them is read a cache line per element.  The smaller one is turned first: k outermost, in the other's order, and
    // its outer index as C has it - the layout the kernel is fastest with.  Below GETT_TURN_MIN products the turn
    // costs more than the scattered reads (323 x 396 x 483: 21 us without, 23 with; 1520 x 1716 x 1435: 830 and 216).
    int ua = -1, ub = -1;
    for (int i = 0; i < k.nd; ++i) {
        ua = k.s0[i] == 1 ? i : ua;
        ub = k.s1[i] == 1 ? i : ub;
    }
    if (ua >= 0 && ub >= 0 && ua != ub && (double)p.M * (double)p.N * (double)p.K >= GETT_TURN_MIN) {
        const bool turn_a = p.M < p.N;
        const int rank = turn_a ? p.rankA : p.rankB, nfree = turn_a ? d.nm : d.nn;
        const int64_t *shape = turn_a ? a_shape : b_shape;
        int32_t perm[8];
        int64_t other[8];
        std::vector<std::pair<int64_t, int32_t>> ks;          // (minus the stride in the other operand, dimension)
        for (int i = 0; i < d.nk; ++i) {
            const int32_t mine = turn_a ? da(d.ak + i) : db(d.bk + i);
            ks.emplace_back(-(turn_a ? sb[db(d.bk + i)] : sa[da(d.ak + i)]), mine);
        }
        std::stable_sort(ks.begin(), ks.end());
        std::vector<std::pair<int64_t, int32_t>> fs;
        for (int i = 0; i < nfree; ++i) {
            const int32_t mine = turn_a ? da(d.am + i) : db(d.bn + i);
            fs.emplace_back(-(turn_a ? sc[dc(d.cm + i)] : sc[dc(d.cn + i)]), mine);
        }
        std::stable_sort(fs.begin(), fs.end());
        int at = 0;
        for (auto &e : ks)
            perm[at++] = e.second;
        for (auto &e : fs)
            perm[at++] = e.second;
        for (int i = 0; i < rank; ++i)
            other[i] = shape[perm[i]];
        Workspace &w = turn_a ? g_tt_a : g_tt_b;
        COMET_CHK(w.ensure(sizeof(double) * (size_t)((turn_a ? p.M : p.N) * p.K), false));
        COMET_CHK(transpose_device(rank, shape, perm, turn_a ? A : B, (double *)w.ptr));
        int64_t st[8];
        strides(other, rank, st);
        int64_t *s_mine = turn_a ? sa : sb;
        for (int i = 0; i < rank; ++i)
            s_mine[perm[i]] = st[i];
        (turn_a ? A : B) = (const double *)w.ptr;
        m = n = k = GettIndex{};
        for (int i = 0; i < d.nm; ++i)
            gett_add_dim(&m, a_shape[da(d.am + i)], sa[da(d.am + i)], sc[dc(d.cm + i)]);
        for (int i = 0; i < d.nn; ++i)
            gett_add_dim(&n, b_shape[db(d.bn + i)], sb[db(d.bn + i)], sc[dc(d.cn + i)]);
        for (int i = 0; i < d.nk; ++i)
            gett_add_dim(&k, a_shape[da(d.ak + i)], sa[da(d.ak + i)], sb[db(d.bk + i)]);
    }
    return gett_device(m, n, k, p.M, p.N, p.K, A, B, C, beta);
}

}  // namespace comet

using namespace comet;

extern "C" int comet_hip_transpose_f64(int32_t rank, const int64_t *in_shape, const int32_t *perm, int64_t in_dptr,
                                       int64_t out_dptr)
{
    COMET_CHK(ensure_init());
    if (!in_shape || !perm || !in_dptr || !out_dptr)
        return set_error(COMET_HIP_ERR_ARG, "null argument to comet_hip_transpose_f64");
    if (in_dptr == out_dptr)
        return set_error(COMET_HIP_ERR_ARG, "in-place transpose is not supported");
    return transpose_device(rank, in_shape, perm, (const double *)in_dptr, (double *)out_dptr);
}

extern "C" int comet_hip_dgemm_f64(int64_t M, int64_t N, int64_t K, int64_t a_dptr, int64_t b_dptr, int64_t c_dptr,
                                   double beta)
{
    COMET_CHK(ensure_init());
    if ((M > 0 && N > 0 && !c_dptr) || (M > 0 && N > 0 && K > 0 && (!a_dptr || !b_dptr)))
        return set_error(COMET_HIP_ERR_ARG, "null matrix passed to comet_hip_dgemm_f64");
    return dgemm_device(M, N, K, (const double *)a_dptr, (const double *)b_dptr, (double *)c_dptr, beta);
}

extern "C" int comet_hip_ttgt_plan(int32_t rankA, const int32_t *a_lab, int32_t rankB, const int32_t *b_lab,
                                   int32_t rankC, const int32_t *c_lab, const int64_t *extent, int32_t which,
                                   comet_ttgt_plan *plan)
{
    if (!a_lab || !b_lab || !c_lab || !extent || !plan)
        return set_error(COMET_HIP_ERR_ARG, "null argument to comet_hip_ttgt_plan");
    return make_plan(rankA, a_lab, rankB, b_lab, rankC, c_lab, extent, which, plan);
}

// Yardstick for the GEMM: back-to-back v_mfma_f64_16x16x4_f64 on registers only, sixteen independent
// accumulators per wavefront (more than the instruction's latency needs), two wavefronts per SIMD on every CU.
__global__ __launch_bounds__(256, 2) void mfma_f64_peak_kernel(int64_t iters, double *__restrict__ out)
{
    double4_t acc[16];
#pragma unroll
    for (int i = 0; i < 16; ++i)
        acc[i] = (double4_t){0.0, 0.0, 0.0, 0.0};
    const double a = 1.0 + threadIdx.x * 1e-9, b = 1.0 - threadIdx.x * 1e-9;
    for (int64_t it = 0; it < iters; ++it) {
#pragma unroll
        for (int i = 0; i < 16; ++i)
            acc[i] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, acc[i], 0, 0, 0);
    }
    double4_t s = acc[0];
#pragma unroll
    for (int i = 1; i < 16; ++i)
        s += acc[i];
    out[(int64_t)blockIdx.x * blockDim.x + threadIdx.x] = s[0] + s[1] + s[2] + s[3];
}

static Workspace g_peak_out;

extern "C" int comet_hip_mfma_f64_peak(int64_t iters, double *tflops)
{
    COMET_CHK(ensure_init());
    if (iters <= 0 || iters > (1ll << 24) || !tflops)
        return set_error(COMET_HIP_ERR_ARG, "bad arguments to comet_hip_mfma_f64_peak");
    const int blocks = num_cus() * 2;        // 8 wavefronts per CU: two per SIMD
    COMET_CHK(g_peak_out.ensure(sizeof(double) * 256 * (size_t)blocks, false));
    hipEvent_t e0, e1;
    COMET_HIPCHK(hipEventCreate(&e0));
    COMET_HIPCHK(hipEventCreate(&e1));
    float best = 0.f;
    for (int rep = 0; rep < 4; ++rep) {      // the first launch warms the clocks up
        COMET_HIPCHK(hipEventRecord(e0, stream()));
        mfma_f64_peak_kernel<<<dim3((unsigned)blocks), dim3(256), 0, stream()>>>(iters, (double *)g_peak_out.ptr);
        COMET_HIPCHK(hipEventRecord(e1, stream()));
        COMET_HIPCHK(hipEventSynchronize(e1));
        float ms = 0.f;
        COMET_HIPCHK(hipEventElapsedTime(&ms, e0, e1));
        if (rep > 0 && (best == 0.f || ms < best))
            best = ms;
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    COMET_HIPCHK(hipGetLastError());
    const double flops = 2.0 * 16 * 16 * 4 * 16.0 * (double)iters * 4.0 * blocks;      // per MFMA x 16 x iters x waves
    *tflops = flops / ((double)best * 1e-3) / 1e12;
    return COMET_HIP_OK;
}

extern "C" int comet_hip_ttgt_contract(const comet_ttgt_plan *plan, const int64_t *a_shape, const int64_t *b_shape,
                                       const int64_t *c_shape, int64_t a_dptr, int64_t b_dptr, int64_t c_dptr,
                                       double beta)
{
    COMET_CHK(ensure_init());
    if (!plan || !a_shape || !b_shape || !c_shape || !a_dptr || !b_dptr || !c_dptr)
        return set_error(COMET_HIP_ERR_ARG, "null argument to comet_hip_ttgt_contract");
    if (beta != 0.0 && beta != 1.0)
        return set_error(COMET_HIP_ERR_ARG, "beta must be 0 or 1 (got %g)", beta);
    // the plan may come from anywhere: ranks index 8-entry arrays and each perm must be a permutation
    auto is_perm = [](const int32_t *perm, int rank) {
        unsigned seen = 0;
        for (int i = 0; i < rank; ++i) {
            if (perm[i] < 0 || perm[i] >= rank || (seen >> perm[i] & 1u))
                return false;
            seen |= 1u << perm[i];
        }
        return true;
    };
    if (plan->rankA < 1 || plan->rankA > 8 || plan->rankB < 1 || plan->rankB > 8 || plan->rankC < 1 || plan->rankC > 8)
        return set_error(COMET_HIP_ERR_ARG, "plan ranks (%d, %d, %d) outside 1..8", plan->rankA, plan->rankB,
                         plan->rankC);
    if ((plan->transA && !is_perm(plan->permA, plan->rankA)) || (plan->transB && !is_perm(plan->permB, plan->rankB)) ||
        (plan->transC && !is_perm(plan->permC, plan->rankC)))
        return set_error(COMET_HIP_ERR_ARG, "a transpose of the plan is not a permutation of its tensor's dimensions");
    const int64_t M = plan->M, N = plan->N, K = plan->K;
    if (M < 0 || N < 0 || K < 0)
        return set_error(COMET_HIP_ERR_ARG, "negative GEMM extent in the plan");
    int64_t ta = 1, tb = 1, tc = 1;
    for (int i = 0; i < plan->rankA; ++i) ta *= a_shape[i];
    for (int i = 0; i < plan->rankB; ++i) tb *= b_shape[i];
    for (int i = 0; i < plan->rankC; ++i) tc *= c_shape[i];
    if (ta != M * K || tb != K * N || tc != M * N)
        return set_error(COMET_HIP_ERR_ARG, "tensor shapes do not match the plan (M,N,K = %lld,%lld,%lld)",
                         (long long)M, (long long)N, (long long)K);
    const double *A = (const double *)a_dptr, *B = (const double *)b_dptr;
    double *C = (double *)c_dptr;
    if (gett_fits(*plan, a_shape, b_shape, c_shape))
        return contract_strided(*plan, a_shape, b_shape, c_shape, A, B, C, beta);
    // a plan whose transposed tensors do not share their dimensions one by one: as matrices, after transposes
    const double *Ause = A, *Buse = B;
    double *Cuse = C;
    if (plan->transA) {
        COMET_CHK(g_tt_a.ensure(sizeof(double) * (size_t)ta, false));
        COMET_CHK(transpose_device(plan->rankA, a_shape, plan->permA, A, (double *)g_tt_a.ptr));
        Ause = (const double *)g_tt_a.ptr;
    }
    if (plan->transB) {
        COMET_CHK(g_tt_b.ensure(sizeof(double) * (size_t)tb, false));
        COMET_CHK(transpose_device(plan->rankB, b_shape, plan->permB, B, (double *)g_tt_b.ptr));
        Buse = (const double *)g_tt_b.ptr;
    }
    double gemm_beta = beta;
    if (plan->transC) {
        COMET_CHK(g_tt_c.ensure(sizeof(double) * (size_t)tc, false));
        Cuse = (double *)g_tt_c.ptr;
        if (beta != 0.0)
            COMET_CHK(transpose_device(plan->rankC, c_shape, plan->permC, C, Cuse));
    }
    if (plan->swapAB)
        COMET_CHK(dgemm_device(N, M, K, Buse, Ause, Cuse, gemm_beta));
    else
        COMET_CHK(dgemm_device(M, N, K, Ause, Buse, Cuse, gemm_beta));
    if (plan->transC) {
        int64_t cp_shape[8];
        int32_t rev[8];
        for (int i = 0; i < plan->rankC; ++i) {
            cp_shape[i] = c_shape[plan->permC[i]];
            rev[plan->permC[i]] = i;
        }
        COMET_CHK(transpose_device(plan->rankC, cp_shape, rev, Cuse, C));
    }
    return COMET_HIP_OK;
}
