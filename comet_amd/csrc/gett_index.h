// The indices of a contraction: what their dimensions are and in which order the kernel walks them.  Plain C++, so
// that the CPU tests compile it by itself.
#pragma once
#include <stdint.h>

#include <algorithm>
#include <vector>

namespace comet {

constexpr int GETT_MAXRANK = 8;

// A multi-index: extents (outermost first) and the strides of its dimensions in the two tensors it appears in.
struct GettIndex {
    int nd;
    int64_t ext[GETT_MAXRANK];
    int64_t s0[GETT_MAXRANK], s1[GETT_MAXRANK];
};

// The innermost dimension of an index comes last: `first` names the tensor (0 or 1) whose contiguous dimension it
// should be, if that dimension is in the index.  Dimensions that follow each other in both tensors are merged.
static bool gett_order(GettIndex *g, int first)
{
    if (g->nd == 0)          // an index of one element: nothing to order, nothing to read
        return false;
    GettIndex in = *g;
    int last = -1;
    for (int pass = 0; pass < 2 && last < 0; ++pass)
        for (int d = 0; d < in.nd; ++d)
            if (((pass == 0) == (first == 0) ? in.s0[d] : in.s1[d]) == 1)
                last = d;
    if (last < 0)
        last = in.nd - 1;
    const bool contiguous = (first == 0 ? in.s0[last] : in.s1[last]) == 1;
    // from the innermost outwards: first whatever continues the dimension before it in the tensor `first`
    std::vector<int> order(1, last), rest;
    for (int d = 0; d < in.nd; ++d)
        if (d != last)
            rest.push_back(d);
    const int64_t *key = first == 0 ? in.s0 : in.s1;
    std::sort(rest.begin(), rest.end(), [&](int x, int y) { return key[x] < key[y]; });
    order.insert(order.end(), rest.begin(), rest.end());
    g->nd = 0;
    int64_t ext[GETT_MAXRANK], s0[GETT_MAXRANK], s1[GETT_MAXRANK];
    int n = 0;
    for (int d : order) {
        if (n > 0 && s0[n - 1] * ext[n - 1] == in.s0[d] && s1[n - 1] * ext[n - 1] == in.s1[d]) {
            ext[n - 1] *= in.ext[d];
        } else {
            ext[n] = in.ext[d];
            s0[n] = in.s0[d];
            s1[n] = in.s1[d];
            ++n;
        }
    }
    g->nd = n;
    for (int d = 0; d < n; ++d) {          // outermost first
        g->ext[d] = ext[n - 1 - d];
        g->s0[d] = s0[n - 1 - d];
        g->s1[d] = s1[n - 1 - d];
    }
    return contiguous;
}

static void gett_add_dim(GettIndex *g, int64_t ext, int64_t s0, int64_t s1)
{
    if (ext == 1)
        return;
    g->ext[g->nd] = ext;
    g->s0[g->nd] = s0;
    g->s1[g->nd] = s1;
    ++g->nd;
}

// One more than the largest offset of an element whose two indices have the strides sx and sy in its tensor.
static int64_t gett_span(const GettIndex &x, const int64_t *sx, const GettIndex &y, const int64_t *sy)
{
    int64_t last = 0;
    for (int d = 0; d < x.nd; ++d)
        last += (x.ext[d] - 1) * sx[d];
    for (int d = 0; d < y.nd; ++d)
        last += (y.ext[d] - 1) * sy[d];
    return last + 1;
}

// Where a contraction is cut in two: dimension d of the index `which` (0: m, 1: n, 2: k), `first` values of it go to
// the first half.  which < 0: it need not be cut.
struct GettCut {
    int which, d;
    int64_t first;
};

// The kernel adds 32-bit byte offsets to the operands, which is what lets it read them without vector arithmetic, so
// an operand of more elements than `limit` is cut along the dimension that spans most of it.  (So are the indices kept
// within 32 bits: none of a piece has more elements than the operands it is in.)  Halves of this size keep every CU busy
// for milliseconds; where the sum is cut, C is read and written once more.  A variant with 64-bit offsets, for operands
// that need them, took 9.4 ms for 1048576 x 520 x 512 and this takes 8.7, 450 and 394 for 24000^3, 2.63 and 0.91 for a
// matrix of 1048577 x 521 and a vector.
static GettCut gett_cut(const GettIndex &m, const GettIndex &n, const GettIndex &k, int64_t limit)
{
    GettCut cut{-1, 0, 0};
    int64_t most = 0;
    const auto look = [&](const GettIndex &x, const int64_t *s, int which) {
        for (int d = 0; d < x.nd; ++d)
            if ((x.ext[d] - 1) * s[d] > most) {
                most = (x.ext[d] - 1) * s[d];
                const int64_t half = x.ext[d] / 2 + x.ext[d] % 2, whole = (half + 127) / 128 * 128;
                cut = GettCut{which, d, whole < x.ext[d] ? whole : half};          // whole tiles, if there are any
            }
    };
    if (gett_span(m, m.s0, k, k.s0) > limit) {
        look(m, m.s0, 0);
        look(k, k.s0, 2);
    } else if (gett_span(n, n.s0, k, k.s1) > limit) {
        look(n, n.s0, 1);
        look(k, k.s1, 2);
    }
    return cut;
}

// The index with `ext` values of dimension d.
static GettIndex gett_part(const GettIndex &g, int d, int64_t ext)
{
    GettIndex out{};
    for (int i = 0; i < g.nd; ++i)
        gett_add_dim(&out, i == d ? ext : g.ext[i], g.s0[i], g.s1[i]);
    return out;
}

}  // namespace comet
