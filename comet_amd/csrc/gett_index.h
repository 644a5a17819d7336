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
    uint32_t ext[GETT_MAXRANK];
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
    uint32_t ext[GETT_MAXRANK];
    int64_t s0[GETT_MAXRANK], s1[GETT_MAXRANK];
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
    g->ext[g->nd] = (uint32_t)ext;
    g->s0[g->nd] = s0;
    g->s1[g->nd] = s1;
    ++g->nd;
}

}  // namespace comet
