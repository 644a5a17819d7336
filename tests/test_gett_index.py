"""The order in which a contraction's indices are walked (csrc/gett_index.h), compiled for the CPU with bounds checks."""
import itertools
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <stdio.h>
#include "gett_index.h"
int main()
{
    int first, nd;
    while (scanf("%d", &first) == 1) {
        if (first < 0) {          // three indices and the most an operand may span: where to cut
            comet::GettIndex x[3] = {};
            long long limit, e, s0, s1;
            for (auto &g : x)
                for (int d = scanf("%d", &nd) == 1 ? 0 : nd; d < nd; ++d)
                    if (scanf("%lld %lld %lld", &e, &s0, &s1) == 3)
                        comet::gett_add_dim(&g, e, s0, s1);
            if (scanf("%lld", &limit) != 1)
                return 1;
            const comet::GettCut c = comet::gett_cut(x[0], x[1], x[2], limit);
            printf("%d %d %lld\n", c.which, c.d, (long long)c.first);
            continue;
        }
        if (scanf("%d", &nd) != 1)
            return 1;
        comet::GettIndex g{};
        for (int d = 0; d < nd; ++d) {
            long long e, s0, s1;
            if (scanf("%lld %lld %lld", &e, &s0, &s1) != 3)
                return 1;
            comet::gett_add_dim(&g, e, s0, s1);
        }
        const bool contiguous = comet::gett_order(&g, first);
        printf("%d %d", contiguous, g.nd);
        for (int d = 0; d < g.nd; ++d)
            printf(" %lld %lld %lld", (long long)g.ext[d], (long long)g.s0[d], (long long)g.s1[d]);
        printf("\n");
    }
}
"""


@pytest.fixture(scope="module")
def order(tmp_path_factory):
    d = tmp_path_factory.mktemp("gett_index")
    (d / "main.cpp").write_text(PROGRAM)
    subprocess.check_call(["g++", "-std=c++17", "-fsanitize=undefined", "-fno-sanitize-recover=undefined", "-I",
                           os.path.join(ROOT, "comet_amd", "csrc"), str(d / "main.cpp"), "-o", str(d / "main")])

    def ask(text):
        return [int(x) for x in subprocess.run([str(d / "main")], input=text, capture_output=True, text=True, check=True).stdout.split()]

    def text_of(dims):
        return f"{len(dims)} " + " ".join(f"{e} {a} {b}" for e, a, b in dims) + " "

    def run(first, dims):
        out = ask(f"{first} " + text_of(dims))
        assert len(out) == 2 + 3 * out[1]
        return bool(out[0]), [tuple(out[2 + 3 * i:5 + 3 * i]) for i in range(out[1])]
    run.cut = lambda m, n, k, limit: ask("-1 " + text_of(m) + text_of(n) + text_of(k) + str(limit))
    return run


def _offsets(dims):
    """Offsets in the two tensors of every value of the index, in the order it is walked."""
    return [tuple(sum(i * d[t] for i, d in zip(at, dims)) for t in (1, 2))
            for at in itertools.product(*(range(e) for e, _, _ in dims))]


@pytest.mark.parametrize("first", [0, 1])
@pytest.mark.parametrize("dims", [[], [(1, 5, 7)], [(1, 1, 1), (1, 3, 9)], [(6, 1, 1)], [(4, 15, 1), (5, 3, 4), (3, 1, 20)],
                                  [(4, 15, 15), (5, 3, 3), (3, 1, 1)], [(2, 40, 4), (1, 8, 8), (4, 10, 1), (5, 2, 8)], [(3, 8, 64)]])
def test_every_index_is_walked_once(order, dims, first):
    contiguous, got = order(first, dims)
    assert sorted(_offsets(got)) == sorted(_offsets(dims))
    assert len(got) <= sum(e > 1 for e, _, _ in dims) and all(e > 1 for e, _, _ in got)
    units = [d for d in dims if d[0] > 1 and d[1 + first] == 1]
    assert contiguous == bool(units)
    if contiguous:          # neighbours of that tensor follow each other
        assert got[-1][1 + first] == 1


def _span(x, sx, y, sy):
    return 1 + sum((d[0] - 1) * d[sx] for d in x) + sum((d[0] - 1) * d[sy] for d in y)


LIMIT = (1 << 29) - 1


@pytest.mark.parametrize("m,n,k", [
    ([(1000, 64, 1)], [(64, 1, 1000)], [(64, 1, 64)]),                                                # nothing to cut
    ([(32768, 32768, 32768)], [(32768, 1, 1)], [(32768, 1, 32768)]),                                  # both operands, m and k
    ([(1 << 29, 1, 1)], [(1, 1, 1)], [(3, 1 << 29, 1)]),                                              # k is outermost
    ([(160, 160**3, 160**3), (160, 160, 160**2)], [(160, 160**3, 1), (160, 160, 160)], [(160, 160**2, 1), (160, 1, 160**2)]),
    ([], [], [((1 << 31) - 1, 1, 1)]), ([((1 << 31) - 1, 1, 1)], [], []),
    ([], [], [((1 << 33) + 3, 1, 1)]), ([((1 << 32) + 1, 1, 1)], [], []), ([], [((1 << 31) + 7, 1, 1)], [(2, 1, (1 << 31) + 7)]), ([(2, 1 << 30, 1)], [(5, 1, 2)], [(1 << 30, 1, 5)])])
def test_pieces_cover_a_large_contraction_once(order, m, n, k):
    drop = lambda x: [d for d in x if d[0] > 1]
    todo, done, total = [(drop(m), drop(n), drop(k))], 0, 1
    for x in todo[0]:
        for d in x:
            total *= d[0]
    while todo:
        m, n, k = todo.pop()
        which, d, first = order.cut(m, n, k, LIMIT)
        if which < 0:
            assert _span(m, 1, k, 1) <= LIMIT and _span(n, 1, k, 2) <= LIMIT
            size = 1
            for x in (m, n, k):
                for e in x:
                    size *= e[0]
            done += size
            continue
        x = (m, n, k)[which]
        assert 0 < first < x[d][0] and (first % 128 == 0 or x[d][0] <= 256)
        for part in (first, x[d][0] - first):
            halves = [m, n, k]
            halves[which] = drop(x[:d] + [(part, *x[d][1:])] + x[d + 1:])
            todo.append(tuple(halves))
        assert len(todo) < 100
    assert done == total
