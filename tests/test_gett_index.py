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
    while (scanf("%d %d", &first, &nd) == 2) {
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

    def run(first, dims):
        text = f"{first} {len(dims)} " + " ".join(f"{e} {a} {b}" for e, a, b in dims)
        out = [int(x) for x in subprocess.run([str(d / "main")], input=text, capture_output=True, text=True,
                                              check=True).stdout.split()]
        assert len(out) == 2 + 3 * out[1]
        return bool(out[0]), [tuple(out[2 + 3 * i:5 + 3 * i]) for i in range(out[1])]
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
