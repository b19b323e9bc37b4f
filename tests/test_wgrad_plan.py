"""Host rules of the direct weight gradient (wgrad_direct.hip), on the CPU: a
small program linked with the library's own objects prints the plan of each
shape.

Lanes with nothing to load use byte offset 2^31, which has to lie past the end
of every buffer resource. The resource over dY starts (2 - pad) rows of dY
above the tensor, the one over x up to one 16-byte chunk, and each is as much
longer.
"""

import pytest

from host_program import build

PROGRAM = """
#include <cstdio>
#include "nova_internal.h"
int main() {
    int B, C, K, H, W, pad;
    while (std::scanf("%d %d %d %d %d %d", &B, &C, &K, &H, &W, &pad) == 6) {
        const nova::WgradDirectPlan p = nova::wgrad_direct_plan(B, C, K, H, W, pad, 256);
        std::printf("%d %d\\n", (int)p.ok, p.lo);
    }
}
"""


@pytest.fixture(scope="module")
def plans(tmp_path_factory):
    return build(tmp_path_factory.mktemp("wgrad_plan"), PROGRAM)


def resource_ends(shape, lo):
    """Bytes of the two resources, for the first channels (the longest), at an
    address 2 past a dword."""
    B, C, K, H, W, pad = shape
    Ho, Wo = H + 2 * pad - 2, W + 2 * pad - 2
    x = 2 * B * C * H * W + 16 * lo + 2
    dy = 2 * B * K * Ho * Wo + 2 * (2 - pad) * Wo + 2
    return (x + 3) & ~3, (dy + 3) & ~3


def test_resources_end_below_the_offset_of_empty_lanes(plans):
    shapes = [(1, 1, 2, 17897, 30002, 0), (1, 1, 1, 17895, 60000, 1)]
    # tensors around 2 GiB, by columns, rows, channels and images
    for pad in (0, 1, 2):
        for Wo in (40, 1000, 16390, 30000, 60000, 120000):
            for K, B in ((1, 1), (3, 1), (1, 2)):
                for d in range(-3, 3):
                    Ho = (2**31 // (2 * Wo * K * B)) + d
                    shapes.append((B, 1, K, Ho + 2 - 2 * pad, Wo + 2 - 2 * pad, pad))
    got = plans(shapes)
    for shape, (ok, lo) in zip(shapes, got):
        if ok:
            assert max(resource_ends(shape, lo)) <= 2**31, shape


def test_smaller_tensors_keep_the_direct_products(plans):
    shapes = [(32, 64, 64, 56, 56, 1), (1, 1, 1, 17000, 60000, 1), (1, 1, 2, 17000, 30002, 0),
              (1, 1, 1, 3, 3, 0), (2, 65, 40, 9, 11, 2),
              (1, 1, 1, 1048543, 1024, 1), (1, 1, 1, 131035, 8194, 0)]  # 66 and 80 KB below 2 GiB
    assert [ok for ok, _ in plans(shapes)] == [1] * len(shapes)
    assert [ok for ok, _ in plans([(1, 4, 4, 8, 8, 3), (0, 4, 4, 8, 8, 1)])] == [0, 0]
