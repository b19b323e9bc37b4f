"""The cache policy of the V stores in front of the Winograd-domain GEMM
(wgemm_stream_v), a host rule, on the CPU: 0 plain, 1 nt where stores are
pieces of lines, 2 nt in any case. Layers of more than 256 channels that the
96- and 160-row tiles read few times were slower with nt unless V's rows lie on
64-byte boundaries and V or M is large."""

import pytest

from host_program import build

PROGRAM = """
#include <cstdio>
#include "nova_internal.h"
int main() {
    int K, Cp, BP;
    while (std::scanf("%d %d %d", &K, &Cp, &BP) == 3)
        std::printf("%d\\n", nova::wgemm_stream_v(K, Cp, BP));
}
"""


@pytest.fixture(scope="module")
def stream_v(tmp_path_factory):
    run = build(tmp_path_factory.mktemp("wgemm_rules"), PROGRAM)
    return lambda rows: [v for v, in run(rows)]


def test_wide_layers_off_64_bytes_or_small_are_not_streamed(stream_v):
    # (K, Cp, BP): 160 -> 320@23^2 batch 36 and 328 -> 320@128^2 took 3 and 25 %
    # longer streamed, 200 -> 480@14^2 batch 48 10 %, 200 -> 384@61^2 batch 3 5 %
    assert stream_v([(320, 160, 576), (320, 328, 484), (480, 200, 432),
                     (384, 200, 363)]) == [0] * 4


def test_streamed_layers(stream_v):
    assert stream_v([(320, 320, 484), (480, 96, 864)]) == [1, 1]
    # up to 256 channels, and 512 from 256 tiles on, at any row length
    assert stream_v([(72, 104, 400), (160, 160, 576), (200, 200, 200), (256, 256, 256),
                     (512, 200, 256)]) == [1] * 5
    assert stream_v([(640, 1280, 72), (640, 1920, 72), (640, 640, 121)]) == [2, 2, 0]
    assert stream_v([(64, 128, 3200), (700, 704, 121)]) == [0, 0]  # V of 50 MB; 11 reads
