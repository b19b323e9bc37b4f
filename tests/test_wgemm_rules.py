"""Host rules of the Winograd-domain GEMM, on the CPU: the tile it takes
(wgemm_name) and the cache policy of the V stores in front of it
(wgemm_stream_v: 0 plain, 1 nt where stores are pieces of lines, 2 nt in any
case). Each case is a layer whose time was measured on both sides."""

import pytest

from host_program import build

PROGRAM = """
#include <cstdio>
#include "nova_internal.h"
int main() {
    int K, Cp, BP;
    while (std::scanf("%d %d %d", &K, &Cp, &BP) == 3) {
        int tk = 0, tb = 0, wk = 0, wb = 0;
        std::sscanf(nova::wgemm_name(K, Cp, BP), "wgemm_lds_kernel<%d, %d, %d, %d", &tk, &tb, &wk,
                    &wb);
        std::printf("%d %d %d %d\\n", nova::wgemm_stream_v(K, Cp, BP), tk, tb, wk * wb);
    }
}
"""


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    return build(tmp_path_factory.mktemp("wgemm_rules"), PROGRAM)


@pytest.fixture(scope="module")
def stream_v(rules):
    return lambda rows: [r[0] for r in rules(rows)]


@pytest.fixture(scope="module")
def tile(rules):
    return lambda rows: [r[1:] for r in rules(rows)]


def test_96_row_tiles_need_workgroups(tile):
    # (K, Cp, BP): 96 of 72 or 96 channels left most CUs idle (480 -> 96@48^2
    # batch 2 18.7 -> 21.4 us); so did 160 rows of 160 channels
    assert tile([(96, 480, 128), (72, 72, 128), (96, 96, 144), (192, 192, 147),
                 (160, 64, 256)]) == [(64, 64, 8)] * 2 + [(64, 64, 4)] * 3
    assert tile([(96, 448, 576), (192, 192, 512), (288, 288, 192), (384, 384, 144),
                 (160, 160, 800)]) == [(96, 96, 4), (96, 128, 8), (96, 96, 4), (96, 96, 4),
                                       (160, 128, 8)]


def test_wide_layers_take_128_rows_from_256_tiles(tile):
    # 640 -> 768@64^2 batch 4 94.6 -> 102.1 us with 96 rows, 768@56^2 likewise
    assert tile([(768, 640, 484), (768, 768, 400), (768, 64, 288), (768, 768, 192)]) == [
        (128, 128, 8), (128, 128, 8), (96, 96, 4), (96, 96, 4)]


def test_64_row_tiles_take_four_waves_from_300_workgroups(tile):
    assert tile([(128, 128, 128), (200, 200, 144), (333, 336, 64), (576, 576, 50),
                 (64, 64, 1024)]) == [(64, 64, 8)] + [(64, 64, 4)] * 4
    # off 4 channels: eight up to 256, four above
    assert tile([(141, 144, 560), (333, 336, 64)]) == [(64, 64, 8), (64, 64, 4)]


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
