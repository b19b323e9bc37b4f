"""The Winograd-domain GEMM's tiles (direct loads to LDS) at the edges of what
each takes: M read back from the caller's workspace against the fp64 products
of the V and U the forward used, with K off the tile, BP off the tile, one and
several 64-channel stages, channel counts that end inside a stage, and M
staged as whole rows or stored in pieces. Each case names the kernel it is for.

Bound per entry: fp32 accumulation of Cp exact products (2 * Cp * 2^-24 *
sum |U||V|) and one rounding to fp16.
"""

import pytest
import torch

from test_gpu_filter_prep import DEV, handle_u

pytestmark = pytest.mark.gpu

# (B, C, K, H, kernel): BP = B * ceil(H / 6)^2
CASES = [
    (9, 40, 280, 28, "<96, 128, 2, 4, 2>"),    # BP 225, K past a tile
    (5, 300, 200, 33, "<64, 64, 2, 2, 2>"),    # BP 180
    (3, 72, 320, 54, "<160, 128, 2, 4, 2>"),   # BP 243, two stages, the last of 8 channels
    (2, 700, 640, 36, "<64, 96, 2, 2, 2>"),    # BP 72, 11 stages
    (2, 1030, 640, 33, "<160, 128, 2, 4, 3>"),  # three buffers; channels end inside a stage
    (6, 136, 288, 30, "<96, 96, 2, 2, 2>"),    # BP 150
    (9, 64, 480, 28, "<96, 128, 2, 4, 2>"),    # BP 225, one stage
    (16, 64, 256, 36, "<128, 192, 2, 4, 2>"),  # BP 576
    (9, 200, 512, 33, "<128, 128, 2, 4, 2>"),  # BP 324
    (2, 129, 1032, 25, "<128, 64, 2, 4, 2>"),  # BP 50, K past a tile
    (3, 80, 512, 36, "<64, 64, 2, 2, 2>"),     # BP 108
    (9, 72, 696, 30, "<64, 128, 2, 4, 2>"),    # BP 225, K past a tile
    (1, 24, 40, 36, "<64, 64, 2, 4, 2>"),      # BP 36, M staged
    # K % 8 != 0: M stored in pieces of four channels, or one by one (odd K)
    (8, 66, 130, 25, "<64, 64, 2, 4, 2>"),     # BP 200
    (8, 66, 132, 25, "<64, 64, 2, 2, 2>"),     # BP 200, four channels a piece
    (5, 9, 33, 30, "<64, 64, 2, 4, 2>"),       # BP 125, one partial stage
    (9, 77, 700, 30, "<64, 128, 2, 4, 2>"),    # BP 225
    (9, 40, 517, 33, "<128, 128, 2, 4, 2>"),   # BP 324
    (2, 129, 1030, 25, "<128, 64, 2, 4, 2>"),  # BP 50
]


@pytest.mark.parametrize("B,C,K,H,kernel", CASES)
def test_products_of_each_tile(B, C, K, H, kernel):
    from nova_winograd.ops import check, compute_tiling, get_lib

    lib = get_lib()
    g = torch.Generator().manual_seed(B * C + K)
    x = torch.randn(B, C, H, H, generator=g).half().to(DEV)
    w = (torch.randn(K, C, 3, 3, generator=g) * (2.0 / (9 * C)) ** 0.5).to(DEV)
    nh, nw, Ho, Wo = compute_tiling(H, H, 1)
    BP, Cp = B * (-(-Ho // 6)) ** 2, (C + 7) // 8 * 8
    while 64 * Cp * BP > 64 * C * B * nh * nw:  # room for V's Cp-wide rows
        nh += 1
    V = torch.zeros(64 * Cp * B * nh * nw, dtype=torch.float16, device=DEV)
    M = torch.full((64 * K * B * nh * nw,), float("nan"), dtype=torch.float16, device=DEV)
    y = torch.empty(B, K, Ho, Wo, dtype=torch.float16, device=DEV)
    h = lib.nova_create()
    try:
        lib.nova_set_path(h, 1)
        lib.nova_set_weights(h, w.data_ptr(), K, C)
        check()
        lib.nova_profile_enable(h, 1)
        torch.cuda.synchronize()
        lib.nova_forward_workspace(h, x.data_ptr(), y.data_ptr(), V.data_ptr(), M.data_ptr(), B,
                                   H, H, 1, nh, nw)
        check()
        torch.cuda.synchronize()
        ran = lib.nova_profile_kernel_name(h, 1).decode()
        print(f"[wgemm tiles] {B} {C}->{K}@{H} BP={BP} {ran}", flush=True)
        u = handle_u(lib, h, K, C).double()
    finally:
        lib.nova_destroy(h)
    assert ran == "wgemm_lds_kernel" + kernel
    got = M[:64 * BP * K].view(64, BP, K)
    assert torch.isfinite(got).all() and torch.isnan(M[64 * BP * K:]).all()
    assert torch.isfinite(y).all()
    v = V[:64 * BP * Cp].view(64, BP, Cp).double()
    for p in range(0, 64, 7):
        want = v[p] @ u[p].t().contiguous()
        mag = v[p].abs() @ u[p].abs().t().contiguous()
        bound = 2 * Cp * 2.0**-24 * mag + 2.0**-11 * want.abs() * 1.01 + 2.0**-24
        assert ((got[p].double() - want).abs() <= bound).all(), p
