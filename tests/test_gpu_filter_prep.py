"""The one-launch filter preparation: U in the product layout against the
oracle's transform, the flipped form against the flipped weights, and both
fragment-ordered copies against U, at both lane widths (8 channels per lane
from 512 pairs per CU on, else 2) and at channel counts off the 8, 16, 32 and
64 blocks. The forwards of the paths that read each copy must agree bit for
bit with the same paths on copies built from U."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda:0")


class DeviceView:
    """The handle's U as an array torch can wrap without a copy."""

    def __init__(self, ptr, shape):
        self.__cuda_array_interface__ = {"shape": shape, "typestr": "<f2", "data": (ptr, False),
                                         "version": 2}


def handle_u(lib, h, K, C):
    torch.cuda.synchronize()
    return torch.as_tensor(DeviceView(lib.nova_get_U_gemm(h), (64, K, (C + 7) // 8 * 8)),
                           device=DEV).clone()


@pytest.mark.parametrize("K,C", [(1, 1), (3, 5), (16, 8), (17, 33), (64, 64), (72, 100),
                                 (130, 24), (24, 130), (500, 264), (264, 500), (520, 256)])
@pytest.mark.parametrize("f16", [False, True])
def test_u_and_flipped_u(oracle, K, C, f16):
    from nova_winograd.ops import check, get_lib

    print(f"[filter prep] K={K} C={C} f16={f16}", flush=True)
    lib = get_lib()
    g = torch.Generator().manual_seed(K + C)
    w = torch.randn(K, C, 3, 3, generator=g) * 0.1
    w = w.half() if f16 else w
    # off a 16-byte address, as a view into a larger parameter may be
    buf = torch.zeros(w.numel() + 3, dtype=w.dtype, device=DEV)
    buf[3:] = w.reshape(-1).to(DEV)
    wd = buf[3:]
    h, hf, hs = lib.nova_create(), lib.nova_create(), lib.nova_create()
    try:
        (lib.nova_set_weights_f16 if f16 else lib.nova_set_weights)(h, wd.data_ptr(), K, C)
        check()
        u = handle_u(lib, h, K, C)
        want = oracle.filter_transform(w.float().numpy())  # [64][C][K]
        want = torch.from_numpy(np.ascontiguousarray(want).view(np.float16)).to(DEV)
        assert torch.equal(u[:, :, :C].view(torch.int16),
                           want.reshape(64, C, K).transpose(1, 2).contiguous().view(torch.int16))
        assert not u[:, :, C:].any()
        lib.nova_set_weights_flipped(hf, wd.data_ptr(), C, K, 1 if f16 else 0)
        check()
        wf = w.flip(2, 3).transpose(0, 1).contiguous().to(DEV)
        (lib.nova_set_weights_f16 if f16 else lib.nova_set_weights)(hs, wf.data_ptr(), C, K)
        check()
        assert torch.equal(handle_u(lib, hf, C, K).view(torch.int16),
                           handle_u(lib, hs, C, K).view(torch.int16))
    finally:
        for x in (h, hf, hs):
            lib.nova_destroy(x)


# paths: those that serve 2 x 13^2 with these channels when asked to
@pytest.mark.parametrize("K,C,paths", [
    (64, 64, (3, 5, 6, 7)), (40, 48, (3, 5, 6, 7)), (17, 9, (3, 5, 6, 7)), (128, 128, (6, 7)),
    (256, 128, (6, 7)), (96, 24, (6, 7)), (512, 512, (6, 7)),
    (1000, 800, (6,))])
def test_copies_match_u(K, C, paths):
    """The copies that set_weights writes, Uf (paths 3 and 5) and Uw (6 and 7),
    against copies built afterwards from U: forwards of the same path, bit for
    bit. Weights are set twice, since some copies are written by set_weights
    only once a forward has used them. Paths 6 and 7 also match path 1, which
    reads U, and 3 and 5 sum the channels in another order."""
    from nova_winograd.ops import check, get_lib

    lib = get_lib()
    g = torch.Generator().manual_seed(K * C)
    B, H = 2, 13
    x = torch.randn(B, C, H, H, generator=g).half().to(DEV)
    w = torch.randn(K, C, 3, 3, generator=g).to(DEV) * 0.05

    def forward(h, path):
        y = torch.empty(B, K, H, H, dtype=torch.float16, device=DEV)
        lib.nova_forward(h, x.data_ptr(), y.data_ptr(), B, H, H, 1)
        check()
        torch.cuda.synchronize()
        ran = lib.nova_get_last_path(h)
        print(f"[filter copies] K={K} C={C} asked {path} ran {ran}", flush=True)
        assert ran == path
        return y

    def written(path):
        """set_weights under the path, twice."""
        h = lib.nova_create()
        try:
            lib.nova_set_path(h, path)
            for scale in (2.0, 1.0):
                ws = w * scale
                lib.nova_set_weights(h, ws.data_ptr(), K, C)
                check()
                y = forward(h, path)
            return y
        finally:
            lib.nova_destroy(h)

    def built(path):
        """U alone by set_weights, the copy from it when the path is asked for."""
        h = lib.nova_create()
        try:
            lib.nova_set_path(h, 1)
            lib.nova_set_weights(h, w.data_ptr(), K, C)
            lib.nova_set_path(h, path)
            check()
            return forward(h, path)
        finally:
            lib.nova_destroy(h)

    base = built(1)
    for path in paths:
        y = written(path)
        assert torch.equal(y, built(path)), path
        if path in (6, 7):
            assert torch.equal(y, base)
        else:
            assert (y.float() - base.float()).norm() <= 5e-3 * base.float().norm()


def test_blocks_are_written_only_while_forwards_read_them():
    """One batch-1 forward reads U's operand blocks; the steps at a larger
    batch that follow, each with new weights, take as long as on a handle that
    never had them (they took twice as long while set_weights went on writing
    the blocks)."""
    from nova_winograd.ops import check, get_lib

    lib = get_lib()
    C, B, H = 1280, 8, 16
    w = torch.randn(C, C, 3, 3, device=DEV) * 0.02
    x, one = (torch.randn(n, C, h, h, device=DEV).half() for n, h in ((B, H), (1, 7)))
    y, y1 = torch.empty_like(x), torch.empty_like(one)

    def step_us(batch_1_first):
        h = lib.nova_create()
        try:
            lib.nova_set_stream(h, torch.cuda.current_stream().cuda_stream)
            lib.nova_set_weights(h, w.data_ptr(), C, C)
            if batch_1_first:
                lib.nova_forward(h, one.data_ptr(), y1.data_ptr(), 1, 7, 7, 1)
            best = float("inf")
            for _ in range(4):
                a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
                a.record()
                for _ in range(10):
                    lib.nova_set_weights(h, w.data_ptr(), C, C)
                    lib.nova_forward(h, x.data_ptr(), y.data_ptr(), B, H, H, 1)
                b.record()
                torch.cuda.synchronize()
                best = min(best, a.elapsed_time(b) * 100)
            check()
            return best
        finally:
            lib.nova_destroy(h)

    fresh, after = step_us(False), step_us(True)
    print(f"[filter blocks] fresh {fresh:.1f} us, after a batch-1 forward {after:.1f}", flush=True)
    assert after <= 1.4 * fresh
