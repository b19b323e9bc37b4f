"""The direct weight gradient (fp16 output gradients, nova_weight_grad) at the
edges of its units: odd widths (staged through registers), widths off the
8-pixel chunk (masked), whole chunks, several images per unit, column strips,
pads 0 to 2, channels off the 32-blocks, and both tensors off every 4-byte
address.

Bound: the products of fp16 values are exact, so each entry's error is that of
an fp32 sum of n = B*Ho*Wo terms, at most n * 2^-23 * sum |dY||x| (one unit in
the last place per addition, whichever way the matrix unit rounds).
"""

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda:0")

# (B, C, K, H, W, pad)
CASES = [
    (3, 33, 31, 7, 7, 1), (17, 32, 64, 7, 7, 1), (1, 1, 1, 3, 3, 0), (2, 65, 40, 9, 11, 2),
    (2, 24, 40, 28, 28, 1), (5, 40, 33, 14, 14, 1), (1, 64, 64, 56, 56, 1), (2, 8, 48, 12, 12, 0),
    (2, 16, 16, 10, 14, 2), (1, 16, 32, 6, 150, 1), (1, 5, 7, 4, 261, 0), (1, 9, 6, 5, 140, 2),
    (2, 3, 70, 33, 64, 1), (1, 640, 320, 16, 16, 1), (1, 320, 640, 16, 18, 1),
    (2, 1280, 640, 8, 8, 1), (40, 4, 4, 5, 5, 2), (9, 96, 96, 1, 8, 1), (4, 30, 30, 8, 1, 1),
]


def weight_grad(x, dy, pad, C, K):
    from nova_winograd.ops import check, get_lib

    lib = get_lib()
    B, _, H, W = x.shape
    gw = torch.full((K, C, 3, 3), float("nan"), device=DEV)
    h = lib.nova_create()
    try:
        lib.nova_set_stream(h, torch.cuda.current_stream().cuda_stream)
        lib.nova_weight_grad(h, x.data_ptr(), dy.data_ptr(), gw.data_ptr(), B, C, K, H, W, pad, 0)
        check()
        torch.cuda.synchronize()
    finally:
        lib.nova_destroy(h)
    return gw


def exact(x, dy, pad):
    """The gradient and sum |dY||x| per entry in fp64, tap by tap."""
    K, C = dy.shape[1], x.shape[1]
    Ho, Wo = dy.shape[2:]
    xp = torch.nn.functional.pad(x.double(), (pad, pad, pad, pad)).transpose(0, 1)
    g = dy.double().transpose(0, 1).reshape(K, -1)
    want = torch.empty(K, C, 3, 3, dtype=torch.float64, device=x.device)
    mag = torch.empty_like(want)
    for r in range(3):
        for s in range(3):
            xs = xp[:, :, r:r + Ho, s:s + Wo].reshape(C, -1).t().contiguous()
            want[:, :, r, s] = g @ xs
            mag[:, :, r, s] = g.abs() @ xs.abs()
    return want, mag


def offset_copy(t, halves):
    """t's values at an address `halves` fp16 elements past an allocation, with
    NaN on both sides."""
    buf = torch.full((t.numel() + halves + 8,), float("nan"), dtype=t.dtype, device=t.device)
    buf[halves:halves + t.numel()] = t.reshape(-1)
    return buf[halves:halves + t.numel()].view(t.shape)


@pytest.mark.parametrize("B,C,K,H,W,pad", CASES)
def test_direct_weight_grad(B, C, K, H, W, pad):
    print(f"[wgrad direct] B={B} C={C} K={K} H={H} W={W} pad={pad}", flush=True)
    g = torch.Generator().manual_seed(H * W + C)
    x = torch.randn(B, C, H, W, generator=g).half().to(DEV)
    # gradients down into fp16's subnormals
    dy = (torch.randn(B, K, H + 2 * pad - 2, W + 2 * pad - 2, generator=g) * 1e-4).half().to(DEV)
    want, mag = exact(x, dy, pad)
    n = dy.numel() // K
    got = weight_grad(x, dy, pad, C, K)
    assert ((got.double() - want).abs() <= n * 2.0**-23 * mag + 1e-30).all()
    # any address and any neighbours in memory: the same bits (an odd offset
    # goes through registers; on a dword even widths stay on the direct loads)
    for xo, go in ((1, 0), (0, 1), (3, 2), (2, 2), (2, 4)):
        again = weight_grad(offset_copy(x, xo), offset_copy(dy, go), pad, C, K)
        assert torch.equal(got, again)


@pytest.mark.parametrize("W", [7, 12, 16])
def test_infinities_stay_in_their_channels(W):
    """An infinite x makes only its own input channel's taps infinite or NaN,
    an infinite dY only its own output channel's: the chunks that reach past a
    row or a channel hold zeros, not a neighbour's values."""
    B, C, K, H = 2, 40, 40, 10
    g = torch.Generator().manual_seed(W)
    x = torch.randn(B, C, H, W, generator=g).half().to(DEV)
    dy = torch.randn(B, K, H, W, generator=g).half().to(DEV)
    base = weight_grad(x, dy, 1, C, K)
    x2, dy2 = x.clone(), dy.clone()
    x2[0, 5, 0, 0] = float("inf")
    x2[1, 9, H - 1, W - 1] = float("-inf")
    got = weight_grad(x2, dy, 1, C, K)
    keep = torch.ones(C, dtype=torch.bool, device=DEV)
    keep[[5, 9]] = False
    assert torch.equal(got[:, keep], base[:, keep])
    assert not torch.isfinite(got[:, 5, 0, 0]).any() and not torch.isfinite(got[:, 9, 2, 2]).any()
    dy2[0, 3, H - 1, W - 1] = float("-inf")
    got = weight_grad(x, dy2, 1, C, K)
    keep = torch.arange(K, device=DEV) != 3
    assert torch.equal(got[keep], base[keep])
    assert not torch.isfinite(got[3, :, 0, 0]).any()


# one strip with and without a masked tail; two strips of 16 segments for 19
# (the first empty one lies right behind the masked chunk) and for 29; odd
@pytest.mark.parametrize("W", [24, 38, 150, 226, 151])
@pytest.mark.parametrize("pad", [0, 1, 2])
def test_infinities_beside_a_row_stay_in_their_channels(W, pad):
    """The chunks at a row's end reach into what follows in memory: the first
    pixels of the next row, and behind a channel's last row those of the next
    channel. Infinities there reach no other channel's gradient."""
    print(f"[wgrad direct, infinities] W={W} pad={pad}", flush=True)
    B, C, K, H = 1, 16, 32, 6
    Ho, Wo = H + 2 * pad - 2, W + 2 * pad - 2
    g = torch.Generator().manual_seed(W + pad)
    x = torch.randn(B, C, H, W, generator=g).half().to(DEV)
    dy = torch.randn(B, K, Ho, Wo, generator=g).half().to(DEV)
    base = weight_grad(x, dy, pad, C, K)
    for row, col in ((0, slice(0, 8)), (H - 1, slice(W - 8, W))):
        x2 = x.clone()
        x2[0, 8, row, col] = float("inf")
        got = weight_grad(x2, dy, pad, C, K)
        keep = torch.arange(C, device=DEV) != 8
        assert torch.equal(got[:, keep], base[:, keep])
        assert not torch.isfinite(got[:, 8]).all()
    for row, col in ((0, slice(0, 8)), (Ho - 1, slice(Wo - 8, Wo))):
        dy2 = dy.clone()
        dy2[0, 8, row, col] = float("-inf")
        got = weight_grad(x, dy2, pad, C, K)
        keep = torch.arange(K, device=DEV) != 8
        assert torch.equal(got[keep], base[keep])
        assert not torch.isfinite(got[8]).all()


@pytest.mark.parametrize("B,C,K,H,W,pad,f32", [
    (3, 33, 31, 7, 7, 1, False), (2, 70, 65, 28, 28, 1, False), (4, 16, 40, 56, 56, 0, False),
    (2, 3, 70, 9, 12, 2, False), (1, 320, 64, 16, 16, 1, False), (2, 8, 9, 10, 10, 1, True),
    (0, 4, 5, 8, 8, 1, False)])
def test_bias_gradient(B, C, K, H, W, pad, f32):
    """nova_weight_bias_grad: the same filter gradient, and the channel sums of
    dY: sums over n = B*Ho*Wo terms, each addition within 2^-24 of its result;
    no chain is longer than n / 8 (8 waves or more share a channel's pixels)
    plus the 8 waves and at most 256 splits."""
    from nova_winograd.ops import check, get_lib

    print(f"[bias grad] B={B} C={C} K={K} H={H} W={W} pad={pad} f32={f32}", flush=True)
    lib = get_lib()
    g = torch.Generator().manual_seed(B + K)
    Ho, Wo = H + 2 * pad - 2, W + 2 * pad - 2
    x = torch.randn(B, C, H, W, generator=g).half().to(DEV)
    dy = torch.randn(B, K, Ho, Wo, generator=g).to(DEV) * 0.01
    dy = dy if f32 else dy.half()
    gw = torch.full((K, C, 3, 3), float("nan"), device=DEV)
    gb = torch.full((K,), float("nan"), device=DEV)
    alone = torch.empty_like(gw)
    h = lib.nova_create()
    try:
        args = (B, C, K, H, W, pad, 1 if f32 else 0)
        lib.nova_weight_bias_grad(h, x.data_ptr(), dy.data_ptr(), gw.data_ptr(), gb.data_ptr(),
                                  *args)
        check()
        lib.nova_weight_grad(h, x.data_ptr(), dy.data_ptr(), alone.data_ptr(), *args)
        check()
        torch.cuda.synchronize()
    finally:
        lib.nova_destroy(h)
    assert torch.equal(gw, alone)
    want = dy.double().sum(dim=(0, 2, 3))
    bound = (B * Ho * Wo / 8 + 264) * 2.0**-24 * dy.double().abs().sum(dim=(0, 2, 3))
    assert ((gb.double() - want).abs() <= bound).all()


def bias_grads(x, dy, pad, K, C, runs=0):
    """nova_weight_bias_grad's results; with `runs`, also the time it takes
    beyond nova_weight_grad and torch's own sums, in us."""
    from nova_winograd.ops import check, get_lib

    lib = get_lib()
    B, _, H, W = x.shape
    gw = torch.full((K, C, 3, 3), float("nan"), device=DEV)
    gb = torch.full((K,), float("nan"), device=DEV)
    args = (B, C, K, H, W, pad, 1 if dy.dtype == torch.float32 else 0)
    h = lib.nova_create()

    def us(call):
        call()
        best = float("inf")
        for _ in range(3):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(runs):
                call()
            b.record()
            torch.cuda.synchronize()
            best = min(best, a.elapsed_time(b) * 1e3 / runs)
        return best

    def alone():
        lib.nova_weight_grad(h, x.data_ptr(), dy.data_ptr(), gw.data_ptr(), *args)

    def both():
        lib.nova_weight_bias_grad(h, x.data_ptr(), dy.data_ptr(), gw.data_ptr(), gb.data_ptr(),
                                  *args)

    try:
        lib.nova_set_stream(h, torch.cuda.current_stream().cuda_stream)
        times = None
        if runs:
            times = (us(both) - us(alone), us(lambda: dy.float().sum(dim=(0, 2, 3))))
        alone()
        want = gw.clone()
        both()
        check()
        torch.cuda.synchronize()
    finally:
        lib.nova_destroy(h)
    assert torch.equal(gw.view(torch.int32), want.view(torch.int32))
    return gb, times


# images of one run and of several, of a whole number of 16-byte words and not,
# channels of one workgroup and of many; few input channels bound the splits
@pytest.mark.parametrize("B,C,K,Ho,Wo", [
    (1, 1, 1, 3, 4), (3, 2, 5, 3, 3), (2, 1, 1, 200, 200), (3, 1, 2, 131, 127), (1, 4, 3, 128, 128),
    (40, 3, 7, 30, 31), (64, 8, 40, 17, 16), (2, 9, 600, 92, 91), (5, 2, 33, 64, 129)])
@pytest.mark.parametrize("f32", [False, True])
def test_bias_sums_of_their_own(B, C, K, Ho, Wo, f32):
    """The sums that the direct products do not take along (padding 2, float32
    dY): added in fp64 and rounded once, from any address, whatever stands
    beside them."""
    print(f"[bias sums] B={B} C={C} K={K} {Ho}x{Wo} f32={f32}", flush=True)
    pad = 1 if f32 else 2
    g = torch.Generator().manual_seed(Ho * Wo + K)
    H, W = Ho + 2 - 2 * pad, Wo + 2 - 2 * pad
    x = torch.randn(B, C, H, W, generator=g).half().to(DEV)
    dy = torch.randn(B, K, Ho, Wo, generator=g).to(DEV)
    dy = dy if f32 else dy.half()
    want = dy.double().sum(dim=(0, 2, 3))
    mag = dy.double().abs().sum(dim=(0, 2, 3))
    for off in (0, 1, 5):
        gb, _ = bias_grads(x, offset_copy(dy, off), pad, K, C)
        bound = 2.0**-24 * want.abs() + B * Ho * Wo * 2.0**-53 * mag
        assert ((gb.double() - want).abs() <= bound).all()
    dy[0, 0, 0, 0] = float("inf")
    gb, _ = bias_grads(x, dy, pad, K, C)
    assert torch.isinf(gb[0]) and torch.isfinite(gb[1:]).all()


@pytest.mark.parametrize("B,C,K,H,pad,f32", [(64, 32, 32, 112, 2, False), (16, 64, 3, 512, 2, False),
                                             (64, 32, 32, 112, 1, True)])
def test_bias_sums_fill_the_chip(B, C, K, H, pad, f32):
    """Few channels of many pixels take no longer than torch's conversion and
    sum (one workgroup per channel took 3 to 150 times as long)."""
    Ho = H + 2 * pad - 2
    x = torch.randn(B, C, H, H, device=DEV).half()
    dy = torch.randn(B, K, Ho, Ho, device=DEV)
    dy = dy if f32 else dy.half()
    _, (own, torchs) = bias_grads(x, dy, pad, K, C, runs=10)
    print(f"[bias sums] B={B} K={K} {Ho}^2 f32={f32}: {own:.1f} us, torch {torchs:.1f}", flush=True)
    assert own <= 1.5 * torchs + 20
