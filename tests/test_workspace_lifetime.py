"""The module's workspace belongs to one stream, and one that a graph capture
took belongs to that capture: it is never handed back while work on another
stream, or a replay, may still write to it. The rule itself is tested on the
CPU with the library's answer in a stub; a captured training step and steps on
two streams run on the GPU."""

from types import SimpleNamespace

import pytest
import torch

from nova_winograd import NovaWinogradConv2d, NovaWinogradConv2dTrainable

DEV = torch.device("cuda:0")


class Handle:
    """The library handle's part in it: a stream, the key of the last weights
    and a layer that needs a workspace."""

    h, key, stream = None, None, 1
    lib = SimpleNamespace(nova_workspace_bytes=lambda h, b, H, W, pad: 1)

    def set_stream(self, device):
        pass

    def set_weights(self, weight):
        pass


@pytest.fixture
def module(monkeypatch):
    state = SimpleNamespace(capturing=False)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: state.capturing)
    mod = NovaWinogradConv2d(8, 8)
    mod._handle = Handle()
    mod.capture = state

    def workspace(batch=2, new_weights=False):
        if new_weights:
            with torch.no_grad():
                mod.weight.add_(1.0)
        mod._ensure_handle()
        mod._ensure_workspace(batch, 14, 14)
        assert mod._V_gemm.numel() == 64 * 8 * batch * 16 and mod._M_gemm.shape == mod._V_gemm.shape
        return mod._V_gemm, mod._M_gemm

    mod.workspace = workspace
    return mod


def other(a, b):
    return a[0] is not b[0] and a[1] is not b[1]


def test_same_stream_and_shape_keep_the_workspace(module):
    a = module.workspace()
    assert not other(a, module.workspace())
    assert not other(a, module.workspace(new_weights=True))
    assert other(a, module.workspace(3))


@pytest.mark.parametrize("new_weights", [False, True])
def test_another_stream_takes_its_own(module, new_weights):
    a = module.workspace()
    module._handle.stream = 2
    b = module.workspace(new_weights=new_weights)
    assert other(a, b)
    assert not other(b, module.workspace())


@pytest.mark.parametrize("new_weights", [False, True])
def test_a_capture_takes_its_own_and_leaves_none(module, new_weights):
    a = module.workspace()
    # on a stream of its own, or with new weights on the eager calls' stream
    module._handle.stream = 1 if new_weights else 2
    module.capture.capturing = True
    b = module.workspace(new_weights=new_weights)
    assert other(a, b)
    module.capture.capturing = False
    c = module.workspace()  # same stream, same shape: not the graph's
    assert other(b, c)
    module._handle.stream = 2 if new_weights else 3
    module.capture.capturing = True  # another capture
    assert other(c, module.workspace(new_weights=new_weights))


def test_a_failed_allocation_leaves_no_record(module, monkeypatch):
    module.workspace()
    module._state = ("record of a cached forward",)

    def fail(*a, **k):
        raise torch.OutOfMemoryError("out of memory")

    monkeypatch.setattr(torch, "empty", fail)
    with pytest.raises(torch.OutOfMemoryError):
        module._ensure_workspace(5, 14, 14)
    assert module._last_config is None and module._state is None


def layer(C, seed):
    torch.manual_seed(seed)
    mod = NovaWinogradConv2dTrainable(C, C, bias=True).to(DEV)
    with torch.no_grad():
        mod.bias.copy_(torch.randn(C))
    return mod


def step(mod, x, gy):
    """Forward, backward and a plain gradient step: the weights are new to the
    next forward. Returns the output and the gradients."""
    mod.zero_grad(set_to_none=True)
    x.grad = None
    y = mod(x)
    y.backward(gy)
    with torch.no_grad():
        mod.weight.sub_(mod.weight.grad, alpha=1e-2)
        mod.bias.sub_(mod.bias.grad, alpha=1e-2)
    return y.detach(), x.grad, mod.weight.grad, mod.bias.grad


@pytest.mark.gpu
@pytest.mark.parametrize("same_stream", [False, True])
def test_captured_training_step_keeps_its_workspace(same_stream):
    C, B, H = 192, 6, 20
    x = torch.randn(B, C, H, H, device=DEV).half().requires_grad_()
    gy = (0.01 * torch.randn(B, C, H, H, device=DEV)).half()
    small = torch.randn(2, C, H, H, device=DEV).half()
    mod, ref = layer(C, 7), layer(C, 7)
    assert torch.equal(mod.weight, ref.weight)
    print("[workspace, captured step] eager reference", flush=True)
    want = []
    for _ in range(6):  # three warm-up steps, then the replays' steps
        want.append([t.clone() for t in step(ref, x, gy)])
    torch.cuda.synchronize()
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        for _ in range(3):
            step(mod, x, gy)
    torch.cuda.current_stream().wait_stream(s)
    torch.cuda.synchronize()
    assert mod._V_gemm is not None  # a layer that needs the workspace
    eager = {mod._V_gemm.data_ptr(), mod._M_gemm.data_ptr()}
    print("[workspace, captured step] capture", flush=True)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s if same_stream else None):
        out = step(mod, x, gy)
    captured = {mod._V_gemm.data_ptr(), mod._M_gemm.data_ptr()}
    assert not eager & captured
    V = mod._V_gemm.numel()
    for i in range(3):
        print(f"[workspace, captured step] replay {i}", flush=True)
        g.replay()
        torch.cuda.synchronize()
        for a, b in zip(out, want[3 + i]):
            assert torch.equal(a, b), i
        # a smaller last batch, then memory of the old workspace's size in use
        with torch.no_grad():
            mod(small)
        assert not captured & {mod._V_gemm.data_ptr(), mod._M_gemm.data_ptr()}
        mine = [torch.full((V,), 3.0, dtype=torch.float16, device=DEV) for _ in range(3)]
        assert not captured & {t.data_ptr() for t in mine}
        torch.cuda.synchronize()
        if i == 2:
            g.replay()
            torch.cuda.synchronize()
        assert all((t == 3.0).all() for t in mine)


@pytest.mark.gpu
def test_steps_on_two_streams():
    C, B, H = 192, 6, 20
    x = torch.randn(B, C, H, H, device=DEV).half().requires_grad_()
    gy = (0.01 * torch.randn(B, C, H, H, device=DEV)).half()
    mod, ref = layer(C, 8), layer(C, 8)
    print("[workspace, two streams]", flush=True)
    want = [[t.clone() for t in step(ref, x, gy)] for _ in range(4)]
    torch.cuda.synchronize()
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    got, seen = [], []
    for i in range(4):
        s = (a, b)[i // 2]
        if i == 2:
            b.wait_stream(a)
        with torch.cuda.stream(s):
            got.append([t.clone() for t in step(mod, x, gy)])
        seen.append(mod._V_gemm)
    assert seen[0] is seen[1] and seen[2] is seen[3]  # new weights keep it
    assert seen[1] is not seen[2]  # the other stream has its own
    torch.cuda.synchronize()
    for g, w in zip(got, want):
        for u, v in zip(g, w):
            assert torch.equal(u, v)
