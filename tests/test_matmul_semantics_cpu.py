"""matmul, matmul_shared_input and swiglu_matmul where torch's own operators
have to see the call: transforms, tracers and subclasses, whose tensors have no
address to read, and sparse tensors.

Without a GPU: the module's source with its GPU tests turned into CPU tests, so
that the routes are decided on CPU tensors, and every launch turned into a
failure."""
import sys
import types
import warnings

import pytest
import torch
from torch.func import grad, jvp, vmap

from lightserve_amd.kernels import tiled_matmul

ROWS = [1, 2, 3, 9, 16, 33, 64, 512, 5000]


@pytest.fixture
def tm(monkeypatch):
    path = tiled_matmul.__file__
    with open(path) as f:
        source = f.read().replace(".is_cuda", ".is_cpu")
    module = types.ModuleType("lightserve_amd.kernels.tiled_matmul_on_cpu")
    module.__package__, module.__file__ = "lightserve_amd.kernels", path
    monkeypatch.setitem(sys.modules, module.__name__, module)
    exec(compile(source, path, "exec"), module.__dict__)

    def launch(*args, **kwargs):
        raise AssertionError("routed to a kernel")
    module._run_group = launch
    return module


def _calls(tm, x, w):
    return [lambda a: tm.matmul(a, w), lambda a: tm.matmul_shared_input(a, [w, w])[1],
            lambda a: tm.swiglu_matmul(a, x, w), lambda a: tm.swiglu_matmul(x, a, w)]


def _operands(m, k=4096, n=256):
    g = torch.Generator().manual_seed(m)
    return (torch.randn(m, k, generator=g).to(torch.bfloat16), torch.randn(m, k, generator=g).to(torch.bfloat16),
            (torch.randn(k, n, generator=g) / k ** 0.5).to(torch.bfloat16))


def test_plain_calls_reach_the_kernels(tm):
    """The stand-in decides as on a GPU: without a transform these are routed."""
    for m in (1, 2, 3, 32, 512):
        x, y, w = _operands(m, n=4096 if m > 16 else 256)
        for f in _calls(tm, x, w)[:2 if m > 32 else 4]:
            with pytest.raises(AssertionError, match="routed to a kernel"):
                f(y)


@pytest.mark.parametrize("m", ROWS)
def test_transforms(tm, m):
    x, y, w = _operands(m, 128, 128)
    for f in _calls(tm, x, w):
        want = f(y.clone().requires_grad_()).detach().float()
        torch.testing.assert_close(vmap(f)(torch.stack([y, y])).float(), torch.stack([want, want]), rtol=2 ** -7, atol=1e-6)
        assert torch.isfinite(grad(lambda a: f(a).float().sum())(y)).all()
        assert torch.isfinite(jvp(f, (y,), (y,))[1]).all()


@pytest.mark.parametrize("m", [1, 16, 64, 600])
def test_compile_traces_the_whole_call(tm, m):
    x, y, w = _operands(m, 128, 128)
    for f in _calls(tm, x, w):
        torch._dynamo.reset()
        assert torch.compile(f, backend="eager", fullgraph=True)(y).shape == (m, 128)


@pytest.mark.parametrize("m", ROWS)
def test_tensors_without_storage(m):
    """Fake GPU tensors through the module itself."""
    from torch._subclasses.fake_tensor import FakeTensorMode
    with FakeTensorMode():
        x = torch.empty(m, 4096, dtype=torch.bfloat16, device="cuda")
        w = torch.empty(4096, 512, dtype=torch.bfloat16, device="cuda")
    # an address read of a fake tensor only warns
    always = torch.is_warn_always_enabled()
    torch.set_warn_always(True)
    warnings.simplefilter("error")
    try:
        assert tiled_matmul.matmul(x, w).shape == (m, 512)
        assert [t.shape for t in tiled_matmul.matmul_shared_input(x, [w, w])] == [(m, 512)] * 2
        assert tiled_matmul.swiglu_matmul(x, x, w).shape == (m, 512)
    finally:
        torch.set_warn_always(always)


@pytest.mark.parametrize("layout", ["to_sparse", "to_sparse_csr", "to_sparse_csc"])
@pytest.mark.parametrize("m", ROWS)
def test_sparse_weights(tm, m, layout, monkeypatch):
    """Sparse operands are torch.matmul's (which has no bf16 sparse product on a CPU)."""
    x, _, w = _operands(m, 128, 128)
    w, got = getattr(w, layout)(), []
    monkeypatch.setattr(torch, "matmul", lambda a, b: got.append((a.shape, b)))
    tm.matmul(x, w)
    tm.matmul_shared_input(x, [w])
    tm.swiglu_matmul(x, x, w)
    assert len(got) == 3 and all(shape == (m, 128) and b is w for shape, b in got)


class _Seen(torch.overrides.TorchFunctionMode):
    def __torch_function__(self, func, types, args=(), kwargs=None):
        self.names.append(func.__name__)
        return func(*args, **(kwargs or {}))


@pytest.mark.parametrize("m", [1, 2, 3, 9, 16])
def test_modes_that_change_nothing(tm, m):
    """A default device and autocast to the operands' own type leave the
    kernels in place; autocast to another type and any other mode do not."""
    x, y, w = _operands(m, n=256)
    mode = _Seen()
    mode.names = []
    for f in _calls(tm, x, w):
        with torch.device("cpu"), pytest.raises(AssertionError, match="routed to a kernel"):
            f(y)
        with mode:
            f(y)
        try:
            torch.set_autocast_enabled("cuda", True)
            torch.set_autocast_dtype("cuda", torch.float16)
            f(y)
            torch.set_autocast_dtype("cuda", torch.bfloat16)
            with pytest.raises(AssertionError, match="routed to a kernel"):
                f(y)
        finally:
            torch.set_autocast_dtype("cuda", torch.float16)
            torch.set_autocast_enabled("cuda", False)
    assert mode.names.count("matmul") == 5  # matmul_shared_input makes two


@pytest.mark.parametrize("m", ROWS)
def test_gradients_are_recorded(tm, m):
    """Every route is differentiable in each of its operands, at every row count."""
    x, y, w = (t.requires_grad_() for t in _operands(m, 128, 128))
    for f, leaves in zip(_calls(tm, x, w), ((y, w), (y, w), (y, x, w), (y, x, w))):
        assert all(torch.isfinite(t).all() for t in torch.autograd.grad(f(y).float().sum(), leaves))


@pytest.mark.parametrize("with_residual", [False, True])
@pytest.mark.parametrize("m", [1, 2])
def test_norm_route_asks_as_well(tm, m, with_residual, monkeypatch):
    """The launch that folds the norm in: not where a gradient is recorded,
    under autocast to another type, or with operands of two devices."""
    from lightserve_amd.kernels import fused_rmsnorm_residual
    x, y, w = _operands(m, 128, 128)
    gain, residual = torch.ones(128, dtype=torch.bfloat16), y if with_residual else None
    with pytest.raises(AssertionError, match="routed to a kernel"):
        tm.add_rmsnorm_matmul_shared_input(x, residual, gain, 1e-6, [w])
    monkeypatch.setattr(fused_rmsnorm_residual, "rmsnorm", lambda a, weight, eps: a)
    monkeypatch.setattr(fused_rmsnorm_residual, "fused_add_rmsnorm", lambda a, r, weight, eps: (a, r))
    (out,), _ = tm.add_rmsnorm_matmul_shared_input(x, residual, gain, 1e-6, [w.clone().requires_grad_()])
    assert out.requires_grad
    monkeypatch.setattr(tm, "matmul_shared_input", lambda a, bs: ["apart"])

    def apart(residual=residual, gain=gain):
        return tm.add_rmsnorm_matmul_shared_input(x, residual, gain, 1e-6, [w])[0] == ["apart"]
    assert apart(gain=gain.to("meta")) and (not with_residual or apart(residual=y.to("meta")))
    try:
        torch.set_autocast_enabled("cuda", True)
        assert torch.get_autocast_dtype("cuda") == torch.float16 and apart()
    finally:
        torch.set_autocast_enabled("cuda", False)


@pytest.mark.parametrize("m,k,n", [(64, 128, 128), (600, 4096, 4096), (64, 4096, 200), (5000, 4096, 4096), (9, 128, 200),
                                   (16, 12, 128),
                                   (9, 1024, 1024), (16, 512, 2048), (17, 4096, 2048), (32, 8192, 512), (128, 4096, 1024),
                                   (512, 4096, 256), (128, 4096, 14336)])
def test_sizes_that_stay_on_torch_are_told_first(tm, m, k, n, monkeypatch):
    """A product that no kernel takes by its size goes on without the other questions."""
    def asked(*args):
        raise AssertionError("asked")
    for name in ("_library_only", "_auto_skinny", "_gemm_ok"):
        monkeypatch.setattr(tm, name, asked)
    monkeypatch.setattr(torch, "matmul", lambda a, b: "torch")
    x, w = torch.empty(m, k, dtype=torch.bfloat16), torch.empty(k, n, dtype=torch.bfloat16)
    assert tm.matmul(x, w) == "torch" and tm.matmul_shared_input(x, [w])[0] == "torch"
    if m > 32:
        assert tm.swiglu_matmul(x, x, w) == "torch"


@pytest.mark.parametrize("rows,k,cols", [(8, 512, (128,)), (9, 1536, (128,)), (16, 768, (3072,)), (9, 512, (256,)), (17, 3072, (3072,)),
                                         (32, 4096, (4096,)), (32, 256, (256, 256, 256)), (64, 4096, (14336,)),
                                         (128, 8192, (1024,)), (200, 4096, (1024,)), (512, 4096, (4096,)), (33, 4096, (2048,)),
                                         (65, 1024, (512, 512)), (129, 512, (1024, 1024)), (192, 256, (256, 256, 256))])
def test_sizes_that_have_a_kernel(rows, k, cols):
    """The other side of the same lines."""
    assert tiled_matmul._sizes_fit(rows, k, cols)
