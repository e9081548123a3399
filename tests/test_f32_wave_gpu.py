"""The fp32 kernels for rows that 16-byte loads can address, at the edges of
their 32-row tiles and of the splits of a row block over waves, against float64
autograd and against the general kernels (the same values in rows of odd
stride, which only those take). Bound: each output element is a chain of at most
three fp32 sums (scores, probabilities, products) of up to N terms, whose
rounding errors add like a random walk: sqrt(N) 2^-24 relative per sum, under
8e-7 at N = 2000; 4e-6 leaves a factor of five."""
import math

import pytest
import torch

from lightserve_amd.kernels.flash_attention_backward import _flash_attention_backward, _flash_attention_forward_lse
from lightserve_amd.kernels.flash_attention_varlen import flash_attention_varlen_forward

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return ((a.double() - b.double()).norm() / b.double().norm().clamp_min(1e-30)).item()


def _odd(t):
    """t's values in rows of odd stride."""
    wide = torch.zeros(*t.shape[:-1], t.shape[-1] + 1 + t.shape[-1] % 2, device=t.device)
    wide[..., :t.shape[-1]] = t
    return wide[..., :t.shape[-1]]


def _run(q, k, v, do, causal):
    o, lse = _flash_attention_forward_lse(q, k, v, causal)
    return (o, *_flash_attention_backward(do, q, k, v, o, lse, causal), lse)


# blocks of 32 rows x heads: one to 128 (four waves a block), 544 (two, or four when causal), 1056 / 2080 (one, or two / one)
@pytest.mark.parametrize("B,H,N,D", [(1, 1, 1, 4), (1, 2, 31, 8), (1, 3, 33, 32), (2, 2, 129, 36), (1, 4, 257, 64), (1, 2, 500, 100),
                                     (1, 3, 640, 128), (4, 8, 513, 64), (4, 16, 515, 32), (8, 16, 490, 20), (8, 20, 385, 128)])
@pytest.mark.parametrize("causal", [True, False])
def test_wave_kernels(B, H, N, D, causal):
    print(f"case f32 wave {B}x{H}x{N}x{D} causal={causal}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(N)
    q, k, v, do = (torch.randn(B, N, H, D, device="cuda", generator=g).transpose(1, 2) for _ in range(4))
    got = _run(q, k, v, do, causal)
    assert all(torch.equal(a, b) for a, b in zip(got, _run(q, k, v, do, causal)))
    general = _run(*(_odd(t) for t in (q, k, v, do)), causal)
    qd, kd, vd = (t[:2, :2].double().requires_grad_() for t in (q, k, v))
    s = qd @ kd.transpose(2, 3) / math.sqrt(D)
    if causal:
        s = s.masked_fill(torch.ones(N, N, dtype=torch.bool, device="cuda").triu(1), -math.inf)
    ref = s.softmax(-1) @ vd
    want = (ref, *torch.autograd.grad(ref, (qd, kd, vd), do[:2, :2].double()))
    for name, a, b, c in zip(("o", "dq", "dk", "dv"), got, want, general):
        if N > 1 or name in ("o", "dv"):  # one key: dq and dk are rounding noise around zero
            assert _rel(a[:2, :2], b) < 4e-6, name
            assert _rel(a, c) < 8e-6, name
    assert (got[4][:2, :2].double() - torch.logsumexp(s, -1)).abs().max() < 1e-5


@pytest.mark.parametrize("causal", [True, False])
def test_wave_forward_packed(causal):
    """Packed sequences with grouped heads: empty sides, rows that see no key,
    more keys than queries and fewer; infinities and NaN as the general kernel
    gives them."""
    print(f"case f32 wave packed causal={causal}", flush=True)
    lq, lk = [40, 0, 1, 130, 64, 3], [17, 3, 1, 300, 0, 200]
    g = torch.Generator(device="cuda").manual_seed(3)
    q = torch.randn(sum(lq), 6, 64, device="cuda", generator=g)
    k, v = (torch.randn(sum(lk), 2, 64, device="cuda", generator=g) for _ in range(2))
    cu = [torch.tensor([0] + n, device="cuda").cumsum(0).to(torch.int32) for n in (lq, lk)]
    for poison in (None, math.inf, math.nan):
        if poison is not None:
            k[sum(lk[:3]) + 7, 1, 5] = poison
        o, lse = flash_attention_varlen_forward(q, k, v, *cu, max(lq), max(lk), causal=causal)
        o2, lse2 = flash_attention_varlen_forward(_odd(q), _odd(k), _odd(v), *cu, max(lq), max(lk), causal=causal)
        assert torch.equal(o.isnan(), o2.isnan()) and torch.equal(lse.isinf(), lse2.isinf())
        torch.testing.assert_close(o, o2, atol=4e-6, rtol=4e-6, equal_nan=True)
        torch.testing.assert_close(lse, lse2, atol=4e-6, rtol=4e-6, equal_nan=True)


def test_wave_kernels_take_only_what_they_can_address():
    """Expanded, transposed and offset operands, and a head dim that is not a
    multiple of four, keep giving the general kernels' results."""
    print("case f32 wave layouts", flush=True)
    q, k, v = (torch.randn(1, 2, 200, 32, device="cuda") for _ in range(3))
    want, _ = _flash_attention_forward_lse(q, k[:, :, :1].expand(1, 2, 200, 32).contiguous(), v, True)
    forms = [(q, k[:, :, :1].expand(1, 2, 200, 32), v),                                    # row stride 0
             (q.transpose(2, 3).contiguous().transpose(2, 3), k[:, :, :1].expand(1, 2, 200, 32), v),  # head-dim stride 200
             (_odd(q), k[:, :, :1].expand(1, 2, 200, 32).contiguous(), v),
             (torch.empty(q.numel() + 1, device="cuda")[1:].view_as(q).copy_(q), k[:, :, :1].expand(1, 2, 200, 32), v)]
    for a, b, c in forms:
        got, _ = _flash_attention_forward_lse(a, b, c, True)
        assert _rel(got, want) < 8e-6
