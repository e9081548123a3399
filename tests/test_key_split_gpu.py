"""The forward with its keys split over workgroups (lsfa_fwd_split,
lsfa_prefill_paged_split) against the unsplit forward of the same library and
the float64 oracle: both take the same tiles with fp32 partial results, so they
agree to one rounding of the output (2^-8 of it in bf16, 2^-11 in fp16), up to
the rounding of p, which follows each split's own exponent offset (another
2^-9 / 2^-12 of the largest |v|, the bound of the unsplit forward itself)."""
import importlib
import math

import pytest
import torch

from lightserve_amd import _lib
from lightserve_amd.kernels.flash_attention_varlen import flash_attention_varlen_forward
from lightserve_amd.kernels.paged_attention import paged_prefill
from oracle.attention import attention_reference

pytestmark = pytest.mark.gpu
fa = importlib.import_module("lightserve_amd.kernels.flash_attention")  # (the package has a function of that name)


def _ulp(dtype):
    return 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11


def _unsplit(monkeypatch):
    monkeypatch.setattr(fa, "SPLIT_MAX_TILES", 0)
    monkeypatch.setattr(_lib, "prefill_paged_workspace_size", lambda args: 0)


def _agree(got, want, v, dtype):
    """Outputs and logsumexps of the two forwards."""
    o, lse = got
    o2, lse2 = want
    torch.testing.assert_close(lse, lse2, atol=2e-5, rtol=1e-5, equal_nan=True)
    bound = _ulp(dtype) * (o2.float().abs() + v.float().abs().max())
    assert ((o.float() - o2.float()).abs() <= bound).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,H,N,D,causal", [(1, 2, 1024, 128, True), (1, 1, 1537, 128, False), (1, 3, 2047, 64, True),
                                            (2, 1, 4001, 40, False), (1, 4, 4096, 128, True), (1, 1, 9000, 24, True)])
def test_dense_split(B, H, N, D, causal, dtype, monkeypatch):
    print(f"case dense split {B}x{H}x{N}x{D} causal={causal} {dtype}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(N)
    q, k, v = (torch.randn(B, N, H, D, device="cuda", generator=g).to(dtype).transpose(1, 2) for _ in range(3))
    seen = []
    real = _lib.fwd_split
    monkeypatch.setattr(_lib, "fwd_split", lambda *a: (seen.append(1), real(*a)))
    got = fa.flash_attention_forward(q, k, v, causal, return_lse=True)
    plain = fa.flash_attention_forward(q, k, v, causal)
    torch.cuda.synchronize()
    assert len(seen) == 2, "the call was not split"
    assert torch.equal(got[0], plain)
    assert torch.equal(got[0], fa.flash_attention_forward(q, k, v, causal))
    _unsplit(monkeypatch)
    _agree(got, fa.flash_attention_forward(q, k, v, causal, return_lse=True), v, dtype)
    o_ref, _ = attention_reference(q[:1, :1].cpu(), k[:1, :1].cpu(), v[:1, :1].cpu(), causal)
    assert (got[0][:1, :1].cpu().double() - o_ref).abs().max() < 2e-2


@pytest.mark.parametrize("lens_q,lens_k", [([1, 130, 0, 65], [2000, 1500, 700, 40]), ([300], [5000]), ([129, 1], [64, 3000]),
                                           ([200, 200], [100, 3000])])
def test_paged_and_packed_split(lens_q, lens_k, monkeypatch):
    """Chunks of several lengths (empty ones among them, rows that see no key,
    items of too few tiles beside items that split) over a paged cache and over
    packed keys."""
    print(f"case paged split {lens_q} {lens_k}", flush=True)
    H, Hkv, D, bs = 6, 2, 128, 16
    g = torch.Generator(device="cuda").manual_seed(sum(lens_k))
    B, nb = len(lens_q), [-(-n // bs) for n in lens_k]
    kc, vc = (torch.randn(sum(nb), bs, Hkv, D, device="cuda", generator=g).to(torch.bfloat16) for _ in range(2))
    bt = torch.full((B, max(nb)), -1, dtype=torch.int32, device="cuda")
    order = torch.randperm(sum(nb), generator=torch.Generator().manual_seed(1)).to(torch.int32).cuda()
    at = 0
    for i, n in enumerate(nb):
        bt[i, :n] = order[at:at + n]
        at += n
    q = torch.randn(sum(lens_q), H, D, device="cuda", generator=g).to(torch.bfloat16)

    def offsets(lens):
        return torch.tensor([0] + lens, device="cuda").cumsum(0).to(torch.int32)
    cu, sl = offsets(lens_q), torch.tensor(lens_k, dtype=torch.int32, device="cuda")
    seen = []
    for name in ("prefill_paged_split", "fwd_split"):
        real = getattr(_lib, name)
        monkeypatch.setattr(_lib, name, lambda *a, real=real, name=name: (seen.append(name), real(*a)))
    kp, vp = (torch.cat([c[bt[i, :nb[i]].long()].flatten(0, 1)[:n] for i, n in enumerate(lens_k)]) for c in (kc, vc))
    for causal in (True, False):
        got = paged_prefill(q, kc, vc, bt, cu, sl, max_seqlen_q=max(lens_q), causal=causal, return_lse=True)
        got2 = flash_attention_varlen_forward(q, kp, vp, cu, offsets(lens_k), max(lens_q), max(lens_k), causal=causal)
        with monkeypatch.context() as m:
            _unsplit(m)
            want = paged_prefill(q, kc, vc, bt, cu, sl, max_seqlen_q=max(lens_q), causal=causal, return_lse=True)
        _agree(got, want, vc, torch.bfloat16)
        _agree(got2, want, vc, torch.bfloat16)
    assert seen.count("prefill_paged_split") == 2 and seen.count("fwd_split") == 2


def test_split_keeps_nan_inf_and_capture(monkeypatch):
    """A NaN or infinite score shows in the rows that see it and nowhere else,
    as unsplit; and a captured split call replays with the eager result."""
    print("case split nan / capture", flush=True)
    q, k, v = (torch.randn(1, 2, 2048, 64, device="cuda").to(torch.bfloat16) for _ in range(3))
    k[0, 0, 1500] = float("nan")
    k[0, 1, 700, 3] = math.inf
    got = fa.flash_attention_forward(q, k, v, True)
    with monkeypatch.context() as m:
        _unsplit(m)
        want = fa.flash_attention_forward(q, k, v, True)
    assert torch.equal(got.isnan(), want.isnan()) and got.isnan().any() and got.isfinite().any()
    k.copy_(torch.randn_like(k))
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        fa.flash_attention_forward(q, k, v, True)
        s.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=s):
            o = fa.flash_attention_forward(q, k, v, True)
    for _ in range(3):
        k.copy_(torch.randn_like(k))
        eager = fa.flash_attention_forward(q, k, v, True)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(o, eager)
