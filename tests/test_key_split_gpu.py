"""The forward with its keys split over workgroups (lsfa_fwd_split,
lsfa_prefill_paged_split) against attention in float64, row by row, and against
the unsplit forward of the same library.

The bound on a row is that of the unsplit forward: partial results and their
merge are fp32, so what is left is one rounding of the output, at most u |o|
(u half an ulp: 2^-9 in bf16, 2^-12 in fp16), and the rounding of p, each p_i off
by at most u p_i with either sign: u sqrt(sum p_i^2 |v_i|^2) if one key carries
the row, 0.58 of that in the mean where many do. Leaving out a fifth of the keys,
or a wrong weight on one split, is a hundred times that."""
import importlib
import math

import pytest
import torch

from lightserve_amd import _lib
from lightserve_amd.kernels.flash_attention_varlen import flash_attention_varlen_forward
from lightserve_amd.kernels.paged_attention import paged_prefill

pytestmark = pytest.mark.gpu
fa = importlib.import_module("lightserve_amd.kernels.flash_attention")  # (the package has a function of that name)


def _unsplit(monkeypatch):
    monkeypatch.setattr(fa, "SPLIT_MAX_TILES", 0)
    monkeypatch.setattr(_lib, "prefill_paged_workspace_size", lambda args: 0)


def _check_head(o, lse, q, k, v, causal):
    """One head's rows [n, D] (and lse [n]) against float64."""
    u = 2.0 ** -9 if o.dtype == torch.bfloat16 else 2.0 ** -12
    q, k, v = q.double(), k.double(), v.double()
    s = (q @ k.T) * q.shape[1] ** -0.5
    if causal:
        s.masked_fill_(torch.ones_like(s, dtype=torch.bool).triu_(k.shape[0] - q.shape[0] + 1), -math.inf)
    want = torch.logsumexp(s, 1)
    p = torch.exp(s - want[:, None]).nan_to_num_(0.0)  # a row that sees no key: o = 0
    ref = p @ v
    bound = u * (ref.norm(dim=1) + (p.square() @ v.square().sum(1)).sqrt())
    err = (o.double() - ref).norm(dim=1)
    worst = (err - bound).argmax()
    assert (err <= bound + 1e-6).all(), (int(worst), float(err[worst]), float(bound[worst]))
    torch.testing.assert_close(lse.double(), want, atol=2e-5, rtol=1e-5)


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
    want = fa.flash_attention_forward(q, k, v, causal, return_lse=True)
    for b in range(B):
        for h in range(H):
            for o, lse in (got, want):
                _check_head(o[b, h], lse[b, h], q[b, h], k[b, h], v[b, h], causal)


@pytest.mark.parametrize("dtype,D", [(torch.bfloat16, 128), (torch.float16, 128), (torch.bfloat16, 64), (torch.float16, 24)])
@pytest.mark.parametrize("lens_q,lens_k", [([1, 130, 0, 65], [2000, 1500, 700, 40]), ([300], [5000]), ([129, 1], [64, 3000]),
                                           ([200, 200], [100, 3000]),
                                           ([3, 0] * 32 + [5], [40, 9, 1100, 2500] * 16 + [5200])])
def test_paged_and_packed_split(lens_q, lens_k, dtype, D, monkeypatch):
    """Chunks of several lengths (empty ones among them, rows that see no key,
    items of too few tiles beside items that split, more sequences than the
    ranking of items takes) over a paged cache and over packed keys."""
    print(f"case paged split {lens_q[:4]} {lens_k[:4]} of {len(lens_q)} {dtype} D={D}", flush=True)
    H, Hkv, bs = (6, 2, 16) if len(lens_q) < 64 else (2, 1, 16)
    g = torch.Generator(device="cuda").manual_seed(sum(lens_k))
    B, nb = len(lens_q), [-(-n // bs) for n in lens_k]
    kc, vc = (torch.randn(sum(nb), bs, Hkv, D, device="cuda", generator=g).to(dtype) for _ in range(2))
    bt = torch.full((B, max(nb)), -1, dtype=torch.int32, device="cuda")
    order = torch.randperm(sum(nb), generator=torch.Generator().manual_seed(1)).to(torch.int32).cuda()
    at = 0
    for i, n in enumerate(nb):
        bt[i, :n] = order[at:at + n]
        at += n
    q = torch.randn(sum(lens_q), H, D, device="cuda", generator=g).to(dtype)

    def offsets(lens):
        return torch.tensor([0] + lens, device="cuda").cumsum(0).to(torch.int32)
    cu, sl = offsets(lens_q), torch.tensor(lens_k, dtype=torch.int32, device="cuda")
    seen = []
    for name in ("prefill_paged_split", "fwd_split"):
        real = getattr(_lib, name)
        monkeypatch.setattr(_lib, name, lambda *a, real=real, name=name: (seen.append(name), real(*a)))
    keys, values = ([c[bt[i, :nb[i]].long()].flatten(0, 1)[:n] for i, n in enumerate(lens_k)] for c in (kc, vc))
    kp, vp = torch.cat(keys), torch.cat(values)
    for causal in (True, False):
        got = paged_prefill(q, kc, vc, bt, cu, sl, max_seqlen_q=max(lens_q), causal=causal, return_lse=True)
        got2 = flash_attention_varlen_forward(q, kp, vp, cu, offsets(lens_k), max(lens_q), max(lens_k), causal=causal)
        with monkeypatch.context() as m:
            _unsplit(m)
            want = paged_prefill(q, kc, vc, bt, cu, sl, max_seqlen_q=max(lens_q), causal=causal, return_lse=True)
        row = 0
        for i, n in enumerate(lens_q):
            r, row = slice(row, row + n), row + n
            for h in range(H if n else 0):
                for o, lse in (got, got2, want):
                    _check_head(o[r, h], lse[h, r], q[r, h], keys[i][:, h // (H // Hkv)], values[i][:, h // (H // Hkv)],
                                causal)
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


@pytest.mark.parametrize("B,chunk,prefix,D", [(2, 512, 0, 128), (2, 512, 256, 128), (1, 512, 0, 64), (4, 128, 256, 128),
                                              (4, 16, 0, 128), (1, 1024, 0, 128), (2, 300, 100, 64)])
def test_wide_table_leaves_short_prompts_whole(B, chunk, prefix, D, monkeypatch):
    """A block table sized for a context limit, over sequences too short to be
    split: the same bits as under a table that just holds them."""
    print(f"case wide table {B} x {prefix}+{chunk} D={D}", flush=True)
    H, Hkv, bs, n = 32, 8, 16, prefix + chunk
    g = torch.Generator(device="cuda").manual_seed(n)
    blocks = -(-n // bs)
    kc, vc = (torch.randn(B * blocks, bs, Hkv, D, device="cuda", generator=g).to(torch.bfloat16) for _ in range(2))
    tight = torch.randperm(B * blocks, device="cuda", generator=g).to(torch.int32).view(B, blocks)
    wide = torch.full((B, 1024), -1, dtype=torch.int32, device="cuda")
    wide[:, :blocks] = tight
    q = torch.randn(B * chunk, H, D, device="cuda", generator=g).to(torch.bfloat16)
    cu = torch.arange(0, (B + 1) * chunk, chunk, dtype=torch.int32, device="cuda")
    sl = torch.full((B,), n, dtype=torch.int32, device="cuda")
    seen = []
    real = _lib.prefill_paged_split
    monkeypatch.setattr(_lib, "prefill_paged_split", lambda *a: (seen.append(1), real(*a)))
    got = paged_prefill(q, kc, vc, wide, cu, sl, max_seqlen_q=chunk, return_lse=True)
    assert seen, "the launch under the wide table has splits to give"
    _unsplit(monkeypatch)
    want = paged_prefill(q, kc, vc, tight, cu, sl, max_seqlen_q=chunk, return_lse=True)
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
