"""Sparse MLA attention with at most 64 heads (the few-head kernels) against the float64 oracle, at the
sizes where their tiles end: head counts around 16 and 32, index rows around one and two key blocks,
rows with padding inside and at the end, rows without a key, and logits that force the second pass.

Tolerance: P (and dS) are rounded to bf16 before their products and outputs to bf16, 2^-9 each on terms
of one sign mixture, so a normalised error of a few 1e-3; 1e-2 as in the other parity tests."""
import pytest
import torch

from oracle import dsa_oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda"
SCALE = 192.0 ** -0.5


def _rows(T, N, K, seed, causal):
    g = torch.Generator().manual_seed(seed)
    idx = torch.full((T, K), -1, dtype=torch.int32)
    for t in range(T):
        lim = min(N, t + 1) if causal else N
        m = min(K, lim)
        pick = torch.randperm(lim, generator=g)[:m].sort().values.to(torch.int32)
        if t % 3 == 1 and K > m:                       # padding first
            idx[t, K - m:] = pick
        else:
            idx[t, :m] = pick
        if t % 4 == 2:                                 # padding inside, an id past the last row
            idx[t, torch.randperm(K, generator=g)[:max(1, K // 5)]] = -1
            idx[t, 0] = N + 3
    idx[min(5, T - 1)] = -1                            # a row without a key
    return idx


def _err(got, ref):
    return ((got.double().cpu() - ref).norm() / (ref.norm() + 1e-30)).item()


@pytest.mark.parametrize("H", [1, 15, 16, 17, 32, 33, 48, 64])
@pytest.mark.parametrize("K", [1, 32, 33, 65, 200])
def test_few_heads_forward(H, K):
    from mcore_bridge_amd import ops
    T, N = 37, 150
    print(f"[few heads] H={H} K={K}", flush=True)
    g = torch.Generator().manual_seed(1000 * H + K)
    q = torch.randn(T, H, 576, generator=g).bfloat16()
    q[3] *= 200.0                                      # overshoots the first block's reference: second pass
    kv = torch.randn(N, 576, generator=g).bfloat16()
    for causal in (False, True):
        idx = _rows(T, N, K, H + K, causal)
        ok = (idx >= 0) & (idx < N)
        if causal:
            ok &= idx <= torch.arange(T)[:, None]
        ref_idx = torch.where(ok, idx, torch.full_like(idx, -1)).long()
        out, lse = ops.sparse_mla_fwd(q.to(DEV), kv.to(DEV), idx.to(DEV), SCALE, causal)
        o_ref, l_ref = O.sparse_mla_fwd(q, kv, ref_idx, SCALE)
        live = torch.isfinite(l_ref)
        assert torch.equal(torch.isfinite(lse.cpu()), live)
        assert _err(out, o_ref) < 1e-2
        assert torch.allclose(lse.cpu().double()[live], l_ref[live], rtol=1e-4, atol=1e-4)
        if not causal:   # the key-split decode form of the same rows
            od, ld = ops.sparse_mla_decode(q.to(DEV), kv.to(DEV), idx.to(DEV), SCALE)
            assert _err(od, o_ref) < 1e-2 and torch.allclose(ld.cpu().double()[live], l_ref[live], rtol=1e-4, atol=1e-4)


@pytest.mark.parametrize("H", [16, 40])
def test_few_heads_forward_sink_without_rope(H):
    from mcore_bridge_amd import ops
    T, N, K = 21, 90, 77
    g = torch.Generator().manual_seed(H)
    q = torch.randn(T, H, 512, generator=g).bfloat16()
    kv = torch.nn.functional.pad(torch.randn(N, 512, generator=g).bfloat16(), (0, 64))
    sinks = torch.randn(H, generator=g)
    idx = _rows(T, N, K, 7, False)
    ref_idx = torch.where((idx >= 0) & (idx < N), idx, torch.full_like(idx, -1)).long()
    out, lse = ops.sparse_mla_fwd_sink(q.to(DEV), kv.to(DEV), idx.to(DEV), sinks.to(DEV), SCALE)
    o, l = O.sparse_mla_fwd(torch.nn.functional.pad(q, (0, 64)), kv, ref_idx, SCALE)
    l_ref = torch.logaddexp(l, sinks.double()[None].expand_as(l))
    o_ref = o * torch.exp(l - l_ref)[..., None]
    assert _err(out, o_ref) < 1e-2
    assert torch.allclose(lse.cpu().double(), l_ref, rtol=1e-4, atol=1e-4)


@pytest.mark.parametrize("H", [16, 32, 48, 64])
@pytest.mark.parametrize("K", [1, 32, 33, 65, 200])
def test_few_heads_backward(H, K):
    from mcore_bridge_amd import ops
    T, N = 37, 150
    print(f"[few heads bwd] H={H} K={K}", flush=True)
    g = torch.Generator().manual_seed(2000 * H + K)
    q = torch.randn(T, H, 576, generator=g).bfloat16()
    kv = torch.randn(N, 576, generator=g).bfloat16()
    dout = torch.randn(T, H, 512, generator=g).bfloat16()
    for causal in (False, True):
        idx = _rows(T, N, K, H + K, causal)
        ok = (idx >= 0) & (idx < N)
        if causal:
            ok &= idx <= torch.arange(T)[:, None]
        ref_idx = torch.where(ok, idx, torch.full_like(idx, -1)).long()
        o_ref, l_ref = O.sparse_mla_fwd(q, kv, ref_idx, SCALE)
        out, lse = o_ref.bfloat16(), l_ref.float()
        dq_ref, dkv_ref = O.sparse_mla_bwd(q, kv, ref_idx, out, dout, l_ref, SCALE)
        a = [x.to(DEV) for x in (q, kv, idx, out, dout, lse)]
        dq, dkv = ops.sparse_mla_bwd(*a, SCALE, causal)
        # a single key has P = 1 and dS = 0 but for out's rounding: dq is then held to dout's scale
        floor = 1e-2 * (dout.double().norm() if K == 1 else 0.0)
        for name, got, ref in (("dq", dq, dq_ref), ("dkv", dkv, dkv_ref)):
            err = (got.double().cpu() - ref).norm().item()
            assert err < 1e-2 * ref.norm().item() + floor, f"{name} causal={causal}: {err} of {ref.norm()}"
        assert torch.equal(dkv, ops.sparse_mla_bwd(*a, SCALE, causal)[1])
