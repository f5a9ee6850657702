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


# (T, N, K, H, causal, q width): key tiles of 128 and subtiles of 32 that end inside, query chunks of 16,
# two LDS passes of the inverse index (N > 16384), one to eight head groups; at each of them a query
# selects a good part of the keys it sees, so dKV is summed by key tiles
_TILED = [(130, 129, 96, 16, False, 576), (128, 128, 128, 48, True, 576), (257, 257, 200, 64, True, 576),
          (513, 300, 256, 128, False, 576), (20, 16500, 1600, 16, False, 576), (145, 161, 160, 32, False, 512)]


@pytest.mark.parametrize("T,N,K,H,causal,dqk", _TILED)
def test_backward_by_key_tiles(T, N, K, H, causal, dqk):
    from mcore_bridge_amd import ops
    print(f"[key tiles] T={T} N={N} K={K} H={H} causal={causal} {dqk}", flush=True)
    g = torch.Generator().manual_seed(T + N + H)
    q = torch.randn(T, H, dqk, generator=g).bfloat16()
    kv = torch.randn(N, 576, generator=g).bfloat16()
    kv[:, dqk:] = 0
    dout = torch.randn(T, H, 512, generator=g).bfloat16()
    idx = _rows(T, N, K, T, causal)
    idx[9, 4], idx[9, 7], idx[10, 1] = idx[9, 2], idx[9, 2], idx[10, 3]   # rows that repeat a key
    ok = (idx >= 0) & (idx < N)
    if causal:
        ok &= idx <= torch.arange(T)[:, None]
    ref_idx = torch.where(ok, idx, torch.full_like(idx, -1)).long()
    qp = torch.nn.functional.pad(q, (0, 576 - dqk))
    o_ref, l_ref = O.sparse_mla_fwd(qp, kv, ref_idx, SCALE)
    out, lse = o_ref.bfloat16(), l_ref.float()
    dq_ref, dkv_ref = O.sparse_mla_bwd(qp, kv, ref_idx, out, dout, l_ref, SCALE)
    a = [x.to(DEV) for x in (q, kv, idx, out, dout, lse)]
    far = torch.full((H,), -1e4, device=DEV)   # 512-wide rows come with a sink: one of no weight

    def bwd(*cap):
        return ops.sparse_mla_bwd(*a, SCALE, causal, *cap) if dqk == 576 else ops.sparse_mla_bwd_sink(*a, far, SCALE, causal)[:2]

    dq, dkv = bwd()
    assert _err(dq, dq_ref[..., :dqk]) < 1e-2 and _err(dkv, dkv_ref) < 1e-2
    assert torch.equal(dkv, bwd()[1])
    if T > 512:   # passes of 256 queries under a cap
        one = ops.bwd_workspace_bytes_chunked(T, N, H, K, 256)
        dq2, dkv2 = bwd(one)
        assert torch.equal(dq2, dq) and _err(dkv2, dkv_ref) < 1e-2
    # a query that is not finite reaches the keys it selects and no other
    a[0][T - 2, H // 2, 3] = float("inf")
    bad = torch.zeros(N, dtype=torch.bool)
    bad[idx[T - 2][ok[T - 2]].long()] = True
    dkv = bwd()[1].cpu()
    assert torch.equal(~torch.isfinite(dkv).all(1), bad)
    rest = O.sparse_mla_bwd(qp, kv, torch.where(torch.arange(T)[:, None] == T - 2, -1, ref_idx), out, dout, l_ref, SCALE)[1]
    assert _err(dkv[~bad], rest[~bad]) < 1e-2
