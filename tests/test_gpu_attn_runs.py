"""Decode attention where a workgroup takes one, two or more steps of 128
positions (four waves of 32) and where a wave has none, at the edges of a step
and of a 32-position group, against the oracle.

Bound: 1e-5 relative per head. The products carry ~22 significant bits and the
sums are in fp32: over p positions, p <= 2^14, the softmax sum and the output
sum in four chains of at most p / 128 steps of 32 terms, a worst case of about
(p / 128 + 40) 2^-24 < 1e-5 of the largest partial sum."""
import numpy as np
import pytest
import torch

from desireeia_amd import _lib, ops

from test_gpu_attn import device_cache, host_cache, rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fused", [False, True])
@pytest.mark.parametrize("hd,n_head,n_kv,pos,cc_start", [
    (64, 8, 4, 31, 0),         # exactly one group
    (64, 16, 16, 8192, 0),     # one group past whole steps
    (64, 64, 64, 5000, 33),    # runs of several steps
    (128, 8, 8, 127, 0),       # exactly one step
    (128, 16, 4, 128, 0),      # one position past it
    (128, 64, 64, 1535, 0),    # the longest runs of one step
    (128, 64, 64, 1568, 0),    # runs of two; the last workgroup with one group
    (128, 64, 32, 9000, 77),   # runs of several, from inside the cache
    (256, 8, 8, 96, 0),        # three of four waves
    (256, 32, 32, 3333, 1),    # runs of several steps
])
def test_attention_runs(gpu, orc, hd, n_head, n_kv, pos, cc_start, fused):
    print(f"attn runs hd={hd} n_head={n_head} n_kv={n_kv} pos={pos} cc_start={cc_start} fused={fused}", flush=True)
    n_old = pos if fused else pos + 1
    kc, vc = host_cache(orc, n_old, n_kv, seed=pos + n_head + hd, hd=hd)
    rng = np.random.default_rng(pos + hd)
    q = rng.standard_normal(n_head * hd).astype(np.float32)
    k, v = (rng.standard_normal(n_kv * hd).astype(np.float32) for _ in range(2))
    # runs are taken where the cache has more steps than 2 workgroups per CU
    cus = torch.cuda.get_device_properties(gpu).multi_processor_count
    n_ctx = max(pos + 5, 128 * (2 * cus // n_kv + 1))
    cache = device_cache(gpu, kc, vc, n_ctx, n_kv, hd=hd)
    dq, dk, dv = (torch.from_numpy(a).to(gpu) for a in (q, k, v))
    if fused:
        table = orc.rope_cache(hd, pos, 10000.0)
        dr = torch.from_numpy(table).to(gpu)
        got = torch.empty(n_head * hd, dtype=torch.float32, device=gpu)
        work = ops.attn_workspace(n_head, n_kv, hd, cache.n_ctx, gpu)
        _lib.check(_lib.load().dq_attn_rope_kv_decode(
            ops._ptr(dq), ops._ptr(dk), ops._ptr(dv), ops._ptr(dr), hd, ops._ptr(cache.k), ops._ptr(cache.v), n_head,
            n_kv, hd, cc_start, pos, None, cache.n_ctx, ops._ptr(got), None, None, None, ops._ptr(work), work.numel(),
            ops._stream()), "dq_attn_rope_kv_decode")
        q = np.concatenate([orc.rope_neox(x, hd, table) for x in q.reshape(n_head, hd)])
        k = np.concatenate([orc.rope_neox(x, hd, table) for x in k.reshape(n_kv, hd)])
        kc = np.concatenate([kc, orc.kv_quantize_row(k)])
        vc = np.concatenate([vc, orc.kv_quantize_row(v)])
        pb = n_kv * hd // 32 * 34
        assert np.array_equal(cache.k.cpu().numpy()[:(pos + 1) * pb], kc)
        assert np.array_equal(cache.v.cpu().numpy()[:(pos + 1) * pb], vc)
    else:
        got = ops.attention_decode(dq, cache, n_head, pos, cc_start)
    want = orc.attn_decode(q, kc, vc, n_head, n_kv, hd, cc_start, pos, f64=True)
    got = got.cpu().numpy().reshape(n_head, hd)
    want = np.asarray(want).reshape(n_head, hd)
    worst = max(rel(g, w) for g, w in zip(got, want))
    print(f"  worst head {worst:.2e}", flush=True)
    assert worst <= 1e-5


@pytest.mark.parametrize("spans", [
    [(0, 128)],                           # the first step of a run's four waves
    [(800, 832), (1920, 2560)],           # a later step of one wave, a whole run
])
def test_attention_runs_minus_infinity(gpu, orc, spans):
    """Positions whose scores are all -inf weigh 0, wherever the steps put them."""
    hd, n_head, n_kv, pos = 128, 64, 32, 9000   # runs of 5 steps
    print(f"attn runs -inf {spans}", flush=True)
    kc, vc = host_cache(orc, pos + 1, n_kv, seed=7, hd=hd)
    rng = np.random.default_rng(7)
    q = rng.standard_normal(n_head * hd).astype(np.float32)
    q.reshape(n_head, hd)[:, :32] = 1.0
    blocks = kc.reshape(pos + 1, n_kv, hd // 32, 34)
    keep = np.ones(pos + 1, bool)
    for a, b in spans:
        blocks[a:b, :, 0, :2] = np.array([np.inf], np.float16).view(np.uint8)
        blocks[a:b, :, 0, 2:] = 255         # quants of -1
        keep[a:b] = False
    n_ctx = max(pos + 5, 128 * (2 * torch.cuda.get_device_properties(gpu).multi_processor_count // n_kv + 1))
    got = ops.attention_decode(torch.from_numpy(q).to(gpu), device_cache(gpu, kc, vc, n_ctx, n_kv, hd=hd), n_head, pos, 0)
    kept = [np.ascontiguousarray(c.reshape(pos + 1, -1)[keep]).reshape(-1) for c in (kc, vc)]
    want = orc.attn_decode(q, *kept, n_head, n_kv, hd, 0, int(keep.sum()) - 1, f64=True)
    got, want = got.cpu().numpy().reshape(n_head, hd), np.asarray(want).reshape(n_head, hd)
    assert max(rel(g, w) for g, w in zip(got, want)) <= 1e-5
