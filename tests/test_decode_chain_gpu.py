"""The chained decode launch (decode_chain) against the separate kernels it
stands for: attention merge, o_proj, gate_up, down and the next layer's qkv,
bit for bit."""
from types import SimpleNamespace

import pytest
import torch

from conftest import announce

pytestmark = pytest.mark.gpu


def _layer(g, dev, hidden, inter, hq, hkv):
    def w(*shape, std=0.03):
        t = torch.randn(*shape, generator=g, device=dev) * std
        return SimpleNamespace(weight=t.to(torch.bfloat16))

    def norm(n):
        return SimpleNamespace(weight=(1 + 0.1 * torch.randn(n, generator=g, device=dev)).bfloat16())

    return SimpleNamespace(
        self_attn=SimpleNamespace(qkv_proj=w((hq + 2 * hkv) * 128, hidden),
                                  o_proj=w(hidden, hq * 128), q_norm=norm(128), k_norm=norm(128)),
        mlp=SimpleNamespace(gate_up_proj=w(2 * inter, hidden), down_proj=w(hidden, inter)),
        input_layernorm=norm(hidden), post_attention_layernorm=norm(hidden))


@pytest.mark.parametrize("hidden, inter, hq, hkv", [
    (1024, 3072, 16, 8),   # Qwen3-0.6B: every register of the weight slabs used
    (128, 2048, 16, 8),    # one k-step per wave of gate_up
    (640, 2304, 18, 9),    # ragged k-steps; the qkv halves are not whole prefetches
    (1024, 2816, 24, 8),   # the widest o_proj
])
@pytest.mark.parametrize("M", [1, 2, 7, 16])
@pytest.mark.parametrize("merge", [True, False])
def test_chain_same_bits_as_separate_kernels(gpu, hidden, inter, hq, hkv, M, merge):
    """Lengths from 1 token to thousands (heads written whole by one wave and
    split over many), a row outside the resident table, with and without the
    merge and the next layer; the counters are left at zero; three launches
    in a row."""
    from qwen3_engine_from_scratch_amd.PagedKVcache import (KVCachePool, PagedKVCache,
                                                            reserve_pages_bulk, set_seq_lens_bulk)
    from qwen3_engine_from_scratch_amd.kernels.model_ops import (
        decode_chain, decode_chain_ok, decode_chain_sync, decode_linear, decode_qkv_rope, embed_ss)
    from qwen3_engine_from_scratch_amd.kernels.paged_attention import (
        paged_attention_decode_hip, paged_attention_decode_partials_hip,
        paged_decode_workspace_bytes)
    from qwen3_engine_from_scratch_amd.kernels.pre_attention import rope_tables

    assert decode_chain_ok(M, hidden, inter, hq, hkv)
    assert not decode_chain_ok(17, hidden, inter, hq, hkv)
    g = torch.Generator(device=gpu).manual_seed(M + hidden)
    a, b = (_layer(g, gpu, hidden, inter, hq, hkv) for _ in range(2))
    lens = [3000, 1, 16, 40, 700, 15, 129][:M] + [33 * i + 5 for i in range(M - 7)]
    pool = KVCachePool(sum(n // 16 + 1 for n in lens) + 2, 2, 16, hkv, 128, device=gpu,
                       dtype=torch.bfloat16, max_seq_len=4096, max_requests=M + 1)
    caches = [PagedKVCache(pool) for _ in range(M)]
    reserve_pages_bulk(caches, [n + 1 for n in lens])
    for c, n in zip(caches, lens):
        c.seq_len = n
    set_seq_lens_bulk(caches)
    rows = [c.row_id for c in caches]
    if M == 7:
        rows[3] = -1
    rows = torch.tensor(rows, dtype=torch.int32, device=gpu)
    pool.k_buffer.normal_(generator=g)
    pool.v_buffer.normal_(generator=g)
    cos, sin = rope_tables(128, 1e6, 4096, device=gpu)
    pos = torch.tensor(lens, device=gpu) if M != 2 else None
    emb = torch.randn(64, hidden, generator=g, device=gpu).bfloat16()
    ids = torch.arange(M, device=gpu)
    q0 = torch.randn(M, hq, 128, generator=g, device=gpu).bfloat16()
    kv = (pool.block_table_2d, pool.seq_lens, rows, 16)
    ws = torch.zeros(paged_decode_workspace_bytes(M, hq, hkv, 128, pool.block_table_2d.shape[1], 16),
                     dtype=torch.uint8, device=gpu)
    eps = 1e-6
    announce(f"decode chain M={M} hidden={hidden} inter={inter} heads={hq}/{hkv} merge={merge}")

    o = paged_attention_decode_hip(q0, pool.k_buffer[:, 0], pool.v_buffer[:, 0], *kv, workspace=ws)
    h, ss = embed_ss(ids, emb)
    mid, ss_mid = torch.empty_like(h), torch.empty_like(ss)
    k0, v0 = pool.k_buffer.clone(), pool.v_buffer.clone()
    want = []
    for nxt in (True, True, False):  # the same layer's work three times in a row
        decode_linear(o.view(M, -1), a.self_attn.o_proj.weight, epilogue="residual", residual=h,
                      residual_out=mid, ss_out=ss_mid)
        act = decode_linear(mid, a.mlp.gate_up_proj.weight, epilogue="silu", ss_in=ss_mid,
                            norm_weight=a.post_attention_layernorm.weight, eps=eps)
        decode_linear(act, a.mlp.down_proj.weight, epilogue="residual", residual=mid,
                      residual_out=h, ss_out=ss)
        q = None
        if nxt:
            q = decode_qkv_rope(h, ss, b.input_layernorm.weight, eps, b.self_attn.qkv_proj.weight,
                                hq, hkv, b.self_attn.q_norm.weight, b.self_attn.k_norm.weight,
                                eps, cos, sin, pool, 1, rows, pos)
        want.append([t.clone() for t in (h, ss, mid, ss_mid, pool.k_buffer, pool.v_buffer)] + [q])
    pool.k_buffer.copy_(k0)
    pool.v_buffer.copy_(v0)

    h, ss = embed_ss(ids, emb)
    mid, ss_mid = torch.full_like(h, float("nan")), torch.full_like(ss, float("nan"))
    sync = decode_chain_sync(gpu)
    whole = o
    for i, nxt in enumerate((True, True, False)):
        if merge:
            o = paged_attention_decode_partials_hip(q0, pool.k_buffer[:, 0], pool.v_buffer[:, 0],
                                                    *kv, ws)
        q = decode_chain(o, h, mid, ss, ss_mid, a, eps, hq, hkv, sync,
                         attn_workspace=ws if merge else None, next_layer=b if nxt else None,
                         head_eps=eps, cos_table=cos, sin_table=sin, pool=pool, next_idx=1,
                         row_ids=rows, positions=pos)
        torch.cuda.synchronize()
        assert torch.equal(o, whole)
        for name, x, y in zip("h ss mid ss_mid k v q".split(),
                              [h, ss, mid, ss_mid, pool.k_buffer, pool.v_buffer, q], want[i]):
            assert (x is None and y is None) or torch.equal(x, y), f"launch {i}: {name}"
        assert not sync.any()


@pytest.mark.parametrize("hidden, hq, hkv", [(1024, 16, 8), (64, 3, 1), (640, 18, 9)])
@pytest.mark.parametrize("M", [1, 16, 17, 33, 64])
def test_qkv_half_heads_same_bits(gpu, hidden, hq, hkv, M):
    """decode_qkv_rope on two workgroups per head against one: rows past a
    16-row block's end, rows outside the resident table, a row stride of the
    residual stream that is not its width; the exchanged words are left zero."""
    from qwen3_engine_from_scratch_amd.PagedKVcache import (KVCachePool, PagedKVCache,
                                                            reserve_pages_bulk, set_seq_lens_bulk)
    from qwen3_engine_from_scratch_amd.kernels.model_ops import (decode_chain_sync,
                                                                 decode_qkv_rope, embed_ss)
    from qwen3_engine_from_scratch_amd.kernels.pre_attention import rope_tables

    g = torch.Generator(device=gpu).manual_seed(M + hidden)
    layer = _layer(g, gpu, hidden, 128, hq, hkv)
    at = layer.self_attn
    lens = [(37 * i) % 200 for i in range(M)]
    pool = KVCachePool(sum(n // 16 + 1 for n in lens) + 2, 2, 16, hkv, 128, device=gpu,
                       dtype=torch.bfloat16, max_seq_len=256, max_requests=M + 1)
    caches = [PagedKVCache(pool) for _ in range(M)]
    reserve_pages_bulk(caches, [n + 1 for n in lens])
    for c, n in zip(caches, lens):
        c.seq_len = n
    set_seq_lens_bulk(caches)
    rows = torch.tensor([c.row_id for c in caches], dtype=torch.int32, device=gpu)
    if M > 16:
        rows[5], rows[16] = -1, 1 << 20
    cos, sin = rope_tables(128, 1e6, 256, device=gpu)
    h, ss = embed_ss(torch.arange(M, device=gpu),
                     torch.randn(64, hidden, generator=g, device=gpu).bfloat16())
    wide = torch.zeros(M, hidden + 64, dtype=h.dtype, device=gpu)
    wide[:, :hidden] = h
    sync = decode_chain_sync(gpu)
    announce(f"qkv half heads M={M} hidden={hidden} heads={hq}/{hkv}")

    def run(x, **kw):
        pool.k_buffer.zero_()
        pool.v_buffer.zero_()
        q = decode_qkv_rope(x, ss, layer.input_layernorm.weight, 1e-6, at.qkv_proj.weight, hq, hkv,
                            at.q_norm.weight, at.k_norm.weight, 1e-5, cos, sin, pool, 1, rows, **kw)
        return q, pool.k_buffer.clone(), pool.v_buffer.clone()

    want = run(h)
    for x in (h, wide[:, :hidden], h):
        for a, b in zip(run(x, sync=sync), want):
            assert torch.equal(a, b)
    assert not sync.any()
