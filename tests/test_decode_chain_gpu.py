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


def _launches(sync):
    """The launches counted in the hand-off words (their first word; the
    blocks' arrivals, on the 33 lines after it, are put back to zero)."""
    words = sync.view(torch.int32)
    assert not words[1:34 * 32].any()
    return words[0].item()


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
    merge and the next layer; three launches in a row, each of which advances
    the launch number."""
    from qwen3_engine_from_scratch_amd.PagedKVcache import (KVCachePool, PagedKVCache,
                                                            reserve_pages_bulk, set_seq_lens_bulk)
    from qwen3_engine_from_scratch_amd.kernels.model_ops import (
        decode_chain, decode_chain_ok, decode_chain_sync, decode_linear, decode_qkv_rope, embed_ss)
    from qwen3_engine_from_scratch_amd.kernels.paged_attention import (
        paged_attention_decode_hip, paged_attention_decode_partials_hip,
        paged_decode_workspace_bytes)
    from qwen3_engine_from_scratch_amd.kernels.pre_attention import rope_tables

    if not decode_chain_ok(M, hidden, inter, hq, hkv):
        pytest.skip("the grid does not fit this device at once")
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
        assert _launches(sync) == i + 1


@pytest.mark.parametrize("hidden, hq, hkv", [(1024, 16, 8), (64, 3, 1), (640, 18, 9)])
@pytest.mark.parametrize("M", [1, 16, 17, 33, 64])
def test_qkv_half_heads_same_bits(gpu, hidden, hq, hkv, M):
    """decode_qkv_rope on two workgroups per head against one: rows past a
    16-row block's end, rows outside the resident table, a row stride of the
    residual stream that is not its width; every launch is counted."""
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
    assert _launches(sync) == 3


class _Chain:
    """A layer's dense work after an attention over M sequences, with the next
    layer's qkv, on a pool, a residual stream and hand-off words of its own."""

    def __init__(self, gpu, M, hidden=1024, inter=3072, hq=16, hkv=8, seed=0):
        from qwen3_engine_from_scratch_amd.PagedKVcache import (KVCachePool, PagedKVCache,
                                                                reserve_pages_bulk,
                                                                set_seq_lens_bulk)
        from qwen3_engine_from_scratch_amd.kernels.model_ops import (decode_chain_ok,
                                                                     decode_chain_sync, embed_ss)
        from qwen3_engine_from_scratch_amd.kernels.paged_attention import (
            paged_decode_workspace_bytes)
        from qwen3_engine_from_scratch_amd.kernels.pre_attention import rope_tables

        if not decode_chain_ok(M, hidden, inter, hq, hkv):
            pytest.skip("the grid does not fit this device at once")
        g = torch.Generator(device=gpu).manual_seed(seed)
        self.M, self.hq, self.hkv = M, hq, hkv
        self.a, self.b = (_layer(g, gpu, hidden, inter, hq, hkv) for _ in range(2))
        lens = [(331 * i + 900) % 1500 + 1 for i in range(M)]
        self.pool = pool = KVCachePool(sum(n // 16 + 1 for n in lens) + 2, 2, 16, hkv, 128,
                                       device=gpu, dtype=torch.bfloat16, max_seq_len=2048,
                                       max_requests=M + 1)
        caches = [PagedKVCache(pool) for _ in range(M)]
        reserve_pages_bulk(caches, [n + 1 for n in lens])
        for c, n in zip(caches, lens):
            c.seq_len = n
        set_seq_lens_bulk(caches)
        self.rows = torch.tensor([c.row_id for c in caches], dtype=torch.int32, device=gpu)
        pool.k_buffer.normal_(generator=g)
        pool.v_buffer.normal_(generator=g)
        self.tables = rope_tables(128, 1e6, 2048, device=gpu)
        self.h0, self.ss0 = embed_ss(
            torch.arange(M, device=gpu),
            torch.randn(64, hidden, generator=g, device=gpu).bfloat16())
        self.q0 = torch.randn(M, hq, 128, generator=g, device=gpu).bfloat16()
        self.ws = torch.zeros(
            paged_decode_workspace_bytes(M, hq, hkv, 128, pool.block_table_2d.shape[1], 16),
            dtype=torch.uint8, device=gpu)
        self.sync = decode_chain_sync(gpu)

    def run(self, merge=True, nxt=True, **kw):
        """One pass from the same inputs, with no synchronisation."""
        from qwen3_engine_from_scratch_amd.kernels.model_ops import decode_chain
        from qwen3_engine_from_scratch_amd.kernels.paged_attention import (
            paged_attention_decode_hip, paged_attention_decode_partials_hip)

        kv = (self.q0, self.pool.k_buffer[:, 0], self.pool.v_buffer[:, 0],
              self.pool.block_table_2d, self.pool.seq_lens, self.rows, 16)
        o = (paged_attention_decode_partials_hip(*kv, self.ws) if merge
             else paged_attention_decode_hip(*kv, workspace=self.ws))
        h, ss = self.h0.clone(), self.ss0.clone()
        mid, ss_mid = torch.empty_like(h), torch.empty_like(ss)
        q = decode_chain(o, h, mid, ss, ss_mid, self.a, 1e-6, self.hq, self.hkv, self.sync,
                         attn_workspace=self.ws if merge else None,
                         next_layer=self.b if nxt else None, head_eps=1e-6,
                         cos_table=self.tables[0], sin_table=self.tables[1], pool=self.pool,
                         next_idx=1, row_ids=self.rows, **kw)
        out = [o, h, ss, mid, ss_mid, self.pool.k_buffer[:, 1].clone(),
               self.pool.v_buffer[:, 1].clone()]
        return out + ([q] if nxt else [])


def _same(x, y):
    """Bit for bit (NaNs too)."""
    return all(torch.equal(a.view(torch.int16), b.view(torch.int16)) for a, b in zip(x, y))


@pytest.mark.parametrize("M", [1, 7, 16])
@pytest.mark.parametrize("merge, nxt", [(True, True), (False, True), (True, False)])
@pytest.mark.parametrize("ticks", [-1, 1, 500])
def test_chain_waits_that_are_not_answered(gpu, M, merge, nxt, ticks):
    """Every wait gives up at its first unanswered poll, or soon after it: the
    blocks run one another's work, several of them the same, with the same
    bits, in place, launch after launch."""
    c = _Chain(gpu, M, seed=M)
    announce(f"decode chain unanswered waits M={M} merge={merge} next={nxt} ticks={ticks}")
    want = c.run(merge, nxt)
    for i in range(4):
        assert _same(c.run(merge, nxt, wait_ticks=ticks), want), f"launch {i}"
    assert _same(c.run(merge, nxt), want)
    assert _launches(c.sync) == 6


@pytest.mark.parametrize("hidden, hq, hkv", [(1024, 16, 8), (64, 3, 1)])
@pytest.mark.parametrize("M", [1, 17, 64])
@pytest.mark.parametrize("ticks", [-1, 1])
def test_qkv_halves_that_do_not_come(gpu, hidden, hq, hkv, M, ticks):
    """The sums of a head's other half do not come in time: a block runs that
    half itself, with the same bits."""
    from types import SimpleNamespace as NS

    from qwen3_engine_from_scratch_amd.kernels.model_ops import (decode_chain_sync,
                                                                 decode_qkv_rope, embed_ss)
    from qwen3_engine_from_scratch_amd.kernels.pre_attention import rope_tables

    g = torch.Generator(device=gpu).manual_seed(M)
    layer = _layer(g, gpu, hidden, 128, hq, hkv)
    at = layer.self_attn
    pool = NS(k_buffer=torch.zeros(M, 1, hkv, 16, 128, dtype=torch.bfloat16, device=gpu),
              v_buffer=torch.zeros(M, 1, hkv, 16, 128, dtype=torch.bfloat16, device=gpu),
              block_table_2d=torch.arange(M, dtype=torch.int32, device=gpu).view(M, 1),
              seq_lens=(torch.arange(M, device=gpu) % 16).to(torch.int32))
    cos, sin = rope_tables(128, 1e6, 64, device=gpu)
    h, ss = embed_ss(torch.arange(M, device=gpu),
                     torch.randn(64, hidden, generator=g, device=gpu).bfloat16())
    sync = decode_chain_sync(gpu)
    announce(f"qkv halves that do not come M={M} hidden={hidden} ticks={ticks}")

    def run(**kw):
        pool.k_buffer.zero_()
        pool.v_buffer.zero_()
        q = decode_qkv_rope(h, ss, layer.input_layernorm.weight, 1e-6, at.qkv_proj.weight, hq, hkv,
                            at.q_norm.weight, at.k_norm.weight, 1e-6, cos, sin, pool, 0, None, **kw)
        return q, pool.k_buffer.clone(), pool.v_buffer.clone()

    want = run()
    for _ in range(3):
        assert _same(run(sync=sync, wait_ticks=ticks), want)
    assert _launches(sync) == 3


def test_chain_launches_that_overlap(gpu):
    """Four models' launches in flight at once, each with hand-off words of its
    own (together more blocks than are resident), waiting as long as they like
    and giving up at once: every one has its own bits."""
    chains = [_Chain(gpu, M, seed=20 + M) for M in (16, 1, 7, 16)]
    want = [c.run() for c in chains]
    streams = [torch.cuda.Stream() for _ in chains]
    torch.cuda.synchronize()
    announce("decode chain: four launches in flight")
    for ticks in (0, -1):
        got = [[] for _ in chains]
        for _ in range(6):
            for c, s, out in zip(chains, streams, got):
                with torch.cuda.stream(s):
                    out.append(c.run(wait_ticks=ticks))
        torch.cuda.synchronize()
        for i, (outs, w) in enumerate(zip(got, want)):
            assert all(_same(x, w) for x in outs), f"stream {i}, ticks {ticks}"
    assert [_launches(c.sync) for c in chains] == [13] * 4


@pytest.mark.parametrize("value", ["nan", "-nan", "inf", "big"])
def test_chain_non_finite_activations(gpu, value):
    """A residual row that is not finite (or whose squares are not) goes through
    the handed-on sums as through the separate kernels: NaN sums of either
    sign are sums, and the other rows have their bits."""
    from qwen3_engine_from_scratch_amd.kernels.model_ops import decode_qkv_rope

    c = _Chain(gpu, 7, seed=5)
    announce(f"decode chain: {value} in the residual stream")
    x = {"nan": float("nan"), "-nan": float("nan"), "inf": float("inf"), "big": 3e38}[value]
    want = c.run()
    c.h0[2, 5] = x
    if value == "-nan":
        c.h0.view(torch.int16)[2, 5] = -1  # every bit set
    c.ss0[2] = c.h0[2].float().square().view(-1, 16).sum(-1)
    got = c.run(nxt=False)
    h, ss = got[1], got[2]
    assert not torch.isfinite(ss[2]).all()
    keep = [0, 1, 3, 4, 5, 6]
    assert _same([h[keep], ss[keep]], [want[1][keep], want[2][keep]])
    # the next layer's heads from that stream, in one workgroup each and in two
    at = c.b.self_attn

    def qkv(**kw):
        q = decode_qkv_rope(h, ss, c.b.input_layernorm.weight, 1e-6, at.qkv_proj.weight, 16, 8,
                            at.q_norm.weight, at.k_norm.weight, 1e-6, *c.tables, c.pool, 1, c.rows,
                            **kw)
        return q, c.pool.k_buffer[:, 1].clone(), c.pool.v_buffer[:, 1].clone()

    one, two = qkv(), qkv(sync=c.sync)
    for a, b in zip(one, two):
        assert torch.equal(a.isnan(), b.isnan()) and torch.equal(a.nan_to_num(), b.nan_to_num())
    q = c.run()[-1]
    assert torch.equal(q.isnan(), one[0].isnan())
    assert torch.equal(q.nan_to_num(), one[0].nan_to_num())


def test_chain_refuses_wrong_tensors(gpu):
    """What the separate wrappers refuse: a norm of another length or type, and
    hand-off words that are too few."""
    from types import SimpleNamespace as NS

    c = _Chain(gpu, 2)
    norm = c.a.post_attention_layernorm
    for bad in (norm.weight[:512], norm.weight.float(), torch.stack([norm.weight] * 2, 1)[:, 0]):
        c.a.post_attention_layernorm = NS(weight=bad)
        with pytest.raises(AssertionError):
            c.run()
    c.a.post_attention_layernorm = norm
    c.b.self_attn.q_norm, q_norm = NS(weight=c.b.self_attn.q_norm.weight[:64]), c.b.self_attn.q_norm
    with pytest.raises(AssertionError):
        c.run()
    c.b.self_attn.q_norm = q_norm
    c.sync, sync = c.sync[:-16], c.sync
    with pytest.raises(AssertionError):
        c.run()
    c.sync = sync
    c.run()


def test_qkv_rows_that_coincide(gpu):
    """Rows that are one row (stride 0) go to the one-workgroup form, hand-off
    words or not."""
    from qwen3_engine_from_scratch_amd.kernels.model_ops import decode_qkv_rope

    c = _Chain(gpu, 3)
    at = c.b.self_attn
    h, ss = c.h0[:1].expand(3, -1), c.ss0[:1].expand(3, -1).contiguous()

    def qkv(x, **kw):
        return decode_qkv_rope(x, ss, c.b.input_layernorm.weight, 1e-6, at.qkv_proj.weight, 16, 8,
                               at.q_norm.weight, at.k_norm.weight, 1e-6, *c.tables, c.pool, 1,
                               c.rows, **kw)

    assert torch.equal(qkv(h, sync=c.sync), qkv(h.contiguous()))
