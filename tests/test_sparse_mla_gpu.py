"""GPU parity of the sparse MLA forward against the CPU oracle.

Tolerance of the path's parity bar: out within atol = rtol = 2e-2 (bf16), lse within 1e-3.
"""
import math

import pytest
import torch

from oracle import dsa_oracle as ref

pytestmark = pytest.mark.gpu


def _inputs(B, S, Skv, H, topk, seed, dtype=torch.bfloat16, q_start=None):
    g = torch.Generator().manual_seed(seed)
    q = (torch.randn(B, S, H, 576, generator=g) * 0.5).to(dtype)
    kv = (torch.randn(B, Skv, 1, 576, generator=g) * 0.5).to(dtype)
    idx = ref.causal_sparse_indices(B, S, Skv, topk, seed=seed, q_start=q_start)
    return q, kv, idx


def _check(out, lse, ro, rl):
    torch.testing.assert_close(out.float().cpu(), ro, atol=2e-2, rtol=2e-2)
    torch.testing.assert_close(lse.cpu(), rl, atol=1e-3, rtol=1e-3)


def test_config1_parity(dsa, dev):
    # The CPU-runnable case C1: B=1, Sq=128, Skv=4096, H=16, topk=512.
    q, kv, idx = _inputs(1, 128, 4096, 16, 512, seed=20261201)
    out, lse = dsa.sparse_mla_fwd(q.to(dev), kv.to(dev), idx.to(dev), 1 / math.sqrt(576))
    _check(out, lse, *ref.sparse_mla_fwd(q, kv, idx))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_prefill_shaped_launch(dsa, dev, dtype):
    # 768 rows x 16 heads: more workgroups than the decode-shaped (single-phase) loop takes, so
    # this runs the two-phase software pipeline that the prefill benchmarks use.
    q, kv, idx = _inputs(1, 768, 4096, 16, 256, seed=21, dtype=dtype)
    out, lse = dsa.sparse_mla_fwd(q.to(dev), kv.to(dev), idx.to(dev), 1 / math.sqrt(576))
    _check(out, lse, *ref.sparse_mla_fwd(q, kv, idx))


@pytest.mark.parametrize("H", [32, 48, 64, 128, 160, 256])
def test_head_counts(dsa, dev, H):
    q, kv, idx = _inputs(1, 4, 2048, H, 256, seed=H)
    out, lse = dsa.sparse_mla_fwd(q.to(dev), kv.to(dev), idx.to(dev))
    _check(out, lse, *ref.sparse_mla_fwd(q, kv, idx))


def test_fp16_inputs(dsa, dev):
    q, kv, idx = _inputs(1, 8, 1024, 128, 256, seed=3, dtype=torch.float16)
    out, lse = dsa.sparse_mla_fwd(q.to(dev), kv.to(dev), idx.to(dev))
    assert out.dtype == torch.float16
    _check(out, lse, *ref.sparse_mla_fwd(q, kv, idx))


def test_decode_paged_h128_topk2048(dsa, dev):
    # Decode shape: B sequences x 1 query, 128 heads, topk 2048 over a paged pool.
    B, Skv, H, topk, bs = 4, 8192, 128, 2048, 64
    g = torch.Generator().manual_seed(31)
    q = (torch.randn(B, 1, H, 576, generator=g) * 0.5).to(torch.bfloat16)
    nblk = Skv // bs
    pool = (torch.randn(B * nblk, bs, 1, 576, generator=g) * 0.5).to(torch.bfloat16)
    table = torch.randperm(B * nblk, generator=g).view(B, nblk).to(torch.int32)
    idx = torch.stack([torch.randperm(Skv, generator=g)[:topk] for _ in range(B)]).view(B, 1, 1, topk).to(torch.int32)
    out, lse = dsa.sparse_mla_fwd(q.to(dev), pool.to(dev), idx.to(dev), block_table=table.to(dev))
    _check(out, lse, *ref.sparse_mla_fwd(q, pool, idx, block_table=table))


def test_padding_causal_and_actual_lengths(dsa, dev):
    B, S, Skv, H, topk = 2, 16, 256, 64, 64
    q, kv, idx = _inputs(B, S, Skv, H, topk, seed=5)
    idx[0, 3, 0, 10:] = -1                  # padded slots
    idx[0, 4, 0, :] = -1                    # empty row -> out 0, lse -inf
    idx[1, 5, 0, :8] = Skv - 1              # future positions masked by causality (duplicates dropped)
    idx[1, 5, 0, 1:8] = -1
    ql = torch.tensor([16, 12], dtype=torch.int32)
    kl = torch.tensor([256, 200], dtype=torch.int32)
    out, lse = dsa.sparse_mla_fwd(q.to(dev), kv.to(dev), idx.to(dev), actual_seq_lengths_query=ql.to(dev),
                                  actual_seq_lengths_kv=kl.to(dev))
    ro, rl = ref.sparse_mla_fwd(q, kv, idx, actual_seq_lengths_query=ql.tolist(), actual_seq_lengths_kv=kl.tolist())
    _check(out, lse, ro, rl)
    assert torch.all(out[0, 4].cpu() == 0) and torch.all(torch.isneginf(lse[0, 4].cpu()))


@pytest.mark.parametrize("topk", [40, 300, 1500])
@pytest.mark.parametrize("paged", [False, True])
def test_decode_rows_edges(dsa, dev, topk, paged):
    # At most 8 query rows: the decode kernel (one workgroup per row and 16 heads up to
    # 256 slots, 128-slot chunks and a combine past that).  Padded rows (out 0, lse -inf),
    # key lengths, the causal bound, -1 and out-of-range slots, an empty 128-slot chunk, fp16.
    B, S, Skv, H, bs = 2, 3, 1800, 32, 48
    for dtype in (torch.bfloat16, torch.float16):
        print(f"sparse_mla decode rows topk={topk} paged={paged} {dtype}", flush=True)
        g = torch.Generator().manual_seed(topk + paged)
        q = (torch.randn(B, S, H, 576, generator=g) * 0.5).to(dtype)
        kv = (torch.randn(B, Skv, 1, 576, generator=g) * 0.5).to(dtype)
        idx = torch.stack([torch.randperm(Skv, generator=g)[:topk] for _ in range(B * S)]).view(B, S, 1, topk)
        idx = idx.to(torch.int32)
        idx[0, 0, 0, : topk // 3] = -1                 # leading empty slots (a whole chunk at topk 1500)
        idx[0, 1, 0, 5] = Skv + 7                      # out of range
        if topk > 256:
            idx[1, 0, 0, 128:256] = -1                 # chunk 1 empty
        ql = torch.tensor([3, 2], dtype=torch.int32)   # row (1, 2) padded
        kl = torch.tensor([Skv, 1000], dtype=torch.int32)
        args = dict(actual_seq_lengths_query=ql.to(dev), actual_seq_lengths_kv=kl.to(dev))
        if paged:
            nblk = (Skv + bs - 1) // bs
            table = torch.randperm(B * nblk, generator=g).view(B, nblk).to(torch.int32)
            pool = torch.zeros(B * nblk, bs, 1, 576, dtype=dtype)
            for b in range(B):
                for j in range(nblk):
                    rows = kv[b, j * bs:(j + 1) * bs]
                    pool[table[b, j], :rows.shape[0]] = rows
            out, lse = dsa.sparse_mla_fwd(q.to(dev), pool.to(dev), idx.to(dev), block_table=table.to(dev), **args)
        else:
            out, lse = dsa.sparse_mla_fwd(q.to(dev), kv.to(dev), idx.to(dev), **args)
        ro, rl = ref.sparse_mla_fwd(q, kv, idx, actual_seq_lengths_query=ql.tolist(),
                                    actual_seq_lengths_kv=kl.tolist())
        _check(out, lse, ro, rl)
        assert torch.all(out[1, 2].cpu() == 0) and torch.all(torch.isneginf(lse[1, 2].cpu()))


def test_split_and_unsplit_agree(dsa, dev):
    # 1 token -> the index list is split across workgroups; 512 tokens -> no split.
    q, kv, idx = _inputs(1, 512, 4096, 128, 512, seed=9)
    qd, kvd, idd = q.to(dev), kv.to(dev), idx.to(dev)
    out_all, lse_all = dsa.sparse_mla_fwd(qd, kvd, idd)
    out_one, lse_one = dsa.sparse_mla_fwd(qd[:, 300:301].contiguous(), kvd, idd[:, 300:301].contiguous(),
                                          actual_seq_lengths_query=torch.tensor([1], device=dev),
                                          actual_seq_lengths_kv=torch.tensor([4096 - 511 + 300], device=dev))
    torch.testing.assert_close(out_one.float(), out_all[:, 300:301].float(), atol=1e-2, rtol=1e-2)
    torch.testing.assert_close(lse_one, lse_all[:, 300:301], atol=1e-4, rtol=1e-4)
    ro, rl = ref.sparse_mla_fwd(q[:, 296:304], kv, idx[:, 296:304], actual_seq_lengths_query=[8],
                                actual_seq_lengths_kv=[4096 - 511 + 303])
    _check(out_all[:, 296:304], lse_all[:, 296:304], ro, rl)


def test_single_index_closed_form(dsa, dev):
    q, kv, _ = _inputs(1, 1, 64, 16, 8, seed=1)
    idx = torch.full((1, 1, 1, 64), -1, dtype=torch.int32)
    idx[0, 0, 0, 37] = 21
    out, lse = dsa.sparse_mla_fwd(q.to(dev), kv.to(dev), idx.to(dev))
    assert torch.equal(out[0, 0].cpu(), kv[0, 21, 0, :512].expand(16, 512))
    want = (q[0, 0].double() @ kv[0, 21, 0].double()) / math.sqrt(576)
    torch.testing.assert_close(lse[0, 0].cpu().double(), want, atol=1e-3, rtol=1e-3)


def test_builder_signature(dsa, dev):
    q, kv, idx = _inputs(1, 32, 2048, 128, 256, seed=8)
    kern = dsa.sparse_attention_fwd(heads=128, dim=512, tail_dim=64, topk=256, kv_stride=1)
    out = kern(q.to(dev), kv.to(dev), idx.to(dev))
    ro, _ = ref.sparse_mla_fwd(q, kv, idx)
    torch.testing.assert_close(out.float().cpu(), ro, atol=2e-2, rtol=2e-2)


def _ramp_inputs(jump_log2, H=128, S=2, topk=256, Skv=1024, seed=12):
    """Scores of later index slots exceed the first tile's by ~jump_log2 (base 2)."""
    g = torch.Generator().manual_seed(seed)
    q = torch.zeros(1, S, H, 576)
    q[..., :64] = 1.0
    q += torch.randn(1, S, H, 576, generator=g) * 0.01
    kv = torch.randn(1, Skv, 1, 576, generator=g) * 0.5
    # t = sm_scale * log2(e) * q.k ~= 64 * c / 24 * 1.4427 for a row with c in its first 64 dims
    c = jump_log2 / (64 / 24 * 1.4426950408889634)
    kv[0, 512:, 0, :64] = c
    idx = torch.empty(1, S, 1, topk, dtype=torch.int32)
    for s in range(S):
        low = torch.randperm(512, generator=g)[:topk // 2]
        high = 512 + torch.randperm(Skv - 512 - S, generator=g)[:topk // 2]
        idx[0, s, 0] = torch.cat([low, high]).to(torch.int32)  # first tiles all low
    return q.to(torch.bfloat16), kv.to(torch.bfloat16), idx


@pytest.mark.parametrize("jump", [40.0, 200.0])  # within the fast path's headroom / beyond it (exact fallback)
@pytest.mark.parametrize("S", [1, 300])          # split index list (+combine) / one workgroup per row
def test_large_score_jumps(dsa, dev, jump, S):
    q, kv, idx = _ramp_inputs(jump, S=S)
    out, lse = dsa.sparse_mla_fwd(q.to(dev), kv.to(dev), idx.to(dev))
    ro, rl = ref.sparse_mla_fwd(q, kv, idx)
    assert torch.isfinite(out.float()).all() and torch.isfinite(lse).all()
    torch.testing.assert_close(out.float().cpu(), ro, atol=2e-2, rtol=2e-2)
    torch.testing.assert_close(lse.cpu(), rl, atol=1e-3, rtol=1e-3)


def _ring_depth(dsa, B, S, H, topk):
    """Stages the 64-head kernel's launch picks: 3 where the grid has at most 256 workgroups of more
    than 512 slots each.  The split count is read off the workspace (split partials of 512 16-bit
    values and an fp32 LSE per row and head, and 256 bytes)."""
    ws = dsa.load_library().dsa_sparse_mla_workspace_size(B, S, H, topk)
    splits = (ws - 256) // (B * S * H * (512 * 2 + 4)) if ws else 1
    per = math.ceil(math.ceil(topk / splits) / 32) * 32
    return 3 if B * S * splits <= 256 and per > 512 else 2


@pytest.mark.parametrize("B,S,H,topk,paged,stages", [
    (1, 9, 16, 31, False, 2), (3, 3, 48, 1100, True, 2), (2, 130, 64, 33, True, 2), (120, 1, 32, 1100, True, 2),
    (1, 120, 64, 1088, False, 2), (1, 300, 48, 2049, False, 2), (1, 128, 64, 2048, False, 3),
    (2, 64, 16, 2048, True, 3), (1, 256, 48, 1100, False, 3), (2, 128, 64, 545, True, 3)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_up_to_64_heads_tile_and_stage_edges(dsa, dev, B, S, H, topk, paged, stages, dtype):
    """The 64-head kernel: both ring depths, splits, ragged last tiles, empty tiles, heads short of 64.

    Slots are emptied by -1 and, in a paged cache, by a block of a negative number; key 0 is NaN and
    never selected, so an empty slot that reads a key instead of zeros shows.
    """
    assert _ring_depth(dsa, B, S, H, topk) == stages
    g = torch.Generator().manual_seed(B * S + H + topk)
    skv, bs = 2112, 64
    q = (torch.randn(B, S, H, 576, generator=g) * 0.5).to(dtype)
    kv = (torch.randn(1, skv, 1, 576, generator=g) * 0.5).to(dtype).expand(B, -1, -1, -1).contiguous()
    idx = torch.stack([1 + torch.randperm(skv - 1, generator=g)[:topk] for _ in range(B * S)])
    idx = idx.view(B, S, 1, topk).to(torch.int32)
    idx[:, ::2, :, 3::5] = -1
    idx[:, 1::3, :, :min(40, topk - 1)] = -1  # the first tile empty
    idx[:, 2::4, :, topk // 2:] = -1
    idx[0, S - 1] = -1 if S > 3 else idx[0, S - 1]
    want_idx, kw = idx, {}
    kv[:, 0] = float("nan")
    if paged:
        # One pool; each sequence its own order of the blocks, block 5 of every sequence missing.
        pool = kv[0].view(skv // bs, bs, 1, 576)
        table = torch.arange(skv // bs, dtype=torch.int32).expand(B, -1).contiguous()
        table[:, 5] = -3
        want_idx = torch.where((idx >= 0) & (idx // bs == 5), torch.full_like(idx, -1), idx)
        kw = dict(block_table=table.to(dev))
    out, lse = dsa.sparse_mla_fwd(q.to(dev), (pool if paged else kv).to(dev), idx.to(dev), 1 / math.sqrt(576), **kw)
    kv[:, 0] = 0
    _check(out, lse, *ref.sparse_mla_fwd(q, kv, want_idx, 1 / math.sqrt(576)))


@pytest.mark.parametrize("H,S,paged,topk", [(16, 300, False, 256), (48, 20, True, 256), (64, 260, True, 256),
                                            (64, 256, True, 1000), (16, 256, False, 1000)])
@pytest.mark.parametrize("jump", [40.0, 200.0])
def test_up_to_64_heads_large_score_jumps(dsa, dev, jump, H, S, paged, topk):
    """The 64-head kernel's headroom and its exact fallback, whose slot table is made after the loop
    (topk 1000: from three stages)."""
    assert _ring_depth(dsa, 1, S, H, topk) == (3 if topk == 1000 else 2)
    q, kv, idx = _ramp_inputs(jump, H=H, S=S, topk=topk, Skv=2048 if topk == 1000 else 1024)
    src, kw = kv, {}
    if paged:
        n = kv.shape[1] // 64
        table = torch.randperm(n, generator=torch.Generator().manual_seed(S)).view(1, n).to(torch.int32)
        src = torch.empty(n, 64, 1, 576, dtype=kv.dtype)
        src[table[0].long()] = kv.view(n, 64, 1, 576)
        kw = dict(block_table=table.to(dev))
    out, lse = dsa.sparse_mla_fwd(q.to(dev), src.to(dev), idx.to(dev), **kw)
    ro, rl = ref.sparse_mla_fwd(q, kv, idx)
    torch.testing.assert_close(out.float().cpu(), ro, atol=2e-2, rtol=2e-2)
    torch.testing.assert_close(lse.cpu(), rl, atol=1e-3, rtol=1e-3)


@pytest.mark.parametrize("T", [1, 2, 8])
@pytest.mark.parametrize("topk", [40, 300])  # one workgroup per row and 16 heads / chunks
@pytest.mark.parametrize("form", ["contiguous", "paged", "parts", "parts_paged"])
def test_decode_rows_read_no_key_for_empty_slots(dsa, dev, T, topk, form):
    """Up to 8 rows: the cache's first row is NaN and never selected; -1 slots, slots past the causal
    bound or the end of the list, and blocks without a valid slot must not bring it in."""
    g = torch.Generator().manual_seed(100 * T + topk)
    H, skv, bs, dt = 32, 640, 64, torch.bfloat16
    apart = form.startswith("parts")
    B, S = (1, T) if apart else (T, 1)
    q = (torch.randn(B, S, H, 576, generator=g) * 0.5).to(dt)
    kv = (torch.randn(B, skv, 1, 576, generator=g) * 0.5).to(dt)
    idx = torch.stack([1 + torch.randperm(skv - 1, generator=g)[:topk] for _ in range(B * S)]).to(torch.int32)
    idx[:, ::3] = -1
    idx[:, 16:33] = -1                                   # a whole block, then past the key length
    idx = idx.view(B, S, 1, topk)
    kl = torch.tensor([skv - 40] * B, dtype=torch.int32)
    want, want_lse = ref.sparse_mla_fwd(q, kv, idx, 0.05, actual_seq_lengths_kv=kl.tolist())
    kv[0, 0] = float("nan")
    src, kw = kv, {}
    if form.endswith("paged"):
        n = skv // bs
        perm = 1 + torch.randperm(B * n, generator=g)
        src = torch.full((B * n + 1, bs, 1, 576), float("nan"), dtype=dt)  # block 0 holds no key
        src[perm] = kv.view(B * n, bs, 1, 576)
        kw = dict(block_table=perm.view(B, n).to(torch.int32).to(dev))
    if apart:
        cut = lambda t: (t[..., :512].contiguous().to(dev), t[..., 512:].contiguous().to(dev))  # noqa: E731
        (ql, qr), (kc, kr) = cut(q[0]), cut(src)
        out = dsa.sparse_attn_tilelang(ql, kc, kc, idx[0].to(dev), 0.05, 1, None, kl.to(dev), query_rope=qr,
                                       key_rope=kr, sparse_mode=3, **kw)
        torch.testing.assert_close(out[None].float().cpu(), want, atol=2e-2, rtol=2e-2)
    else:
        out, lse = dsa.sparse_mla_fwd(q.to(dev), src.to(dev), idx.to(dev), 0.05, actual_seq_lengths_kv=kl.to(dev), **kw)
        _check(out, lse, want, want_lse)
