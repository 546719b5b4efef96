"""GPU parity of the gathered-index V4 attention with sinks (``sparse_attn``) and of the
SFA decode entry ``sparse_attn_tilelang`` against the CPU oracle.

``sparse_attn`` (examples/deepseek_v4/sparse_attention.py:171-241): the reference
test's own shape (b=1, m=256, n=256, h=64, d=512, topk=128, indices from randint, so
duplicates occur, bf16 randn inputs, fp32 sinks), plus -1 slots, batches, 128 heads,
fp16 and the split path (long index lists on few rows).  The output is the fp32
accumulator, as the reference kernel writes it (sparse_attention.py:56): out within
rtol = 2e-3 of the exact oracle, atol 2e-3 for fp16 and 4e-3 for bf16 (the reference
test's own bar is 1e-2; the probabilities enter P V rounded to the input dtype, which on
unit-scale data moves an output by up to ~2e-3 for bf16), and most elements not
representable in 16 bits: a 16-bit rounding of the output (2^-9 relative for bf16) would
slip under those bars, so that check is what sees it.  LSE within 1e-3 of the exact oracle.

``sparse_attn_tilelang`` (examples/sparse_flash_attention/bench_sfa/bench_sfa.py:10-120):
the benchmark's inputs (T=1, 128 heads, 512 + 64 rope, paged KV in 128-row blocks,
topk 2048 drawn by topk of uniform noise over act_kv_s = 2560, scale 0.5, values of
std 0.5), out within atol = rtol = 2e-2 of the exact oracle (the benchmark itself
compares two kernels at 1e-2).
"""
import pytest
import torch

from oracle import dsa_oracle as ref

pytestmark = pytest.mark.gpu


def _inputs(b, m, n, h, d, topk, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    q = torch.randn((b, m, h, d), generator=g).to(dtype)
    kv = torch.randn((b, n, d), generator=g).to(dtype)
    sink = torch.randn((h,), generator=g)
    idx = torch.randint(0, n, (b, m, topk), generator=g, dtype=torch.int32)
    return q, kv, sink, idx


def _run(dsa, dev, q, kv, sink, idx, scale):
    out = dsa.sparse_attn(q.to(dev), kv.to(dev), None if sink is None else sink.to(dev), idx.to(dev), scale)
    torch.cuda.synchronize()
    return out.cpu()


def _check_out(out, want, dtype):
    """fp32 output within the bar of the oracle, and not a 16-bit value widened."""
    assert out.dtype == torch.float32
    torch.testing.assert_close(out, want, rtol=2e-3, atol=4e-3 if dtype == torch.bfloat16 else 2e-3)
    nz = out != 0
    if nz.sum() > 0:
        exact16 = (out[nz].to(dtype).float() == out[nz]).float().mean().item()
        assert exact16 < 0.05, f"{exact16:.3f} of the outputs are {dtype} values"


def _lse(dsa, dev, q, kv, sink, idx, scale):
    """The LSE the kernel writes, read through the C ABI."""
    b, m, h, d = q.shape
    lib = dsa.load_library()
    qd, kvd, idxd = q.to(dev), kv.to(dev), idx.to(dev)
    sk = None if sink is None else sink.to(dev)
    out = torch.empty((b, m, h, d), dtype=torch.float32, device=dev)
    lse = torch.empty((b, m, h), dtype=torch.float32, device=dev)
    nbytes = lib.dsa_sparse_attn_sink_workspace_size(b, m, h, idx.shape[2])
    ws = torch.empty((max(nbytes, 1),), dtype=torch.uint8, device=dev)
    kind = 1 if q.dtype == torch.bfloat16 else 2
    rc = lib.dsa_sparse_attn_sink(kind, qd.data_ptr(), kvd.data_ptr(), idxd.data_ptr(), b, m, h, kv.shape[1], d,
                                  idx.shape[2], None if sk is None else sk.data_ptr(), scale, out.data_ptr(),
                                  lse.data_ptr(), ws.data_ptr(), nbytes, torch.cuda.current_stream(dev).cuda_stream)
    assert rc == 0
    torch.cuda.synchronize()
    return lse.cpu()


def test_reference_test_shape(dsa, dev):
    """sparse_attention.py:216-241: shape 1, bf16, scale 512**-0.5 (the reference's bar is 1e-2)."""
    print("sparse_attn reference shape b=1 m=256 n=256 h=64 topk=128", flush=True)
    q, kv, sink, idx = _inputs(1, 256, 256, 64, 512, 128, torch.bfloat16, 41)
    scale = 512 ** -0.5
    out = _run(dsa, dev, q, kv, sink, idx, scale)
    want, want_lse = ref.sparse_attn_sink(q, kv, sink, idx, scale)
    assert out.shape == (1, 256, 64, 512)
    _check_out(out, want, torch.bfloat16)
    torch.testing.assert_close(_lse(dsa, dev, q, kv, sink, idx, scale), want_lse, rtol=1e-3, atol=1e-3)


def test_reference_small_shape_via_builder(dsa, dev):
    """Shape 2 of the reference test (b=1, m=6, n=6, h=16, topk=6) through the builder."""
    q, kv, sink, idx = _inputs(1, 6, 6, 16, 512, 6, torch.bfloat16, 42)
    kernel = dsa.sparse_attn_kernel(h=16, d=512, scale=512 ** -0.5)
    out = kernel(q.to(dev), kv.to(dev), sink.to(dev), idx.to(dev)).cpu()
    want, _ = ref.sparse_attn_sink(q, kv, sink, idx, 512 ** -0.5)
    _check_out(out, want, torch.bfloat16)
    # Default scale is 1/sqrt(d), as in the reference builder.
    out2 = dsa.sparse_attn_kernel(h=16, d=512)(q.to(dev), kv.to(dev), sink.to(dev), idx.to(dev)).cpu()
    torch.testing.assert_close(out2, out, rtol=0, atol=0)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_masked_slots_batches_and_heads(dsa, dev, dtype):
    """-1 slots (masked), out-of-range slots (masked), two batches (row bases b*n), 128 heads."""
    print(f"sparse_attn masked b=2 h=128 {dtype}", flush=True)
    q, kv, sink, idx = _inputs(2, 40, 300, 128, 512, 200, dtype, 43)
    g = torch.Generator().manual_seed(44)
    drop = torch.rand(idx.shape, generator=g) < 0.3
    idx = torch.where(drop, torch.full_like(idx, -1), idx)
    idx[0, 0, :] = -1                      # no valid slot: out 0, lse = sink
    idx[1, 1, 5] = 300                     # past n: masked
    scale = 0.05
    out = _run(dsa, dev, q, kv, sink, idx, scale)
    want, want_lse = ref.sparse_attn_sink(q, kv, sink, idx, scale)
    _check_out(out, want, dtype)
    torch.testing.assert_close(_lse(dsa, dev, q, kv, sink, idx, scale), want_lse, rtol=1e-3, atol=1e-3)
    assert torch.count_nonzero(out[0, 0]) == 0


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_decode_rows_masked_slots(dsa, dev, dtype):
    """At most 8 query rows with at most 256 slots each: the decode-shaped kernel in one workgroup
    per row and 16 heads (slots across the waves); -1 and out-of-range slots, an all-empty row, a
    block of 16 slots with none valid."""
    print(f"sparse_attn decode rows b=2 m=3 topk=150 {dtype}", flush=True)
    q, kv, sink, idx = _inputs(2, 3, 300, 32, 512, 150, dtype, 46)
    g = torch.Generator().manual_seed(47)
    drop = torch.rand(idx.shape, generator=g) < 0.3
    idx = torch.where(drop, torch.full_like(idx, -1), idx)
    idx[0, 1, :] = -1                      # no valid slot: out 0, lse = sink
    idx[1, 0, 16:32] = -1                  # a whole 16-slot block masked
    idx[1, 2, 7] = 300                     # past n: masked
    scale = 0.05
    for sk in (sink, None):
        out = _run(dsa, dev, q, kv, sk, idx, scale)
        want, want_lse = ref.sparse_attn_sink(q, kv, sk, idx, scale)
        _check_out(out, want, dtype)
        torch.testing.assert_close(_lse(dsa, dev, q, kv, sk, idx, scale), want_lse, rtol=1e-3, atol=1e-3)
        assert torch.count_nonzero(out[0, 1]) == 0


@pytest.mark.parametrize("m,topk", [(1, 150), (3, 150), (4, 1000)])
def test_decode_rows_read_no_key_for_empty_slots(dsa, dev, m, topk):
    """At most 8 query rows: key 0 is NaN and never selected; -1 slots and those past the list's end
    must not bring it in."""
    print(f"sparse_attn decode rows, NaN in key 0: b=2 m={m} topk={topk}", flush=True)
    q, kv, sink, idx = _inputs(2, m, 300, 32, 512, topk, torch.bfloat16, 48)
    idx = idx.clamp(min=1)
    idx[:, :, ::3] = -1
    idx[1, 0, 16:32] = -1
    want, want_lse = ref.sparse_attn_sink(q, kv, sink, idx, 0.05)
    kv[0, 0] = float("nan")
    _check_out(_run(dsa, dev, q, kv, sink, idx, 0.05), want, torch.bfloat16)
    torch.testing.assert_close(_lse(dsa, dev, q, kv, sink, idx, 0.05), want_lse, rtol=1e-3, atol=1e-3)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_decode_rows_chunked(dsa, dev, dtype):
    """At most 8 query rows with 257..1024 slots: the decode kernel in 128-slot chunks whose
    partials a combine kernel merges (sinks join there); an all-empty row, a chunk with no valid
    slot, a last chunk that is partly past the list."""
    print(f"sparse_attn decode chunks b=2 m=2 topk=600 {dtype}", flush=True)
    q, kv, sink, idx = _inputs(2, 2, 900, 64, 512, 600, dtype, 48)
    idx[0, 1, :] = -1                      # no valid slot: out 0, lse = sink
    idx[1, 0, 128:256] = -1                # chunk 1 empty
    idx[1, 1, 590:] = 900                  # past n: masked
    scale = 0.05
    for sk in (sink, None):
        out = _run(dsa, dev, q, kv, sk, idx, scale)
        want, want_lse = ref.sparse_attn_sink(q, kv, sk, idx, scale)
        _check_out(out, want, dtype)
        torch.testing.assert_close(_lse(dsa, dev, q, kv, sk, idx, scale), want_lse, rtol=1e-3, atol=1e-3)
        assert torch.count_nonzero(out[0, 1]) == 0


def test_split_path_and_no_sink(dsa, dev):
    """Few rows with long index lists take the split + combine path (sinks join in the combine)."""
    print("sparse_attn split path b=2 m=1 topk=4096", flush=True)
    q, kv, sink, idx = _inputs(2, 1, 5000, 64, 512, 4096, torch.bfloat16, 45)
    scale = 512 ** -0.5
    for sk in (sink, None):
        out = _run(dsa, dev, q, kv, sk, idx, scale)
        want, want_lse = ref.sparse_attn_sink(q, kv, sk, idx, scale)
        _check_out(out, want, torch.bfloat16)
        torch.testing.assert_close(_lse(dsa, dev, q, kv, sk, idx, scale), want_lse, rtol=1e-3, atol=1e-3)


@pytest.mark.parametrize("jump", [40.0, 200.0])  # within the fixed reference's headroom / beyond it
def test_row_lists_large_score_jumps(dsa, dev, jump):
    """40 rows of 64 heads (the two-stage row-list kernel) whose last four tiles score ~jump (base 2)
    above the first four: within the bf16 headroom of the fixed reference max, and beyond it, where
    the workgroup recomputes exactly (its scratch and flags in the two-stage LDS layout)."""
    b, m, n, h, d, topk = 1, 40, 1024, 64, 512, 256
    g = torch.Generator().manual_seed(21)
    q = torch.zeros(b, m, h, d)
    q[..., :64] = 1.0
    q += torch.randn(b, m, h, d, generator=g) * 0.01
    kv = torch.randn(b, n, d, generator=g) * 0.5
    scale = 512 ** -0.5
    # base-2 score = scale * log2(e) * q.k ~= 64 * c * scale * log2(e) for a row with c in its first 64 dims
    kv[0, 512:, :64] = jump / (64 * scale * 1.4426950408889634)
    idx = torch.empty(b, m, topk, dtype=torch.int32)
    for t in range(m):
        low = torch.randperm(512, generator=g)[:topk // 2]
        high = 512 + torch.randperm(512, generator=g)[:topk // 2]
        idx[0, t] = torch.cat([low, high]).to(torch.int32)  # the first four tiles all low
    sink = torch.randn(h, generator=g)
    q, kv = q.to(torch.bfloat16), kv.to(torch.bfloat16)
    print(f"sparse_attn row lists b=1 m=40 h=64 topk=256 jump={jump}", flush=True)
    out = _run(dsa, dev, q, kv, sink, idx, scale)
    want, want_lse = ref.sparse_attn_sink(q, kv, sink, idx, scale)
    assert torch.isfinite(out).all()
    torch.testing.assert_close(out, want, atol=2e-2, rtol=2e-2)
    torch.testing.assert_close(_lse(dsa, dev, q, kv, sink, idx, scale), want_lse, rtol=1e-3, atol=1e-3)


def test_rejects_bad_shapes(dsa, dev):
    q, kv, sink, idx = _inputs(1, 2, 8, 16, 512, 4, torch.bfloat16, 46)
    with pytest.raises(ValueError):
        dsa.sparse_attn(q[..., :256].contiguous().to(dev), kv[..., :256].contiguous().to(dev), sink.to(dev),
                        idx.to(dev), 0.1)
    with pytest.raises(ValueError):
        dsa.sparse_attn(q.to(dev), kv.to(dev), sink[:8].to(dev), idx.to(dev), 0.1)
    with pytest.raises(ValueError):
        dsa.sparse_attn_kernel(h=16, d=256)


# ------------------------------------------------------------- sparse_attn_tilelang
def _bench_sfa_inputs(T, KV_S, act_kv_s, Q_N, topk, block_size, seed):
    """bench_sfa.py:19-45 with a CPU generator."""
    g = torch.Generator().manual_seed(seed)
    nb = KV_S // block_size
    query = (torch.randn((T, Q_N, 512), generator=g) * 0.5).to(torch.bfloat16)
    key = (torch.randn((nb, block_size, 1, 512), generator=g) * 0.5).to(torch.bfloat16)
    query_rope = (torch.randn((T, Q_N, 64), generator=g) * 0.5).to(torch.bfloat16)
    key_rope = (torch.randn((nb, block_size, 1, 64), generator=g) * 0.5).to(torch.bfloat16)
    _, ind = torch.topk(torch.rand((T, 1, act_kv_s), generator=g), topk, dim=-1)
    block_table = torch.arange(nb, dtype=torch.int32).view(1, nb)
    return query, key, query_rope, key_rope, ind.to(torch.int32), block_table


@pytest.mark.parametrize("KV_S,T,sparse_mode", [(2560, 1, 0), (6400, 1, 0), (6400, 4, 3)])
def test_sparse_attn_tilelang_bench_sfa(dsa, dev, KV_S, T, sparse_mode):
    print(f"sparse_attn_tilelang KV_S={KV_S} T={T} mode={sparse_mode}", flush=True)
    act_kv_s, block_size = 2560, 128
    query, key, qr, kr, ind, bt = _bench_sfa_inputs(T, KV_S, act_kv_s, 128, 2048, block_size, 47 + KV_S + T)
    aq = torch.tensor([T], dtype=torch.int32)
    akv = torch.tensor([act_kv_s], dtype=torch.int32)
    out = dsa.sparse_attn_tilelang(query.to(dev), key.to(dev), key.to(dev), ind.to(dev), 0.5, 1, aq.to(dev),
                                   akv.to(dev), query_rope=qr.to(dev), key_rope=kr.to(dev), layout_query="TND",
                                   layout_kv="PA_BSND", sparse_mode=sparse_mode, block_table=bt.to(dev),
                                   attention_mode=2)
    torch.cuda.synchronize()
    assert out.shape == (T, 128, 512) and out.dtype == torch.bfloat16
    q = torch.cat((query, qr), dim=-1).unsqueeze(0)
    kv = torch.cat((key, kr), dim=-1)
    want, _ = ref.sparse_mla_fwd(q, kv, ind.view(1, T, 1, -1), 0.5, block_table=bt, actual_seq_lengths_query=[T],
                                 actual_seq_lengths_kv=[act_kv_s], is_causal=sparse_mode == 3)
    torch.testing.assert_close(out.cpu().float(), want[0], rtol=2e-2, atol=2e-2)


def test_torch_op_equals_wrapper(dsa, dev):
    """torch.ops.dsa.sparse_attn gives the wrapper's output and the C entry's LSE."""
    q, kv, sink, idx = _inputs(1, 32, 256, 64, 512, 128, torch.bfloat16, 48)
    ops = dsa.load_torch_ops()
    o, l = ops.sparse_attn(q.to(dev), kv.to(dev), sink.to(dev), idx.to(dev), 512 ** -0.5)
    torch.cuda.synchronize()
    assert torch.equal(o.cpu(), _run(dsa, dev, q, kv, sink, idx, 512 ** -0.5))
    assert torch.equal(l.cpu(), _lse(dsa, dev, q, kv, sink, idx, 512 ** -0.5))


@pytest.mark.parametrize("T,N,topk,nb", [(1, 16, 40, 3), (3, 48, 300, 20), (8, 128, 2048, 21)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_decode_parts_equal_the_joined_call(dsa, dev, T, N, topk, nb, dtype):
    """Latent and rope parts read where they lie against sparse_mla_fwd on their joined rows: bit-equal
    (one workgroup per row, chunks with a ragged last one, the largest shape; -1 slots, a key length)."""
    g = torch.Generator().manual_seed(T * N + topk)
    bs = 128
    q, qr = torch.randn(T, N, 512, generator=g).to(dtype), torch.randn(T, N, 64, generator=g).to(dtype)
    k, kr = (torch.randn(nb, bs, 1, d, generator=g).to(dtype) for d in (512, 64))
    idx = torch.stack([torch.randperm(nb * bs, generator=g)[:topk] for _ in range(T)]).to(torch.int32)
    idx[:, 1::7] = -1
    bt = torch.randperm(nb, generator=g).to(torch.int32).view(1, nb)
    ql, kl = torch.tensor([T], dtype=torch.int32), torch.tensor([nb * bs - 5], dtype=torch.int32)
    q, qr, k, kr, idx, bt, ql, kl = (x.to(dev) for x in (q, qr, k, kr, idx, bt, ql, kl))
    for mode in (0, 3):
        out = dsa.sparse_attn_tilelang(q, k, k, idx.view(T, 1, topk), 0.05, 1, ql, kl, query_rope=qr, key_rope=kr,
                                       sparse_mode=mode, block_table=bt)
        want, _ = dsa.sparse_mla_fwd(torch.cat((q, qr), -1).unsqueeze(0), torch.cat((k, kr), -1),
                                     idx.view(1, T, 1, topk), 0.05, block_table=bt, actual_seq_lengths_query=ql,
                                     actual_seq_lengths_kv=kl, is_causal=mode == 3)
        assert torch.equal(out, want[0])
        # A transposed query layout cannot be read in place: the joined call takes it, same result.
        qt = q.transpose(0, 1).contiguous().transpose(0, 1)
        same = dsa.sparse_attn_tilelang(qt, k, k, idx.view(T, 1, topk), 0.05, 1, ql, kl, query_rope=qr, key_rope=kr,
                                        sparse_mode=mode, block_table=bt)
        assert torch.equal(out, same)


@pytest.mark.parametrize("h", [16, 32, 48, 64, 80])
@pytest.mark.parametrize("topk", [1, 31, 33, 200, 2080])
def test_row_lists_head_and_tile_edges(dsa, dev, h, topk):
    """More than 8 rows, so the row-list kernels: both sides of their head counts (four waves of 16
    heads with missing blocks and with every block, four of 32) by list lengths of less than a tile, a
    tile and one row, many tiles, and more slots than one workgroup holds (split partials); -1 slots
    leave the first, a middle or every tile of some rows empty.  Bars as the module's bf16 ones."""
    g = torch.Generator().manual_seed(h + topk)
    m, n = 10, 2200
    q = (torch.randn(1, m, h, 512, generator=g) * 0.5).to(torch.bfloat16)
    kv = (torch.randn(1, n, 512, generator=g) * 0.5).to(torch.bfloat16)
    idx = torch.stack([torch.randperm(n, generator=g)[:topk] for _ in range(m)]).to(torch.int32).view(1, m, topk)
    idx[0, 1, :32] = -1
    idx[0, 2, 32:96] = -1
    idx[0, 3] = -1
    sink = torch.randn(h, generator=g)
    scale = 512 ** -0.5
    out = _run(dsa, dev, q, kv, sink, idx, scale)
    want, want_lse = ref.sparse_attn_sink(q, kv, sink, idx, scale)
    torch.testing.assert_close(out, want, atol=4e-3, rtol=2e-3)
    torch.testing.assert_close(_lse(dsa, dev, q, kv, sink, idx, scale), want_lse, rtol=1e-3, atol=1e-3)
