"""The wrappers' native host path against their Python path (the same call with the native path
returning None): equal results on plain arguments, the same exception on refused ones, and the
arguments it must leave to the wrapper (other dtypes, layouts, host lengths) still accepted."""
import importlib

import pytest
import torch

pytestmark = pytest.mark.gpu


class _Off:
    """A host path that takes nothing."""

    def __getattr__(self, name):
        return lambda *a: None


class _Seen:
    """The native path, counting the calls it took."""

    def __init__(self, native):
        self.native, self.took = native, 0

    def __getattr__(self, name):
        def call(*a):
            r = getattr(self.native, name)(*a)
            self.took += r is not None
            return r
        return call


def _calls(dsa, dev):
    g = torch.Generator(device=dev).manual_seed(5)

    def rn(*s, dt=torch.bfloat16):
        return torch.randn(s, generator=g, device=dev).to(dt)

    def ints(*v):
        return torch.tensor(v, dtype=torch.int32, device=dev)

    f8 = torch.float8_e4m3fn
    idx = torch.stack([torch.randperm(300, generator=g, device=dev)[:64] for _ in range(6)]).to(torch.int32)
    x, q, kv, pool = rn(5, 900, dt=torch.float32), rn(2, 3, 32, 576), rn(2, 300, 1, 576), rn(10, 64, 1, 576)
    table = torch.randperm(10, generator=g, device=dev).to(torch.int32).view(2, 5)
    iq, ik, iw = rn(2, 6, 24, 128, dt=f8), rn(2, 700, 1, 128, dt=f8), rn(2, 6, 24, dt=torch.float32)
    ks = rn(2, 700, dt=torch.float32).abs()
    ipool, itable = rn(24, 32, 1, 128), torch.arange(24, device=dev).to(torch.int32).view(2, 12)
    v4q, ori, cmp = rn(7, 16, 512), rn(8, 32, 1, 512), rn(4, 32, 1, 512)
    obt, cbt = torch.arange(8, device=dev).to(torch.int32).view(2, 4), torch.arange(4, device=dev).to(torch.int32).view(2, 2)
    sel = torch.arange(7 * 9, device=dev).view(7, 1, 9).remainder(20).to(torch.int32)
    v4 = dict(ori_kv=ori, ori_block_table=obt, cu_seqlens_q=ints(0, 3, 7), seqused_kv=ints(100, 121),
              sinks=rn(16, dt=torch.float32), softmax_scale=0.05, return_softmax_lse=True)
    parts = dict(query_rope=rn(2, 16, 64), key_rope=rn(10, 64, 1, 64), block_table=table[:1].contiguous())
    return {
        "topk": lambda **k: dsa.topk_selector(x, **{**dict(top_k=100, return_values=True), **k}),
        "topk_len": lambda **k: dsa.topk_selector(x, 50, **{**dict(row_len=ints(900, 1, 0, 77, 400)), **k}),
        "quant": lambda **k: dsa.act_quant(x, **{**dict(round_scale=True, dtype=f8), **k}),
        "mla": lambda **k: dsa.sparse_mla_fwd(q, kv, idx.view(2, 3, 1, 64), **k),
        "mla_paged": lambda **k: dsa.sparse_mla_fwd(q, pool, idx.view(2, 3, 64), 0.04, **{**dict(
            block_table=table, actual_seq_lengths_query=ints(3, 2), actual_seq_lengths_kv=ints(300, 290)), **k}),
        "gqa": lambda **k: dsa.sparse_gqa_fwd(rn(1, 3, 16, 128), rn(1, 300, 2, 128), idx.view(1, 3, 2, 64), **k)[0].shape,
        "parts": lambda **k: dsa.sparse_attn_tilelang(rn(2, 16, 512) * 0 + 1, ori.view(4, 64, 1, 512), None,
                                                      idx[:2].view(2, 1, 64).remainder(256), 0.04, 1, None, ints(256),
                                                      **{**parts, "key_rope": parts["key_rope"][:4].contiguous(),
                                                         "block_table": ints(3, 1, 0, 2).view(1, 4), **k}),
        "indexer": lambda **k: dsa.lightning_indexer(iq, ik, iw, **{**dict(key_scale=ks, sparse_count=200,
                                                                           return_value=True), **k}),
        "indexer_lens": lambda **k: dsa.lightning_indexer(iq, ik, iw, **{**dict(
            actual_seq_lengths_query=ints(6, 4), actual_seq_lengths_key=ints(700, 650), sparse_count=200), **k}),
        "indexer_paged": lambda **k: dsa.lightning_indexer(iq.to(torch.bfloat16), ipool, iw, **{**dict(
            actual_seq_lengths_query=ints(6, 5), actual_seq_lengths_key=ints(384, 301), block_table=itable,
            layout_key="PA_BSND", sparse_count=64), **k}),
        "indexer_packed": lambda **k: dsa.lightning_indexer(
            iq.view(12, 24, 128), ik.view(1400, 1, 128), iw.view(12, 24), **{**dict(
                actual_seq_lengths_query=ints(5, 11), actual_seq_lengths_key=ints(600, 1399), layout_query="TND",
                layout_key="TND", sparse_count=100, return_value=True, key_scale=ks), **k}),
        "indexer_packed_paged": lambda **k: dsa.lightning_indexer(
            iq.to(torch.bfloat16).view(12, 24, 128), ipool, iw.view(12, 24), **{**dict(
                actual_seq_lengths_query=ints(5, 12), actual_seq_lengths_key=ints(384, 200), block_table=itable,
                layout_query="TND", layout_key="PA_BSND", sparse_count=100), **k}),
        "v4_swa": lambda **k: dsa.sparse_flash_mla(v4q, **{**v4, **k}),
        "v4_hca": lambda **k: dsa.sparse_flash_mla(v4q, cmp_kv=cmp, cmp_block_table=cbt, **{**v4, **dict(cmp_ratio=4), **k}),
        "v4_csa": lambda **k: dsa.sparse_flash_mla(v4q, cmp_kv=cmp, cmp_block_table=cbt, cmp_sparse_indices=sel,
                                                   **{**v4, **dict(cmp_ratio=4), **k}),
    }


NAMES = ["topk", "topk_len", "quant", "mla", "mla_paged", "gqa", "parts", "indexer", "indexer_lens", "indexer_paged",
         "indexer_packed", "indexer_packed_paged", "v4_swa", "v4_hca", "v4_csa"]


def _both(monkeypatch, fn):
    """(result or exception type of the native path, of the Python path, whether the native path took it)."""
    lib = importlib.import_module("tilelang_ascend_amd._lib")
    native = lib.host_path()
    got = []
    seen = _Seen(native)
    for path in (seen, _Off()):
        monkeypatch.setattr(lib, "_host_path", path)
        try:
            got.append(fn())
        except Exception as e:  # noqa: BLE001
            got.append(type(e))
    monkeypatch.setattr(lib, "_host_path", native)
    return got[0], got[1], seen.took


def _equal(a, b):
    if isinstance(a, torch.Tensor):
        return (a.dtype == b.dtype and a.shape == b.shape and a.is_contiguous() and
                torch.equal(a.view(torch.uint8) if a.numel() else a, b.view(torch.uint8) if b.numel() else b))
    if isinstance(a, tuple):
        return type(a) is type(b) and len(a) == len(b) and all(_equal(x, y) for x, y in zip(a, b))
    return a == b


@pytest.mark.parametrize("name", NAMES)
def test_plain_arguments(dsa, dev, monkeypatch, name):
    a, b, took = _both(monkeypatch, _calls(dsa, dev)[name])
    assert took == 1, "the native path must take plain arguments"
    assert not isinstance(a, type) and _equal(a, b)


OTHER = [
    ("topk", dict(top_k=0)), ("topk", dict(top_k=9000)), ("topk_len", dict(row_len=[1])),
    ("topk", dict(return_values=1)), ("topk", dict(sorted=False)), ("quant", dict(dtype=torch.int16)),
    ("quant", dict(round_scale=0)), ("mla", dict(sm_scale=-1.0)), ("mla", dict(sm_scale=1)),
    ("mla_paged", dict(block_table=None)), ("mla_paged", dict(actual_seq_lengths_kv=[300, 290])),
    ("parts", dict(query_rope=None)), ("parts", dict(sparse_mode=0)), ("indexer", dict(sparse_count=3000)),
    ("indexer", dict(sparse_mode=1)), ("indexer", dict(fuse_topk=True)), ("indexer", dict(pre_tokens=4)),
    ("indexer_lens", dict(actual_seq_lengths_query=[7, 4])), ("indexer_lens", dict(actual_seq_lengths_key=[701, 4])),
    ("indexer_paged", dict(return_value=True)), ("indexer_paged", dict(actual_seq_lengths_key=None)),
    ("indexer_paged", dict(layout_key="BSND")), ("indexer_packed", dict(actual_seq_lengths_query=[11, 5])),
    ("indexer_packed", dict(actual_seq_lengths_key=[600, 1401])), ("indexer_packed", dict(block_n=64)),
    ("v4_swa", dict(cu_seqlens_q=[0, 3, 8])), ("v4_swa", dict(cu_seqlens_q=[0, 4, 3])), ("v4_swa", dict(sinks=None)),
    ("v4_hca", dict(cmp_ratio=None)), ("v4_csa", dict(cmp_ratio=None)), ("v4_csa", dict(topk_cmp=4)),
    ("v4_csa", dict(ori_win_left=-1)), ("v4_swa", dict(return_softmax_lse=False)), ("v4_swa", dict(softmax_scale=1)),
    ("topk", dict(top_k=2**64 + 100)), ("topk", dict(top_k=-2**70)), ("indexer", dict(sparse_count=2**64 + 200)),
    ("indexer", dict(sparse_mode=2**32 + 3)), ("indexer_packed", dict(sparse_mode=2**64)),
    ("v4_swa", dict(ori_win_left=2**64 + 127)), ("v4_csa", dict(cmp_ratio=2**64 + 4))]


# Length lists run twice: as device tensors (which the native path reads) and as they are (which it leaves alone).
@pytest.mark.parametrize("name,change,on_device", [
    (name, change, dev) for name, change in OTHER
    for dev in ((True, False) if any(isinstance(v, list) for v in change.values()) else (False,))])
def test_other_arguments(dsa, dev, monkeypatch, name, change, on_device):
    """Refused calls raise the same exception, odd ones give the same result."""
    if on_device:
        change = {k: torch.tensor(v, dtype=torch.int32, device=dev) if isinstance(v, list) else v
                  for k, v in change.items()}
    fn = _calls(dsa, dev)[name]
    a, b, _ = _both(monkeypatch, lambda: fn(**change))
    assert (a is b) if isinstance(b, type) else _equal(a, b)
