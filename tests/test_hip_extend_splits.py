"""Extend attention whose key tiles several workgroups share (mi355_extend_attention_ws with splits): the unsplit kernel is the reference,
itself checked against the oracle in test_hip_ops.py and test_hip_extend_rows.py."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture(scope="module")
def ops():
    from sglang_custom_amd import ops as o

    return o


def _call(ops, q, k, v, kb, vb, qo, kv, slots, mask, splits, rows=None):
    T, hq, d = q.shape
    lib, o = ops._lib_(), torch.full((T, hq, d), 7.0, dtype=q.dtype, device=DEV)
    need = lib.mi355_extend_attention_workspace_bytes(T, hq, d, splits)
    ws = torch.full((max(need, 16) // 4,), float("nan"), dtype=torch.float32, device=DEV)
    longest = int((qo[1:] - qo[:-1]).max())
    ops.check(lib.mi355_extend_attention_ws(
        q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), kb.data_ptr(), vb.data_ptr(), qo.data_ptr(), kv.data_ptr(), slots.data_ptr(),
        mask[0].data_ptr() if mask else None, mask[1].data_ptr() if mask else None, 1, 0, qo.numel() - 1, longest, hq, k.shape[1], d, d,
        q.stride(0), k.stride(0), v.stride(0), kb.shape[0], d ** -0.5, 0.0, -1, ops._kvdt(q, kb, vb), T, splits, ws.data_ptr(), need,
        ops._stream(q)), "extend")
    torch.cuda.synchronize()
    return o


# blocks of one and several tiles, prefixes that end inside a tile, sequences of which one has a single token, more splits than tiles
@pytest.mark.parametrize("splits", [2, 3, 16])
@pytest.mark.parametrize("ext,pre", [([1], [300]), ([130, 1, 70], [0, 513, 255]), ([257], [0]), ([64, 65], [64, 1000])])
@pytest.mark.parametrize("d,kv8,dtype", [(64, False, torch.bfloat16), (64, True, torch.float16), (128, False, torch.float16), (128, True, torch.bfloat16)])
def test_splits_of_the_keys(ops, splits, ext, pre, d, kv8, dtype):
    """Both sides round the same fp32 quotient to 16 bits once; their sums differ by the order of at most 1300 additions and, at 128, by which
    weights rounded relative to which maximum: 2^-8 (bf16) or 2^-11 (fp16) of the values' scale allows for one rounding boundary."""
    g = torch.Generator().manual_seed(sum(ext) + sum(pre) + d)
    T, P, hq, hkv = sum(ext), sum(pre), 4, 2
    r = lambda *s: torch.randn(*s, generator=g).to(dtype).to(DEV)
    q, k, v, kb, vb = r(T + 3, hq, d), r(T + 3, hkv, d), r(T + 3, hkv, d), r(P + 9, hkv, d), r(P + 9, hkv, d)
    if kv8:
        kb, vb = kb.to(torch.float8_e4m3fn), vb.to(torch.float8_e4m3fn)
    ind = lambda x: torch.tensor([0] + list(torch.tensor(x).cumsum(0)), dtype=torch.int32, device=DEV)
    qo, kv = ind(ext), ind(pre)
    slots = (torch.randperm(P + 8, generator=g)[: max(P, 1)] + 1).to(torch.int32).to(DEV)
    one, many = (_call(ops, q, k, v, kb, vb, qo, kv, slots, None, s) for s in (1, splits))
    eps = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    assert ((one.float() - many.float()).abs() <= 4 * eps * (one.float().abs() + 0.05)).all()
    assert (many[T:] == 7.0).all()          # rows of no sequence are not written
    if d == 64:
        # a triangle for a mask gives the causal rule's bits here too, and values that are no numbers reach the queries that see them alone
        rows = [torch.ones(e, p + e).tril(p) for e, p in zip(ext, pre)]
        mask = (torch.cat([x.flatten() for x in rows]).to(torch.uint8).to(DEV),
                torch.tensor([0] + list(torch.tensor([x.numel() for x in rows]).cumsum(0)), dtype=torch.int64, device=DEV))
        assert torch.equal(_call(ops, q, k, v, kb, vb, qo, kv, slots, mask, splits), many)
        v[T - 1] = float("inf")             # the last sequence's newest token: its own query alone
        odd = _call(ops, q, k, v, kb, vb, qo, kv, slots, None, splits)
        assert torch.equal(odd[: T - 1], many[: T - 1]) and torch.isinf(odd[T - 1]).all()


@pytest.mark.parametrize("rows,bs,longest,prefix,hq,d,want", [
    (88, 1, 88, 1933, 32, 128, 7), (1730, 4, 490, 7000, 32, 128, 1), (591, 3, 197, 4842, 32, 64, 2), (1148, 1, 1148, 0, 32, 64, 1),
    (400, 1, 400, 300, 32, 128, 1), (100, 1, 100, 30000, 8, 128, 8), (100, 1, 100, 30000, 8, 96, 1),
    (2048, 1, 2048, 1, 8, 128, 1), (4096, 1, 4096, 0, 8, 128, 1), (99, 1, 99, 511, 32, 128, 1), (99, 1, 99, 640, 32, 128, 2)])
def test_rule(ops, rows, bs, longest, prefix, hq, d, want):
    f = ops._lib_().mi355_extend_attention_splits
    assert f(rows, bs, longest, prefix, 0, hq, d, d, 0.1, 0.0, -1, 1) == want
    assert f(rows, bs, longest, prefix, 0, hq, d, d, 0.1, 30.0, -1, 1) == 1 and f(rows, bs, longest, prefix, 0, hq, d, d, 0.1, 0.0, 64, 1) == 1
    assert f(rows, bs, longest, prefix, 0, hq, d, d, 0.1, 0.0, -1, 0) == 1          # fp32 has no matrix-core kernel


def test_layers_of_a_step_share_the_rule_and_its_memory(ops, monkeypatch):
    """The second launch of a step asks nothing and gives the same bits; another shape under the same dict has an entry of its own."""
    lib, asked = ops._lib_(), []
    rule = lib.mi355_extend_attention_splits

    class Counting:
        def __getattr__(self, name):
            return getattr(lib, name)

        def mi355_extend_attention_splits(self, *a):
            asked.append(rule(*a))
            return asked[-1]

    monkeypatch.setattr(ops, "_lib_", lambda: Counting())
    g, d, hkv, pre = torch.Generator().manual_seed(5), 64, 2, 1000
    r = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16).to(DEV)
    kb, vb = r(pre + 9, hkv, d), r(pre + 9, hkv, d)
    slots = (torch.randperm(pre + 8, generator=g)[:pre] + 1).to(torch.int32).to(DEV)
    kv, shared = torch.tensor([0, pre], dtype=torch.int32, device=DEV), {}
    for ext, hq in ((70, 4), (70, 8), (200, 4)):
        q, k, v = r(ext, hq, d), r(ext, hkv, d), r(ext, hkv, d)
        qo, out = torch.tensor([0, ext], dtype=torch.int32, device=DEV), []
        for kw in ({}, {"shared": shared}, {"shared": shared}):
            o = torch.empty_like(q)
            ops.extend_attention_fwd(q, k, v, o, kb, vb, qo, kv, slots, None, True, None, ext, d ** -0.5, **kw)
            out.append(o)
        assert torch.equal(out[0], out[1]) and torch.equal(out[0], out[2])
    assert len(asked) == 6 and asked[0] > 1 and len(shared) == 3


def test_a_model_step_asks_once(monkeypatch):
    """An extend over cached tokens through a model: one entry for all of its layers, none without a prefix."""
    from sglang_custom_amd import bench_one_batch as bob, ops_backend
    from sglang_custom_amd.configs.model_config import ModelConfig
    from sglang_custom_amd.distributed import parallel_state
    from sglang_custom_amd.managers.schedule_batch import Req
    from sglang_custom_amd.model_executor.model_runner import ModelRunner
    from sglang_custom_amd.model_loader.synthetic import hf_config_dict, make_synthetic_llama_weights
    from sglang_custom_amd.server_args import ServerArgs

    ops_backend.set_ops_backend(None)
    parallel_state.init_distributed_environment(1, 0)
    cfg = hf_config_dict("tiny-llama-d64", "bfloat16")
    w = make_synthetic_llama_weights(cfg, seed=1, dtype=torch.bfloat16)
    mr = ModelRunner(ModelConfig(cfg, dtype="bfloat16"), ServerArgs(dtype="bfloat16", max_total_tokens=1024, max_running_requests=2, disable_cuda_graph=True),
                     weights={k: v.to(DEV) for k, v in w.items()})
    tokens = torch.randint(0, cfg["vocab_size"], (600,), generator=torch.Generator().manual_seed(2)).tolist()
    _, _, batch = bob.extend([Req(0, tokens[:520])], mr)
    assert mr.attn_backend.forward_metadata.extend_shared is None
    req = Req(1, tokens)
    req.init_next_round_input(mr.req_to_token_pool.req_to_token[int(batch.req_pool_indices[0]), :520].clone())
    bob.extend([req], mr)
    assert len(mr.attn_backend.forward_metadata.extend_shared) == 1
