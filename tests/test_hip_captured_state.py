"""Captured decode steps of the families that keep state per sequence (Fudonex) or latent rows (Silatar without matrix memories), against
the whole-sequence oracles: eager prompts between the replays, padded batches, requests that end and begin again in their rows, and a
request at row 0 of the request table that waits while padded batches of others run (its state is its own)."""
import gc
import weakref

import pytest

import fudonex_util as fu
import lomazen_util as lu
import silatar_util as su
from oracle import fudonex_ref, silatar_ref
from sglang_custom_amd.managers.trace_replay import TraceReplayer

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture(autouse=True)
def _product_ops():
    from sglang_custom_amd import ops_backend
    from sglang_custom_amd.distributed import parallel_state

    ops_backend.set_ops_backend(None)      # the HIP library (get_ops() loads it and raises if it is missing)
    parallel_state.init_distributed_environment(1, 0)
    yield


# the families' own engine tests take the same limits
@pytest.mark.parametrize("family,dtype,tol", [("fudonex", "float32", 3e-5), ("fudonex", "bfloat16", 6e-2), ("silatar", "float32", 3e-5),
                                              ("silatar", "bfloat16", 6e-2)])
def test_replays_against_the_oracle(family, dtype, tol):
    if family == "fudonex":
        u, ref, cfg = fu, fudonex_ref, fu.make_config()
    else:
        u, ref, cfg = su, silatar_ref, su.make_config(layers=[(su.latent(), su.dense(96)), (su.latent(kv_rank=24), su.dense(64)), (su.latent(), None)], width=96,
                                                      loop=(0, 2, 2))
    w = u.make_weights(cfg, seed=4)
    prompts = u.random_prompts(cfg, [40, 25, 18, 22, 9], seed=6)
    want = {k: ref.forward(cfg, w, p) for k, p in prompts.items()}
    mr = u.build_runner(cfg, w, dtype=dtype, device=DEV, max_total_tokens=160, max_running_requests=5, cuda_graph_bs=[1, 4])
    assert mr.graph_runner is not None
    sched = [[("r0", 20), ("r1", 5)], [("r2", 3), ("r3", 7)]]                  # r0 holds row 0
    sched += [[("r1", 1), ("r2", 1), ("r3", 1)]] * 6                           # three in a graph of four while r0 waits
    sched += [[("r0", 1)]] * 5 + [[("r0", 1), ("r1", 1)]] * 4                  # alone, and two of four
    sched += [[("r0", 4), ("r4", 2)]]                                          # a portion between the replays
    sched += [[("r0", 1), ("r1", 1), ("r2", 1), ("r3", 1)]] * 7                # whole
    sched += [[("r1", 1), ("r2", 1), ("r4", 1)], [("r1", 2), ("r2", 1), ("r3", 2), ("r4", 6)]]
    assert {k: sum(n for s in sched for r, n in s if r == k) for k in prompts} == {k: len(p) for k, p in prompts.items()}
    for _ in range(2):       # the second time over used slots and rows
        u.replay_and_compare(mr, cfg, w, prompts, sched, tol, want_all=want)
        assert mr.req_to_token_pool.available_size() == mr.req_to_token_pool.size
        assert mr.token_to_kv_pool_allocator.available_size() == mr.max_total_num_tokens
        assert not mr.req_to_token_pool.table[mr.req_to_token_pool.pad_row].any()


@pytest.mark.parametrize("family,dtype,tol", [("fudonex", "float32", 3e-5), ("fudonex", "bfloat16", 6e-2), ("silatar", "bfloat16", 6e-2)])
def test_replays_with_many_key_ranges(family, dtype, tol, monkeypatch):
    """A captured step has its key ranges from the model's context length: at 8192 tokens ten and sixteen (windows and averaged blocks) and 64 (latent rows),
    of which sequences of up to 78 tokens leave all but one to three without a key and padded rows all but one.  Silatar's with mixtures."""
    from sglang_custom_amd import ops
    from sglang_custom_amd.configs.model_config import ModelConfig
    from sglang_custom_amd.model_executor.model_runner import ModelRunner
    from sglang_custom_amd.server_args import ServerArgs

    ranges = []
    for name in ("window_attention_splits", "latent_window_attention_splits"):
        monkeypatch.setattr(ops, name, lambda *a, rule=getattr(ops, name), **kw: (ranges.append(rule(*a, **kw)), ranges[-1])[1])
    if family == "fudonex":
        u, ref, cfg = fu, fudonex_ref, fu.make_config()
    else:
        moe = [su.moe(experts=3, top=3, ff=40, shared=(24, 1.1)), su.moe(experts=2, top=2, ff=32, shared=None)]
        u, ref, cfg = su, silatar_ref, su.make_config(layers=[(su.latent(), moe[0]), (su.latent(kv_rank=24), su.dense(64)), (su.latent(), moe[1])], width=96,
                                                      loop=(0, 2, 2))
    w = u.make_weights(cfg, seed=4)
    prompts = u.random_prompts(cfg, [78, 25, 12], seed=6)
    want = {k: ref.forward(cfg, w, p) for k, p in prompts.items()}
    mr = ModelRunner(ModelConfig(cfg, dtype=dtype, context_length=8192),
                     ServerArgs(dtype=dtype, device=DEV, max_total_tokens=160, max_running_requests=4, context_length=8192, cuda_graph_bs=[1, 4]),
                     weights={k: v.to(DEV) for k, v in w.items()})
    assert mr.graph_runner is not None and set(ranges) == ({10, 16} if family == "fudonex" else {64})
    sched = [[("r0", 60), ("r1", 5)]] + [[("r0", 1)]] * 4 + [[("r2", 2)]] + [[("r0", 1), ("r1", 1), ("r2", 1)]] * 10 + [[("r0", 1), ("r1", 1)]] * 4
    sched += [[("r1", 1)]] * 6
    for _ in range(2):
        u.replay_and_compare(mr, cfg, w, prompts, sched, tol, want_all=want)


def test_what_a_graph_was_recorded_over_stays(monkeypatch):
    """A captured step's kernels keep the addresses of its batch's tensors, which the graphs' memory pool does not hold."""
    from sglang_custom_amd.model_executor.forward_batch_info import ForwardBatch

    made, init = [], ForwardBatch._init_seq_state

    def recording(self, runner):
        init(self, runner)
        made.append(weakref.ref(self.seq_state.h_last))

    monkeypatch.setattr(ForwardBatch, "_init_seq_state", recording)
    cfg = fu.make_config()
    mr = fu.build_runner(cfg, fu.make_weights(cfg, seed=4), dtype="bfloat16", device=DEV, max_total_tokens=160, cuda_graph_bs=[1, 4])
    gc.collect()
    assert mr.graph_runner is not None and len(made) == 2 and all(t() is not None for t in made)


@pytest.mark.parametrize("family", ["fudonex", "silatar", "lomazen"])
def test_streams_of_a_decode_step(family):
    """A list in capture_streams receives the residual behind every layer of a decode step too, though the model's steps are captured."""
    u = {"fudonex": fu, "silatar": su, "lomazen": lu}[family]
    cfg = su.make_config(layers=[(su.latent(), su.dense())] * 2, loop=None) if family == "silatar" else u.make_config()
    mr = u.build_runner(cfg, u.make_weights(cfg, seed=4), dtype="bfloat16", device=DEV, max_total_tokens=160, cuda_graph_bs=[1])
    rp, tokens = TraceReplayer(mr), u.random_prompts(cfg, [4], seed=6)["r0"]
    step = lambda t: rp.step([dict(id="r0", tokens=t, want=[0])])
    step(tokens[:2])
    mr.model.model.capture_streams = got = []
    step(tokens[2:3])
    n = len(mr.model_config.layer_runs) if family != "fudonex" else len(cfg["layers"])
    assert mr.graph_runner is not None and [tuple(x.shape) for x in got] == [(1, cfg["width"])] * n
    mr.model.model.capture_streams = None
    step(tokens[3:])
    assert len(got) == n
