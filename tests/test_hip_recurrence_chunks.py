"""GPU: the recurrences with one decay per head and token over many tokens at a time (chunks of 64), against float64 token by
token: chunk edges, ragged batches, starting and continued states, narrow keys and values, grouped keys, strong and weak decays."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _case(lens, H, G, dk, dv, qk_dtype, v_dtype, seed, rate):
    g = torch.Generator().manual_seed(seed)
    T = sum(lens)
    pad = 8
    c = dict(q=torch.randn(T, G * dk + pad, generator=g), k=torch.nn.functional.normalize(torch.randn(T, G, dk, generator=g), dim=-1).reshape(T, G * dk),
             v=torch.randn(T, H, dv, generator=g), z=2.0 * torch.randn(T, H, generator=g), beta=torch.randn(T, H, generator=g),
             bias=0.1 * torch.randn(H, generator=g), rate=rate + 0.3 * torch.randn(H, generator=g), skip=torch.randn(H, generator=g),
             state=torch.randn(len(lens) + 3, H, dk, dv, generator=g))
    c["q"], c["k"], c["v"] = c["q"].to(qk_dtype), c["k"].to(qk_dtype), c["v"].to(v_dtype)
    B = len(lens)
    c["slots"] = torch.randperm(B + 2, generator=g)[:B] + 1
    c["start"] = torch.tensor([sum(lens[:i]) for i in range(B)], dtype=torch.int32)
    # every other sequence starts afresh, the others go on from their slot
    c["pos"] = torch.cat([torch.arange(n) + (0 if i % 2 == 0 else 5) for i, n in enumerate(lens)])
    return c


def _exact(c, lens, H, G, dk, dv, delta, q_scale):
    q = c["q"][:, : G * dk].double().view(-1, G, dk).repeat_interleave(H // G, 1) * q_scale
    k = c["k"].double().view(-1, G, dk).repeat_interleave(H // G, 1)
    v = c["v"].double()
    dt = torch.nn.functional.softplus(c["z"].double() + c["bias"].double())
    keep = torch.exp(-torch.exp(c["rate"].double()) * dt)
    beta = torch.sigmoid(c["beta"].double())
    out, states = torch.empty_like(v), []
    for b, n in enumerate(lens):
        s0 = int(c["start"][b])
        S = torch.zeros(H, dk, dv, dtype=torch.float64) if int(c["pos"][s0]) == 0 else c["state"][int(c["slots"][b])].double()
        for t in range(s0, s0 + n):
            S = S * keep[t][:, None, None]
            u = beta[t][:, None] * (v[t] - torch.einsum("hdv,hd->hv", S, k[t])) if delta else dt[t][:, None] * v[t]
            S = S + k[t][:, :, None] * u[:, None]
            out[t] = torch.einsum("hdv,hd->hv", S, q[t]) + (0 if delta else c["skip"].double()[:, None] * v[t])
        states.append(S)
    return out, torch.stack(states)


@pytest.mark.parametrize("lens", [(1, 16, 17), (63, 64, 65, 2), (15, 200, 128), (331,)])
@pytest.mark.parametrize("H,G,dk,dv,qk,vt,rate", [(4, 2, 64, 128, torch.float32, torch.bfloat16, -2.0), (2, 2, 40, 33, torch.bfloat16, torch.bfloat16, 0.0),
                                                  (3, 1, 64, 32, torch.float32, torch.float32, 2.0), (1, 1, 7, 6, torch.float16, torch.float16, -4.0)])
@pytest.mark.parametrize("delta", [False, True])
def test_chunks_match_token_by_token(lens, H, G, dk, dv, qk, vt, rate, delta):
    """fp32 inside: a chunk's sums round 64 + 64 times (2^-24 each, randomly: 1e-6 of the terms' scale at most); 4e-6 of the result's
    norm is allowed.  The delta rule's solve repeats that over 16-token blocks: 1e-5."""
    from sglang_custom_amd import ops

    c = _case(lens, H, G, dk, dv, qk, vt, len(lens) * 10 + dk, rate)
    want, states = _exact(c, lens, H, G, dk, dv, delta, 0.25)
    T, B = sum(lens), len(lens)
    d = {n: t.to(DEV) for n, t in c.items()}
    state = d["state"].clone()
    req_to_state = torch.zeros(B, dtype=torch.int32, device=DEV)
    req_to_state[:] = d["slots"].int()
    out = torch.full((T, H, dv), float("nan"), device=DEV)
    seg_len = torch.tensor(lens, dtype=torch.int32, device=DEV)
    tok = torch.repeat_interleave(torch.arange(B, dtype=torch.int32), torch.tensor(lens)).to(DEV)
    q = d["q"][:, : G * dk].view(T, G, dk)
    seg = dict(tok_req=tok, seg_start=d["start"], seg_len=seg_len)
    args = (req_to_state, torch.arange(B, device=DEV), d["pos"], 0.25)
    if delta:
        ops.gated_delta_rule(q, d["k"].view(T, G, dk), d["v"], d["beta"], d["z"], d["bias"], d["rate"], out, state, *args, **seg)
    else:
        ops.linear_recurrence(q, d["k"].view(T, G, dk), d["v"], out, state, *args, dt_logits=d["z"], dt_bias=d["bias"], rate_log=d["rate"],
                              skip=d["skip"], **seg)
    tol = 1e-5 if delta else 4e-6
    got, gs = out.cpu().double(), state.cpu().double()
    assert (got - want).norm() <= tol * want.norm()
    assert (gs[c["slots"]] - states).norm() <= tol * states.norm()
    others = [i for i in range(state.shape[0]) if i not in c["slots"].tolist()]
    assert torch.equal(gs[others], c["state"][others].double())


@pytest.mark.parametrize("delta", [False, True])
def test_total_forgetting_stays_finite(delta):
    """Decays that underflow to zero, for some tokens or all."""
    from sglang_custom_amd import ops

    c = _case((130,), 2, 2, 64, 32, torch.float32, torch.float32, 3, 1.0)
    c["z"][::3] = 1e6
    c["rate"][1] = 60.0
    if not delta:
        c["z"][::3] = 50.0
    want, _ = _exact(c, (130,), 2, 2, 64, 32, delta, 1.0)
    d = {n: t.to(DEV) for n, t in c.items()}
    out = torch.empty((130, 2, 32), device=DEV)
    seg = dict(tok_req=torch.zeros(130, dtype=torch.int32, device=DEV), seg_start=d["start"], seg_len=torch.tensor([130], dtype=torch.int32, device=DEV))
    args = (d["slots"].int(), torch.zeros(1, dtype=torch.int64, device=DEV), d["pos"], 1.0)
    q, k = d["q"][:, :128].view(130, 2, 64), d["k"].view(130, 2, 64)
    if delta:
        ops.gated_delta_rule(q, k, d["v"], d["beta"], d["z"], d["bias"], d["rate"], out, d["state"], *args, **seg)
    else:
        ops.linear_recurrence(q, k, d["v"], out, d["state"], *args, dt_logits=d["z"], dt_bias=d["bias"], rate_log=d["rate"], skip=d["skip"], **seg)
    assert (out.cpu().double() - want).norm() <= 1e-5 * want.norm()


@pytest.mark.parametrize("what,delta", [(w, d) for w in ("v", "k", "q", "z", "beta", "state") for d in (False, True) if d or w != "beta"])
def test_non_finite_inputs_reach_no_earlier_token(what, delta):
    """An infinity or a NaN in the middle of a chunk, and the tokens behind it: finite outputs are where the token-by-token form
    has them, and right there (the bound of the tests above)."""
    from sglang_custom_amd import ops

    lens, H, G, dk, dv = (150, 130), 2, 1, 40, 33
    c = _case(lens, H, G, dk, dv, torch.float32, torch.float32, 11, -1.0)
    nan, inf = float("nan"), float("inf")
    if what == "v":
        c["v"][70, 1, 5], c["v"][150 + 127, 0, 32] = inf, nan
    elif what in ("k", "q"):
        c[what][21, 7], c[what][150 + 64, 39] = nan, inf
    elif what in ("z", "beta"):
        c[what][100, 0], c[what][150 + 3, 1] = nan, nan
    else:
        c["state"][c["slots"][1], 0, 3, 4], c["state"][c["slots"][1], 1, 39, 32] = nan, inf
    want, states = _exact(c, lens, H, G, dk, dv, delta, 0.25)
    d = {n: t.to(DEV) for n, t in c.items()}
    T, B = sum(lens), len(lens)
    out = torch.empty((T, H, dv), device=DEV)
    seg = dict(tok_req=torch.repeat_interleave(torch.arange(B, dtype=torch.int32), torch.tensor(lens)).to(DEV), seg_start=d["start"],
               seg_len=torch.tensor(lens, dtype=torch.int32, device=DEV))
    args = (d["slots"].int(), torch.arange(B, device=DEV), d["pos"], 0.25)
    q, k = d["q"][:, : G * dk].view(T, G, dk), d["k"].view(T, G, dk)
    if delta:
        ops.gated_delta_rule(q, k, d["v"], d["beta"], d["z"], d["bias"], d["rate"], out, d["state"], *args, **seg)
    else:
        ops.linear_recurrence(q, k, d["v"], out, d["state"], *args, dt_logits=d["z"], dt_bias=d["bias"], rate_log=d["rate"], skip=d["skip"], **seg)
    for got, ref in ((out.cpu().double(), want), (d["state"].cpu().double()[c["slots"]], states)):
        ok = ref.isfinite()
        assert torch.equal(got.isfinite(), ok)
        assert (got - ref)[ok].norm() <= 1e-5 * ref[ok].norm()


@pytest.mark.parametrize("lens", [(449,), (200, 0, 64, 331, 1), tuple(900 if i == 69 else 130 if i % 9 == 1 else 0 for i in range(70)), (2000, 65)])
@pytest.mark.parametrize("H,G,dk,dv,qk,vt", [(4, 2, 64, 128, torch.float32, torch.bfloat16), (2, 1, 40, 33, torch.bfloat16, torch.bfloat16)])
@pytest.mark.parametrize("delta", [False, True])
def test_records_in_front_change_no_bits(lens, H, G, dk, dv, qk, vt, delta, monkeypatch):
    """What depends on no state from a launch of its own: the same operations, so the same bits, for sequences of none to many chunks
    whose segments lie in any order."""
    from sglang_custom_amd import ops

    c = _case(lens, H, G, dk, dv, qk, vt, len(lens) + dk, -1.0)
    T, B = sum(lens), len(lens)
    order = torch.randperm(B, generator=torch.Generator().manual_seed(7))      # the sequences' order, not their segments'
    n = torch.tensor(lens, dtype=torch.int32)[order]
    start = torch.where(n > 0, c["start"][order], 0).to(torch.int32)
    d = {k: t.to(DEV) for k, t in c.items()}
    seg = dict(tok_req=torch.zeros(T, dtype=torch.int32, device=DEV), seg_start=start.to(DEV), seg_len=n.to(DEV), longest=max(lens))
    args = (d["slots"].int()[order.to(DEV)], torch.arange(B, device=DEV), d["pos"], 0.25)
    q, k = d["q"][:, : G * dk].view(T, G, dk), d["k"].view(T, G, dk)
    wanted = ops._chunk_records

    def run(records):
        monkeypatch.setattr(ops, "_chunk_records", records)
        out, state = torch.full((T, H, dv), float("nan"), device=DEV), d["state"].clone()
        if delta:
            ops.gated_delta_rule(q, k, d["v"], d["beta"], d["z"], d["bias"], d["rate"], out, state, *args, **seg)
        else:
            ops.linear_recurrence(q, k, d["v"], out, state, *args, dt_logits=d["z"], dt_bias=d["bias"], rate_log=d["rate"], skip=d["skip"], **seg)
        return out, state

    assert wanted(delta, B, H, dk, dv, T, max(lens), DEV)[1] > 0, "the case is for the chunks"
    got, want = run(wanted), run(lambda *a: (None, 0))
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1]) and got[0].isfinite().all()


@pytest.mark.parametrize("what,delta", [(w, d) for w in ("v", "k", "q", "z", "beta", "state") for d in (False, True) if d or w != "beta"])
def test_records_with_values_that_are_no_numbers(what, delta, monkeypatch):
    """An infinity and a NaN in a middle chunk: with records in front every output and state is what it is without them, and the tokens before are
    finite."""
    from sglang_custom_amd import ops

    lens, H, G, dk, dv = (449, 330), 2, 1, 40, 33
    c = _case(lens, H, G, dk, dv, torch.float32, torch.float32, 12, -1.0)
    bad = {"v": (c["v"][200, 1, 5:6], c["v"][449 + 127, 0, 32:]), "k": (c["k"][200, 7:8], c["k"][449 + 127, 39:]), "q": (c["q"][200, 7:8], c["q"][449 + 127, 39:40]),
           "z": (c["z"][200, :1], c["z"][449 + 127, 1:]), "beta": (c["beta"][200, :1], c["beta"][449 + 127, 1:]),
           "state": (c["state"][int(c["slots"][1]), 0, 3, :1], c["state"][int(c["slots"][1]), 1, 5, 32:])}[what]
    bad[0].fill_(float("inf") if what in ("v", "k", "state") else float("nan"))
    bad[1].fill_(float("nan"))
    d, T = {k: t.to(DEV) for k, t in c.items()}, sum(lens)
    seg = dict(tok_req=torch.zeros(T, dtype=torch.int32, device=DEV), seg_start=d["start"], seg_len=torch.tensor(lens, dtype=torch.int32, device=DEV), longest=max(lens))
    args = (d["slots"].int(), torch.arange(2, device=DEV), d["pos"], 0.25)
    q, k = d["q"][:, : G * dk].view(T, G, dk), d["k"].view(T, G, dk)
    wanted, results = ops._chunk_records, []
    assert wanted(delta, 2, H, dk, dv, T, max(lens), DEV)[1] > 0, "the case is for the records"
    for records in (wanted, lambda *a: (None, 0)):
        monkeypatch.setattr(ops, "_chunk_records", records)
        out, state = torch.zeros(T, H, dv, device=DEV), d["state"].clone()
        if delta:
            ops.gated_delta_rule(q, k, d["v"], d["beta"], d["z"], d["bias"], d["rate"], out, state, *args, **seg)
        else:
            ops.linear_recurrence(q, k, d["v"], out, state, *args, dt_logits=d["z"], dt_bias=d["bias"], rate_log=d["rate"], skip=d["skip"], **seg)
        results.append((out, state))
    for a, b in zip(*results):
        assert torch.equal(a.isnan(), b.isnan()) and torch.equal(a.nan_to_num(0.0), b.nan_to_num(0.0))
    out = results[0][0]
    assert out[:200].isfinite().all() and not out.isfinite().all()
    assert what == "state" or out[449: 449 + 127].isfinite().all()
