"""The softmax and the draw over chunks whose highest entries are listed: one fused call against the two calls, and the draw against
float64, where the lists hold the cut, where they do not, and where chunks have none."""
import pytest
import torch

DEV = "cuda"


@pytest.fixture(scope="module")
def ops():
    from sglang_custom_amd import ops

    return ops


def _drawn(p, k, tp, mp, u):
    """Per row the interval of the float64 inverse CDF in index order over the kept set: lower and upper ends of every entry, total."""
    p = p.double()
    vals, order = p.sort(descending=True, stable=True)
    above = torch.searchsorted(-vals, -vals, right=False)
    mass = torch.cat([torch.zeros(1, dtype=torch.float64), vals.cumsum(0)])[above]
    keep = torch.zeros(p.numel(), dtype=torch.bool)
    keep[order] = (above < k) & (mass <= (tp if tp < 1.0 else float("inf"))) & (vals > 0) & (vals >= mp * vals[0])
    cdf = torch.where(keep, p, torch.zeros((), dtype=torch.float64)).cumsum(0)
    return keep, cdf


@pytest.mark.gpu
@pytest.mark.parametrize("rows,vocab,pad", [(1, 4096, 0), (2, 16384, 0), (3, 32771, 1), (5, 128257, 3), (64, 65536, 0), (40, 131075, 1), (130, 140000, 0)])
def test_fused_call_equals_the_two(ops, rows, vocab, pad):
    """(130 rows: chunks past what a workgroup holds in registers, no lists; 4096: one chunk; odd strides: no 16-byte loads.)  Row 0 has its
    largest entries in the last vocab % 4, row 1 tied with the cut, the last all its mass in one chunk.  Draws: inside float64's interval of
    the entry, 2e-5 of the total wide for the fp32 probabilities' own sum."""
    g = torch.Generator().manual_seed(rows + vocab)
    logits = 2.5 * torch.randn((rows, vocab), generator=g)
    logits[0, -1] = logits[0].max() + 0.25
    logits[0, -2] = logits[0, -1] - 0.5
    if rows > 2:
        logits[1, torch.randperm(vocab, generator=g)[:300]] = 14.0
        logits[-1, : vocab // 64] += 12.0
    temps = (0.6 + 0.6 * torch.rand(rows, generator=g)).to(DEV)
    for k, tp, mp in ((2, 1.0, 0.0), (50, 0.9, 0.0), (1000, 0.999, 0.0), (1 << 30, 0.6, 0.0), (1 << 30, 1.0, 0.0), (300, 0.95, 0.05)):
        ks = torch.full((rows,), k, dtype=torch.int32, device=DEV)
        tps, mps = torch.full((rows,), tp, device=DEV), torch.full((rows,), mp, device=DEV) if mp else None
        u = torch.rand(rows, generator=g).to(DEV)
        a = torch.zeros((rows, vocab + pad), device=DEV)[:, :vocab]
        b = torch.zeros((rows, vocab + pad), device=DEV)[:, :vocab]
        a.copy_(logits)
        b.copy_(logits)
        ids = ops.softmax_sample_(a, temps, ks, tps, mps, u)
        ops.softmax_temperature_(b, temps)
        assert torch.equal(a, b)
        assert torch.equal(ids, ops.top_k_top_p_min_p_sample(b, ks, tps, mps, u)), (k, tp, mp)
        for r in {0, min(1, rows - 1), rows - 1}:
            p, i = b[r].cpu(), int(ids[r])
            ok = False
            for slack in (0.0, -1e-5, 1e-5):      # entries within rounding of the mass limit may go either way
                keep, cdf = _drawn(p, k, tp + (slack if tp < 1.0 else 0.0), mp, u)
                t = float(u[r]) * float(cdf[-1])
                ok |= bool(keep[i]) and cdf[i] >= t - 2e-5 * cdf[-1] and cdf[i] - p[i].double() <= t + 2e-5 * cdf[-1]
            assert ok, (r, k, tp, mp, i)


@pytest.mark.gpu
@pytest.mark.parametrize("vocab", [20000, 65537])
def test_softmax_at_temperatures_that_do_not_divide_once(ops, vocab):
    """Small, large, subnormal, zero, negative and NaN temperatures, and infinite entries, against x / t in the same precision: NaN where
    that has NaN, finite rows within 2e-6 of float64 over the rounded quotients (the quotient's rounding is 2^-24 of up to 100)."""
    g = torch.Generator().manual_seed(vocab)
    temps = torch.tensor([1e-3, 2.0, 7e29, 1e-39, 0.0, -1.5, float("nan"), 1.0, 1.0, 1e31, float("inf")])
    x = torch.randn((len(temps), vocab), generator=g) * 2.0
    x[0] *= 1e-3
    x[7, 5] = float("inf")
    x[8, vocab // 2:] = float("-inf")
    got = x.to(DEV)
    ops.softmax_temperature_(got, temps.to(DEV))
    z = (x / temps[:, None]).double()
    ref = torch.softmax(z, -1)
    got = got.cpu().double()
    bad = ref.isnan().any(-1)
    # an infinite maximum: inf - inf
    bad |= z.amax(-1) == float("inf")
    assert torch.equal(got.isnan().any(-1), bad), (got.isnan().any(-1), bad)
    assert (got[~bad] - ref[~bad]).norm() <= 1e-5 * ref[~bad].norm()
