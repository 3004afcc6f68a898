"""Per-head norms, rotations and gates where lanes share a row in 16-byte pieces: widths, rotations and strides at the edges of that form."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _rows(x, w, eps, pos, freq, rot, interleaved, mag, norm=True):
    """float64 (values, the magnitude that rounding errors of the fp32 steps scale with)"""
    x = x.double()
    if norm:
        x = x / (x.pow(2).mean(-1, keepdim=True) + eps).sqrt()
    if w is not None:
        x = x * w.double()
    size = x.abs()
    if rot:
        ang = (pos.float()[:, None] * freq[None, : rot // 2]).double()[:, None]
        c, s = ang.cos() * mag, ang.sin() * mag
        a, b = (x[..., 0:rot:2], x[..., 1:rot:2]) if interleaved else (x[..., : rot // 2], x[..., rot // 2: rot])
        na, nb, m = a * c - b * s, b * c + a * s, (a.abs() + b.abs()) * mag
        x, size = x.clone(), size.clone()
        if interleaved:
            x[..., 0:rot:2], x[..., 1:rot:2], size[..., 0:rot:2], size[..., 1:rot:2] = na, nb, m, m
        else:
            x[..., : rot // 2], x[..., rot // 2: rot], size[..., : rot // 2], size[..., rot // 2: rot] = na, nb, m, m
    return x, size


def _close(got, want, size, what):
    """u of the stored value and 32 fp32 roundings (sum of squares, root, sine) of what went into it"""
    u = 0.0 if got.dtype == torch.float32 else torch.finfo(got.dtype).eps / 2
    tiny = 0.0 if got.dtype != torch.float16 else 2.0 ** -25
    err = (got.double() - want).abs()
    bound = u * want.abs() + 32 * 2.0 ** -24 * size * (1 + u) + tiny
    assert bool((err <= bound).all()), (what, (err / bound).max().item())


# (d, dv, rot, interleaved): one lane a row; idle lanes in a row (24, 96); the widest; one past it and a rotation that is no
# multiple of a piece (the form for any width); 37 tokens, and as many as lead rows narrower than 128 and more than one pass of a
# token's rows through a workgroup there
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,d,dv,rot,interleaved", [(2300, 8, 8, 8, True), (600, 24, 16, 16, False), (300, 64, 64, 64, False), (200, 96, 64, 48, False),
                                                    (1030, 128, 96, 64, True), (1030, 64, 512, 64, False)] + [(37, *c) for c in [(8, 8, 8, True), (24, 16, 16, False), (64, 128, 64, False), (96, 64, 48, False), (128, 96, 64, True),
                                                  (512, 256, 512, False), (128, 128, 0, False), (520, 64, 16, False), (64, 64, 20, False), (60, 64, 16, True)]])
def test_norm_rotate_and_write(dt, T, d, dv, rot, interleaved):
    from sglang_custom_amd import ops

    g = torch.Generator().manual_seed(d + dv + rot)
    H, G, eps, mag = 5, 3, 1e-5, 1.25
    rows = torch.randn(T, (H + G) * d + G * dv, generator=g).to(dt).to(DEV)
    q, k, v = rows[:, : H * d].view(T, H, d), rows[:, H * d: (H + G) * d].view(T, G, d), rows[:, (H + G) * d:].view(T, G, dv)
    wq, wk = (torch.randn(2, d, generator=g) + 1).to(dt).to(DEV)
    pos = torch.randint(0, 9000, (T,), generator=g).to(DEV)
    freq = (torch.rand(max(rot // 2, 1), generator=g) * 0.7).to(DEV)
    loc = torch.randperm(T + 4, generator=g)[:T].to(DEV)
    kc = torch.full((T + 4, G, d), 7.0, dtype=dt, device=DEV)
    vc = torch.full((T + 4, G, dv), 7.0, dtype=dt, device=DEV)
    got = ops.qkv_norm_rope_write(q, k, v, wq, wk, eps, pos, freq, rot, interleaved, mag, kc, vc, loc)
    _close(got, *_rows(q, wq, eps, pos, freq, rot, interleaved, mag), "q")
    _close(kc[loc], *_rows(k, wk, eps, pos, freq, rot, interleaved, mag), "k")
    _close(vc[loc], *_rows(v, None, eps, pos, freq, 0, interleaved, mag), "v")
    rest = torch.ones(T + 4, dtype=torch.bool, device=DEV)
    rest[loc] = False
    assert bool((kc[rest] == 7).all()) and bool((vc[rest] == 7).all())
    # the same rows one by one: with and without a norm, in fp32, and from rows that start off a 16-byte piece
    wide = torch.zeros(T, H * d + 3, dtype=dt, device=DEV)
    wide[:, 1: 1 + H * d] = q.reshape(T, H * d)
    for src, w, out in ((q, wq, torch.float32), (q, None, dt), (wide[:, 1: 1 + H * d].view(T, H, d), wq, dt)):
        want, size = _rows(q, w, eps, pos, freq, rot, interleaved, mag, norm=w is not None)
        _close(ops.head_norm_rope(src, w, eps, pos, freq, rot, interleaved, 0.5, out, rot_mag=mag), want * 0.5, size * 0.5, "rows")


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,H,dv,pad", [(37, 5, 8, 0), (37, 3, 96, 8), (5, 4, 128, 1), (9, 2, 512, 0), (9, 1, 520, 0), (7, 3, 36, 0), (6600, 5, 8, 0), (1000, 3, 96, 8), (600, 4, 128, 1), (600, 4, 128, 8)])
def test_norm_and_gate(dt, T, H, dv, pad):
    from sglang_custom_amd import ops

    g = torch.Generator().manual_seed(T * dv + H)
    o = torch.randn(T, H, dv, generator=g).to(DEV)
    gate = torch.randn(T, H * dv + pad, generator=g).to(dt).to(DEV)[:, : H * dv]
    z = gate.double().view(T, H, dv)
    for act, n_w in (("silu", 0), ("silu", dv), ("sigmoid", H * dv)):
        w = (torch.randn(n_w, generator=g) + 1).to(dt).to(DEV) if n_w else None
        f = torch.sigmoid(z) * (z if act == "silu" else 1.0)
        want = _rows(o, None if w is None else w.view(-1, dv), 1e-6, None, None, 0, False, 1.0)[0] * f
        _close(ops.head_rmsnorm_gate_act(o, w, gate, 1e-6, dt, act).view(T, H, dv), want, want.abs() + 1e-6, act)
    w = (torch.randn(H * dv, generator=g) + 1).to(dt).to(DEV)
    y = o.view(T, H * dv).double() * (gate.double() * torch.sigmoid(gate.double()))
    want = _rows(y.view(T, H, dv), w.view(H, dv), 1e-6, None, None, 0, False, 1.0)[0].view(T, H * dv)
    _close(ops.gated_group_rmsnorm(o.view(T, H * dv), gate, w, H, 1e-6), want, want.abs() + 1e-6, "groups")
