"""The Sekulorn design on the GPU against the plain restatement in oracle/sekulorn.py: each mechanism's kernels alone, then the model through
its engine, scheduler and generate().  Inputs are made so that a fault shows: keys that stand out just inside and just outside a window,
states that decay slowly, sizes that differ from each other."""
import json

import pytest
import torch

from oracle import sekulorn as O

pytestmark = pytest.mark.gpu


def rel(got, ref):
    """Largest deviation over the reference's root mean square; a bf16 result has its last rounding (2^-8 of the value) for free."""
    free = 2.0 ** -8 if got.dtype == torch.bfloat16 else 0.0
    got, ref = got.detach().double().cpu(), ref.detach().double().cpu()
    assert got.shape == ref.shape
    return float(((got - ref).abs() - free * ref.abs()).max() / ref.pow(2).mean().sqrt().clamp_min(1e-30))


TOL = {torch.float32: 2e-5, torch.bfloat16: 4e-2}  # (the tiles round rotated q and the weights to bf16 in front of loud scores)


# ---------------------------------------------------------------------------------------- window attention
def attention_case(T, H, G, dim, vdim, window, rot, dtype, seed=0, gate=True):
    """Packed projections of one sequence and the oracle's output.  Row window is asked for by three queries: it is the largest key for
    the query that just sees it and for the one that just does not."""
    gen = torch.Generator().manual_seed(seed)
    pad = lambda n: (n + 15) // 16 * 16
    off_q, off_k = 0, pad(H * dim)
    off_v = off_k + pad(G * dim)
    off_g = off_v + pad(G * vdim)
    p = torch.randn((T, off_g + pad(H)), generator=gen)
    q, k, v = p[:, :H * dim].view(T, H, dim), p[:, off_k:off_k + G * dim].view(T, G, dim), p[:, off_v:off_v + G * vdim].view(T, G, vdim)
    for j in range(0, T - 1, max(1, T // 7)):  # key j stands out for the queries at both sides of the window's edge
        loud = torch.randn((G, dim), generator=gen)
        loud[:, :rot] = 0  # (unrotated dimensions: the same direction at every position)
        if dim > rot:
            loud = loud / loud.norm(dim=-1, keepdim=True) * dim ** 0.5
            k[j] = 2 * loud
            for i in (j + window - 1, j + window):
                if i < T:
                    q[i] = 2 * loud.repeat_interleave(H // G, 0)
            v[j] += 3
    p = p.to(dtype)
    pd = p.double()
    base = 5000.0
    q, k = pd[:, :H * dim].view(T, H, dim), pd[:, off_k:off_k + G * dim].view(T, G, dim)
    v, g = pd[:, off_v:off_v + G * vdim].view(T, G, vdim), pd[:, off_g:off_g + H]
    scale = 1.3 * dim ** -0.5
    ref = O.window_attention(O.rotate_pairs(q, rot, base), O.rotate_pairs(k, rot, base), v, scale, window)
    if gate:
        ref = ref * torch.sigmoid(g)[:, :, None]
    inv = torch.tensor([base ** (-2.0 * i / rot) for i in range(rot // 2)], dtype=torch.float64) if rot else None
    kw = dict(heads=H, scale=scale, window=window, off_q=off_q, off_k=off_k, off_v=off_v, off_g=off_g if gate else -1)
    return p, ref.reshape(T, -1), kw, inv


def run_portions(dev, p, kw, inv, dims, cuts, ring, slot=1, path=0, split=False):
    from lit_llama_amd import ops

    G, dim, vdim = dims
    kr = torch.full((3, G, ring, dim), 7.0, dtype=p.dtype, device=dev)  # (a slot somebody used before)
    vr = torch.full((3, G, ring, vdim), 9.0, dtype=p.dtype, device=dev)
    part = torch.zeros(1 << 20, device=dev) if split else None
    out, at = [], 0
    for n in cuts:
        b = ops.PackedBatch([n], [slot], [at], dev)
        out.append(ops.window_attention(p[at:at + n].contiguous().to(dev), b, kr, vr, inv_freq=inv.to(dev) if inv is not None else None,
                                        path=path, partials=part, **kw))
        at += n
    assert at == p.shape[0]
    assert (kr[0] == 7).all() and (kr[2] == 7).all() and (vr[0] == 9).all()
    return torch.cat(out)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("H,G,dim,vdim,window,rot", [(4, 2, 40, 24, 37, 16), (6, 1, 64, 64, 64, 32), (3, 3, 18, 10, 20, 6), (8, 2, 128, 128, 130, 64),
                                                     (10, 1, 72, 200, 1, 8), (2, 1, 32, 16, 500, 0)])
def test_window_attention(dev, dtype, H, G, dim, vdim, window, rot):
    T = 210
    p, ref, kw, inv = attention_case(T, H, G, dim, vdim, window, rot, dtype)
    ring = min(window, T)
    whole = run_portions(dev, p, kw, inv, (G, dim, vdim), [T], ring)
    assert rel(whole, ref) < TOL[dtype]
    for cuts in ([2] * 3 + [T - 6], [100, 1, 64, T - 165], [T - 70] + [1] * 70):
        assert rel(run_portions(dev, p, kw, inv, (G, dim, vdim), cuts, ring), ref) < TOL[dtype], cuts
    assert rel(run_portions(dev, p, kw, inv, (G, dim, vdim), [T], ring, path=1), ref) < TOL[dtype]


def test_window_attention_split_decode_and_larger_ring(dev):
    T, H, G, dim, vdim, window, rot = 700, 4, 1, 64, 32, 600, 64
    p, ref, kw, inv = attention_case(T, H, G, dim, vdim, window, rot, torch.float32, gate=False)
    out = run_portions(dev, p, kw, inv, (G, dim, vdim), [T - 60] + [1] * 60, 640, split=True)
    assert rel(out, ref) < TOL[torch.float32]


DECODE_FORMS = [  # heads, key heads, dim, vdim, window, ring, options
    (8, 2, 128, 128, 1000, 1000, {}), (4, 4, 64, 64, 300, 320, dict(rot=64)), (10, 2, 64, 40, 77, 90, dict(keep=3, slope=True)), (16, 2, 256, 256, 200, 256, dict(rot=32, gate="values")),
    (6, 2, 128, 200, 500, 500, dict(keep=40, sink=True, gate="heads")), (4, 1, 256, 64, 33, 33, dict(softcap=3.0, sink=True)), (8, 1, 64, 128, 600, 700, dict(chunked=True, head_scale=True)),
    (3, 1, 128, 8, 1, 1, dict(gate="heads")), (8, 2, 128, 128, 400, 512, dict(unit=True, rot=64, unit_v=True, gate="heads")), (8, 8, 64, 128, 2000, 2000, dict(unit=True, rot=16, v_first=True, slope=True)),
    (4, 1, 128, 128, 256, 256, dict(borrows=True, rot=128)),
]


@pytest.mark.parametrize("split", [False, True])
@pytest.mark.parametrize("H,G,dim,vdim,window,ring,o", DECODE_FORMS)
def test_decode_rows_on_the_matrix_cores_against_rows(dev, H, G, dim, vdim, window, ring, o, split, odd=False):
    """window_keys_kernel takes what window_rows_kernel takes (path 1), wherever a run of keys ends: first positions, the ring's wrap, the row's own key.  Both sum f32 products in f32
    (1e-4 of a head's size covers the order of up to 2000 terms), so what differs is a rounding of the result now and then: a step of bf16's 8 bits, 2^-7 of it at most.  The cache rows are the same bits."""
    from lit_llama_amd import ops

    gen = torch.Generator(device=dev).manual_seed(H * dim + vdim + window)
    rnd = lambda *s: torch.randn(s, generator=gen, device=dev)  # noqa: E731
    keep, pos = o.get("keep", 0), [0, 1, 31, 32, 33, ring - 1, ring, ring + 5, 3 * ring + 17, 127, 1500]
    kept, B = (keep + 3) // 4 * 4, len(pos)
    off = [0, H * dim, (H + G) * dim, (H + G) * dim + G * vdim]
    proj = rnd(B, off[3] + H * vdim).bfloat16()
    rings = rnd(B, G, kept + ring, dim).bfloat16(), rnd(B, G, kept + ring, vdim).bfloat16()
    if odd:  # of the last key head: an infinite value, one of each sign in one dimension, infinite keys; an infinite value of a row's own
        for b in range(0, B, 2):
            rings[1][b, -1, 0, 1], rings[1][b, -1, ring // 2, 5], rings[1][b, -1, ring // 3, 5] = float("inf"), float("inf"), -float("inf")
        rings[0][2::3, -1, ring // 4, 3] = float("inf")
        proj[1::4, off[3] - vdim + 2] = -float("inf")
    rot = o.get("rot", 0)
    kw = dict(heads=H, scale=1.5 * dim ** -0.5, window=window, off_q=off[0], off_k=off[1], off_v=off[2], off_g=off[3] if "gate" in o else -1, gate_values=o.get("gate") == "values",
              keep=keep, kept=kept, softcap=o.get("softcap", 0.0), chunked=o.get("chunked", False), inv_freq=5000.0 ** (-torch.arange(rot // 2, device=dev).double() * 2 / rot) if rot else None,
              partials=torch.zeros(1 << 22, device=dev) if split else None)
    for name, size in (("sink", H), ("slope", H), ("head_scale", H)):
        if name in o:
            kw[name] = rnd(size).abs() * (0.02 if name == "slope" else 1)
    if "unit" in o:
        kw.update(unit_eps=1e-6, q_norm=rnd(dim).abs(), k_norm=rnd(dim).abs())
    if "unit_v" in o:
        kw["unit_v_eps"] = 1e-6
    if "v_first" in o:
        kw.update(v_first=rnd(B, G * vdim).bfloat16(), v_mix=0.3)
    if "borrows" in o:
        kw.update(role="borrows", kv_rows=rnd(B * G * (dim + vdim)).bfloat16())
    b, got = ops.PackedBatch([1] * B, list(range(B))[::-1], pos, dev), []
    for path in (0, 1):
        kr, vr = rings[0].clone(), rings[1].clone()
        got.append((ops.window_attention(proj, b, kr, vr, path=path, **kw).double(), kr, vr))
    (y, kr, vr), (ref, kr1, vr1) = got
    for kind in (torch.isposinf, torch.isneginf, torch.isnan):
        assert torch.equal(kind(y), kind(ref)), kind
    assert torch.isfinite(ref).all() != odd and ref.nan_to_num(0, 0, 0).abs().max() > 0.1
    y, ref = y.nan_to_num(0, 0, 0), ref.nan_to_num(0, 0, 0)
    size = ref.view(B, H, vdim).square().mean(-1, keepdim=True).sqrt().expand(B, H, vdim).reshape(ref.shape)
    bad = (y - ref).abs() > 2.0 ** -7 * ref.abs() + 1e-4 * size
    assert not bad.any()
    assert torch.equal(kr.view(torch.int16), kr1.view(torch.int16)) and torch.equal(vr.view(torch.int16), vr1.view(torch.int16))


@pytest.mark.parametrize("split", [False, True])
@pytest.mark.parametrize("H,G,dim,vdim,window,ring,o", [f for f in DECODE_FORMS if f[4] > 32 and not {"unit", "rot", "v_first", "borrows"} & set(f[6])] + [(16, 2, 128, 64, 400, 450, {})])
def test_infinite_keys_and_values_of_decode_rows(dev, H, G, dim, vdim, window, ring, o, split):
    """Three bf16 to a weight, one of them 0 as a rule: infinities stay infinities, a key whose score is -inf has no weight, and what is NaN over rows is NaN here."""
    test_decode_rows_on_the_matrix_cores_against_rows(dev, H, G, dim, vdim, window, ring, o, split, odd=True)


@pytest.mark.parametrize("H,G,dim,vdim", [(32, 8, 128, 128), (8, 8, 64, 64), (16, 4, 256, 256), (32, 2, 64, 128), (4, 4, 128, 256), (8, 2, 256, 128)])
def test_decode_rows_on_the_matrix_cores_cost_no_precision(dev, H, G, dim, vdim):
    """The f32 sums of the splits, joined in 64 bits: their error is no larger than window_rows_kernel's (path 1), three lengths and inputs together."""
    from lit_llama_amd import ops

    errors = [0.0, 0.0]
    for seed, (B, keys) in enumerate([(4, 1900), (8, 512), (8, 200)]):
        g = torch.Generator(device=dev).manual_seed(seed)
        rnd = lambda *s: torch.randn(s, generator=g, device=dev).bfloat16()  # noqa: E731
        off = [0, H * dim, (H + G) * dim, (H + G) * dim + G * vdim]
        proj, kr, vr = rnd(B, off[3]), rnd(B, G, keys, dim), rnd(B, G, keys, vdim)
        b = ops.PackedBatch([1] * B, list(range(B)), [keys - 1] * B, dev)
        for path in (0, 1):
            part = torch.full((1 << 21,), float("nan"), device=dev)
            ops.window_attention(proj, b, kr, vr, heads=H, scale=dim ** -0.5, window=keys, off_q=off[0], off_k=off[1], off_v=off[2], path=path, partials=part)
            rec = part[~part.isnan()].view(B, H, -1, vdim + 2).double()
            assert rec.shape[2] > 1
            w = torch.exp(rec[..., 0] - rec[..., 0].amax(-1, keepdim=True))
            y = (rec[..., 2:] * w[..., None]).sum(2) / (rec[..., 1] * w).sum(-1, keepdim=True)
            score = (proj[:, : H * dim].float() * dim ** -0.5).double().view(B, G, H // G, dim) @ kr.double().transpose(-1, -2).contiguous()
            ref = (torch.softmax(score, -1) @ vr.double()).view(B, H, vdim)
            errors[path] += float((y - ref).square().sum() / ref.square().sum())
    assert errors[0] <= errors[1]


def test_far_positions_keep_their_angle(dev):
    """Two rows a million positions in: rotation depends on the distance only."""
    from lit_llama_amd import ops

    H, G, dim, vdim, window, rot = 2, 1, 32, 16, 8, 32
    p, ref, kw, inv = attention_case(6, H, G, dim, vdim, window, rot, torch.float32)
    kr, vr = torch.zeros((1, G, 8, dim), device=dev), torch.zeros((1, G, 8, vdim), device=dev)
    b = ops.PackedBatch([6], [0], [1_000_003], dev)
    kr.zero_()
    kw = dict(kw, window=6)
    y = ops.window_attention(p.to(dev), b, kr, vr, inv_freq=inv.to(dev), **kw)
    # rows 0..4 see cached rows that were never written (zeros here); the last row sees exactly the portion
    ref6 = attention_case(6, H, G, dim, vdim, 6, rot, torch.float32)[1]
    want = O.window_attention(O.rotate_pairs(p[:, :H * dim].double().view(6, H, dim), rot, 5000.0),
                              O.rotate_pairs(p[:, kw["off_k"]:kw["off_k"] + G * dim].double().view(6, G, dim), rot, 5000.0),
                              p[:, kw["off_v"]:kw["off_v"] + G * vdim].double().view(6, G, vdim), kw["scale"], 6)
    want = want * torch.sigmoid(p[:, kw["off_g"]:kw["off_g"] + H].double())[:, :, None]
    assert ref6.shape == want.reshape(6, -1).shape
    assert rel(y[5], want[5].reshape(-1)) < 2e-5


# ---------------------------------------------------------------------------------------- recurrences
def rec_case(kind, T, H, G, dim, vdim, dtype, taps=4, rank=8, tau=8.0, seed=0, strong=False):
    gen = torch.Generator().manual_seed(seed)
    pad = lambda n: (n + 15) // 16 * 16
    sizes = dict(q=G * dim, k=G * dim, v=H * vdim, g=H * vdim, **({"a": H, "b": H} if kind == "delta" else {"a": rank}))
    off, n = {}, 0
    for name, s in sizes.items():
        off[name] = n
        n += pad(s)
    p = torch.randn((T, n), generator=gen)
    if strong:  # decays that nearly erase the state next to ones that keep it, repeated keys with beta near 1
        p[::9, off["a"]:off["a"] + sizes["a"]] *= 30
        p[1::2, off["k"]:off["k"] + G * dim] = p[:1, off["k"]:off["k"] + G * dim]
        if kind == "delta":
            p[:, off["b"]:off["b"] + H] += 4
    p = p.to(dtype)
    w = dict(head_norm=1 + 0.2 * torch.randn(vdim, generator=gen), eps=3e-3)
    if kind == "delta":
        w.update(conv=tuple(0.5 * torch.randn((c, taps), generator=gen) for c in (G * dim, G * dim, H * vdim)),
                 a_log=torch.randn(H, generator=gen) - 1, dt_bias=torch.randn(H, generator=gen))
    else:
        w.update(a2=torch.randn((H * dim, rank), generator=gen) * rank ** -0.5, a2_bias=torch.randn(H * dim, generator=gen) + 1, tau=tau)
    d = p.double()
    part = lambda name: d[:, off[name]:off[name] + sizes[name]]
    if kind == "delta":
        q, k, v = (O.silu(O.short_conv(part(x), w["conv"][i].double())) for i, x in enumerate("qkv"))
        q = O.unit_vector(q.view(T, G, dim)) * dim ** -0.5
        k = O.unit_vector(k.view(T, G, dim))
        g = torch.exp(-torch.exp(w["a_log"].double()) * O.softplus(part("a") + w["dt_bias"].double()))
        o = O.delta_rule(q, k, v.view(T, H, vdim), g, torch.sigmoid(part("b")))
    else:
        z = part("a") @ w["a2"].double().T + w["a2_bias"].double()
        alpha = torch.exp(-O.softplus(-z) / tau).view(T, H, dim)
        o = O.gated_linear_attention(part("q").view(T, H, dim) * dim ** -0.5, part("k").view(T, H, dim), part("v").view(T, H, vdim), alpha)
    ref = O.rms_norm(o, w["head_norm"].double(), w["eps"]).reshape(T, -1) * O.silu(part("g"))
    return p, ref, off, w


def run_rec(dev, kind, p, off, w, H, G, dim, vdim, cuts, path=0, taps=4, slots=(1,)):
    from lit_llama_amd import ops

    state = torch.full((3, H, dim, vdim), 5.0, device=dev)
    ring = torch.full((3, taps, 2 * G * dim + H * vdim), 3.0, dtype=p.dtype, device=dev)
    state[slots[0]] = 0
    kw = {k: (tuple(t.to(dev) for t in v) if isinstance(v, tuple) else v.to(dev) if torch.is_tensor(v) else v) for k, v in w.items()}
    out, at = [], 0
    for n in cuts:
        b = ops.PackedBatch([n], [slots[0]], [at], dev)
        out.append(ops.recurrent(kind, p[at:at + n].contiguous().to(dev), b, state, off=off, kv_heads=G, conv_ring=ring, path=path, **kw))
        at += n
    assert at == p.shape[0]
    assert (state[0] == 5).all() and (state[2] == 5).all() and (ring[0] == 3).all()
    return torch.cat(out)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("kind,H,G,dim,vdim,taps", [("delta", 4, 2, 24, 40, 4), ("delta", 3, 3, 64, 32, 2), ("delta", 2, 1, 130, 70, 5), ("delta", 2, 2, 16, 144, 1),
                                                    ("delta", 1, 1, 33, 17, 9),
                                                    ("gla", 3, 3, 24, 40, 0), ("gla", 2, 2, 130, 70, 0), ("gla", 1, 1, 64, 128, 0)])
def test_recurrences(dev, dtype, kind, H, G, dim, vdim, taps):
    T = 203
    p, ref, off, w = rec_case(kind, T, H, G, dim, vdim, dtype, taps=taps or 4)
    args = (dev, kind, p, off, w, H, G, dim, vdim)
    tol = 5e-5  # (bf16: only the inputs and the stored outputs are rounded)
    for path, cuts in ((1, [T]), (2, [T]), (0, [2, 2, 3, 64, 65, T - 136]), (0, [T - 40] + [1] * 40), (2, [1, 1, 127, T - 129])):
        assert rel(run_rec(*args, cuts, path=path, taps=taps or 4), ref) < tol, (path, cuts)


@pytest.mark.parametrize("kind,H,G,dim,vdim", [("delta", 4, 2, 128, 128), ("delta", 6, 3, 130, 70), ("gla", 4, 4, 128, 128), ("gla", 4, 4, 40, 200), ("delta", 5, 5, 100, 300)])
def test_decode_steps_of_many_sequences_give_those_of_few(dev, kind, H, G, dim, vdim):
    """More workgroups than CUs have four waves, fewer eight: the same f32 sums in another order (300 terms, 2e-6 of their size; three steps of it)."""
    from lit_llama_amd import ops

    B, steps = 300 // H, 3
    p, _, off, w = rec_case(kind, B * steps, H, G, dim, vdim, torch.float32)
    kw = {k: (tuple(t.to(dev) for t in v) if isinstance(v, tuple) else v.to(dev) if torch.is_tensor(v) else v) for k, v in w.items()}
    p = p.view(steps, B, -1).to(dev)
    gen = torch.Generator().manual_seed(7)
    state0, ring0 = torch.randn((B, H, dim, vdim), generator=gen).to(dev), torch.randn((B, 4, 2 * G * dim + H * vdim), generator=gen).to(dev)
    got = []
    for size in (B, 9):
        state, ring, out = state0.clone(), ring0.clone(), []
        for i in range(steps):
            for at in range(0, B, size):
                n = min(size, B - at)
                b = ops.PackedBatch([1] * n, list(range(at, at + n)), [11 + i] * n, dev)
                out.append(ops.recurrent(kind, p[i, at:at + n].contiguous(), b, state, off=off, kv_heads=G, conv_ring=ring, path=1, **kw))
        got.append((torch.cat(out), state, ring))
    assert rel(got[0][0], got[1][0].double().cpu()) < 1e-5 and rel(got[0][1], got[1][1].double().cpu()) < 1e-5
    assert torch.equal(got[0][2], got[1][2])


@pytest.mark.parametrize("counts", [[3, 0, 2], [0, 2, 1], [0, 20, 0, 9]])
@pytest.mark.parametrize("kind,H,dim,vdim", [("delta", 4, 128, 128), ("delta", 2, 16, 144), ("delta", 1, 64, 1000), ("gla", 4, 128, 128)])
def test_sequences_without_rows_keep_their_state(dev, kind, H, dim, vdim, counts):
    """An empty portion between others: its slot's state and ring keep their bits, the other sequences give the bits that they give without it."""
    from lit_llama_amd import ops

    p, _, off, w = rec_case(kind, sum(counts), H, H, dim, vdim, torch.float32)
    kw = {k: (tuple(t.to(dev) for t in v) if isinstance(v, tuple) else v.to(dev) if torch.is_tensor(v) else v) for k, v in w.items()}
    gen = torch.Generator().manual_seed(5)
    state0, ring0 = torch.randn((len(counts), H, dim, vdim), generator=gen).to(dev), torch.randn((len(counts), 4, 2 * H * dim + H * vdim), generator=gen).to(dev)
    for path in (0, 1) + ((2,) if vdim <= 256 else ()):
        got = []
        for keep in (range(len(counts)), [i for i, n in enumerate(counts) if n]):
            state, ring = state0.clone(), ring0.clone()
            b = ops.PackedBatch([counts[i] for i in keep], list(keep), [7] * len(keep), dev)
            got.append((ops.recurrent(kind, p.to(dev), b, state, off=off, kv_heads=H, conv_ring=ring, path=path, **kw), state, ring))
        for a, b in zip(*got):
            assert torch.isfinite(a).all() and torch.equal(a, b), path
        for i in [i for i, n in enumerate(counts) if n == 0]:
            assert torch.equal(got[0][1][i], state0[i]) and torch.equal(got[0][2][i], ring0[i]), path


@pytest.mark.parametrize("kind,H,dim,vdim,counts,rows", [
    ("delta", 32, 128, 128, list(range(1, 25)), True), ("gla", 32, 128, 128, list(range(9, 33)), True), ("delta", 16, 100, 120, [16], True), ("gla", 8, 128, 96, [17, 3], True),
    ("delta", 16, 128, 128, [40], False), ("gla", 4, 64, 128, [12, 12], False), ("delta", 4, 128, 200, [9], False), ("gla", 32, 128, 128, [65] * 8, False),
])
def test_short_prompts_go_by_rows_or_in_chunks(dev, kind, H, dim, vdim, counts, rows):
    """What the estimate takes, bit for bit, and the other path: the same f32 recurrence in another order.  Bound: each is within 5e-5 of 64 bits by this measure (test_recurrences; rows whose norm is
    near sqrt(eps) are stretched by the output norm), so 1e-4 of each other."""
    from lit_llama_amd import ops

    G = H // 2 if kind == "delta" else H
    p, _, off, w = rec_case(kind, sum(counts), H, G, dim, vdim, torch.float32)
    kw = {k: (tuple(t.to(dev) for t in v) if isinstance(v, tuple) else v.to(dev) if torch.is_tensor(v) else v) for k, v in w.items()}
    got = {}
    for path in (0, 1, 2):
        state = torch.zeros((len(counts), H, dim, vdim), device=dev)
        ring = torch.zeros((len(counts), 4, 2 * G * dim + H * vdim), device=dev)
        b = ops.PackedBatch(counts, list(range(len(counts))), [0] * len(counts), dev)
        y = ops.recurrent(kind, p.to(dev), b, state, off=off, kv_heads=G, conv_ring=ring, path=path, **kw)
        got[path] = y, state, ring
    assert all(torch.equal(a, b) for a, b in zip(got[0], got[1 if rows else 2]))
    assert rel(got[1][0], got[2][0].double().cpu()) < 1e-4 and rel(got[1][1], got[2][1].double().cpu()) < 1e-4
    assert torch.equal(got[1][2], got[2][2])


@pytest.mark.parametrize("kind,tau", [("delta", 1.0), ("gla", 1.0), ("gla", 16.0)])
def test_recurrences_with_strong_decays_and_repeated_keys(dev, kind, tau):
    T, H, G, dim, vdim = 300, 2, 2, 48, 32
    p, ref, off, w = rec_case(kind, T, H, G, dim, vdim, torch.float32, tau=tau, strong=True, seed=3)
    for path in (1, 2):
        out = run_rec(dev, kind, p, off, w, H, G, dim, vdim, [T], path=path)
        assert torch.isfinite(out).all()
        assert rel(out, ref) < 2e-4, path


# ---------------------------------------------------------------------------------------- the model
def small_config(**kw):
    att = lambda **m: {"type": "attention", "mixer": {"heads": 4, "kv_heads": 2, "dim": 24, "vdim": 40, "scale": 0.3, "mask": {"size": 19},
                                                      "rot": {"base": 900.0, "dims": 8}, **m}, "mlp": {"kind": "dense", "ff": 72}}
    gla = {"type": "gla", "mixer": {"heads": 3, "dim": 20, "vdim": 28, "tau": 4.0}, "mlp": {"kind": "dense", "ff": 40}}
    delta = {"type": "delta", "mixer": {"heads": 6, "kv_heads": 2, "dim": 12, "vdim": 20, "conv": 3}, "mlp": None}
    return {"architecture": "Sekulorn", "vocab": 211, "width": 104, "norm": {"eps": 3e-5}, "residual_mult": 0.45,
            "layers": [delta, att(), {**att(kv_heads=4, dim=32, vdim=8), "mlp": None}, gla], "loop": {"start": 1, "stop": 3, "times": 3}, **kw}


def build(config, dtype, dev, seed=1):
    from lit_llama_amd import synth
    from lit_llama_amd.registry import build_model

    sd = synth.make_hybrid_state_dict(config, seed=seed, rank=5)
    m = build_model(config, dtype, dev)
    m.load_state_dict(sd)
    return m, sd


def tokens_of(n, vocab=211, seed=0):
    return torch.randint(0, vocab, (n,), generator=torch.Generator().manual_seed(seed)).tolist()


CONFIGS = {
    "mixed": small_config(),
    "no loop, unit multiplier": small_config(loop=None, residual_mult=1.0),
    "no rotation, no window": small_config(layers=[{"type": "attention", "mixer": {"heads": 3, "kv_heads": 1, "dim": 16, "vdim": 16, "scale": 0.25},
                                                    "mlp": None}], loop=None, width=64),
    "all looped": small_config(loop={"start": 0, "stop": 4, "times": 2}, width=97, vocab=130),
}


@pytest.mark.parametrize("name", CONFIGS)
def test_model_layer_by_layer_and_logits(dev, name):
    from lit_llama_amd.hybrid_engine import Entry

    config = CONFIGS[name]
    m, sd = build(config, torch.float32, dev)
    eng = m.engine()
    eng.ensure(2, 128)
    toks = tokens_of(61, config["vocab"])
    logits, trail = O.forward(config, sd, toks)
    assert eng.run_layers == O.layer_order(config)
    for r in range(1, len(trail) + 1):
        s = eng.acquire()
        assert rel(eng.residual_after([Entry(s, 0, toks, [])], r), trail[r - 1]) < 5e-5, r
        eng.release(s)
    s = eng.acquire()
    assert rel(eng.step([Entry(s, 0, toks, range(61))]), logits) < 5e-5
    eng.release(s)


@pytest.mark.parametrize("runs", [3, 40])  # (one launch's regions, and more)
def test_a_slot_is_cleared_in_every_run_and_no_other_slot_is(dev, runs):
    import ctypes as C

    from lit_llama_amd import _native as nat

    sizes = [(3, 5, 7), (4, 128, 128), (1, 1, 1), (2, 64, 33)]
    layers, states, shifts = (nat.HybridLayer * runs)(), [], []
    for i in range(runs):
        H, d, v = sizes[i % 4]
        states.append(torch.ones((4, H, d, v), device=dev))
        shifts.append(torch.ones((4, 30), device=dev))
        l = layers[i]
        l.mixer, l.n_mix, l.shift = 1, i % 2, shifts[i].data_ptr()
        l.rec.heads, l.rec.dim, l.rec.vdim, l.rec.state = H, d, v, states[i].data_ptr()
    m = nat.HybridModel()
    m.n_runs, m.width, m.layers = runs, 30, layers
    stream = torch.cuda.current_stream().cuda_stream
    slots = torch.tensor([3, 0], dtype=torch.int32, device=dev)
    nat.check(nat.lib().mi355_hybrid_reset_slot(C.byref(m), 1, stream), "reset_slot")
    for live in ([0, 2, 3], [2]):
        for i in range(runs):
            for t, cleared in ((states[i], True), (shifts[i], i % 2 == 1)):
                assert [bool((t[s] == 1).all()) for s in range(4)] == [s in live or not cleared for s in range(4)], (i, live)
                assert not cleared or all(bool((t[s] == 0).all()) for s in range(4) if s not in live)
        nat.check(nat.lib().mi355_hybrid_reset_slots(C.byref(m), slots.data_ptr(), 2, stream), "reset_slots")


def test_more_slots_are_cleared_than_a_grid_is_high(dev):
    import ctypes as C

    from lit_llama_amd import _native as nat

    states = [torch.ones((5, 2, 3, 4), device=dev), torch.ones((5, 1, 1, 3), device=dev)]
    layers = (nat.HybridLayer * 2)()
    for l, t in zip(layers, states):
        l.mixer = 1
        l.rec.heads, l.rec.dim, l.rec.vdim, l.rec.state = *t.shape[1:], t.data_ptr()
    m = nat.HybridModel()
    m.n_runs, m.width, m.layers = 2, 30, layers
    slots = torch.tensor([1, 4], dtype=torch.int32, device=dev).repeat(40000)
    nat.check(nat.lib().mi355_hybrid_reset_slots(C.byref(m), slots.data_ptr(), slots.numel(), torch.cuda.current_stream().cuda_stream), "reset_slots")
    for t in states:
        assert [bool((t[s] == (s not in (1, 4))).all()) for s in range(5)] == [True] * 5


def test_tokens_in_any_form(dev):
    """Lists of numbers, of scalars on the device or the host, arrays, tensors: the same step."""
    from lit_llama_amd.hybrid_engine import Entry

    m, _ = build(CONFIGS["mixed"], torch.float32, dev)
    eng = m.engine()
    eng.ensure(2, 64)
    toks, got = tokens_of(7), []
    for form in (list, tuple, torch.tensor, lambda t: torch.tensor(t, device=dev), lambda t: list(torch.tensor(t, device=dev)), lambda t: [torch.tensor(t[0]), *t[1:]], lambda t: torch.tensor(t).numpy()):
        slots = [eng.acquire(), eng.acquire()]
        out = [eng.step([Entry(slots[0], 0, form(toks[:5]), [1, 4]), Entry(slots[1], 0, form(toks[5:6]), [0])]).clone()]
        out.append(eng.step([Entry(slots[0], 5, form(toks[5:6]), [0]), Entry(slots[1], 1, form(toks[6:]), [0])]).clone())
        got.append(torch.cat(out))
        for s in slots:
            eng.release(s)
    assert got[0].shape[0] == 5 and all(torch.equal(g, got[0]) for g in got[1:])


@pytest.mark.parametrize("name,dtype,tol", [("mixed", torch.float32, 1e-4), ("mixed", torch.bfloat16, 0.12), ("all looped", torch.bfloat16, 0.12)])
def test_portions_batches_slots_and_decoding(dev, name, dtype, tol):
    """Unequal requests in one batch, cut differently, decoded together, their slots used again: the logits of each alone."""
    from lit_llama_amd.hybrid_engine import Entry

    config = CONFIGS[name]
    m, sd = build(config, dtype, dev)
    eng = m.engine()
    eng.ensure(4, 200)
    seqs = [tokens_of(n, config["vocab"], seed=n) for n in (150, 9, 64, 33)]
    refs = [O.forward(config, sd, s)[0] for s in seqs]
    for first in ((100, 2, 31, 32), (64, 8, 1, 3)):  # (the second time in the slots of the first)
        slots = [eng.acquire() for _ in seqs]
        at = [0] * 4
        got = [[] for _ in seqs]

        def feed(counts):
            es = []
            for i, n in enumerate(counts):
                n = min(n, len(seqs[i]) - at[i])
                if n:
                    es.append((i, Entry(slots[i], at[i], seqs[i][at[i]:at[i] + n], range(n))))
            lg = eng.step([e for _, e in es]).clone().split([len(e.tokens) for _, e in es])
            for (i, e), x in zip(es, lg):
                got[i].append(x)
                at[i] += len(e.tokens)

        feed(first)
        feed((2, 1, 2, 30))      # a mixed batch: two-row portions and single rows
        while any(a < len(s) for a, s in zip(at, seqs)):
            feed((1, 1, 1, 1))
        for i in range(4):
            assert rel(torch.cat(got[i]), refs[i]) < tol, (i, first)
        for s in slots:
            eng.release(s)
    assert eng.slots.live == 0


def test_a_step_larger_than_the_scratch_is_cut(dev):
    from lit_llama_amd.hybrid_engine import Entry, HybridEngine

    config = CONFIGS["mixed"]
    m, sd = build(config, torch.float32, dev)
    eng = HybridEngine(m, max_rows=48)
    eng.ensure(3, 200)
    seqs = [tokens_of(n, seed=n) for n in (130, 17, 60)]
    slots = [eng.acquire() for _ in seqs]
    out = eng.step([Entry(s, 0, t, [0, len(t) - 1]) for s, t in zip(slots, seqs)])
    ref = torch.cat([O.forward(config, sd, t)[0][[0, len(t) - 1]] for t in seqs])
    assert rel(out, ref) < 1e-4


def test_bad_input_is_an_error_on_the_host(dev):
    from lit_llama_amd._native import NativeError
    from lit_llama_amd.hybrid_engine import Entry

    m, _ = build(CONFIGS["mixed"], torch.float32, dev)
    eng = m.engine()
    eng.ensure(1, 16)
    s = eng.acquire()
    for entry in (Entry(s, 0, [0] * 17, []), Entry(s, 0, [211], []), Entry(s, 0, [-1], []), Entry(s, 0, [1, 2], [1, 0])):
        with pytest.raises(NativeError):
            eng.step([entry])


def greedy_reference(config, sd, prompt, n, margin):
    """Greedy continuation by the oracle, up to the first near tie."""
    seq = list(prompt)
    for _ in range(n):
        top = torch.topk(O.forward(config, sd, seq)[0][-1], 2)
        if float(top.values[0] - top.values[1]) < margin:
            break
        seq.append(int(top.indices[0]))
    return seq[len(prompt):]


def test_greedy_generation_through_generate_and_the_scheduler(dev):
    import lit_llama_amd
    from lit_llama_amd.batching import generate_batch

    config = CONFIGS["mixed"]
    m, sd = build(config, torch.float32, dev)
    prompts = [tokens_of(n, seed=n) for n in (23, 3, 40, 1, 18)]
    refs = [greedy_reference(config, sd, p, 12, 1e-3) for p in prompts]
    assert sum(map(len, refs)) > 30
    outs = generate_batch(m, prompts, 12, top_k=1, max_batch=3, portion=16)  # (requests wait, enter late, are cut)
    for o, r in zip(outs, refs):
        assert len(o) == 12 and o[:len(r)] == r
    assert m.engine().slots.live == 0
    for p, r in zip(prompts[:2], refs):
        y = lit_llama_amd.generate(m, torch.tensor(p, device=dev), 12, top_k=1).tolist()
        assert y[:len(p)] == p and len(y) == len(p) + 12 and y[len(p):len(p) + len(r)] == r
    again = lit_llama_amd.generate(m, torch.tensor(prompts[0], device=dev), 12, top_k=1).tolist()
    assert again[len(prompts[0]):] == outs[0]
    # a batch behind generate() that needs longer rings than its sequence
    fresh, _ = build(config, torch.float32, dev)
    lit_llama_amd.generate(fresh, torch.tensor([1, 2, 3], device=dev), 2, top_k=1)
    assert generate_batch(fresh, prompts[:2], 12, top_k=1) == outs[:2]
    # eos ends a request early and the others go on
    eos = outs[0][4]
    cut = generate_batch(m, prompts, 12, top_k=1, eos_id=eos)
    assert cut[0] == outs[0][:outs[0].index(eos)]


def test_sampled_generation(dev):
    import lit_llama_amd
    from lit_llama_amd.batching import generate_batch

    config = CONFIGS["mixed"]
    m, _ = build(config, torch.bfloat16, dev)
    p = tokens_of(20)
    torch.manual_seed(5)
    a = lit_llama_amd.generate(m, torch.tensor(p, device=dev), 40, temperature=0.7, top_k=20)
    torch.manual_seed(5)
    b = lit_llama_amd.generate(m, torch.tensor(p, device=dev), 40, temperature=0.7, top_k=20)
    assert torch.equal(a, b) and int(a.max()) < 211
    x = generate_batch(m, [p, p[:7]], 15, temperature=0.9, top_k=50, seed=3)
    y = generate_batch(m, [p, p[:7]], 15, temperature=0.9, top_k=50, seed=3)
    assert x == y and [len(o) for o in x] == [15, 15]


def test_a_dropped_model_frees_its_engine_without_the_collector(dev):
    import gc
    import weakref

    from lit_llama_amd.hybrid_engine import Entry

    m, _ = build(CONFIGS["mixed"], torch.float32, dev)
    eng = m.engine()
    eng.ensure(1, 16)
    s = eng.acquire()
    for i in range(4):  # (a captured step included)
        eng.step([Entry(s, i, [i], [0])])
    alive = weakref.ref(eng)
    gc.collect()
    gc.disable()
    try:
        del eng, m
        assert alive() is None
    finally:
        gc.enable()


def test_long_decoding_matches_the_prompt_pass(dev):
    """Hundreds of decoded tokens (windows pass over them, graphs replayed, eager work in between) against one prompt pass."""
    from lit_llama_amd.hybrid_engine import Entry

    config = CONFIGS["mixed"]
    m, sd = build(config, torch.float32, dev)
    eng = m.engine()
    eng.ensure(2, 400)
    toks = tokens_of(380)
    s, t = eng.acquire(), eng.acquire()
    whole = eng.step([Entry(s, 0, toks, range(380))]).clone()
    rows = [eng.step([Entry(t, 0, toks[:5], range(5))]).clone()]
    for i in range(5, 380):
        rows.append(eng.step([Entry(t, i, toks[i:i + 1], [0])]).clone())
        if i % 50 == 0:
            torch.randn(1000, device=dev).sum().item()
    assert rel(torch.cat(rows), whole) < 2e-4
    assert rel(whole[-1:], O.forward(config, sd, toks)[0][-1:]) < 1e-4


def test_module_forward_and_cache_reset(dev):
    config = CONFIGS["mixed"]
    m, sd = build(config, torch.float32, dev)
    toks = torch.tensor([tokens_of(30, seed=1), tokens_of(30, seed=2)], device=dev)
    out = m(toks)
    for i in range(2):
        assert rel(out[i], O.forward(config, sd, toks[i].tolist())[0]) < 1e-4
    for _ in range(2):
        a = m(toks[:1, :29], 64, torch.arange(29, device=dev))
        b = m(toks[:1, 29:], 64, torch.tensor([29], device=dev))
        assert rel(torch.cat([a[0], b[0]]), out[0]) < 1e-4
        m.reset_cache()


def test_trace_replay_and_command_line(dev, tmp_path, capsys, monkeypatch):
    import io

    import numpy as np
    from safetensors.torch import save_file

    from lit_llama_amd import __main__ as cli
    from lit_llama_amd import synth, trace

    config = CONFIGS["all looped"]
    sd = synth.make_hybrid_state_dict(config, seed=9, rank=3)
    (tmp_path / "config.json").write_text(json.dumps(config))
    save_file(sd, str(tmp_path / "model.safetensors"))
    a, b = tokens_of(25, 130, 1), tokens_of(11, 130, 2)
    steps = [{"step": 0, "entries": [{"id": "a", "tokens": a[:20], "want": [0, 19]}, {"id": "b", "tokens": b[:8], "want": []}], "end": []},
             {"step": 1, "entries": [{"id": "a", "tokens": a[20:21], "want": [0]}, {"id": "b", "tokens": b[8:9], "want": [0]}], "end": ["b"]},
             {"step": 2, "entries": [{"id": "a", "tokens": a[21:22], "want": []}], "end": ["a"]}]
    monkeypatch.setattr("sys.stdin", io.StringIO("\n".join(map(json.dumps, steps)) + "\n"))
    assert trace.main(["--model", str(tmp_path), "--dtype", "float32", "--out", str(tmp_path), "--max-tokens", "64"]) == 0
    assert capsys.readouterr().out.split("\n")[:3] == ["done 0", "done 1", "done 2"]
    ra, rb = O.forward(config, sd, a)[0], O.forward(config, sd, b)[0]
    got = [torch.from_numpy(np.fromfile(tmp_path / f"{i}.f32", "<f4").reshape(-1, 130)) for i in (0, 1)]
    assert rel(got[0], ra[[0, 19]]) < 1e-4 and rel(got[1], torch.stack([ra[20], rb[8]])) < 1e-4
    assert not (tmp_path / "2.f32").exists()
    assert cli.main(["--model", str(tmp_path), "--dtype", "float32", "--prompt-ids", ",".join(map(str, a)), "--prompt-ids", "1,2", "--top-k", "1",
                     "--max-new-tokens", "5"]) == 0
    lines = capsys.readouterr().out.strip().split("\n")
    assert len(lines) == 2 and lines[0].startswith(",".join(map(str, a))) and len(lines[0].split(",")) == 30


@pytest.mark.parametrize("width,batch", [(1024, 9), (1152, 16), (4096, 33), (8192, 10), (8320, 10)])
def test_norm_behind_the_slices_of_a_residual_product(dev, width, batch):
    """Batches whose residual products are cut along K, the norm of the next product taken with their sum (rows of up to 8192) or by itself, in front of
    products of either kind of layer, the next layer's and the head: the logits of each sequence alone, whose norms are taken in the row kernel."""
    from lit_llama_amd.hybrid_engine import Entry

    att = {"type": "attention", "mixer": {"heads": 9, "kv_heads": 3, "dim": 128, "vdim": 128, "scale": 0.09, "mask": {"size": 19}}}
    config = small_config(layers=[{**att, "mlp": {"kind": "dense", "ff": 1280}}, {**att, "mlp": None}], loop=None, width=width)
    m, _ = build(config, torch.bfloat16, dev)
    eng = m.engine()
    eng.ensure(batch + 1, 64)
    seqs = [tokens_of(3, seed=i) for i in range(batch)]

    def steps(group):
        slots = [eng.acquire() for _ in group]
        out = [eng.step([Entry(s, j, t[j:j + 1], [0]) for s, t in zip(slots, group)]).clone() for j in range(3)]
        for s in slots:
            eng.release(s)
        return torch.stack(out)

    got = steps(seqs)
    for i, t in enumerate(seqs):
        # (both sides round the same values to bf16; a value at the edge of a rounding falls either way: a few 2^-9 of the terms over four products)
        assert rel(got[:, i].float(), steps([t])[:, 0].float()) < 4e-2, i


@pytest.mark.parametrize("batch,taken", [(4, False), (8, False), (9, True)])
def test_norm_of_rows_only_in_front_of_a_product_that_takes_it(dev, batch, taken):
    """Hidden rows of more than 12288 leave through the tiled product from 3 rows on, with its K-slices' sum; what stands behind them takes rows that are normed
    already only if it is tiled too, from 9 rows on.  Before that nobody writes (or reads) normed rows."""
    from lit_llama_amd.hybrid_engine import Entry

    att = {"type": "attention", "mixer": {"heads": 9, "kv_heads": 3, "dim": 128, "vdim": 128, "scale": 0.09, "mask": {"size": 19}}}
    config = small_config(layers=[{**att, "mlp": {"kind": "dense", "ff": 12416}}, {**att, "mlp": None}], loop=None, width=1024)
    m, _ = build(config, torch.bfloat16, dev)
    eng = m.engine()
    eng.ensure(batch + 1, 64)
    seqs = [tokens_of(3, seed=i) for i in range(batch)]
    normed = next(t for t in eng._keep if t.data_ptr() == eng.m.xb)

    def steps(group):
        slots = [eng.acquire() for _ in group]
        out = [eng.step([Entry(s, j, t[j:j + 1], [0]) for s, t in zip(slots, group)]).clone() for j in range(3)]
        for s in slots:
            eng.release(s)
        return torch.stack(out)

    normed.fill_(7.0)
    got = steps(seqs)
    assert bool((normed != 7.0).any()) == taken
    for i, t in enumerate(seqs):
        # (the same values rounded to bf16 on both sides, a value at the edge of a rounding either way: a few 2^-9 of the terms over four products)
        assert rel(got[:, i].float(), steps([t])[:, 0].float()) < 4e-2, i


@pytest.mark.parametrize("width,batch", [(128, 9), (1024, 16), (1152, 33), (4096, 20), (8192, 12)])
def test_norm_taken_with_a_sum_of_slices(dev, width, batch):
    """What the sum of the last residual product's slices leaves for the head: bf16(x rinv scale) of the rows that it writes, to one step of bf16 (its own rounding;
    the factors in front of it are f32)."""
    from lit_llama_amd.hybrid_engine import Entry

    att = {"type": "attention", "mixer": {"heads": 9, "kv_heads": 3, "dim": 128, "vdim": 128, "scale": 0.09, "mask": {"size": 19}}}
    m, sd = build(small_config(layers=[{**att, "mlp": None}, {**att, "mlp": {"kind": "dense", "ff": 1280}}], loop=None, width=width), torch.bfloat16, dev)
    eng = m.engine()
    eng.ensure(batch, 64)
    normed = next(t for t in eng._keep if t.data_ptr() == eng.m.xb)
    normed.fill_(7.0)
    eng.step([Entry(eng.acquire(), 0, tokens_of(1, seed=i), [0]) for i in range(batch)])
    got = normed[:batch * width].view(batch, width).double()
    x = eng.x.view(-1, eng.m.ldx)[:batch, :width].double()
    ref = x * (x.square().mean(1, keepdim=True) + 3e-5).rsqrt() * sd["final.norm"].to(torch.bfloat16).to(dev).double()
    assert ((got - ref).abs() <= 2.0 ** -8 * ref.abs() + 1e-6).all()
