"""LLM.int8 products of many rows where their outlier columns begin and end: none, one, a block of 64 and its neighbours, columns past the first 16 384, all of
them, more than their region holds; cut into K-slices and not."""
import ctypes as C

import pytest
import torch

from lit_llama_amd import _native as nat
from lit_llama_amd import ops, synth

pytestmark = pytest.mark.gpu


def _reference(x, cb, scb):
    """The restated algorithm in 64 bits but for its own roundings: int8 part, outlier part, the latter's terms by size."""
    xh = x.half().double()
    big = xh.abs() >= 6
    cols = big.any(0)
    sca = xh.masked_fill(big, 0).abs().amax(1)
    inv = torch.where(sca > 0, torch.full_like(sca, 127.0, dtype=torch.float32) / sca.float(), torch.zeros_like(sca, dtype=torch.float32))
    ca = torch.round(xh.float() * inv[:, None]).double()
    ca[:, cols] = 0
    acc = ca @ cb.double().T
    main = ((acc.float() * 6.200012e-05) * sca.float()[:, None]) * scb[None, :]
    w = ((cb[:, cols].float() * scb[:, None]) / torch.full_like(scb, 127.0)[:, None]).half().double()
    return main.half().float(), xh[:, cols] @ w.T, xh[:, cols].abs() @ w.abs().T


@pytest.mark.parametrize("M,N,K,outliers", [
    (33, 72, 200, 1), (64, 4096, 4096, 63), (200, 4096, 4096, 64), (130, 1000, 1024, 65), (257, 4096, 11008, 700), (48, 4096, 22016, 300),
    (1030, 4096, 640, 129), (2050, 1040, 512, 33), (40, 11008, 4096, 4096), (512, 4096, 1024, 0),
    (33, 1001, 4096, 3), (64, 1001, 4096, 5), (64, 4098, 4096, 70), (129, 1003, 2048, 0),  # K-slices whose rows are not whole vectors of four sums
    (2, 4096, 11008, 40), (7, 1001, 4096, 3), (17, 12288, 4096, 70), (31, 260, 4100, 9),  # a few rows
    (100, 12292, 1152, 20), (200, 4100, 4096, 70), (257, 4096, 1030, 9), (65, 260, 12416, 2000),  # blocks of 64 tokens; rows staged element by element, up to 24 fours a thread
])
@pytest.mark.parametrize("epi", ["store", "accum", "pair"])
def test_outlier_columns(dev, M, N, K, outliers, epi):
    """Integer sums are exact; the outlier part is an f32 sum of exact products, so its f16 rounding may fall on either side: one f16 step of that part,
    and one of the sum that it moves; 2^-22 of its terms' sizes for the sum itself."""
    _check_outlier_columns(dev, M, N, K, outliers, epi)


@pytest.mark.parametrize("K", [1024, 1028, 2048, 2052, 4096, 4100, 8192, 8196, 12288, 12292, 16384, 16388, 20480, 20484, 24576, 24580])
def test_rows_at_the_ends_of_what_a_staging_thread_holds(dev, K):
    """1, 2, 4, 8, 12, 16, 20 or 24 groups of four columns a thread, longer rows element by element: outliers in the last four columns, bounds as above."""
    _check_outlier_columns(dev, 40, 132, K, 4, "store", last=True)


@pytest.mark.parametrize("M,N,K,outliers,epi,waves,slices", [
    (40, 32000, 4096, 2100, "store", 4, 1), (150, 32000, 4096, 2100, "store", 8, 1), (260, 32000, 4096, 2100, "accum", 4, 1), (129, 32000, 4096, 2100, "accum", 8, 1),
    (100, 16384, 8192, 4200, "store", 4, 1),
    (64, 8192, 22016, 8200, "store", 4, 3), (150, 8192, 22016, 8200, "accum", 8, 3),
    (150, 22016, 8192, 1480, "pair", 4, 1), (40, 22016, 8192, 1480, "pair", 8, 1), (64, 4096, 22016, 8200, "pair", 4, 3), (33, 5632, 12288, 6000, "pair", 8, 4),
])
def test_more_outlier_columns_than_their_region_holds(dev, M, N, K, outliers, epi, waves, slices):
    """16-bit weights of the outlier columns (whole 64 of them, whole tiles of 16 rows) beyond the region's 128 MB: each is gathered in the product's own blocks, 64 columns a pass, in
    blocks of 4 and 8 waves, of one token block and several, behind K-slices in the launch that sums them.  Bounds as above."""
    R = 2 if epi == "pair" else 1
    assert (N + 15) // 16 * 16 * R * ((outliers + 63) // 64 * 64) * 2 > 128 << 20
    got = C.c_int(0), C.c_int(0)
    nat.lib().mi355_linear_int8_gemm_plan(M, N, K, R, C.byref(got[0]), C.byref(got[1]))
    assert (got[0].value, got[1].value) == (waves, slices)
    _check_outlier_columns(dev, M, N, K, outliers, epi)


def _check_outlier_columns(dev, M, N, K, outliers, epi, last=False):
    g = torch.Generator(device=dev).manual_seed(M + N + K + outliers)
    x = torch.randn((M, K), generator=g, device=dev).clamp_(-5.9, 5.9)
    at = torch.arange(K - outliers, K, device=dev) if last else torch.randperm(K, generator=g, device=dev)[:outliers]
    x[torch.randint(0, M, (outliers,), generator=g, device=dev), at] = 6.0 + 2 * torch.rand(outliers, generator=g, device=dev)
    x = x.to(torch.bfloat16)
    mats = [ops.int8_quant_rows(torch.randn((N, K), generator=g, device=dev) * K ** -0.5) for _ in range(2 if epi == "pair" else 1)]
    stream = ops.repack_i8(mats[0][0], mats[1][0] if epi == "pair" else None, len(mats))
    parts = [_reference(x, *m) for m in mats]
    refs = [(a + b.half().float()).half().float() for a, b, _ in parts]
    tols = [2.0 ** -10 * (b.abs().float() + r.abs()) + 2.0 ** -24 + 2.0 ** -22 * s.float() for (_, b, s), r in zip(parts, refs)]
    if epi == "pair":
        got = ops.linear_int8_gemm(x, stream, mats[0][1], 2, N, K, scb2=mats[1][1], epi=nat.EPI_SWIGLU, out_dtype=torch.float32)
        ref = torch.nn.functional.silu(refs[0]) * refs[1]
        tol = 1.1 * (tols[0] * refs[1].abs() + tols[1] * refs[0].abs()) + 1e-6 + 1e-6 * ref.abs()
    elif epi == "accum":
        base = torch.randn((M, N), generator=g, device=dev)
        got = ops.linear_int8_gemm(x, stream, mats[0][1], 1, N, K, epi=nat.EPI_ACCUM, out=base.clone())
        ref, tol = base + refs[0], tols[0] + 2.0 ** -22 * (base.abs() + refs[0].abs())
    else:
        got = ops.linear_int8_gemm(x, stream, mats[0][1], 1, N, K, out_dtype=torch.float32)
        ref, tol = refs[0], tols[0]
    assert bool(((got - ref).abs() <= tol).all())
    if outliers == 0 and epi == "store":
        assert torch.equal(got, ref)


@pytest.mark.parametrize("T", [32, 100, 300])
def test_a_chain_of_products_clears_the_mask_of_the_next(dev, T):
    """A prompt's LLM.int8 products share a mask of outlier columns that each clears for the next; driven segment by segment each has its own and clears it first: the same
    bits.  Norm scales bring some columns of c_attn, of the c_fc pair and of the head above the threshold, larger rows of the value and c_fc weights some of c_proj and mlp.c_proj, others
    in each layer."""
    from lit_llama_amd import LLaMA, LLaMAConfig
    from lit_llama_amd.utils import EmptyInitOnDevice

    cfg = LLaMAConfig(block_size=320, n_layer=3, n_head=4, n_embd=512, vocab_size=512)
    with EmptyInitOnDevice(device=dev, dtype=torch.bfloat16, quantization_mode="llm.int8"):
        model = LLaMA(cfg)
    sd = synth.make_state_dict(cfg, seed=5, mode="llm.int8", device="cuda", dtype=torch.bfloat16)
    g = torch.Generator().manual_seed(6)
    for k in sd:
        if k.endswith(".scale"):
            sd[k] = (sd[k].float().cpu() * (1 + 4 * (torch.rand(512, generator=g) < 0.02))).to(torch.bfloat16).to(dev)
        if k.endswith(("c_attn.weight", "c_fc1.weight", "c_fc2.weight")):
            larger = 1 + 7 * (torch.rand((sd[k].shape[0], 1), generator=g) < 0.02)
            if k.endswith("c_attn.weight"):
                larger[:1024] = 1  # (queries and keys)
            sd[k] = (sd[k].float().cpu() * larger).to(torch.bfloat16).to(dev)
    model.load_state_dict(sd)
    model.eval()
    eng = model.engine()
    assert eng is not None and eng.gemm_ws is not None, model._engine_failed
    idx = synth.make_prompt(T, vocab=512).to(dev)
    with torch.no_grad():
        got = [model(idx.view(1, -1), 320, torch.arange(T, device=dev))[0].clone() for _ in range(2)]
        torch.cuda.synchronize()
        s = eng.stream.cuda_stream
        with torch.cuda.stream(eng.stream):
            eng.set_step(idx.reshape(-1), T, 0)
            nat.check(nat.lib().mi355_forward_embed(C.byref(eng.m), T, s), "embed")
            columns = []
            for layer in range(cfg.n_layer):
                for seg in range(4):
                    nat.check(nat.lib().mi355_forward_segment(C.byref(eng.m), T, layer, seg, seg + 1, s), "segment")
                    if seg % 2 == 0:  # what c_proj or mlp.c_proj reads
                        rows = (eng.att if seg == 0 else eng.hbuf)[:T]
                        columns.append((rows.abs() >= 6).any(0))
            nat.check(nat.lib().mi355_forward_head(C.byref(eng.m), T, 2, 0, s), "head")
        torch.cuda.synchronize()
    assert all(0 < int(c.sum()) < len(c) for c in columns)
    want = eng.logits[:T]
    assert torch.equal(got[0], want) and torch.equal(got[1], want)
