"""The tiled products at the sizes where their blocks, K-slices and pipelines end: every number of tokens per block, odd rows and columns, slices of
few units, launches that are cut and launches that are not."""
import ctypes as C

import pytest
import torch

from lit_llama_amd import _native as nat
from lit_llama_amd import ops, synth
from lit_llama_amd.model import LLaMA, LLaMAConfig
from lit_llama_amd.utils import EmptyInitOnDevice

pytestmark = pytest.mark.gpu

SHAPES = [  # M, N, K
    (1, 16, 128), (9, 144, 300), (15, 4096, 4096), (16, 1000, 640), (17, 4096, 1024), (31, 528, 2048), (32, 272, 4224), (33, 4096, 4096),
    (48, 12288, 512), (64, 128, 11008), (65, 4096, 4096), (127, 2064, 896), (128, 11008, 384), (129, 4096, 1664), (200, 260, 1024),
    (300, 12288, 256), (1030, 4096, 384), (2048, 4096, 256), (2050, 8200, 128), (160, 5120, 5120), (330, 6656, 5120), (640, 4096, 11008), (100, 528, 2048),
    (33, 68, 384), (40, 4100, 1024), (64, 6148, 2048), (100, 6144, 2048), (256, 2052, 640), (200, 4112, 4096),  # int4: blocks of 64 rows
]
INT4_WHOLE = [  # M, N, K, pair: blocks of 64, 96, 160 and 192 tokens x 8 waves, whole rows
    (65, 1028, 1024, 1), (500, 2756, 3328, 0), (193, 2752, 3840, 1), (300, 12292, 4096, 0), (130, 12292, 300, 1), (700, 6148, 2048, 0), (390, 5124, 256, 1), (1300, 4100, 1664, 0), (257, 16388, 512, 1),
    (770, 12292, 640, 0), (785, 6148, 512, 1), (450, 16388, 1664, 0), (330, 12292, 1024, 1), (385, 16388, 1280, 1), (810, 12292, 4096, 0),
]


@pytest.mark.parametrize("epi", ["store", "accum", "pair"])
@pytest.mark.parametrize("fmt", ["q4", "bf16"])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_tiled_product_against_64_bits(dev, fmt, M, N, K, epi):
    """The operands are exact in bf16 and summed in f32: the bf16 stream within sqrt(K) roundings of its terms, the int4 stream within those of terms 30
    times the result's (levels enter as 128 + q, the offset is taken off at the end): 1e-3 of the result covers both at K = 11008."""
    g = torch.Generator(device=dev).manual_seed(M * 31 + N + K)
    x = torch.randn((M, K), generator=g, device=dev).to(torch.bfloat16)
    n_mats = 2 if epi == "pair" else 1
    if fmt == "q4":
        qs = [torch.randint(0, 16, (N, K), generator=g, device=dev, dtype=torch.uint8) for _ in range(n_mats)]
        ss = [(torch.rand((N,), generator=g, device=dev) * 0.02 + 0.005).to(torch.bfloat16) for _ in range(n_mats)]
        zs = [torch.randint(5, 11, (N,), generator=g, device=dev).to(torch.bfloat16) for _ in range(n_mats)]
        pk = [synth.pack_colblock(q, 4) for q in qs] if K % 2 == 0 else None
        stream = ops.repack_q4(pk[0], pk[1] if n_mats == 2 else None, N, K, n_mats)
        kw = dict(scales=ss[0], zeros=zs[0])
        if n_mats == 2:
            kw.update(scales2=ss[1], zeros2=zs[1])
        ws = [(q.double() - z.double()[:, None]) * s.double()[:, None] for q, s, z in zip(qs, ss, zs)]
    else:
        mats = [(torch.randn((N, K), generator=g, device=dev) * 0.05).to(torch.bfloat16) for _ in range(n_mats)]
        stream = ops.repack_bf16(mats[0], mats[1] if n_mats == 2 else None, n_mats)
        kw, ws = dict(fmt=nat.W_BF16), [m.double() for m in mats]
    prods = [x.double() @ w.T for w in ws]
    if epi == "pair":
        ref = torch.nn.functional.silu(prods[0]) * prods[1]
        got = ops.linear_gemm(x, stream, 2, N, K, epi=nat.EPI_SWIGLU, out_dtype=torch.bfloat16, **kw).double()
        assert (got - ref).abs().max() <= 2.0 ** -8 * ref.abs().max() + 2e-3 * ref.square().mean().sqrt()  # one rounding to bf16
        return
    if epi == "accum":
        base = torch.randn((M, N), generator=g, device=dev)
        ref = prods[0] + base.double()
        got = ops.linear_gemm(x, stream, 1, N, K, epi=nat.EPI_ACCUM, out=base.clone(), **kw).double()
    else:
        ref = prods[0]
        got = ops.linear_gemm(x, stream, 1, N, K, out_dtype=torch.float32, **kw).double()
    assert (got - ref).abs().max() <= 1e-3 * ref.square().mean().sqrt()


@pytest.mark.parametrize("M,N,K,run", [
    (33, 4096, 4096, 4), (64, 4096, 4096, 4), (65, 4096, 4096, 4), (128, 4096, 11008, 11), (129, 4096, 4096, 8), (256, 4096, 11008, 22), (321, 4096, 4096, 16),
    (512, 4096, 11008, 43), (100, 12288, 4096, 16), (40, 5120, 13824, 14), (24, 4096, 4032, 4), (50, 4096, 4000, 4),
])
def test_int4_sums_beside_a_large_activation(dev, M, N, K, run):
    """Levels are summed as 128 + q: beside an activation of 2^17 an f32 sum is 2^24 and more, and each product of 32 columns costs it a rounding of that size.
    An accumulator sums `run` units of four such products (of the N = 12288 products 1 / 2 of K, of the others 1 / 8 up to 128 tokens, 1 / 4 up to 256, 1 / 2 up to
    640), and only the one with that activation is so large.  A product adds its 32 terms in a few steps, five roundings to the nearest at most: 5 / 12 of a squared
    last bit each, so the rms is sqrt(4 run 5 / 12) last bits (the operand sum's own roundings and the sample: 6 %).  The activation's own levels are its rows' zero points: its share of the result is 0."""
    g = torch.Generator(device=dev).manual_seed(M + N + K)
    q = torch.randint(0, 16, (N, K), generator=g, device=dev, dtype=torch.uint8)
    z = torch.randint(5, 11, (N,), generator=g, device=dev)
    q[:, 0] = z.to(torch.uint8)
    s = torch.full((N,), 2.0 ** -6, device=dev).to(torch.float32 if M < 32 else torch.bfloat16)
    x = torch.randn((M, K), generator=g, device=dev).to(torch.bfloat16)
    x[:, 0] = 2.0 ** 17
    ref = x.double() @ ((q.double() - z.double()[:, None]) * 2.0 ** -6).T
    stream = ops.repack_q4(synth.pack_colblock(q, 4), None, N, K, 1)
    got = ops.linear_gemm(x, stream, 1, N, K, scales=s, zeros=z.to(s.dtype), out_dtype=torch.float32).double()
    last_bit = 2.0 ** -6 * 2.0  # 128 x 2^17 = 2^24 and up to 2^24.2
    assert (got - ref).square().mean().sqrt() <= 1.06 * (4 * run * 5 / 12) ** 0.5 * last_bit


@pytest.mark.parametrize("M,N,K,pair", INT4_WHOLE)
def test_int4_blocks_of_whole_rows_against_64_bits(dev, M, N, K, pair):
    """A few tokens or rows more than whole blocks, rows shorter than the pipeline and ends of it, runs and none (tests/test_host_logic.py compares the list with the rule)."""
    test_tiled_product_against_64_bits(dev, "q4", M, N, K, "pair" if pair else "accum")


BF16_BLOCKS = [
    (512, 4096, 1664, 0), (257, 12288, 1664, 0), (257, 1000, 1664, 0), (449, 4112, 1664, 0), (512, 4112, 1664, 0), (193, 12288, 2176, 0), (500, 6160, 640, 0),
    (320, 12288, 2176, 0), (512, 12288, 640, 0), (1025, 6160, 256, 0), (769, 12288, 2176, 0), (1281, 6160, 2176, 0), (1281, 8200, 256, 0), (1025, 12288, 2048, 0),
    (512, 1000, 2176, 1), (193, 4112, 1664, 1), (320, 4112, 1664, 1), (320, 6160, 2176, 1), (641, 4112, 384, 1), (1281, 4096, 2176, 1), (449, 12288, 2048, 1), (1281, 12288, 128, 1),
    (600, 12288, 1152, 0), (600, 11012, 1664, 1), (70, 4100, 2176, 0), (129, 4100, 4224, 0), (66, 4100, 3200, 0), (300, 4096, 11008, 0), (135, 11012, 8448, 0),
    (70, 2816, 1664, 1), (70, 4100, 2176, 1), (66, 2052, 3200, 1), (129, 11012, 4224, 1),
    (482, 16400, 1664, 0), (674, 16400, 640, 0), (386, 8200, 640, 1), (962, 6160, 384, 1), (1930, 8280, 384, 0), (1165, 3340, 8448, 0),
    (770, 6148, 640, 1), (390, 13124, 640, 1), (785, 13124, 1152, 0),
]


@pytest.mark.parametrize("M,N,K,pair", BF16_BLOCKS)
def test_bf16_blocks_of_every_size_against_64_bits(dev, M, N, K, pair):
    """Blocks of 64 / 96 / 128 tokens x 4 waves and 64 / 128 / 160 / 192 / 208 / 256 x 8, whole rows and K-slices, pairs too (tests/test_host_logic.py compares the list with the rule): a few
    tokens or rows more than whole blocks, rounds of units that end early, row blocks that share an XCD and such that are cut between two.  Bounds: as in test_tiled_product_against_64_bits."""
    g = torch.Generator(device=dev).manual_seed(M * 31 + N + K)
    x = torch.randn((M, K), generator=g, device=dev).to(torch.bfloat16)
    mats = [(torch.randn((N, K), generator=g, device=dev) * 0.05).to(torch.bfloat16) for _ in range(1 + pair)]
    stream = ops.repack_bf16(mats[0], mats[1] if pair else None, 1 + pair)
    prods = [x.double() @ m.double().T for m in mats]
    if pair:
        ref = torch.nn.functional.silu(prods[0]) * prods[1]
        got = ops.linear_gemm(x, stream, 2, N, K, epi=nat.EPI_SWIGLU, out_dtype=torch.bfloat16, fmt=nat.W_BF16).double()
        assert (got - ref).abs().max() <= 2.0 ** -8 * ref.abs().max() + 2e-3 * ref.square().mean().sqrt()
        return
    base = torch.randn((M, N), generator=g, device=dev)
    ref = prods[0] + base.double()
    got = ops.linear_gemm(x, stream, 1, N, K, epi=nat.EPI_ACCUM, out=base.clone(), fmt=nat.W_BF16).double()
    assert (got - ref).abs().max() <= 1e-3 * ref.square().mean().sqrt()


def _chain_against_staging(dev, monkeypatch, width, T, mode):
    cfg = LLaMAConfig(block_size=T + 4, n_layer=2, n_head=width // 128, n_embd=width, vocab_size=512)
    with EmptyInitOnDevice(device=dev, dtype=torch.bfloat16, quantization_mode=mode):
        model = LLaMA(cfg)
    model.load_state_dict(synth.make_state_dict(cfg, seed=3, mode=mode, device="cuda", dtype=torch.bfloat16))
    model.eval()
    idx = synth.make_prompt(T, vocab=512).to(dev)
    out = []
    for fuse in ("1", "0"):
        monkeypatch.setenv("MI355_GEMM_FUSE", fuse)
        model.reset_cache()
        with torch.no_grad():
            out.append(model(idx.view(1, -1), T + 4, torch.arange(T, device=dev))[0].float())
    assert not torch.equal(*out)  # (the chain was on)
    assert (out[0] - out[1]).abs().max() <= 0.02 * out[1].std()


INT4_CHAIN = [(2048, 130), (2048, 400), (2048, 730), (2048, 850), (4096, 180), (4096, 300), (4096, 450), (4096, 700), (4096, 777), (4096, 850)]


@pytest.mark.parametrize("width,T", INT4_CHAIN)
def test_fused_prompt_chain_of_int4_layers_in_blocks_of_whole_rows(dev, monkeypatch, width, T):
    """As test_fused_prompt_chain_of_bf16_layers, for the blocks of 64, 96, 160 and 192 tokens x 8 waves of one scale per row."""
    _chain_against_staging(dev, monkeypatch, width, T, "gptq.int4")


INT4_NARROW_CHAIN = [(640, 32), (640, 40), (640, 60), (2048, 32), (2048, 40), (2048, 64)]


@pytest.mark.parametrize("width,T", INT4_NARROW_CHAIN)
def test_fused_prompt_chain_of_int4_layers_in_blocks_of_64_rows(dev, monkeypatch, width, T):
    """As test_fused_prompt_chain_of_bf16_layers, for c_attn and residual products in waves of one row tile: shares of 64 rows, slices of one run and of several."""
    _chain_against_staging(dev, monkeypatch, width, T, "gptq.int4")


BF16_CHAIN = [
    (640, 65), (640, 1094), (1024, 709), (1280, 65), (1280, 1731), (1920, 65), (1920, 646), (1920, 1633), (2048, 261), (2560, 65), (2560, 1542), (2560, 1605), (3072, 65),
    (4096, 135), (4096, 300), (4096, 400), (4096, 777), (4096, 1100), (4096, 1300), (5120, 1542), (6656, 100), (6656, 135), (6656, 1542), (6656, 1731), (6656, 1878),
]


@pytest.mark.parametrize("width,T", BF16_CHAIN)
def test_fused_prompt_chain_of_bf16_layers(dev, monkeypatch, width, T):
    """The chain's shares, rotations and cache rows in every block that its products take (tests/test_host_logic.py compares the list with the rule), a last block that is not
    whole.  0.02 of the logits' spread as in test_runs_of_shares_in_the_fused_prompt_chain."""
    _chain_against_staging(dev, monkeypatch, width, T, None)


@pytest.mark.parametrize("x_dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("M,N,K,cols", [(1, 16, 256, 128), (16, 144, 2176, 128), (17, 4096, 1280, 256), (33, 12288, 512, 128), (64, 128, 11008, 512), (65, 4096, 4096, 128),
                                        (129, 1000, 896, 256), (257, 2064, 2560, 1024), (700, 11008, 384, 128), (1030, 4100, 512, 64), (2050, 8200, 256, 128),
                                        (385, 15364, 1280, 128), (1300, 4100, 256, 128), (770, 12292, 640, 256), (1500, 6148, 128, 128), (450, 16388, 1664, 128)])
def test_tiled_product_of_grouped_scales_against_64_bits(dev, M, N, K, cols, x_dtype):
    """Groups of whole units: the products of a unit are sums of 128 terms of up to 143 x, the zero points a sum of their own: 1e-3 of the result as above.
    Rows whose addresses are no multiple of 16 B take the staging pass of single loads."""
    g = torch.Generator(device=dev).manual_seed(M * 31 + N + K)
    ld = K + (4 if M % 2 else 3)
    x = torch.randn((M, ld), generator=g, device=dev).to(x_dtype)[:, :K]
    ng = -(-K // cols)
    q = torch.randint(0, 16, (N, K), generator=g, device=dev, dtype=torch.uint8)
    s = (torch.rand((N, ng), generator=g, device=dev) * 0.02 + 0.005).to(torch.bfloat16)
    z = torch.randint(5, 11, (N, ng), generator=g, device=dev).to(torch.bfloat16)
    wide = lambda t: t.double().repeat_interleave(cols, 1)[:, :K]  # noqa: E731
    ref = x.to(torch.bfloat16).double() @ ((q.double() - wide(z)) * wide(s)).T
    stream = ops.repack_q4(synth.pack_colblock(q, 4), None, N, K, 1)
    got = ops.linear_gemm(x, stream, 1, N, K, scales=s.reshape(-1), zeros=z.reshape(-1), group_cols=cols, out_dtype=torch.float32).double()
    assert (got - ref).abs().max() <= 1e-3 * ref.square().mean().sqrt()


GROUPED_BLOCKS = [  # M, N, K, columns of a group, pair: blocks of 96 and 160 tokens x 8 waves
    (321, 12292, 1664, 128, 0), (577, 8196, 1664, 256, 0), (1025, 4100, 2176, 128, 0), (641, 12292, 2176, 256, 0), (450, 16388, 1664, 128, 0),
    (67, 16388, 2176, 128, 1), (385, 6148, 2176, 256, 1), (482, 12292, 128, 256, 1), (450, 8196, 1664, 128, 1), (641, 6148, 2176, 256, 1),
]


@pytest.mark.parametrize("M,N,K,cols,epi", [(*shape[:4], epi) for shape in GROUPED_BLOCKS for epi in (["pair"] if shape[4] else ["store", "accum"])])
def test_grouped_blocks_of_96_and_160_tokens_against_64_bits(dev, M, N, K, cols, epi):
    """A few tokens and rows more than whole blocks, in each epilogue (tests/test_host_logic.py compares the list with the rule).  Bounds: as in test_tiled_product_against_64_bits."""
    g = torch.Generator(device=dev).manual_seed(M * 31 + N + K)
    x = torch.randn((M, K), generator=g, device=dev).to(torch.bfloat16)
    mats, ng = 2 if epi == "pair" else 1, -(-K // cols)
    qs = [torch.randint(0, 16, (N, K), generator=g, device=dev, dtype=torch.uint8) for _ in range(mats)]
    ss = [(torch.rand((N, ng), generator=g, device=dev) * 0.02 + 0.005).to(torch.bfloat16) for _ in range(mats)]
    zs = [torch.randint(5, 11, (N, ng), generator=g, device=dev).to(torch.bfloat16) for _ in range(mats)]
    wide = lambda t: t.double().repeat_interleave(cols, 1)[:, :K]  # noqa: E731
    prods = [x.double() @ ((q.double() - wide(z)) * wide(s)).T for q, s, z in zip(qs, ss, zs)]
    pk = [synth.pack_colblock(q, 4) for q in qs]
    stream = ops.repack_q4(pk[0], pk[1] if mats == 2 else None, N, K, mats)
    kw = dict(scales=ss[0].reshape(-1), zeros=zs[0].reshape(-1), group_cols=cols)
    if epi == "pair":
        kw.update(scales2=ss[1].reshape(-1), zeros2=zs[1].reshape(-1))
        ref = torch.nn.functional.silu(prods[0]) * prods[1]
        got = ops.linear_gemm(x, stream, 2, N, K, epi=nat.EPI_SWIGLU, out_dtype=torch.bfloat16, **kw).double()
        assert (got - ref).abs().max() <= 2.0 ** -8 * ref.abs().max() + 2e-3 * ref.square().mean().sqrt()  # one rounding to bf16
        return
    ref = prods[0]
    if epi == "accum":
        base = torch.randn((M, N), generator=g, device=dev)
        ref = ref + base.double()
        got = ops.linear_gemm(x, stream, 1, N, K, epi=nat.EPI_ACCUM, out=base.clone(), **kw).double()
    else:
        got = ops.linear_gemm(x, stream, 1, N, K, out_dtype=torch.float32, **kw).double()
    assert (got - ref).abs().max() <= 1e-3 * ref.square().mean().sqrt()


@pytest.mark.parametrize("mode", ["gptq.int4", None])
@pytest.mark.parametrize("T", [2, 8, 9, 10, 11, 16, 17, 31, 33, 64, 65, 130, 257])
def test_prompt_pass_of_any_length_matches_single_tokens(dev, mode, T):
    """A prompt in one pass against the same tokens one by one (the row kernels): logits of every position within the spread of bf16 operands."""
    cfg = LLaMAConfig(block_size=288, n_layer=2, n_head=8, n_embd=1024, vocab_size=512)
    with EmptyInitOnDevice(device=dev, dtype=torch.bfloat16, quantization_mode=mode):
        model = LLaMA(cfg)
    model.load_state_dict(synth.make_state_dict(cfg, seed=1, mode=mode, device="cuda", dtype=torch.bfloat16))
    model.eval()
    idx = synth.make_prompt(T, vocab=512).to(dev)
    with torch.no_grad():
        one = model(idx.view(1, -1), 288, torch.arange(T, device=dev))[0]
        model.reset_cache()
        rows = torch.cat([model(idx[t:t + 1].view(1, 1), 288, torch.tensor([t], device=dev))[0] for t in range(T)])
    assert (one - rows).abs().max() <= 0.05 * rows.std()


@pytest.mark.parametrize("M", [1, 5])
@pytest.mark.parametrize("N,K", [(16, 64), (32000, 128), (33000, 384), (260, 512)])
def test_short_rows_in_four_waves_give_the_bits_of_eight(dev, N, K, M):
    """Rows of at most four units: a wave has one unit or none with four waves as with eight, so the sums are the same."""
    g = torch.Generator(device=dev).manual_seed(N + K + M)
    x = torch.randn((M, K), generator=g, device=dev).to(torch.bfloat16)
    q = torch.randint(0, 16, (N, K), generator=g, device=dev, dtype=torch.uint8)
    kw = dict(scales=(torch.rand((N,), generator=g, device=dev) * 0.02).to(torch.bfloat16), zeros=torch.full((N,), 7.0, device=dev).to(torch.bfloat16),
              out_dtype=torch.float32)
    stream = ops.repack_q4(synth.pack_colblock(q, 4), None, N, K, 1)
    assert torch.equal(ops.linear_fast(x, stream, nat.W_Q4, 1, N, K, **kw), ops.linear_fast(x, stream, nat.W_Q4, 1, N, K, waves=8, **kw))


@pytest.mark.parametrize("T", [33, 64, 100])
def test_runs_of_shares_in_the_fused_prompt_chain(dev, monkeypatch, T):
    """Slices of several runs whose operand sums come as shares of the producer: one per unit, or two (c_fc1 / c_fc2 in blocks of 64 rows, up to 64 tokens).  The
    chain with staging passes in place of shares rounds the same operands and sums in another order, as does the rotation of q and k: 0.02 of the logits' spread, the
    bound of the chain at 7B width; a run that took another one's sum would be off by the spread of 135 operands."""
    cfg = LLaMAConfig(block_size=128, n_layer=2, n_head=15, n_embd=1920, vocab_size=512)  # hidden rows of 5120: 40 units
    with EmptyInitOnDevice(device=dev, dtype=torch.bfloat16, quantization_mode="gptq.int4"):
        model = LLaMA(cfg)
    model.load_state_dict(synth.make_state_dict(cfg, seed=3, mode="gptq.int4", device="cuda", dtype=torch.bfloat16))
    model.eval()
    idx = synth.make_prompt(T, vocab=512).to(dev)
    out = []
    for fuse in ("1", "0"):
        monkeypatch.setenv("MI355_GEMM_FUSE", fuse)
        model.reset_cache()
        with torch.no_grad():
            out.append(model(idx.view(1, -1), 128, torch.arange(T, device=dev))[0].float())
    assert not torch.equal(*out)  # (the chain was on)
    assert (out[0] - out[1]).abs().max() <= 0.02 * out[1].std()


def test_an_int4_engine_holds_no_scratch_of_int8_products(dev):
    cfg = LLaMAConfig(block_size=128, n_layer=1, n_head=2, n_embd=256, vocab_size=512)
    with EmptyInitOnDevice(device=dev, dtype=torch.bfloat16, quantization_mode="gptq.int4"):
        model = LLaMA(cfg)
    model.load_state_dict(synth.make_state_dict(cfg, seed=3, mode="gptq.int4", device="cuda", dtype=torch.bfloat16))
    eng = model.eval().engine()
    assert eng.gemm_ws.numel() == nat.lib().mi355_linear_gemm_workspace_bytes(eng.max_T, eng.n_hidden)


def test_few_rows_of_more_outputs_than_a_table_holds(dev):
    """Few int4 rows of one scale per row are summed as one group, whose table has a region of 32 MB: beyond 4.19 million rows of the matrix without it."""
    M, N, K = 8, (1 << 22) + 16, 128
    g = torch.Generator(device=dev).manual_seed(5)
    x = torch.randn((M, K), generator=g, device=dev).to(torch.bfloat16)
    q = torch.randint(0, 16, (N, K), generator=g, device=dev, dtype=torch.uint8)
    s = (torch.rand((N,), generator=g, device=dev) * 0.02 + 0.005).to(torch.bfloat16)
    z = torch.randint(5, 11, (N,), generator=g, device=dev).to(torch.bfloat16)
    got = ops.linear_gemm(x, ops.repack_q4(synth.pack_colblock(q, 4), None, N, K, 1), 1, N, K, scales=s, zeros=z, out_dtype=torch.float32)
    for rows in (slice(0, 4096), slice(N - 4096, N)):
        ref = x.double() @ ((q[rows].double() - z[rows].double()[:, None]) * s[rows].double()[:, None]).T
        assert (got[:, rows].double() - ref).abs().max() <= 1e-3 * ref.square().mean().sqrt()


def _wide_model(dev, cfg, mode, cols):
    with EmptyInitOnDevice(device=dev, dtype=torch.bfloat16, quantization_mode=mode):
        model = LLaMA(cfg)
    if cols:
        from lit_llama_amd.quantization import ColBlockQuantizedLinear

        for mod in model.modules():
            if isinstance(mod, ColBlockQuantizedLinear):
                mod.tile_cols = cols
                mod.scales, mod.zeros = (torch.empty((mod.out_features, mod.in_features // cols), device=dev, dtype=torch.bfloat16) for _ in range(2))
    model.load_state_dict(synth.make_state_dict(cfg, seed=2, mode=mode, device="cuda", dtype=torch.bfloat16, group_cols=cols))
    return model.eval()


def _chunk_and_rows(dev, model, T):
    """Logits of T tokens in one pass and one by one (the row kernels)."""
    S = model.config.block_size
    idx = synth.make_prompt(T, vocab=512).to(dev)
    with torch.no_grad():
        one = model(idx.view(1, -1), S, torch.arange(T, device=dev))[0].float()
        model.reset_cache()
        rows = torch.cat([model(idx[t:t + 1].view(1, 1), S, torch.tensor([t], device=dev))[0].float() for t in range(T)])
    model.reset_cache()
    return one, rows


@pytest.mark.parametrize("mode,cols", [("gptq.int4", 0), ("gptq.int4", 128), ("gptq.int4", 256), (None, 0)])
def test_chunks_of_8_to_31_rows_at_a_width_that_tiles_them(dev, mode, cols):
    """7B width, where the row kernel would read the weights of 8 to 14 rows and more twice (mlp.c_proj's: of 8): on both sides of each product's change of kernel,
    single scales, groups of 128 and 256 columns, bf16."""
    model = _wide_model(dev, LLaMAConfig(block_size=32, n_layer=1, n_head=32, n_embd=4096, vocab_size=512), mode, cols)
    assert model.engine() is not None, model._engine_failed
    for T in (7, 8, 10, 11, 12, 13, 14, 16, 17, 31):
        one, rows = _chunk_and_rows(dev, model, T)
        assert (one - rows).abs().max() <= 0.05 * rows.std(), T


@pytest.mark.parametrize("case", ["tables", "workspace", "stream"])
def test_short_chunks_that_the_tiled_product_refuses_stay_in_the_row_kernel(dev, case):
    """24 tokens at a width where the row kernel reads the weights twice: with group tables of a vocabulary that exceeds their region, a workspace sized for less,
    a head in tiles of 32 rows: as the tokens one by one."""
    cfg = LLaMAConfig(block_size=32, n_layer=1, n_head=32, n_embd=4096, vocab_size=260_000 if case == "tables" else 512)
    model = _wide_model(dev, cfg, None if case == "stream" else "gptq.int4", 128 if case == "tables" else 0)
    eng = model.engine()
    assert eng is not None, model._engine_failed
    if case == "workspace":
        eng.m.gemm_ws_bytes = 4096
    if case == "stream":
        head = ops.repack_bf16(model.lm_head.weight, None, 2)
        eng.m.lm_head.w, eng.m.lm_head.R = head.data_ptr(), 2
    one, rows = _chunk_and_rows(dev, model, 24)
    assert (one - rows).abs().max() <= 0.05 * rows.std()


@pytest.mark.parametrize("T", [40, 150, 700])
def test_fused_prompt_chain_over_layers_of_different_formats(dev, monkeypatch, T):
    """Int4 and bf16 layers in turn: what a producer leaves is cut by its own format, and the chain holds over both.  0.02 of the logits' spread as for one format
    (other orders of f32 sums in front of bf16 roundings)."""
    cfg = LLaMAConfig(block_size=704, n_layer=3, n_head=15, n_embd=1920, vocab_size=512)
    with EmptyInitOnDevice(device=dev, dtype=torch.bfloat16, quantization_mode="gptq.int4"):
        model = LLaMA(cfg)
    model.load_state_dict(synth.make_state_dict(cfg, seed=3, mode="gptq.int4", device="cuda", dtype=torch.bfloat16))
    g = torch.Generator(device=dev).manual_seed(4)
    for layer, names in ((0, ["attn.c_proj"]), (1, ["attn.c_attn", "attn.c_proj", "mlp.c_fc1", "mlp.c_fc2", "mlp.c_proj"]), (2, ["mlp.c_proj"])):
        for name in names:
            part, attr = name.split(".")
            owner = getattr(model.transformer.h[layer], part)
            q = getattr(owner, attr)
            dense = torch.nn.Linear(q.in_features, q.out_features, bias=False, device=dev, dtype=torch.bfloat16)
            dense.weight.data = (torch.randn(dense.weight.shape, generator=g, device=dev) * q.in_features ** -0.5).to(torch.bfloat16)
            setattr(owner, attr, dense)
    model.eval()
    idx = synth.make_prompt(T, vocab=512).to(dev)
    out = []
    for fuse in ("1", "0"):
        monkeypatch.setenv("MI355_GEMM_FUSE", fuse)
        model.reset_cache()
        with torch.no_grad():
            out.append(model(idx.view(1, -1), 704, torch.arange(T, device=dev))[0].float())
    assert model.engine() is not None, model._engine_failed
    assert not torch.equal(*out)  # (the chain was on)
    assert (out[0] - out[1]).abs().max() <= 0.02 * out[1].std()


@pytest.mark.parametrize("epi", ["store", "pair", "accum"])
@pytest.mark.parametrize("M", [5, 16, 17, 32, 33, 64])
@pytest.mark.parametrize("N,K", [(64, 128), (68, 1000), (96, 4096), (100, 640), (4096, 2048), (8200, 384), (12352, 1024), (16512, 512)])
def test_few_bf16_rows_in_blocks_of_2_to_4_waves(dev, N, K, M, epi, flags=0):
    """Block edges at 64, 96 and 128 rows, slices, a last unit that is not whole.  The bound of the tiled product."""
    g = torch.Generator(device=dev).manual_seed(M * 31 + N + K)
    x = torch.randn((M, K), generator=g, device=dev).to(torch.bfloat16)
    ws = [(torch.randn((N, K), generator=g, device=dev) * K ** -0.5).to(torch.bfloat16) for _ in range(2)]
    prods = [x.double() @ w.double().T for w in ws]
    if epi == "pair":
        ref = torch.nn.functional.silu(prods[0]) * prods[1]
        got = ops.linear_gemm(x, ops.repack_bf16(ws[0], ws[1], 2), 2, N, K, epi=nat.EPI_SWIGLU, out_dtype=torch.bfloat16, fmt=nat.W_BF16, flags=flags).double()
        assert (got - ref).abs().max() <= 2.0 ** -8 * ref.abs().max() + 2e-3 * ref.square().mean().sqrt()
        return
    base = torch.randn((M, N), generator=g, device=dev) if epi == "accum" else torch.zeros((M, N), device=dev)
    ref = prods[0] + base.double()
    got = ops.linear_gemm(x, ops.repack_bf16(ws[0], None, 1), 1, N, K, epi=nat.EPI_ACCUM if epi == "accum" else nat.EPI_STORE, out=base.clone(), fmt=nat.W_BF16, flags=flags).double()
    assert (got - ref).abs().max() <= 1e-3 * ref.square().mean().sqrt()


@pytest.mark.parametrize("epi", ["store", "accum"])
@pytest.mark.parametrize("M", [9, 16, 17, 32, 33, 64])
@pytest.mark.parametrize("N,K", [(1000, 1900), (1500, 2700), (2052, 2200), (640, 3968)])
def test_few_bf16_rows_in_slices_of_2_and_3_units(dev, N, K, M, epi):
    """Slices no longer than the buffers that are filled ahead, some of 2 and some of 3 units, the last one not whole.  The bound of longer slices."""
    out = [C.c_int(0) for _ in range(3)]
    nat.lib().mi355_linear_gemm_cut_streamed(M, N, K, 1, C.c_bool(False), *[C.byref(v) for v in out])
    assert -(-K // 128) // out[2].value in (2, 3)
    test_few_bf16_rows_in_blocks_of_2_to_4_waves(dev, N, K, M, epi, flags=nat.LF_STREAMED)


@pytest.mark.parametrize("M", [2, 16, 24, 32, 40, 48, 49, 64, 65])
@pytest.mark.parametrize("N,K,fmt", [(128, 640, "bf16"), (33024, 384, "bf16"), (70000, 128, "bf16"), (4096, 4096, "bf16"), (640, 1024, "g128"), (4096, 1152, "q4"), (1000, 4096, "q4")])
def test_weights_past_the_caches_or_through_them(dev, N, K, fmt, M):
    """Weights requested non-temporal (one token block) or not, of 2 to 8 waves: f32 sums of exact products (see test_tiled_product_against_64_bits), the same bits where the cut is the same."""
    g = torch.Generator(device=dev).manual_seed(M + N)
    x = torch.randn((M, K), generator=g, device=dev).to(torch.bfloat16)
    if fmt == "bf16":
        w = (torch.randn((N, K), generator=g, device=dev) * 0.05).to(torch.bfloat16)
        kw, ref = dict(fmt=nat.W_BF16), x.double() @ w.double().T
        stream = ops.repack_bf16(w, None, 1)
    else:
        groups = K // 128 if fmt == "g128" else 1
        q = torch.randint(0, 16, (N, K), generator=g, device=dev, dtype=torch.uint8)
        scales, zeros = (torch.rand((N, groups), generator=g, device=dev) * 0.01 + 0.01).bfloat16(), torch.full((N, groups), 8.0, device=dev).bfloat16()
        stream = ops.repack_q4(synth.pack_colblock(q, 4), None, N, K, 1)
        kw = dict(scales=scales if groups > 1 else scales.view(-1), zeros=zeros if groups > 1 else zeros.view(-1), **({"group_cols": 128} if groups > 1 else {}))
        wide = lambda t: t.double().repeat_interleave(K // groups, 1)  # noqa: E731
        ref = x.double() @ ((q.double() - wide(zeros)) * wide(scales)).T
    got = [ops.linear_gemm(x, stream, 1, N, K, out_dtype=torch.float32, flags=f, **kw).double() for f in (0, nat.LF_STREAMED)]
    for y in got:
        assert (y - ref).abs().max() <= 1e-3 * ref.square().mean().sqrt()
    assert torch.equal(*got)


def test_engines_say_which_weights_are_streamed(dev, monkeypatch):
    """Every product of a model, or none (a model of this size)."""
    from lit_llama_amd import synth
    from lit_llama_amd.model import LLaMA, LLaMAConfig
    from lit_llama_amd.utils import EmptyInitOnDevice

    cfg = LLaMAConfig(n_layer=2, n_head=4, n_embd=256, vocab_size=512)
    for want in (0, nat.LF_STREAMED):
        if want:
            monkeypatch.setattr(nat, "streamed", lambda n: nat.LF_STREAMED if n == bytes_of else 0)
        with EmptyInitOnDevice(device=dev, dtype=torch.bfloat16):
            model = LLaMA(cfg)
        model.load_state_dict(synth.make_state_dict(cfg, seed=1, dtype=torch.bfloat16))
        model.eval()
        with torch.no_grad():
            model(torch.arange(9, device=dev).view(1, -1), 32, torch.arange(9, device=dev))
        eng = model.engine()
        bytes_of = sum(p.stream_bytes for p in eng.packed)
        assert bytes_of == sum(p.numel() * 2 for n, p in model.named_parameters() if n == "lm_head.weight" or (p.dim() == 2 and "wte" not in n))
        assert {w.flags for L in eng.layers for w in (L.attn, L.proj, L.fc, L.mproj)} | {eng.m.lm_head.flags} == {want}


OPERAND_SLICES = [(9, 256, 9, 4096), (16, 512, 5, 4096), (24, 256, 22, 4096), (32, 256, 65, 128), (32, 3072, 2, 4096), (40, 256, 65, 256), (40, 256, 18, 4096), (64, 256, 66, 256), (64, 512, 11, 4096)]


@pytest.mark.parametrize("M,rows,n,K", OPERAND_SLICES)
def test_operand_slices_of_few_bf16_rows(dev, M, rows, n, K):
    """Products of these rows and columns that read one operand take blocks of 3 waves, 96 rows, which do not divide the slices (tests/test_host_logic.py): one bf16 rounding of the result and
    the sums' 1e-3 of the tiled product."""
    g = torch.Generator(device=dev).manual_seed(M + rows + n)
    x = torch.randn((n, M + 1, K), generator=g, device=dev).to(torch.bfloat16)
    w = (torch.randn((n * rows, K), generator=g, device=dev) * K ** -0.5).to(torch.bfloat16)
    y = torch.zeros((M, n * rows), dtype=torch.bfloat16, device=dev)
    stream = ops.repack_bf16(w, None, 1)
    a = nat.LinearArgs()
    a.fmt, a.R, a.w, a.N, a.K, a.x, a.x_dtype, a.M, a.ldx = nat.W_BF16, 1, nat.ptr(stream), n * rows, K, nat.ptr(x), nat.BF16, M, x.stride(1)
    a.epi, a.y, a.y_dtype, a.ldy, a.alpha, a.slice_rows, a.slice_stride = nat.EPI_STORE, nat.ptr(y), nat.BF16, y.stride(0), 1.0, rows, x.stride(0)
    ws = torch.empty(nat.lib().mi355_linear_gemm_workspace_bytes(M, K), dtype=torch.uint8, device=dev)
    nat.check(nat.lib().mi355_linear_gemm(C.byref(a), nat.ptr(ws), ws.numel(), nat.stream_ptr()))
    ref = torch.cat([x[i, :M].double() @ w[i * rows:(i + 1) * rows].double().T for i in range(n)], 1)
    assert ((y.double() - ref).abs() <= 2.0 ** -8 * ref.abs() + 1e-3 * ref.square().mean().sqrt()).all()


GROUPED_CHAIN = [(128, 15, 33), (128, 15, 64), (128, 15, 65), (128, 15, 500), (128, 32, 40), (128, 32, 300), (128, 32, 777), (256, 32, 130), (256, 32, 600),
                 (128, 32, 180), (256, 32, 450), (128, 32, 650), (128, 32, 1100), (256, 32, 1250), (128, 40, 1650)]


@pytest.mark.parametrize("cols,heads,T", GROUPED_CHAIN)
def test_fused_prompt_chain_over_grouped_scales(dev, monkeypatch, cols, heads, T):
    """Groups of whole units in the chain: one share per unit, or two (c_fc1 / c_fc2 in blocks of 64 hidden rows); slices and whole sums; tables of several layers from one
    launch and the next.  Against the same layers with staging passes, 0.02 of the logits' spread as for one scale per row."""
    size = 784 if T < 784 else T + 4
    model = _wide_model(dev, LLaMAConfig(block_size=size, n_layer=5 if heads == 15 else 3, n_head=heads, n_embd=128 * heads, vocab_size=512), "gptq.int4", cols)
    idx = synth.make_prompt(T, vocab=512).to(dev)
    out = []
    for fuse in ("1", "0"):
        monkeypatch.setenv("MI355_GEMM_FUSE", fuse)
        model.reset_cache()
        with torch.no_grad():
            out.append(model(idx.view(1, -1), size, torch.arange(T, device=dev))[0].float())
    assert model.engine() is not None, model._engine_failed
    assert not torch.equal(*out)  # (the chain was on)
    assert (out[0] - out[1]).abs().max() <= 0.02 * out[1].std()


@pytest.mark.parametrize("T", [40, 150, 700])
def test_fused_prompt_chain_over_groups_rows_and_bf16(dev, monkeypatch, T):
    """Layers of groups of 128 columns, of one scale per row and of bf16 in one chain: K-slices of the latter take the room of the former's tables, which are laid out
    again behind them.  The bound as above."""
    cfg = LLaMAConfig(block_size=704, n_layer=4, n_head=15, n_embd=1920, vocab_size=512)
    model = _wide_model(dev, cfg, "gptq.int4", 128)
    rows = _wide_model(dev, cfg, "gptq.int4", 0)
    g = torch.Generator(device=dev).manual_seed(4)
    for layer, name, kind in ((0, "attn.c_proj", "rows"), (1, "attn.c_attn", "bf16"), (1, "mlp.c_proj", "bf16"), (2, "mlp.c_fc1", "rows"), (2, "mlp.c_fc2", "rows"), (2, "attn.c_proj", "bf16"),
                              (3, "attn.c_attn", "rows")):
        part, attr = name.split(".")
        owner = getattr(model.transformer.h[layer], part)
        q = getattr(owner, attr)
        if kind == "rows":
            new = getattr(getattr(rows.transformer.h[layer], part), attr)
        else:
            new = torch.nn.Linear(q.in_features, q.out_features, bias=False, device=dev, dtype=torch.bfloat16)
            new.weight.data = (torch.randn(new.weight.shape, generator=g, device=dev) * q.in_features ** -0.5).to(torch.bfloat16)
        setattr(owner, attr, new)
    idx = synth.make_prompt(T, vocab=512).to(dev)
    out = []
    for fuse in ("1", "0"):
        monkeypatch.setenv("MI355_GEMM_FUSE", fuse)
        model.reset_cache()
        with torch.no_grad():
            out.append(model(idx.view(1, -1), 704, torch.arange(T, device=dev))[0].float())
    assert model.engine() is not None, model._engine_failed
    assert not torch.equal(*out)  # (the chain was on)
    assert (out[0] - out[1]).abs().max() <= 0.02 * out[1].std()


@pytest.mark.parametrize("M", [9, 40, 100, 300, 600])
@pytest.mark.parametrize("fmt", ["q4", "g128", "g32", "bf16", "i8"])
def test_rows_that_are_not_finite_stay_by_themselves(dev, fmt, M):
    """NaN and infinities in two rows (LLM.int8: NaN alone, an infinity makes its columns everyone's outliers): the other rows keep their bits, in blocks with and
    without empty rows, slices, runs and groups."""
    N, K = 4096, 4096
    g = torch.Generator(device=dev).manual_seed(M)
    x = torch.randn((M, K), generator=g, device=dev).to(torch.bfloat16)
    bad = x.clone()
    bad[2], bad[M - 1, 100:300] = float("nan"), float("nan") if fmt == "i8" else float("inf")
    if fmt == "i8":
        cb, scb = ops.int8_quant_rows(torch.randn((N, K), generator=g, device=dev) * K ** -0.5)
        stream = ops.repack_i8(cb, None, 1)
        run = lambda v: ops.linear_int8_gemm(v, stream, scb, 1, N, K, out_dtype=torch.float32)  # noqa: E731
    elif fmt == "bf16":
        stream = ops.repack_bf16((torch.randn((N, K), generator=g, device=dev) * 0.05).to(torch.bfloat16), None, 1)
        run = lambda v: ops.linear_gemm(v, stream, 1, N, K, fmt=nat.W_BF16, out_dtype=torch.float32)  # noqa: E731
    else:
        cols = int(fmt[1:]) if fmt != "q4" else 0
        ng = K // cols if cols else 1
        stream = ops.repack_q4(synth.pack_colblock(torch.randint(0, 16, (N, K), generator=g, device=dev, dtype=torch.uint8), 4), None, N, K, 1)
        s = (torch.rand((N * ng,), generator=g, device=dev) * 0.02 + 0.005).to(torch.bfloat16)
        z = torch.randint(5, 11, (N * ng,), generator=g, device=dev).to(torch.bfloat16)
        run = lambda v: ops.linear_gemm(v, stream, 1, N, K, scales=s, zeros=z, group_cols=cols, out_dtype=torch.float32)  # noqa: E731
    clean, got = run(x).clone(), run(bad)
    others = torch.ones(M, dtype=torch.bool, device=dev)
    others[2] = others[M - 1] = False
    assert torch.equal(got[others], clean[others]) and bool(clean.isfinite().all())
    if fmt != "i8":
        assert not bool(got[2].isfinite().any()) and not bool(got[M - 1].isfinite().any())


@pytest.mark.parametrize("vocab", [512, 514])
def test_logits_of_a_prompt_in_portions(dev, vocab):
    """The head writes a portion's logits where they are returned; rows of 514 values put the second portion 8 bytes off a 16-byte line, which goes through the engine's
    buffer.  A portion's products are cut by its own rows: the spread of bf16 operands against the prompt in one pass."""
    cfg = LLaMAConfig(block_size=128, n_layer=2, n_head=4, n_embd=512, vocab_size=vocab)
    with EmptyInitOnDevice(device=dev, dtype=torch.bfloat16):
        model = LLaMA(cfg)
    model.load_state_dict(synth.make_state_dict(cfg, seed=7, mode=None, device="cuda", dtype=torch.bfloat16))
    model.eval()
    eng = model.engine()
    assert eng is not None, model._engine_failed
    idx, pos = synth.make_prompt(70, vocab=vocab).to(dev).view(1, -1), torch.arange(70, device=dev)
    with torch.no_grad():
        whole = model(idx, 128, pos)[0].clone()
        model.reset_cache()
        eng.max_T = 33
        parts = model(idx, 128, pos)[0]
    assert parts.shape == whole.shape and (parts - whole).abs().max() <= 0.05 * whole.std()
