"""GPU parity of the thin tiles (csrc/thin.hip): products of few rows an expert.

Linears, MoE layers and dense FFNs at the edges of the tiles (16 tokens an MFMA, 32 or 64 rows
a tile, stages of 4, 2 and 1 super-blocks, row tiles past the last row) and of the rule that
chooses them, in every device format, against float64 products on the oracle's weights.

A linear's bound: fp16 rounding of each weight (2^-11 of it at most; the K-quants' integer
codes are exact) and fp32 sums of K products, so |d| <= 2^-11 sum |x w| + K 2^-23 sum |x| (|w| +
offset part); the second term is held at 2^-13 sum |x w| with room for the offset part.
"""

import numpy as np
import pytest

import oracle
from gpu_helpers import build_pair, check_forward_routing, check_layer_output, log
from pgmoe.synth import DenseSpec, LayerSpec, SyntheticDense, random_blocks

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

F16, Q4_1, Q8_0, Q4_K, Q5_K, Q6_K = 1, 3, 8, 12, 13, 14


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    yield
    torch.cuda.empty_cache()


@pytest.mark.parametrize("qt", [Q4_1, Q8_0, Q4_K, Q5_K, Q6_K])
@pytest.mark.parametrize("N,K,xs", [(68, 256, 1.0), (260, 1280, 1.0), (1540, 768, 1.0), (132, 2304, 3e4)])
def test_linear_tiles(qt, N, K, xs):
    from pgmoe import GGUFQuantLinear
    dev = torch.device("cuda", 0)
    rng = np.random.default_rng(N + K + qt)
    raw = random_blocks(rng, qt, N, K, 0.01)
    bias = torch.from_numpy(rng.standard_normal(N).astype(np.float32))
    lin = GGUFQuantLinear("w8", K, N, qt, raw=raw, bias=bias, device=dev)
    w = oracle.dequant(qt, raw, N, K).astype(np.float64)
    x = (np.clip(rng.standard_normal((300, K)), -2, 2) * xs).astype(np.float16)
    ref = x.astype(np.float64) @ w.T + bias.numpy()
    bound = (2.0 ** -11 + 2.0 ** -13) * (np.abs(x.astype(np.float64)) @ np.abs(w).T) + 1e-5
    for M in (9, 16, 17, 32, 33, 48, 64, 65, 96, 128, 129, 300):
        log(f"thin linear qt={qt} N={N} K={K} x*{xs} M={M}")
        xm = torch.from_numpy(x[:M]).to(dev)
        got = lin(xm.float()).cpu().numpy()
        assert np.all(np.abs(got - ref[:M]) <= bound[:M]), f"M={M}: {np.max(np.abs(got - ref[:M]) / bound[:M]):.2f}"
        if xs == 1.0:  # fp16 output: the fp32 result rounded
            assert np.array_equal(lin(xm).cpu().numpy(), got.astype(np.float16))


@pytest.mark.parametrize("qt", [Q4_K, Q5_K, Q6_K])
@pytest.mark.parametrize("K", [256, 1280, 2304])
def test_decode_linear_of_many_rows(qt, K):
    """3 .. 8 tokens of an output head: exact products in fp32 sums of K / 32 + K / 128 terms, each
    rounded to 2^-24 of a partial sum, at most 90 x 6e-8 = 5.4e-6 of the result's norm (a weight
    rounded to fp16 would show 1e-4); either side of the rule's tokens and rows agrees."""
    from pgmoe import GGUFQuantLinear
    dev = torch.device("cuda", 0)
    rng = np.random.default_rng(K + qt)
    N = 32768 + 36
    raw = random_blocks(rng, qt, N, K, 0.01)
    bias = torch.from_numpy(rng.standard_normal(N).astype(np.float32))
    lin = GGUFQuantLinear("w8", K, N, qt, raw=raw, bias=bias, device=dev)
    w = torch.from_numpy(oracle.dequant(qt, raw, N, K)).to(dev).double()
    x = torch.from_numpy(rng.standard_normal((9, K)).astype(np.float16)).to(dev)
    ref = x.double() @ w.T + bias.to(dev).double()
    for M in (1, 2, 3, 5, 8, 9):
        log(f"thin decode linear qt={qt} K={K} M={M}")
        got = lin(x[:M].float())
        err = float((got.double() - ref[:M]).norm() / ref[:M].norm())
        assert err <= (5.4e-6 if 3 <= M <= 8 else 1e-3), (M, err)
        assert torch.equal(lin(x[:M]), got.to(torch.float16))


@pytest.mark.parametrize("gate_up,down", [(Q4_K, Q6_K), (Q5_K, Q4_K), (Q6_K, Q5_K), (Q8_0, Q8_0), (Q4_1, Q4_1),
                                          (F16, F16)])
def test_layer_tiles(gate_up, down):
    """A skewed router: with M tokens the first expert holds about M pairs (tiles of 32 and a
    remainder), the others few or none; M = 120 / 121 lie on both sides of 30 pairs an expert, 96 / 97 of
    24 (Q8_0; F16 takes the 256-row tiles from 9 tokens on)."""
    spec = LayerSpec("thin", 768, 8, 2, 512, (gate_up, gate_up, down), shared_inter=256,
                     shared_qtypes=(gate_up, gate_up, down), shared_gate=True)
    # float weights at their own scale: at 0.01 (2e-4) the SwiGLU rows, near 1e-6, fall among
    # fp16's subnormals (spacing 6e-8), and their fp16 form alone is off by up to 3e-2 a value
    lay, ol, mod = build_pair(spec, seed=5, scale=1.0 if gate_up == F16 else 0.01)
    bias = np.array([6, 1, 0, 0, -1, -1, -2, -8], np.float32)
    mod.set_router_bias(torch.from_numpy(bias))
    ol = oracle.OracleLayer.from_gguf(lay.gguf, lay.config, router_bias=bias)
    for M in (9, 16, 33, 47, 96, 97, 120, 121, 160, 161):
        log(f"thin layer {gate_up}/{down} M={M}")
        x = lay.draw_x(M)
        got = mod(torch.from_numpy(x).to("cuda:0")).cpu().numpy()
        _, idx, w = ol.route(x)
        check_forward_routing(mod, M, idx, w)
        check_layer_output(got, ol.forward_tokens(x, idx, w))


@pytest.mark.parametrize("gate_up,down", [(Q4_K, Q6_K), (Q5_K, Q4_K), (Q6_K, Q5_K)])
@pytest.mark.parametrize("H,I", [(256, 108800), (2304, 12544), (12544, 2304)])
def test_decode_dense_on_thin_tiles(gate_up, down, H, I):
    """3 .. 8 tokens against float64 on the decoded weights: gate and up within 5.4e-6 of their
    norms as above, their product and the down sums the same again, the split rows 2^-22: 2e-5 of
    the result's norm in all.  Rows that differ by 2^16 in size keep their own accuracy."""
    from pgmoe import HipDenseMLP
    dev = torch.device("cuda", 0)
    lay = SyntheticDense(DenseSpec("thin", H, I, (gate_up, gate_up, down)), seed=3, scale=0.01)
    mod = HipDenseMLP(lay.gguf, lay.config, 0, dev)
    g, u, d = (torch.from_numpy(oracle.dequant(t.qtype, lay.tensor(f"ffn_{p}.weight"), *t.shape)).to(dev).double()
               for p in ("gate", "up", "down") for t in [lay.gguf.tensors[f"blk.0.ffn_{p}.weight"]])
    x = torch.from_numpy(lay.draw_x(9)).to(dev)
    x[1] *= 2.0 ** -8
    x[2] = 0
    ref = (torch.nn.functional.silu(x.double() @ g.T) * (x.double() @ u.T)) @ d.T
    for M in (3, 5, 8):
        log(f"thin decode dense {gate_up}/{down} H={H} I={I} M={M}")
        got = mod(x[:M].clone()).double()
        assert torch.all(got[2] == 0)
        err = (got - ref[:M]).norm(dim=1) / ref[:M].norm(dim=1).clamp_min(1e-300)
        assert float(err.max()) <= 2e-5, (M, err)


def test_dense_sides_of_the_rule_and_replays():
    """Both products on thin tiles (9 tokens), only gate / up (100, 256), only the down one (257) and
    neither (600); a captured forward on thin tiles equals the eager one at every replay."""
    from pgmoe import HipDenseMLP
    dev = torch.device("cuda", 0)
    lay = SyntheticDense(DenseSpec("thin", 1024, 25600, (Q4_K, Q4_K, Q6_K)), seed=2, scale=0.01)
    mod = HipDenseMLP(lay.gguf, lay.config, 0, dev)
    mats = [(t.qtype, *t.shape, lay.tensor(f"ffn_{p}.weight")) for p in ("gate", "up", "down")
            for t in [lay.gguf.tensors[f"blk.0.ffn_{p}.weight"]]]
    for M in (9, 100, 256, 257, 600):
        log(f"thin dense M={M}")
        x = lay.draw_x(M)
        toks = np.unique(np.linspace(0, M - 1, 5).astype(np.int64))
        got = mod(torch.from_numpy(x).to(dev)).cpu().numpy()
        check_layer_output(got[toks], oracle.dense_forward(x, *mats, tokens=toks))
    x = torch.from_numpy(lay.draw_x(40)).to(dev)
    side = torch.cuda.Stream(dev)
    side.wait_stream(torch.cuda.current_stream(dev))
    with torch.cuda.stream(side):
        mod(x)
    side.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=side):
        out = mod(x)
    for seed in range(3):
        x.copy_(torch.randn(x.shape, generator=torch.Generator().manual_seed(seed)).to(torch.float16))
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, mod(x))


@pytest.mark.parametrize("qt", [Q4_1, Q8_0, Q4_K, Q5_K, Q6_K])
@pytest.mark.parametrize("N,K", [(68, 256), (260, 1280), (4100, 512)])
def test_tokens_that_are_not_finite(qt, N, K):
    """Infinities in a token give what the sum over their terms gives with the weights rounded to
    fp16 (+-inf where they agree in sign, else NaN), a NaN gives NaN, and the other tokens of the
    tile are bit-equal to a run without them.  Weights near zero, whose sign the rounding of the
    decoded value decides, are left out."""
    from pgmoe import GGUFQuantLinear
    dev = torch.device("cuda", 0)
    rng = np.random.default_rng(N + K + qt)
    raw = random_blocks(rng, qt, N, K, 0.01)
    lin = GGUFQuantLinear("w8", K, N, qt, raw=raw, device=dev)
    w = oracle.dequant(qt, raw, N, K)
    x = rng.standard_normal((65, K)).astype(np.float16)
    bad = x.copy()
    terms = {3: {7: np.inf}, 8: {K - 1: -np.inf}, 16: {40: np.inf, 200: np.inf}, 32: {0: np.inf, 131: -np.inf}}
    for t, at in terms.items():
        for k, v in at.items():
            bad[t, k] = v
    bad[5, 99] = np.nan
    touched = np.isin(np.arange(65), [*terms, 5])
    for M in (9, 17, 33, 65):
        log(f"thin non-finite qt={qt} N={N} K={K} M={M}")
        clean = lin(torch.from_numpy(x[:M]).to(dev).float()).cpu().numpy()
        got = lin(torch.from_numpy(bad[:M]).to(dev).float()).cpu().numpy()
        assert np.array_equal(got[~touched[:M]], clean[~touched[:M]])
        assert np.all(np.isnan(got[5]))
        for t, at in terms.items():
            if t < M:
                cols = np.all([np.abs(w[:, k]) > 1e-3 * np.abs(w).max() for k in at], axis=0)
                with np.errstate(invalid="ignore"):
                    ref = sum(w[:, k].astype(np.float16) * np.float16(v) for k, v in at.items())
                assert cols.sum() > N // 4 and np.array_equal(got[t, cols], ref[cols], equal_nan=True), (M, t)


def _int_ffn(gate, up, down, arch="qwen3"):
    """A dense FFN of whole-number weights: gate and up [I, H] (0 .. 15) as Q4_K, down [H, I] (-32 ..
    31) as Q6_K, every scale 1 and every minimum 0."""
    from pgmoe import HipDenseMLP
    from pgmoe.gguf import InMemoryGGUF

    def q4(c):
        c = c.reshape(-1, 4, 2, 32).astype(np.uint8)
        qs = (c[:, :, 0] | (c[:, :, 1] << 4)).reshape(-1, 128)
        head = np.frombuffer(np.float16(1).tobytes() + bytes(2) + bytes([1] * 4 + [0] * 4 + [1] * 4), np.uint8)
        return np.concatenate([np.broadcast_to(head, (len(qs), 16)), qs], 1)

    def q6(c):
        c = (c + 32).reshape(-1, 2, 4, 32).astype(np.uint8)
        ql = np.concatenate([(c[:, :, 0] & 15) | ((c[:, :, 2] & 15) << 4), (c[:, :, 1] & 15) | ((c[:, :, 3] & 15) << 4)], 2)
        qh = sum((c[:, :, s] >> 4) << (2 * s) for s in range(4))
        tail = np.frombuffer(bytes([1] * 16) + np.float16(1).tobytes(), np.uint8)
        return np.concatenate([ql.reshape(-1, 128), qh.reshape(-1, 64), np.broadcast_to(tail, (len(ql), 18))], 1)

    I, H = gate.shape
    g = InMemoryGGUF({"general.architecture": arch, f"{arch}.embedding_length": H, f"{arch}.feed_forward_length": I})
    g.add_tensor("blk.0.ffn_gate.weight", (I, H), Q4_K, q4(gate))
    g.add_tensor("blk.0.ffn_up.weight", (I, H), Q4_K, q4(up))
    g.add_tensor("blk.0.ffn_down.weight", (H, I), Q6_K, q6(down))
    return HipDenseMLP(g, g.build_model_config(), 0, torch.device("cuda", 0))


@pytest.mark.parametrize("arch", ["qwen3", "gemma3"])
def test_decode_dense_activation(arch):
    """Each output is one activation times a whole number.  SiLU of -38 .. -3 in fp32: expf 2^-23,
    1 + x, the quotient and the product 2^-24 each, the rows' pieces and their sum 2^-23: 4.2e-7
    (the hardware exp2 of a rounded argument is off by up to 2.4e-6 alone).  GELU of 3 .. 38:
    2z to 4 x 2^-24 of itself, which moves 1 - 1 / (1 + e^2z) by at most 0.3 of that; 1e-6."""
    H, I, M = 1024, 10240, 8
    gate, up, down = np.zeros((I, H), np.int64), np.zeros((I, H), np.int64), np.zeros((H, I), np.int64)
    i, h = np.arange(I), np.arange(H)
    gate[:, 0], up[:, 1] = 12 + i % 4, 1 + i % 7  # (a row's values within 2^12 of one another)
    at = (10 * h + 3 * (h // 64)) % I
    down[h, at] = 1
    x = np.zeros((M, H), np.float16)
    x[:, 0] = (1 if arch == "gemma3" else -1) * np.array([0.25, 0.5, 0.75, 1, 1.25, 1.75, 2, 2.5])
    x[:, 1] = 1
    got = _int_ffn(gate, up, down, arch)(torch.from_numpy(x).to("cuda:0")).double().cpu()
    g = torch.from_numpy(x[:, :1].astype(np.float64) * gate[at, 0])
    a = torch.nn.functional.gelu(g, approximate="tanh") if arch == "gemma3" else torch.nn.functional.silu(g)
    ref = a * torch.from_numpy(up[at, 1].astype(np.float64))
    assert float(((got - ref) / ref).abs().max()) <= (1e-6 if arch == "gemma3" else 6e-7)


@pytest.mark.parametrize("M", [5, 8])
def test_decode_dense_rows_keep_24_bits(M):
    """Activations of up to 24 bits (whole numbers: SiLU of 10000 is 10000) less their neighbours: every
    sum is a whole number below 2^24, so the fp32 value of each activation shows in full."""
    H, I = 2048, 256 * (-(-250000000 // (M * 3 * 2048 * 256)))
    gate, up, down = np.zeros((I, H), np.int64), np.zeros((I, H), np.int64), np.zeros((H, I), np.int64)
    i, h = np.arange(I), np.arange(H)
    gate[:, 0], up[:, 1] = 9 + 2 * (i % 4), 1 + 2 * (i // 4 % 4)
    a, b = 2 * h % I, (2 * h + 1 + 2 * (h // 16)) % I  # one even, one odd: not the same
    down[h, a], down[h, b] = 1, -1
    x = np.zeros((M, H), np.float16)
    x[:, 0], x[:, 1] = 1021 + 2 * np.arange(M), 135 + 2 * np.arange(M)
    got = _int_ffn(gate, up, down)(torch.from_numpy(x).to("cuda:0")).cpu().numpy()
    act = x[:, :1].astype(np.int64) * gate[:, 0] * (x[:, 1:2].astype(np.int64) * up[:, 1])
    assert act.max() < 2 ** 24 and np.array_equal(got, (act[:, a] - act[:, b]).astype(np.float32))


@pytest.mark.parametrize("qt", [Q4_K, Q6_K])
@pytest.mark.parametrize("rows", [(16384, 16420), (32769, 32768)])
def test_packed_projections_equal_separate_ones(qt, rows):
    """Up to 8 tokens a projection has the same bits packed and alone, also where only the pack, or
    each member too, has the rows of an output head."""
    from pgmoe import FusedLinearPack, GGUFQuantLinear
    dev = torch.device("cuda", 0)
    rng = np.random.default_rng(sum(rows) + qt)
    lins = [GGUFQuantLinear("w8", 512, n, qt, raw=random_blocks(rng, qt, n, 512, 0.01), device=dev) for n in rows]
    pack = FusedLinearPack(lins)
    for M in (1, 2, 3, 5, 8):
        log(f"packed qt={qt} rows={rows} M={M}")
        x = torch.from_numpy(rng.standard_normal((M, 512)).astype(np.float16)).to(dev)
        for got, lin in zip(pack(x.float()), lins):
            assert torch.equal(got, lin(x.float()))


def test_layer_on_few_experts_at_both_sides_of_the_rule():
    """Every token on the same two experts: 96 tokens take thin tiles (three an expert), 97 not."""
    spec = LayerSpec("conc", 4096, 8, 2, 8192, (Q4_K, Q4_K, Q4_K))
    lay, ol, mod = build_pair(spec, seed=6, scale=0.01)
    bias = np.array([0, 40, 0, 0, 0, 0, 40, 0], np.float32)
    mod.set_router_bias(torch.from_numpy(bias))
    ol = oracle.OracleLayer.from_gguf(lay.gguf, lay.config, router_bias=bias)
    for M in (64, 96, 97):
        log(f"thin layer on two experts M={M}")
        x = lay.draw_x(M)
        got = mod(torch.from_numpy(x).to("cuda:0")).cpu().numpy()
        _, idx, w = ol.route(x)
        assert set(idx.reshape(-1).tolist()) == {1, 6}
        check_forward_routing(mod, M, idx, w)
        toks = np.array([0, 31, 32, M - 1])
        check_layer_output(got[toks], ol.forward_tokens(x[toks], idx[toks], w[toks]))


def test_layer_tiles_of_fp16_experts():
    """fp16 experts take thin tiles up to two pairs an expert (48 tokens here)."""
    spec = LayerSpec("thin16", 512, 48, 2, 256, (F16, F16, F16))
    lay, ol, mod = build_pair(spec, seed=7)
    bias = np.where(np.arange(48) == 5, 3.0, 0.0).astype(np.float32)  # one expert of up to M pairs
    mod.set_router_bias(torch.from_numpy(bias))
    ol = oracle.OracleLayer.from_gguf(lay.gguf, lay.config, router_bias=bias)
    for M in (9, 17, 33, 48, 49):
        log(f"thin layer fp16 M={M}")
        x = lay.draw_x(M)
        got = mod(torch.from_numpy(x).to("cuda:0")).cpu().numpy()
        _, idx, w = ol.route(x)
        check_forward_routing(mod, M, idx, w)
        check_layer_output(got, ol.forward_tokens(x, idx, w))


@pytest.mark.parametrize("bad", [np.inf, np.nan])
def test_decode_calls_keep_other_tokens_clean(bad):
    """One token of 3 .. 8 with an infinity or NaN: the head's and the FFN's other rows are bit-equal to a
    run without it, in the one 16-row tile and in the two that 6 and more tokens' pieces fill."""
    from pgmoe import GGUFQuantLinear, HipDenseMLP
    dev = torch.device("cuda", 0)
    raw = random_blocks(np.random.default_rng(1), Q6_K, 32768, 512, 0.01)
    head = GGUFQuantLinear("w8", 512, 32768, Q6_K, raw=raw, device=dev)
    lay = SyntheticDense(DenseSpec("thin", 2304, 12544, (Q4_K, Q4_K, Q6_K)), seed=4, scale=0.01)
    ffn = HipDenseMLP(lay.gguf, lay.config, 0, dev)
    for M in (3, 5, 6, 8):
        log(f"thin decode non-finite {bad} M={M}")
        for call, K in ((head, 512), (ffn, 2304)):
            x = torch.randn((M, K), generator=torch.Generator().manual_seed(M)).to(torch.float16).to(dev)
            y = x.clone()
            y[1, K // 3] = bad
            clean, got = call(x), call(y)
            keep = torch.arange(M, device=dev) != 1
            assert torch.equal(got[keep], clean[keep]) and not torch.isfinite(got[1]).any()
