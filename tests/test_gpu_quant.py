"""GPU parity of the quantizers against the CPU oracle: bit-exact bytes and scales.

Cases follow the reference's own byte-exact tests (tests/test_dynamic_fp8_pack.py:7-38,
scripts/qualify_sm89_fp8.py:42-80): shapes (40,2048), (256,5120), (1,16); magnitudes 0,
1e-20, 1e30; every finite bf16 bit pattern; fixed midpoint scales; NaN/inf propagation;
plus every K of the five benchmark configurations, ragged and strided layouts.
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _bits(t: torch.Tensor) -> np.ndarray:
    return t.detach().cpu().contiguous().view(torch.int16).numpy().view(np.uint16)


def _q(t: torch.Tensor) -> np.ndarray:
    return t.detach().cpu().contiguous().view(torch.uint8).numpy()


def _f(t: torch.Tensor) -> np.ndarray:
    return t.detach().cpu().numpy()


def _nan_eq_bytes(got, exp):
    """Byte equality; a NaN code only has to be NaN (sign/payload immaterial,
    scripts/qualify_sm89_fp8.py:71-74)."""
    g, e = np.asarray(got, np.uint8), np.asarray(exp, np.uint8)
    nan_e = (e & 0x7F) == 0x7F
    assert np.array_equal((g & 0x7F) == 0x7F, nan_e)
    bad = np.nonzero((g != e) & ~nan_e)
    assert bad[0].size == 0, f"{bad[0].size} differing bytes, first at {tuple(b[0] for b in bad)}"


def _check_rows(x: torch.Tensor, oracle_mod):
    from instinctflash_amd.kernels import quant_rows
    q, s = quant_rows(x)
    torch.cuda.synchronize()
    xo = _bits(x) if x.dtype == torch.bfloat16 else _f(x).astype(np.float32)
    eq, es = oracle_mod.quant_rows(xo)
    gs = _f(s)
    assert np.array_equal(np.isnan(gs), np.isnan(es))
    assert np.array_equal(gs[~np.isnan(es)].view(np.uint32), es[~np.isnan(es)].view(np.uint32))
    _nan_eq_bytes(_q(q), eq)


def all_finite_bf16():
    pat = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(torch.bfloat16)
    return pat[torch.isfinite(pat)].contiguous()  # 65280 values


def test_known_answer_scale(gpu):
    # tests/test_sm89_fp8.py:48-56: amax 0.0361328125 -> scale 0x38A92493.
    from instinctflash_amd.kernels import quant_rows
    x = torch.full((1, 16), 0.0361328125, dtype=torch.bfloat16, device=gpu)
    _, s = quant_rows(x)
    assert s.cpu().view(torch.int32).item() == 0x38A92493


@pytest.mark.parametrize("shape,mag", [((40, 2048), 1.0), ((256, 5120), 1.0), ((1, 16), 0.0),
                                       ((1, 16), 1e-20), ((1, 16), 1e30)])
def test_reference_cases(gpu, oracle_mod, shape, mag):
    g = torch.Generator().manual_seed(11)
    x = (torch.randn(shape, generator=g) * mag).to(torch.bfloat16).to(gpu)
    _check_rows(x, oracle_mod)


def test_all_finite_bf16_one_row(gpu, oracle_mod):
    _check_rows(all_finite_bf16().reshape(1, -1).to(gpu), oracle_mod)


def test_all_finite_bf16_many_rows(gpu, oracle_mod):
    # 255 rows x 256: each row gets its own scale; exercises the register path.
    x = all_finite_bf16().reshape(255, 256)
    _check_rows(x.to(gpu), oracle_mod)
    # and rows shuffled so magnitudes mix within a row
    perm = torch.randperm(x.numel(), generator=torch.Generator().manual_seed(1))
    _check_rows(x.reshape(-1)[perm].reshape(255, 256).to(gpu), oracle_mod)


@pytest.mark.parametrize("K", [16, 24, 1024, 1536, 2048, 3072, 6144, 11008, 14336, 16384, 20000])
def test_config_widths(gpu, oracle_mod, K):
    g = torch.Generator().manual_seed(K)
    x = torch.randn((37, K), generator=g)
    mask = torch.rand((37, K), generator=g) < 0.01
    x = torch.where(mask, torch.randn((37, K), generator=g) * 20, x)
    _check_rows(x.to(torch.bfloat16).to(gpu), oracle_mod)


@pytest.mark.parametrize("K", [1, 13, 1000, 1003])
def test_ragged_widths(gpu, oracle_mod, K):
    g = torch.Generator().manual_seed(K)
    _check_rows(torch.randn((9, K), generator=g).to(torch.bfloat16).to(gpu), oracle_mod)


def test_strided_rows(gpu, oracle_mod):
    from instinctflash_amd.kernels import quant_rows
    g = torch.Generator().manual_seed(5)
    big = torch.randn((20, 3072), generator=g).to(torch.bfloat16).to(gpu)
    x = big[:, 1024:2048]  # row stride 3072
    qbig = torch.zeros((20, 2048), dtype=torch.float8_e4m3fn, device=gpu)
    q = qbig[:, 512:1536]
    s = torch.empty(20, device=gpu)
    quant_rows(x, q, s)
    eq, es = oracle_mod.quant_rows(_bits(x))
    assert np.array_equal(_f(s).view(np.uint32), es.view(np.uint32))
    assert np.array_equal(_q(q), eq)
    assert not _q(qbig[:, :512]).any() and not _q(qbig[:, 1536:]).any()


def test_rows_past_4gib(gpu, oracle_mod):
    # bf16 input of 4.3 GB and its 2.1 GB e4m3 output: 64-bit row addressing;
    # sampled rows (those past the 4 GiB input offset included) bit-exact
    from instinctflash_amd.kernels import quant_rows
    M, K = 262400, 8192
    assert M * K * 2 >= 1 << 32
    gg = torch.Generator(device=gpu).manual_seed(21)
    x = torch.randn((M, K), device=gpu, generator=gg, dtype=torch.bfloat16)
    q, s = quant_rows(x)
    torch.cuda.synchronize()
    first_past = (1 << 32) // (2 * K)
    rows = torch.as_tensor([0, M // 2, first_past - 1, first_past, first_past + 77, M - 1], device=gpu)
    eq, es = oracle_mod.quant_rows(_bits(x[rows]))
    assert np.array_equal(_f(s[rows]).view(np.uint32), es.view(np.uint32))
    assert np.array_equal(_q(q[rows]), eq)
    del x, q, s
    torch.cuda.empty_cache()


def test_empty_rows(gpu):
    from instinctflash_amd.kernels import quant_rows
    q, s = quant_rows(torch.empty((0, 64), dtype=torch.bfloat16, device=gpu))
    assert q.shape == (0, 64) and s.shape == (0,)


def test_nonfinite_propagation(gpu, oracle_mod):
    for bad in (float("nan"), float("inf"), -float("inf")):
        x = torch.ones((4, 1024), dtype=torch.bfloat16)
        x[0, 0] = bad
        x[2, 700] = bad
        _check_rows(x.to(gpu), oracle_mod)


def test_fp32_weight_rows(gpu, oracle_mod):
    g = torch.Generator().manual_seed(3)
    w = torch.randn((96, 1536), generator=g) * 0.02
    w[5] = 0.0
    w[7, 3] = 1e-30
    _check_rows(w.to(gpu), oracle_mod)
    _check_rows(w[:, :1000].contiguous().to(gpu), oracle_mod)


def test_quantize_weight_matches_recipe(gpu, oracle_mod):
    from instinctflash_amd.kernels import quantize_weight
    g = torch.Generator().manual_seed(4)
    w = torch.randn((4096, 1024), generator=g) * 0.02
    b = torch.randn(4096, generator=g)
    fw = quantize_weight(w, b, device=gpu)
    eq, es = oracle_mod.quant_rows(w.numpy())
    assert np.array_equal(_q(fw.w), eq)
    assert np.array_equal(_f(fw.scale).view(np.uint32), es.view(np.uint32))
    assert torch.equal(fw.bias.cpu(), b)


@pytest.mark.parametrize("scale", [1.0, 1.0 + 2.0 ** -23, 1.0 - 2.0 ** -24, 2.0 ** -16, 1.0 / 448.0])
def test_fixed_scale_pack_all_patterns(gpu, oracle_mod, scale):
    # scripts/qualify_sm89_fp8.py:58-67: exact E4M3 midpoints and scales beside one.
    from instinctflash_amd.kernels import pack_tensor
    x = all_finite_bf16()
    s = torch.tensor([scale], dtype=torch.float32)
    q = pack_tensor(x.to(gpu), s.to(gpu))
    _nan_eq_bytes(_q(q), oracle_mod.pack_fixed(_bits(x), float(s.item())))


@pytest.mark.parametrize("shape,mag", [((40, 2048), 1.0), ((256, 5120), 1.0), ((1, 16), 0.0),
                                       ((1, 16), 1e-20), ((1, 16), 1e30), ((3, 100003), 1.0)])
def test_per_tensor_quant(gpu, oracle_mod, shape, mag):
    from instinctflash_amd.kernels import quantize_tensor
    g = torch.Generator().manual_seed(9)
    x = (torch.randn(shape, generator=g) * mag).to(torch.bfloat16)
    q, s = quantize_tensor(x.to(gpu))
    eq, es = oracle_mod.quant_tensor(_bits(x))
    assert _f(s).view(np.uint32)[0] == es.view(np.uint32)[0]
    _nan_eq_bytes(_q(q), eq)


@pytest.mark.parametrize("count", [8, 8184, 8192, 8200, 131072, 131080])
def test_per_tensor_one_launch_edges(gpu, oracle_mod, count):
    # up to 16 chunks of 8192 elements in one launch, two launches above; the largest value in the last group
    from instinctflash_amd.kernels import quantize_tensor
    x = torch.randn(count, generator=torch.Generator().manual_seed(count)).to(torch.bfloat16)
    x[-1] = -37.0
    q, s = quantize_tensor(x.to(gpu))
    eq, es = oracle_mod.quant_tensor(_bits(x))
    assert _f(s).view(np.uint32)[0] == es.view(np.uint32)[0]
    _nan_eq_bytes(_q(q), eq)
    x[count // 2] = float("nan")
    q, s = quantize_tensor(x.to(gpu))
    assert torch.isnan(s).all() and ((_q(q) & 0x7F) == 0x7F).all()


def test_per_tensor_all_patterns_and_nan(gpu, oracle_mod):
    from instinctflash_amd.kernels import quantize_tensor
    x = all_finite_bf16().reshape(1, -1)
    q, s = quantize_tensor(x.to(gpu))
    eq, es = oracle_mod.quant_tensor(_bits(x))
    assert _f(s).view(np.uint32)[0] == es.view(np.uint32)[0]
    _nan_eq_bytes(_q(q), eq)
    y = torch.full((40, 2048), float("nan"), dtype=torch.bfloat16, device=gpu)
    _, s = quantize_tensor(y)
    assert torch.isnan(s).all()


def test_row_quant_affine_bit_exact(gpu, oracle_mod):
    # reference kernels/norm.py:127-158 without gelu: v = x*row*col + bias in FP32.
    from instinctflash_amd.kernels import row_quant
    g = torch.Generator().manual_seed(21)
    M, D = 50, 2560
    x = torch.randn((M, D), generator=g).to(torch.bfloat16)
    row, col, bias = torch.rand(M, generator=g), torch.rand(D, generator=g), torch.randn(D, generator=g)
    q = torch.empty((M, D), dtype=torch.float8_e4m3fn, device=gpu)
    s = torch.empty(M, device=gpu)
    row_quant(x.to(gpu), q, s, row=row.to(gpu), col=col.to(gpu), bias=bias.to(gpu))
    v = (oracle_mod.bf16_to_f32(_bits(x)) * row.numpy()[:, None]).astype(np.float32)
    v = (v * col.numpy()[None, :]).astype(np.float32) + bias.numpy()[None, :]
    eq, es = oracle_mod.quant_rows(v.astype(np.float32))
    assert np.array_equal(_f(s).view(np.uint32), es.view(np.uint32))
    assert np.array_equal(_q(q), eq)


def _deq(q, s):
    return q.float() * s[:, None]


def _adjacent_codes(got, want):
    """Every differing E4M3 code is one step from the recipe's (signed magnitude order)."""
    a, b = got.astype(np.int32), want.astype(np.int32)
    order = lambda c: np.where(c & 0x80, -(c & 0x7F), c & 0x7F)  # noqa: E731
    d = a != b
    return bool(np.all(np.abs(order(a) - order(b))[d] <= 1))


def test_row_quant_gelu(gpu, oracle_mod):
    from instinctflash_amd.kernels import row_quant
    g = torch.Generator().manual_seed(22)
    M, D = 16, 6144
    x = (torch.randn((M, D), generator=g) * 3).to(torch.bfloat16)
    q = torch.empty((M, D), dtype=torch.float8_e4m3fn, device=gpu)
    s = torch.empty(M, device=gpu)
    row_quant(x.to(gpu), q, s, gelu=True)
    h = oracle_mod.gelu_tanh(oracle_mod.bf16_to_f32(_bits(x)))
    eq, es = oracle_mod.quant_rows(h)
    # GELU uses the hardware exp2/rcp (a few ulp from numpy's tanh): values may
    # straddle a rounding boundary, so require scales within 8 ulp, >= 99.9%
    # identical bytes, and the reference's own envelope
    # (tests/test_gi_kernels.py:127: |deq - h| / amax < 0.07).
    assert np.all(np.abs(_f(s).view(np.int32).astype(np.int64) - es.view(np.int32)) <= 8)
    assert (_q(q) == eq).mean() > 0.999
    assert _adjacent_codes(_q(q), eq)
    err = np.abs(_deq(q, s).cpu().numpy() - h) / np.abs(h).max(axis=1, keepdims=True)
    assert err.max() < 0.07


@pytest.mark.parametrize("M,D", [(50, 2048), (7, 520), (300, 1024)])
def test_row_quant_fp16_input(gpu, oracle_mod, M, D):
    # the pi05 engine quantizes its fp16 attention output (engines/pi05/engine.py:205):
    # fp16 -> fp32 is exact, so bytes and scales are bit-exact to the oracle recipe
    from instinctflash_amd.kernels import row_quant
    g = torch.Generator().manual_seed(M + D)
    x = (torch.randn((M, D), generator=g) * 2).to(torch.float16)
    q = torch.empty((M, D), dtype=torch.float8_e4m3fn, device=gpu)
    s = torch.empty(M, device=gpu)
    row_quant(x.to(gpu), q, s)
    eq, es = oracle_mod.quant_rows(x.float().numpy())
    assert np.array_equal(_q(q), eq) and np.array_equal(_f(s), es)
    row = torch.rand(M, generator=g) + 0.5
    col = torch.rand(D, generator=g) + 0.5
    row_quant(x.to(gpu), q, s, row=row.to(gpu), col=col.to(gpu))
    v = (x.float().numpy() * row.numpy()[:, None]).astype(np.float32) * col.numpy()[None, :]
    eq, es = oracle_mod.quant_rows(v.astype(np.float32))
    assert np.array_equal(_q(q), eq) and np.array_equal(_f(s), es)


@pytest.mark.parametrize("M,D", [(96, 2048), (5, 1000)])
def test_row_quant_fp32_input(gpu, oracle_mod, M, D):
    # the GR00T engine quantizes its float32 encoder rows (engines/groot_n17/engine.py:144):
    # bytes and scales bit-exact to the oracle recipe, also with the affine terms
    from instinctflash_amd.kernels import row_quant
    g = torch.Generator().manual_seed(M * D)
    x = torch.randn((M, D), generator=g) * 3
    x[1] = 0.0  # an all-zero row takes the scale floor
    q = torch.empty((M, D), dtype=torch.float8_e4m3fn, device=gpu)
    s = torch.empty(M, device=gpu)
    row_quant(x.to(gpu), q, s)
    eq, es = oracle_mod.quant_rows(x.numpy())
    assert np.array_equal(_q(q), eq) and np.array_equal(_f(s).view(np.uint32), es.view(np.uint32))
    row, col, bias = torch.rand(M, generator=g) + 0.5, torch.rand(D, generator=g) + 0.5, torch.randn(D, generator=g)
    row_quant(x.to(gpu), q, s, row=row.to(gpu), col=col.to(gpu), bias=bias.to(gpu))
    v = ((x.numpy() * row.numpy()[:, None]).astype(np.float32) * col.numpy()[None, :]).astype(np.float32)
    eq, es = oracle_mod.quant_rows((v + bias.numpy()[None, :]).astype(np.float32))
    assert np.array_equal(_q(q), eq) and np.array_equal(_f(s).view(np.uint32), es.view(np.uint32))


@pytest.mark.parametrize("act", [0, 1])
def test_gated_act_quant(gpu, oracle_mod, act):
    from instinctflash_amd.kernels import gated_act_quant
    g = torch.Generator().manual_seed(23 + act)
    M, F = 9, 4096
    gu = torch.randn((M, 2 * F), generator=g).to(torch.bfloat16)
    row, col = torch.rand(M, generator=g), torch.rand(2 * F, generator=g)
    q = torch.empty((M, F), dtype=torch.float8_e4m3fn, device=gpu)
    s = torch.empty(M, device=gpu)
    gated_act_quant(gu.to(gpu), q, s, row=row.to(gpu), col=col.to(gpu), act=act)
    x = oracle_mod.bf16_to_f32(_bits(gu)) * row.numpy()[:, None] * col.numpy()[None, :]
    gg, uu = x[:, :F].astype(np.float32), x[:, F:].astype(np.float32)
    h = (oracle_mod.gelu_tanh(gg) if act == 0 else oracle_mod.silu(gg)) * uu
    eq, es = oracle_mod.quant_rows(h.astype(np.float32))
    assert np.all(np.abs(_f(s).view(np.int32).astype(np.int64) - es.view(np.int32)) <= 8)
    assert (_q(q) == eq).mean() > 0.999
    assert _adjacent_codes(_q(q), eq)
    err = np.abs(_deq(q, s).cpu().numpy() - h) / np.abs(h).max(axis=1, keepdims=True)
    assert err.max() < 0.07


def test_dequant_rows(gpu):
    from instinctflash_amd.kernels import dequant_rows
    g = torch.Generator().manual_seed(24)
    M, D = 50, 4096
    x = torch.randn((M, D), generator=g).to(torch.bfloat16)
    row, col, bias = torch.rand(M, generator=g), torch.rand(D, generator=g), torch.randn(D, generator=g)
    y = torch.empty((M, D), device=gpu)
    dequant_rows(x.to(gpu), y, row=row.to(gpu), col=col.to(gpu), bias=bias.to(gpu))
    exp = (x.float() * row[:, None]) * col + bias
    assert torch.equal(y.cpu(), exp)
    yb = torch.empty((M, D), dtype=torch.bfloat16, device=gpu)
    dequant_rows(x.to(gpu), yb, row=row.to(gpu), col=col.to(gpu), bias=bias.to(gpu))
    assert torch.equal(yb.cpu(), exp.to(torch.bfloat16))
    # any float dtypes in and out (the reference's GR00T engine writes fp16 q|k|v
    # and cross K/V): float32 arithmetic in the same order, one rounding at the store
    for xd in (torch.float16, torch.float32):
        for yd in (torch.float16, torch.bfloat16, torch.float32):
            xs = x.to(xd)
            yo = torch.empty((M, D), dtype=yd, device=gpu)
            dequant_rows(xs.to(gpu), yo, row=row.to(gpu), col=col.to(gpu), bias=bias.to(gpu))
            ex = ((xs.float() * row[:, None]) * col + bias).to(yd)
            assert torch.equal(yo.cpu(), ex), (xd, yd)
    # strided rows (a column slice of a wider accumulator)
    wide = torch.randn((M, 3 * D // 2), generator=g).to(torch.bfloat16)
    ys = torch.empty((M, D // 2), dtype=torch.float16, device=gpu)
    dequant_rows(wide.to(gpu)[:, D:], ys, col=col[: D // 2].to(gpu))
    assert torch.equal(ys.cpu(), (wide[:, D:].float() * col[: D // 2]).to(torch.float16))


def test_graph_replay_matches_eager(gpu, oracle_mod):
    # tests/test_dynamic_fp8_pack.py:24-35: captured launches give the eager bytes.
    from instinctflash_amd.kernels import quant_rows
    x = torch.randn((40, 2048), device=gpu).to(torch.bfloat16)
    q = torch.empty((40, 2048), dtype=torch.float8_e4m3fn, device=gpu)
    s = torch.empty(40, device=gpu)
    st = torch.cuda.Stream()
    st.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(st):
        for _ in range(3):
            quant_rows(x, q, s)
    torch.cuda.current_stream().wait_stream(st)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=st):
        quant_rows(x, q, s)
    for mag in (0.0, 1e-4, 20.0, 1.0):
        x.copy_(torch.randn_like(x) * mag)
        graph.replay()
        torch.cuda.synchronize()
        qe, se = quant_rows(x)
        torch.cuda.synchronize()
        assert torch.equal(s, se)
        assert torch.equal(q.view(torch.uint8), qe.view(torch.uint8))


@pytest.mark.parametrize("seed", [0, 1, 2])
def test_random_wide_range_stress(gpu, oracle_mod, seed):
    # 64 rows x 65536 fp32 values spanning ~80 binades, random signs, exact zeros,
    # values at and beside every E4M3 midpoint of the row's scale: the fast
    # division/packing path must give the oracle's bytes everywhere.
    rng = np.random.default_rng(seed)
    R, K = 64, 65536
    mag = np.exp2(rng.uniform(-60, 20, size=(R, K))).astype(np.float32)
    x = (mag * rng.choice([-1.0, 1.0], size=(R, K))).astype(np.float32)
    x[:, :64] = 0.0
    amax = np.abs(x).max(axis=1)
    s = (np.maximum(amax, np.float32(1e-12)) * (np.float32(1) / np.float32(448))).astype(np.float32)
    pos = np.unique(oracle_mod.E4M3_VALUES[~np.isnan(oracle_mod.E4M3_VALUES)]).astype(np.float64)
    pos = pos[pos > 0]
    mids = ((pos[1:] + pos[:-1]) / 2)[:, None] * s[None, :].astype(np.float64)   # [n_mid, R]
    n = mids.shape[0]
    for k, eps in enumerate((0.0, 1.0, -1.0)):
        v = (mids * (1 + eps * 2.0 ** -23)).astype(np.float32).T                    # [R, n_mid]
        x[:, 64 + k * n:64 + (k + 1) * n] = np.minimum(v, amax[:, None])
    _check_rows(torch.from_numpy(x).to(gpu), oracle_mod)
    _check_rows(torch.from_numpy(x).to(torch.bfloat16).to(gpu), oracle_mod)


# Every width form of the row engine (lanes per row x 8-value groups per lane),
# for each row source: (M, K) pairs that select them -- fewer than 256 rows give
# each row a whole block (256 / 512 / 1024 lanes), more rows pack 64-256 lanes per
# row, K % 8 != 0 takes the generic kernel.
_FORMS = [(20, 1024), (20, 4096), (20, 8192), (20, 16384), (20, 32768), (20, 1004),
          (260, 512), (260, 1024), (260, 2048), (260, 3072), (260, 4096), (260, 8192), (260, 16384),
          (260, 32768)]
_SOURCES = ["bf16", "f32", "affine", "affine_col", "affine_bias_gelu", "gelu", "gated_gelu_col", "gated_silu"]


@pytest.mark.parametrize("M,K", _FORMS)
@pytest.mark.parametrize("src", _SOURCES)
def test_row_engine_forms(gpu, oracle_mod, src, M, K):
    from instinctflash_amd.kernels import gated_act_quant, quant_rows, row_quant
    gated = src.startswith("gated")
    if gated and K > 16384:
        pytest.skip("gated_act_quant takes hidden widths up to 16384 (the reference's contract)")
    g = torch.Generator().manual_seed(M * 131 + K + len(src))
    cols = 2 * K if gated else K
    x = (torch.randn((M, cols), generator=g) * 2).to(torch.float32 if src == "f32" else torch.bfloat16)
    row, col = torch.rand(M, generator=g) + 0.5, torch.rand(cols, generator=g) + 0.5
    bias = torch.randn(cols, generator=g)
    xf = x.numpy() if src == "f32" else oracle_mod.bf16_to_f32(_bits(x))
    q = torch.empty((M, K), dtype=torch.float8_e4m3fn, device=gpu)
    s = torch.empty(M, device=gpu)
    exact = True
    if src in ("bf16", "f32"):
        q, s = quant_rows(x.to(gpu))
        v = xf
    elif src.startswith("affine") or src == "gelu":
        use_col = src in ("affine", "affine_col")
        use_bias = src in ("affine", "affine_bias_gelu")
        gelu = src.endswith("gelu")
        row_quant(x.to(gpu), q, s, row=row.to(gpu), col=col.to(gpu) if use_col else None,
                  bias=bias.to(gpu) if use_bias else None, gelu=gelu)
        v = (xf * row.numpy()[:, None]).astype(np.float32)
        if use_col:
            v = (v * col.numpy()[None, :]).astype(np.float32)
        if use_bias:
            v = (v + bias.numpy()[None, :]).astype(np.float32)
        if gelu:
            v, exact = oracle_mod.gelu_tanh(v), False
    else:
        use_col = src.endswith("col")
        act = 0 if "gelu" in src else 1
        gated_act_quant(x.to(gpu), q, s, row=row.to(gpu), col=col.to(gpu) if use_col else None, act=act)
        h = (xf * row.numpy()[:, None]).astype(np.float32)
        if use_col:
            h = (h * col.numpy()[None, :]).astype(np.float32)
        gg, uu = h[:, :K], h[:, K:]
        v, exact = ((oracle_mod.gelu_tanh(gg) if act == 0 else oracle_mod.silu(gg)) * uu).astype(np.float32), False
    torch.cuda.synchronize()
    eq, es = oracle_mod.quant_rows(np.ascontiguousarray(v, dtype=np.float32))
    if exact:
        assert np.array_equal(_f(s).view(np.uint32), es.view(np.uint32)), f"{src} {M}x{K}: scales"
        assert np.array_equal(_q(q), eq), f"{src} {M}x{K}: bytes"
    else:
        # hardware exp2 / rcp: the bars of the GELU and gated tests above
        assert np.all(np.abs(_f(s).view(np.int32).astype(np.int64) - es.view(np.int32)) <= 8)
        assert (_q(q) == eq).mean() > 0.999
        err = np.abs(_deq(q, s).cpu().numpy() - v) / np.abs(v).max(axis=1, keepdims=True)
        assert err.max() < 0.07
