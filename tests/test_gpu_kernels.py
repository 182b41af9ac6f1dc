"""Kernel-level parity of the HIP path against the CPU oracle, through the C ABI.

Bar: bit-exact for every GEMM output (int32 accumulators + the f32 fma epilogue)
and every int8 activation / scale on identical inputs; attention (f32, a
different summation order) within the tolerance stated in its test.
"""
import numpy as np
import pytest

import arctic_embed_amd as ae
import oracle as orc

pytestmark = pytest.mark.gpu
f32 = np.float32
# (n, k): the model's four, plus K = 1152 (an even number of 64-deep K steps off
# the model's sizes) and K = 448 (an odd number: the small-M forms hand it to the
# tiled kernel)
SHAPES = [(1152, 384), (384, 384), (1536, 384), (384, 1536), (768, 384), (384, 1152), (384, 448)]


def dev(torch, a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def bits(a):
    return np.ascontiguousarray(a, f32).view(np.uint32)


def linear_inputs(n, k, seed):
    rng = np.random.default_rng(seed)
    w = rng.integers(-127, 128, (n, k), dtype=np.int8)
    ws = (0.05 / 127 * rng.uniform(0.5, 1.5, n)).astype(f32)
    b = rng.normal(0, 0.02, n).astype(f32)
    s = rng.uniform(0.5, 2.0, k).astype(f32) ** -1
    return w, ws, b, s.astype(f32)


@pytest.mark.parametrize("n,k", SHAPES)
@pytest.mark.parametrize("m", [1, 37, 200])
@pytest.mark.parametrize("with_res", [False, True])
def test_gemm_bit_exact(torch_gpu, n, k, m, with_res):
    torch = torch_gpu
    w, ws, b, s = linear_inputs(n, k, n + k + m)
    rng = np.random.default_rng(m)
    a = rng.integers(-127, 128, (m, k), dtype=np.int8)
    sa = rng.uniform(0.01, 0.1, m).astype(f32)
    res = rng.normal(0, 1, (m, n)).astype(f32) if with_res else None
    lin = ae.Linear(w, ws, b, s)
    a_d, sa_d = dev(torch, a), dev(torch, sa)
    res_d = dev(torch, res) if with_res else None
    out_d = torch.full((m, n), float("nan"), dtype=torch.float32, device="cuda")
    lin.gemm(m, a_d.data_ptr(), sa_d.data_ptr(), res_d.data_ptr() if with_res else None, out_d.data_ptr())
    torch.cuda.synchronize()
    ref = orc.gemm(a, sa, w, ws, b, res)
    assert np.array_equal(bits(out_d.cpu().numpy()), bits(ref))


@pytest.mark.parametrize("k,n", [(384, 1152), (384, 384), (384, 1536), (1536, 384)])
@pytest.mark.parametrize("m", [128, 4096, 32768])
def test_gemm_configs1_microbench_shapes(torch_gpu, m, k, n):
    """The standalone W8A8 GEMM microbench that bench.py --gemm times, at its
    own sizes and distributions: A int8 U[-127,127] with row scales U(0.01,0.1), W [K x N] int8
    U[-127,127] (stored [N,K]) with column scales U(0.0002,0.0006), bias N(0,0.02), f32 out.
    GEMM rows are independent, so every row at M = 128 and 64 rows otherwise (the first and
    last 8 and 48 random ones) are checked bit for bit against the oracle's gemm_scalar_fused."""
    torch = torch_gpu
    rng = np.random.default_rng(1000 * m + n + k)
    w = rng.integers(-127, 128, (n, k), dtype=np.int8)
    ws = rng.uniform(0.0002, 0.0006, n).astype(f32)
    b = rng.normal(0, 0.02, n).astype(f32)
    a = rng.integers(-127, 128, (m, k), dtype=np.int8)
    sa = rng.uniform(0.01, 0.1, m).astype(f32)
    lin = ae.Linear(w, ws, b, np.ones(k, f32))
    a_d, sa_d = dev(torch, a), dev(torch, sa)
    out_d = torch.full((m, n), float("nan"), dtype=torch.float32, device="cuda")
    lin.gemm(m, a_d.data_ptr(), sa_d.data_ptr(), None, out_d.data_ptr())
    torch.cuda.synchronize()
    out = out_d.cpu().numpy()
    lin.close()
    if m <= 128:
        rows = np.arange(m)
    else:
        rows = np.unique(np.concatenate([np.arange(8), np.arange(m - 8, m), rng.choice(m, 48, replace=False)]))
    ref = orc.gemm(a[rows], sa[rows], w, ws, b)
    assert np.array_equal(bits(out[rows]), bits(ref))
    assert np.all(np.isfinite(out))


@pytest.mark.parametrize("m,n", [(24576, 1152), (40000, 1152), (32761, 768)])
def test_gemm_row_stationary_tiles(torch_gpu, m, n):
    """Many-row int8 GEMMs without residual run A-stationary (an A tile of 48 or 64 rows kept in LDS
    while the workgroup walks every column tile): 24,576 rows in exactly 512 tiles of 48, 40,000
    rows (48-row tiles, the last one partial) and 32,761 rows (64-row tiles, the last one partial).
    Rows of the first, last and random tiles bit for bit against the oracle."""
    torch = torch_gpu
    k = 384
    w, ws, b, s = linear_inputs(n, k, m + n)
    rng = np.random.default_rng(m)
    a = rng.integers(-127, 128, (m, k), dtype=np.int8)
    sa = rng.uniform(0.01, 0.1, m).astype(f32)
    lin = ae.Linear(w, ws, b, s)
    a_d, sa_d = dev(torch, a), dev(torch, sa)
    out_d = torch.full((m, n), float("nan"), dtype=torch.float32, device="cuda")
    lin.gemm(m, a_d.data_ptr(), sa_d.data_ptr(), None, out_d.data_ptr())
    torch.cuda.synchronize()
    out = out_d.cpu().numpy()
    lin.close()
    rows = np.unique(np.concatenate([np.arange(72), np.arange(m - 72, m), rng.choice(m, 96, replace=False)]))
    assert np.array_equal(bits(out[rows]), bits(orc.gemm(a[rows], sa[rows], w, ws, b)))
    assert np.all(np.isfinite(out))


@pytest.mark.parametrize("m,n,k", [(1025, 384, 384), (2048, 1152, 384), (2049, 1152, 384), (1537, 1536, 384),
                                   (1025, 384, 1536), (4096, 384, 1536), (4097, 384, 1536), (6144, 384, 1536),
                                   (6145, 384, 1536), (1100, 768, 1024), (1536, 1152, 1024)])
@pytest.mark.parametrize("with_res", [False, True])
def test_gemm_int8_tile_heights(torch_gpu, m, n, k, with_res):
    """Both sides of the rule that keeps 16-row workgroups beyond 1,024 rows, with partial last tiles;
    the first, last and 48 random rows bit for bit."""
    torch = torch_gpu
    w, ws, b, s = linear_inputs(n, k, n + k + m)
    rng = np.random.default_rng(m)
    a, sa = rng.integers(-127, 128, (m, k), dtype=np.int8), rng.uniform(0.01, 0.1, m).astype(f32)
    res = rng.normal(0, 1, (m, n)).astype(f32) if with_res else None
    lin = ae.Linear(w, ws, b, s)
    a_d, sa_d = dev(torch, a), dev(torch, sa)
    res_d = dev(torch, res) if with_res else None
    out_d = torch.full((m, n), float("nan"), dtype=torch.float32, device="cuda")
    lin.gemm(m, a_d.data_ptr(), sa_d.data_ptr(), res_d.data_ptr() if with_res else None, out_d.data_ptr())
    torch.cuda.synchronize()
    lin.close()
    rows = np.unique(np.r_[0:16, m - 17:m, rng.integers(0, m, 48)])
    out = out_d.cpu().numpy()
    assert not np.isnan(out).any()
    assert np.array_equal(bits(out[rows]), bits(orc.gemm(a[rows], sa[rows], w, ws, b, res[rows] if with_res else None)))


def test_gemm_extreme_accumulators(torch_gpu):
    torch = torch_gpu
    n, k, m = 384, 1536, 3
    w = np.full((n, k), 127, np.int8)
    w[1::2] = -127
    a = np.full((m, k), 127, np.int8)
    a[1] = -127
    a[2, ::3] = -127
    lin = ae.Linear(w, np.ones(n, f32), np.zeros(n, f32), np.ones(k, f32))
    a_d, sa_d = dev(torch, a), dev(torch, np.ones(m, f32))
    out_d = torch.zeros((m, n), dtype=torch.float32, device="cuda")
    lin.gemm(m, a_d.data_ptr(), sa_d.data_ptr(), None, out_d.data_ptr())
    torch.cuda.synchronize()
    ref = orc.gemm(a, np.ones(m, f32), w, np.ones(n, f32), np.zeros(n, f32))
    assert np.array_equal(bits(out_d.cpu().numpy()), bits(ref))
    assert ref[0, 0] == f32(1536 * 127 * 127)


@pytest.mark.parametrize("smooth", [True, False])
@pytest.mark.parametrize("n,k", [(384, 384), (384, 1536)])
def test_gemm_quantize_on_load_bit_exact(torch_gpu, smooth, n, k):
    """attn_out / FFN-down GEMM: A = smooth_quantize(f32 rows) inside the GEMM prologue."""
    torch = torch_gpu
    m = 70
    w, ws, b, s = linear_inputs(n, k, 7 + k)
    rng = np.random.default_rng(k)
    x = rng.normal(0, 1.5, (m, k)).astype(f32)
    x[3] = 0.0  # zero row -> max_abs floor 1e-8
    res = rng.normal(0, 1, (m, n)).astype(f32)
    sv = s if smooth else np.ones(k, f32)
    rowmax = np.maximum(np.abs(x * sv).max(1), f32(1e-8)).astype(f32)
    lin = ae.Linear(w, ws, b, s)
    x_d, rm_d, res_d = dev(torch, x), dev(torch, rowmax.view(np.uint32).astype(np.int32)), dev(torch, res)
    s_d = dev(torch, s)
    out_d = torch.zeros((m, n), dtype=torch.float32, device="cuda")
    lin.gemm_quant_a(m, x_d.data_ptr(), rm_d.data_ptr(), s_d.data_ptr() if smooth else None, res_d.data_ptr(),
                     out_d.data_ptr())
    torch.cuda.synchronize()
    q, sc = orc.smooth_quant_rows(x, sv)  # src/simd_math.rs:513-530
    ref = orc.gemm(q, sc, w, ws, b, res)
    assert np.array_equal(bits(out_d.cpu().numpy()), bits(ref))


@pytest.mark.parametrize("m", [37, 1500, 2000, 4101, 16387])
def test_gemm_then_layernorm_bit_exact(torch_gpu, m):
    """The attention output GEMM and LN1 in one kernel (16-row workgroups up to 4,096 rows, 32-row ones
    of 8 waves up to 16,384, then of 4, with partial last tiles): f32 LN rows, int8 rows and scales
    bit for bit against the oracle's smooth_quantize -> gemm_scalar_fused(residual) ->
    layernorm_smooth_quantize.  Rows include a zero ctx row, a residual row whose mean and variance
    depend on the summation order (+-1e8 against small values) and a constant output row."""
    torch = torch_gpu
    n = k = 384
    w, ws, b, s = linear_inputs(n, k, 11)
    rng = np.random.default_rng(m + 5)
    x = rng.normal(0, 1.5, (m, k)).astype(f32)
    x[3] = 0.0
    res = rng.normal(0, 1, (m, n)).astype(f32)
    res[5, :] = rng.normal(0, 1e-3, n).astype(f32)
    res[5, 0], res[5, 1] = f32(1e8), f32(-1e8)
    res[m - 1, :] = f32(2.5)
    x[m - 1] = 0.0  # output row = bias + 2.5 (constant up to the bias)
    gamma = (1 + rng.normal(0, 0.05, n)).astype(f32)
    beta = rng.normal(0, 0.02, n).astype(f32)
    ln_s = (rng.uniform(0.5, 2.0, n) ** -1).astype(f32)
    rowmax = np.maximum(np.abs(x * s).max(1), f32(1e-8)).astype(f32)
    lin = ae.Linear(w, ws, b, s)
    x_d, rm_d, res_d = dev(torch, x), dev(torch, rowmax.view(np.uint32).astype(np.int32)), dev(torch, res)
    s_d, g_d, b_d, ls_d = dev(torch, s), dev(torch, gamma), dev(torch, beta), dev(torch, ln_s)
    dst_d = torch.full((m, n), float("nan"), dtype=torch.float32, device="cuda")
    q_d = torch.zeros((m, n), dtype=torch.int8, device="cuda")
    sc_d = torch.zeros(m, dtype=torch.float32, device="cuda")
    lin.gemm_ln(m, x_d.data_ptr(), rm_d.data_ptr(), s_d.data_ptr(), res_d.data_ptr(), g_d.data_ptr(), b_d.data_ptr(),
                ls_d.data_ptr(), dst_d.data_ptr(), q_d.data_ptr(), sc_d.data_ptr())
    torch.cuda.synchronize()
    lin.close()
    q, sc = orc.smooth_quant_rows(x, s)
    out = orc.gemm(q, sc, w, ws, b, res)
    ry, rq, rsc = orc.ln_quant_rows(out, gamma, beta, ln_s)
    assert np.array_equal(bits(dst_d.cpu().numpy()), bits(ry))
    assert np.array_equal(q_d.cpu().numpy(), rq)
    assert np.array_equal(bits(sc_d.cpu().numpy()), bits(rsc))


@pytest.mark.parametrize("m", [1025, 4095, 4096, 4097, 16384, 16385])
def test_gemm_then_layernorm_tile_heights(torch_gpu, m):
    """The same on both sides of the rules for the tile height (16 rows while one workgroup per
    compute unit covers them, 32 beyond, with 8 waves up to two per compute unit, then with 4), with
    partial last tiles, the output in the residual's place."""
    torch = torch_gpu
    n = k = 384
    w, ws, b, s = linear_inputs(n, k, 12)
    rng = np.random.default_rng(m)
    x, res = rng.normal(0, 1.5, (m, k)).astype(f32), rng.normal(0, 1, (m, n)).astype(f32)
    gamma, beta = (1 + rng.normal(0, 0.05, n)).astype(f32), rng.normal(0, 0.02, n).astype(f32)
    ln_s = (rng.uniform(0.5, 2.0, n) ** -1).astype(f32)
    rowmax = np.maximum(np.abs(x * s).max(1), f32(1e-8)).astype(f32)
    lin = ae.Linear(w, ws, b, s)
    x_d, rm_d, res_d = dev(torch, x), dev(torch, rowmax.view(np.uint32).astype(np.int32)), dev(torch, res)
    s_d, g_d, b_d, ls_d = dev(torch, s), dev(torch, gamma), dev(torch, beta), dev(torch, ln_s)
    q_d = torch.zeros((m, n), dtype=torch.int8, device="cuda")
    sc_d = torch.zeros(m, dtype=torch.float32, device="cuda")
    lin.gemm_ln(m, x_d.data_ptr(), rm_d.data_ptr(), s_d.data_ptr(), res_d.data_ptr(), g_d.data_ptr(), b_d.data_ptr(),
                ls_d.data_ptr(), res_d.data_ptr(), q_d.data_ptr(), sc_d.data_ptr())
    torch.cuda.synchronize()
    lin.close()
    q, sc = orc.smooth_quant_rows(x, s)
    ry, rq, rsc = orc.ln_quant_rows(orc.gemm(q, sc, w, ws, b, res), gamma, beta, ln_s)
    assert np.array_equal(bits(res_d.cpu().numpy()), bits(ry))
    assert np.array_equal(q_d.cpu().numpy(), rq)
    assert np.array_equal(bits(sc_d.cpu().numpy()), bits(rsc))


@pytest.mark.parametrize("m", [1, 45, 130])
def test_gemm_gelu_epilogue_bit_exact(torch_gpu, m):
    """FFN-up GEMM with the GELU * inv_smooth epilogue and the row absmax."""
    torch = torch_gpu
    n, k = 1536, 384
    w, ws, b, s = linear_inputs(n, k, 99)
    rng = np.random.default_rng(m + 5)
    a = rng.integers(-127, 128, (m, k), dtype=np.int8)
    sa = rng.uniform(0.01, 0.1, m).astype(f32)
    g_smooth = rng.uniform(0.5, 2.0, n).astype(f32) ** -1
    g_smooth = g_smooth.astype(f32)
    lin = ae.Linear(w, ws, b, s)
    a_d, sa_d, gs_d = dev(torch, a), dev(torch, sa), dev(torch, g_smooth)
    rm_d = dev(torch, np.full(m, f32(1e-8)).view(np.uint32).astype(np.int32))
    out_d = torch.zeros((m, n), dtype=torch.float32, device="cuda")
    lin.gemm_gelu(m, a_d.data_ptr(), sa_d.data_ptr(), gs_d.data_ptr(), out_d.data_ptr(), rm_d.data_ptr())
    torch.cuda.synchronize()
    pre = orc.gemm(a, sa, w, ws, b)
    g, q, sc = orc.gelu_quant_rows(pre, g_smooth)  # src/simd_math.rs:1295-1312
    assert np.array_equal(bits(out_d.cpu().numpy()), bits(g))
    rowmax = rm_d.cpu().numpy().astype(np.int64).astype(np.uint32).view(f32)
    assert np.array_equal(rowmax / f32(127), sc)


@pytest.fixture(params=[16, 32, 64, -64], ids=["rows16", "rows32", "rows64", "mixed64"])
def ffn_rows(request, torch_gpu):
    """Every fused-FFN test runs with 16-, 32- and 64-row workgroups, and with the
    first 64 rows in a 64-row workgroup and the rest in a second launch of 32-row
    ones."""
    ae.set_ffn_rows(request.param)
    yield request.param
    ae.set_ffn_rows(0)


@pytest.mark.parametrize("m,in_place", [(1, False), (31, False), (33, True), (64, False), (100, False),
                                        (4133, True)])
def test_ffn_fused_bit_exact(torch_gpu, ffn_rows, m, in_place):
    """The one-kernel FFN block (FFN-up + GELU * inv_smooth + row absmax int8
    quantization + FFN-down + bias + residual) against the oracle's three steps
    (src/model.rs:725-755): bit-exact, including partial last workgroups (and
    partial second passes of 64-row ones) and out == res."""
    torch = torch_gpu
    print("ffn rows", ffn_rows, "m", m, flush=True)
    w1, ws1, b1, s1 = linear_inputs(1536, 384, 7)
    w2, ws2, b2, s2 = linear_inputs(384, 1536, 8)
    rng = np.random.default_rng(m + 11)
    a = rng.integers(-127, 128, (m, 384), dtype=np.int8)
    a[0, :] = 0  # a row whose GELU outputs are GELU(bias) only
    sa = rng.uniform(0.01, 0.1, m).astype(f32)
    res = rng.normal(0, 1, (m, 384)).astype(f32)
    up, down = ae.Linear(w1, ws1, b1, s1), ae.Linear(w2, ws2, b2, s2)
    a_d, sa_d, res_d = dev(torch, a), dev(torch, sa), dev(torch, res)
    out_d = res_d if in_place else torch.full((m, 384), float("nan"), dtype=torch.float32, device="cuda")
    up.ffn(down, m, a_d.data_ptr(), sa_d.data_ptr(), res_d.data_ptr(), out_d.data_ptr())
    torch.cuda.synchronize()
    pre = orc.gemm(a, sa, w1, ws1, b1)
    _, q, sc = orc.gelu_quant_rows(pre, s2)  # src/simd_math.rs:1295-1312
    ref = orc.gemm(q, sc, w2, ws2, b2, res)
    assert np.array_equal(bits(out_d.cpu().numpy()), bits(ref))


def test_ffn_fused_extreme_rows(torch_gpu, ffn_rows):
    """The fused FFN on rows that drive the GELU to its extremes: saturated int8
    rows (|pre-activation| up to ~1e3, GELU -> 0 or x), tiny scales (GELU near
    0, the 1e-8 absmax floor), a single nonzero column, and rows of equal values
    (quantization ties); the same rows again from row 32 (the second pass of a
    64-row workgroup)."""
    torch = torch_gpu
    w1, ws1, b1, s1 = linear_inputs(1536, 384, 21)
    w2, ws2, b2, s2 = linear_inputs(384, 1536, 22)
    m = 72
    rng = np.random.default_rng(23)
    a = rng.integers(-127, 128, (m, 384), dtype=np.int8)
    sa = rng.uniform(0.01, 0.1, m).astype(f32)
    for o in (0, 32):
        a[o + 1:o + 5] = 127
        a[o + 5:o + 9] = -127
        a[o + 9] = 0
        a[o + 10] = 0
        a[o + 10, 17] = 127
        a[o + 11:o + 14] = 64
        sa[o + 1:o + 3] = 40.0                  # huge pre-activations
        sa[o + 14:o + 18] = np.float32(1e-30)   # GELU inputs ~ bias only
        sa[o + 18] = 0.0
    res = rng.normal(0, 1, (m, 384)).astype(f32)
    up, down = ae.Linear(w1, ws1, b1, s1), ae.Linear(w2, ws2, b2, s2)
    a_d, sa_d, res_d = dev(torch, a), dev(torch, sa), dev(torch, res)
    out_d = torch.full((m, 384), float("nan"), dtype=torch.float32, device="cuda")
    up.ffn(down, m, a_d.data_ptr(), sa_d.data_ptr(), res_d.data_ptr(), out_d.data_ptr())
    torch.cuda.synchronize()
    pre = orc.gemm(a, sa, w1, ws1, b1)
    _, q, sc = orc.gelu_quant_rows(pre, s2)
    ref = orc.gemm(q, sc, w2, ws2, b2, res)
    assert np.array_equal(bits(out_d.cpu().numpy()), bits(ref))


def test_gelu_fast_certified_on_every_float(torch_gpu):
    """The fused FFN's fast GELU against the reference's GELU (gelu_exact, itself bit-exact with
    the oracle's scalar_gelu: test_gelu_bit_exact_over_float_sample) on all 2^32 f32 inputs, as
    the kernels evaluate both: no input outside the certified bound |G - G'| <= 2^-21 |G'| +
    0x1.64p-24, NaN only for NaN and +-inf inputs, and the saturated ranges (G(v) = v from
    5.3474278, G(v) = 0 below -5.5430403) exact.  The same enumeration with half the absolute
    term finds violations, so the bound is near tight and the check is not vacuous."""
    c = ae.gelu_fast_certify()
    assert c[5] == 1 << 32
    assert c[0] == 0 and c[1] == 0, c
    assert c[2] == 0 and c[3] == 0, c
    assert c[4] > 0, c


def _ffn_ref(a, sa, w1, ws1, b1, w2, ws2, b2, s2, res):
    pre = orc.gemm(a, sa, w1, ws1, b1)
    _, q, sc = orc.gelu_quant_rows(pre, s2)  # src/simd_math.rs:1295-1312
    return orc.gemm(q, sc, w2, ws2, b2, res)


def test_ffn_fast_gelu_repairs_are_exact(torch_gpu, ffn_rows):
    """Inputs built so that the fast GELU cannot decide: (1) the row maximum is exactly 127 in two
    columns of one lane (columns 0 and 16: all-zero weights, bias 63.5, inv_smooth 2, GELU
    saturated), a tie the kernel settles by recomputing every element that can reach it; (2)
    zero-weight columns whose GELU * inv_smooth lands exactly on k + 0.5 or one ulp either side of
    it (and a negative inv_smooth), so that x = g * (127 / 127) is undecided and the tile is
    recomputed from its pre-activations.  Bit-exact with the oracle, the repair counters move,
    and the exact-GELU kernel gives the same bits."""
    torch = torch_gpu
    w1, ws1, b1, s1 = linear_inputs(1536, 384, 31)
    w2, ws2, b2, s2 = linear_inputs(384, 1536, 32)
    for c in (0, 16):  # the row maximum, tied inside lane (wave 0, column 0)
        w1[c] = 0
        b1[c] = 63.5
        s2[c] = 2.0
    targets = [10.5, 20.5, 100.5, 6.5, np.nextafter(f32(10.5), f32(0)), np.nextafter(f32(10.5), f32(99)),
               np.nextafter(f32(6.5), f32(0)), 50.5, 126.5, 7.5]
    cols = [37, 200, 399, 401, 777, 1000, 1201, 1535, 512, 95]
    for c, t in zip(cols, targets):
        w1[c] = 0
        b1[c] = t
        s2[c] = 1.0
    s2[95] = -1.0  # x = -7.5: rounds away to -8
    m = 100
    rng = np.random.default_rng(33)
    a = rng.integers(-127, 128, (m, 384), dtype=np.int8)
    sa = rng.uniform(0.01, 0.1, m).astype(f32)
    res = rng.normal(0, 1, (m, 384)).astype(f32)
    up, down = ae.Linear(w1, ws1, b1, s1), ae.Linear(w2, ws2, b2, s2)
    a_d, sa_d, res_d = dev(torch, a), dev(torch, sa), dev(torch, res)
    ref = _ffn_ref(a, sa, w1, ws1, b1, w2, ws2, b2, s2, res)
    pre = orc.gemm(a, sa, w1, ws1, b1)
    _, _, sc = orc.gelu_quant_rows(pre, s2)
    assert np.all(sc == f32(127) / f32(127))  # every row's maximum is the tied 127
    outs = []
    try:
        for exact in (False, True):
            ae.set_ffn_exact_gelu(exact)
            ae.ffn_repairs(reset=True)
            out_d = torch.full((m, 384), float("nan"), dtype=torch.float32, device="cuda")
            up.ffn(down, m, a_d.data_ptr(), sa_d.data_ptr(), res_d.data_ptr(), out_d.data_ptr())
            torch.cuda.synchronize()
            outs.append(out_d.cpu().numpy())
            tiles, rows = ae.ffn_repairs()
            print("exact" if exact else "fast", "repairs: tiles", tiles, "16-row groups", rows, flush=True)
            if exact:
                assert tiles == 0 and rows == 0
            else:
                assert tiles >= len(cols) * ((m + 15) // 16) and rows >= (m + 15) // 16, (tiles, rows)
    finally:
        ae.set_ffn_exact_gelu(False)
    for o in outs:
        assert np.array_equal(bits(o), bits(ref))


def test_ffn_fast_and_exact_gelu_kernels_agree(torch_gpu):
    """The fast-GELU and exact-GELU fused FFN kernels give the same bits on a large random batch (by
    the launch's plan 16,384 rows in 64-row workgroups, the rest in a second launch of 16-row ones),
    and equal the oracle at the first rows, across that line and at the last, partial workgroup; the
    fast kernel's repair count is reported."""
    torch = torch_gpu
    w1, ws1, b1, s1 = linear_inputs(1536, 384, 41)
    w2, ws2, b2, s2 = linear_inputs(384, 1536, 42)
    m = 19999
    rng = np.random.default_rng(43)
    a = rng.integers(-127, 128, (m, 384), dtype=np.int8)
    sa = rng.uniform(0.01, 0.1, m).astype(f32)
    res = rng.normal(0, 1, (m, 384)).astype(f32)
    up, down = ae.Linear(w1, ws1, b1, s1), ae.Linear(w2, ws2, b2, s2)
    a_d, sa_d, res_d = dev(torch, a), dev(torch, sa), dev(torch, res)
    outs = []
    try:
        for exact in (False, True):
            ae.set_ffn_exact_gelu(exact)
            ae.ffn_repairs(reset=True)
            out_d = torch.full((m, 384), float("nan"), dtype=torch.float32, device="cuda")
            up.ffn(down, m, a_d.data_ptr(), sa_d.data_ptr(), res_d.data_ptr(), out_d.data_ptr())
            torch.cuda.synchronize()
            outs.append(out_d.cpu().numpy())
            print("exact" if exact else "fast", "repairs (tiles, 16-row groups):", ae.ffn_repairs(), flush=True)
    finally:
        ae.set_ffn_exact_gelu(False)
    assert np.array_equal(bits(outs[0]), bits(outs[1]))
    for r in (slice(0, 300), slice(16384 - 80, 16384 + 80), slice(m - 72, m)):
        ref = _ffn_ref(a[r], sa[r], w1, ws1, b1, w2, ws2, b2, s2, res[r])
        assert np.array_equal(bits(outs[0][r]), bits(ref)), r


@pytest.mark.parametrize("m", [1, 15, 16, 17, 47, 1025, 4096, 4097, 8193])
def test_ffn_fused_by_the_batch_bit_exact(torch_gpu, m):
    """The fused FFN with the workgroup height that the launch picks: 16 rows up to 4,096 of them
    (partial last tiles included), 32 from there on."""
    torch = torch_gpu
    w1, ws1, b1, s1 = linear_inputs(1536, 384, 51)
    w2, ws2, b2, s2 = linear_inputs(384, 1536, 52)
    rng = np.random.default_rng(m)
    a = rng.integers(-127, 128, (m, 384), dtype=np.int8)
    sa = rng.uniform(0.001, 0.1, m).astype(f32)
    res = rng.normal(0, 1, (m, 384)).astype(f32)
    up, down = ae.Linear(w1, ws1, b1, s1), ae.Linear(w2, ws2, b2, s2)
    a_d, sa_d, res_d = dev(torch, a), dev(torch, sa), dev(torch, res)
    out_d = torch.full((m, 384), float("nan"), dtype=torch.float32, device="cuda")
    up.ffn(down, m, a_d.data_ptr(), sa_d.data_ptr(), res_d.data_ptr(), out_d.data_ptr())
    torch.cuda.synchronize()
    ref = _ffn_ref(a, sa, w1, ws1, b1, w2, ws2, b2, s2, res)
    assert np.array_equal(bits(out_d.cpu().numpy()), bits(ref))


@pytest.mark.parametrize("m", [5, 70])
def test_ffn_row_maximum_candidates(torch_gpu, ffn_rows, m):
    """Row maxima that the fused FFN's first candidate scan cannot settle: rows whose largest
    pre-activation is small (GELU far below its bound, a large inv_smooth on a negative column, every
    column alike so that the candidates overflow a wave's list) and infinite or NaN row scales."""
    torch = torch_gpu
    w1, ws1, b1, s1 = linear_inputs(1536, 384, 61)
    w2, ws2, b2, s2 = linear_inputs(384, 1536, 62)
    rng = np.random.default_rng(63)
    a = rng.integers(-127, 128, (m, 384), dtype=np.int8)
    sa = rng.uniform(1e-5, 1e-3, m).astype(f32)  # |v| up to about 0.3
    res = rng.normal(0, 1, (m, 384)).astype(f32)
    sa[0] = 0.0                       # v = b1 alone
    sa[1], sa[2] = np.inf, np.nan
    s2[7] = 40.0                      # a negative GELU may be the row maximum
    w1[7], b1[7] = 0, -0.75
    outs = []
    for flat in (False, True):
        if flat:  # every column the same value: all of them candidates
            w1, b1, s2 = np.zeros_like(w1), np.full_like(b1, 0.3), np.ones_like(s2)
        up, down = ae.Linear(w1, ws1, b1, s1), ae.Linear(w2, ws2, b2, s2)
        a_d, sa_d, res_d = dev(torch, a), dev(torch, sa), dev(torch, res)
        out_d = torch.full((m, 384), float("nan"), dtype=torch.float32, device="cuda")
        up.ffn(down, m, a_d.data_ptr(), sa_d.data_ptr(), res_d.data_ptr(), out_d.data_ptr())
        torch.cuda.synchronize()
        outs.append((out_d.cpu().numpy(), _ffn_ref(a, sa, w1, ws1, b1, w2, ws2, b2, s2, res)))
    for got, ref in outs:
        nan = np.isnan(ref)
        assert np.array_equal(nan, np.isnan(got))
        assert np.array_equal(bits(got)[~nan], bits(ref)[~nan])


@pytest.mark.parametrize("exact", [False, True], ids=["fast", "exact"])
def test_ffn_with_layernorm_special_rows(torch_gpu, exact):
    """The FFN kernel with LN2 in its epilogue on rows that its repairs and its in-order sums decide:
    tied row maxima and values on a half-integer in every row, zero, infinite and NaN row scales, a
    residual row whose mean and variance depend on the order of summation (+-1e8 against small
    values) and a constant one in the last, partial workgroup; in place of the inputs as in a pass.
    f32 rows, LN rows, int8 rows and scales bit for bit (NaN for NaN) against the oracle's steps."""
    torch = torch_gpu
    w1, ws1, b1, s1 = linear_inputs(1536, 384, 71)
    w2, ws2, b2, s2 = linear_inputs(384, 1536, 72)
    m = 75
    for c in (0, 16):  # the row maximum 127, twice
        w1[c], b1[c], s2[c] = 0, 63.5, 2.0
    for c, t in ((37, 10.5), (200, 20.5), (399, np.nextafter(f32(6.5), f32(0))), (1535, 100.5)):
        w1[c], b1[c], s2[c] = 0, t, 1.0
    rng = np.random.default_rng(73)
    a = rng.integers(-127, 128, (m, 384), dtype=np.int8)
    sa = rng.uniform(0.001, 0.02, m).astype(f32)
    sa[1], sa[2], sa[33] = np.inf, np.nan, 0.0
    res = rng.normal(0, 1, (m, 384)).astype(f32)
    res[5, :] = rng.normal(0, 1e-3, 384).astype(f32)
    res[5, 0], res[5, 1] = f32(1e8), f32(-1e8)
    res[m - 1], a[m - 1] = f32(2.5), 0
    gamma, beta = (1 + rng.normal(0, 0.05, 384)).astype(f32), rng.normal(0, 0.02, 384).astype(f32)
    ln_s = (rng.uniform(0.5, 2.0, 384) ** -1).astype(f32)
    up, down = ae.Linear(w1, ws1, b1, s1), ae.Linear(w2, ws2, b2, s2)
    a_d, sa_d, res_d = dev(torch, a), dev(torch, sa), dev(torch, res)
    g_d, b_d, ls_d = dev(torch, gamma), dev(torch, beta), dev(torch, ln_s)
    out_d = torch.zeros((m, 384), dtype=torch.float32, device="cuda")
    ae.set_ffn_exact_gelu(exact)
    try:
        up.ffn_ln(down, m, a_d.data_ptr(), sa_d.data_ptr(), res_d.data_ptr(), out_d.data_ptr(), g_d.data_ptr(),
                  b_d.data_ptr(), ls_d.data_ptr(), res_d.data_ptr(), a_d.data_ptr(), sa_d.data_ptr())
        torch.cuda.synchronize()
    finally:
        ae.set_ffn_exact_gelu(False)
    ref = _ffn_ref(a, sa, w1, ws1, b1, w2, ws2, b2, s2, res)
    ry, rq, rsc = orc.ln_quant_rows(ref, gamma, beta, ln_s)
    for got, want in ((out_d, ref), (res_d, ry), (sa_d, rsc)):
        got = got.cpu().numpy()
        nan = np.isnan(want)
        assert np.array_equal(nan, np.isnan(got))
        assert np.array_equal(bits(got)[~nan], bits(want)[~nan])
    assert np.array_equal(a_d.cpu().numpy(), rq)


@pytest.mark.parametrize("m", [1, 31, 33, 100])
def test_layernorm_quant_bit_exact(torch_gpu, m):
    torch = torch_gpu
    rng = np.random.default_rng(m)
    x = rng.normal(0.2, 3.0, (m, 384)).astype(f32)
    if m > 2:
        x[1] = 0.0
        x[2, 0], x[2, -1] = 1e8, -1e8  # order-sensitive row
    g = (1 + 0.05 * rng.normal(size=384)).astype(f32)
    b = (0.02 * rng.normal(size=384)).astype(f32)
    s = (rng.uniform(0.5, 2, 384) ** -1).astype(f32)
    x_d, g_d, b_d, s_d = dev(torch, x), dev(torch, g), dev(torch, b), dev(torch, s)
    q_d = torch.zeros((m, 384), dtype=torch.int8, device="cuda")
    sc_d = torch.zeros(m, dtype=torch.float32, device="cuda")
    ae.layernorm_smooth_quantize(m, x_d.data_ptr(), g_d.data_ptr(), b_d.data_ptr(), s_d.data_ptr(), q_d.data_ptr(),
                                 sc_d.data_ptr())
    torch.cuda.synchronize()
    y, q, sc = orc.ln_quant_rows(x, g, b, s)
    assert np.array_equal(bits(x_d.cpu().numpy()), bits(y))
    assert np.array_equal(q_d.cpu().numpy(), q)
    assert np.array_equal(bits(sc_d.cpu().numpy()), bits(sc))


@pytest.mark.parametrize("gelu", [False, True])
@pytest.mark.parametrize("n", [384, 1536])
def test_row_quantizers_bit_exact(torch_gpu, gelu, n):
    torch = torch_gpu
    m = 9
    rng = np.random.default_rng(n + gelu)
    x = rng.normal(0, 2.5, (m, n)).astype(f32)
    x[0] = 0.0
    x[1, :4] = [np.inf, -np.inf, np.nan, 1.0]
    s = (rng.uniform(0.5, 2, n) ** -1).astype(f32)
    x_d, s_d = dev(torch, x), dev(torch, s)
    q_d = torch.zeros((m, n), dtype=torch.int8, device="cuda")
    sc_d = torch.zeros(m, dtype=torch.float32, device="cuda")
    fn = ae.gelu_smooth_quantize if gelu else ae.smooth_quantize
    fn(m, n, x_d.data_ptr(), s_d.data_ptr(), q_d.data_ptr(), sc_d.data_ptr())
    torch.cuda.synchronize()
    if gelu:
        gx, q, sc = orc.gelu_quant_rows(x, s)
        assert np.array_equal(bits(x_d.cpu().numpy()), bits(gx))
    else:
        q, sc = orc.smooth_quant_rows(x, s)
    assert np.array_equal(q_d.cpu().numpy(), q)
    assert np.array_equal(bits(sc_d.cpu().numpy()), bits(sc))


def test_gelu_bit_exact_over_float_sample(torch_gpu):
    """GPU GELU (exact glibc-expf restatement) vs the oracle on every 61st f32 bit pattern."""
    torch = torch_gpu
    pat = np.arange(0, 2 ** 32, 61, dtype=np.uint64).astype(np.uint32)
    x = pat.view(f32)
    x_d = dev(torch, x)
    y_d = torch.empty_like(x_d)
    ae.gelu_map(x_d.data_ptr(), y_d.data_ptr(), x.size)
    torch.cuda.synchronize()
    y = y_d.cpu().numpy()
    ref = orc.gelu(x)
    nan = np.isnan(ref)
    assert np.array_equal(np.isnan(y), nan)
    assert np.array_equal(bits(y)[~nan], bits(ref)[~nan])


# exact attention has five code paths: register-resident rows (longest <= 32, <= 64),
# the latency form for small batches and mixed ones (LATENCY_LENS below), else the tiled
# kernel with the wide (mean > 48) or the narrow operand layout, which runs the rows
# of more than 400 keys in a launch of their own when the batch's mean length is at
# most 448 ("tiled_long": both sides of 400, with short rows; "tiled_long_mean410"), else
# every row in one launch ("tiled_long32").  test_attention_latency_form_choices takes
# the "tiled" sets, which are small, through the tiled kernel
ATTN_LENS = {"tiled_wide": [1, 2, 17, 31, 32, 33, 64, 65, 130, 512, 3],
             "tiled_long": [384, 385, 17, 400, 401, 408, 409, 431, 1, 449, 480, 500, 511, 512, 24, 25, 200],
             "tiled_long_mean410": [512, 500, 450, 400, 385, 512, 480, 449, 33, 384],
             "tiled_long32": [512, 500, 480, 512, 449, 512, 470, 300, 505, 512, 490, 401],
             "tiled_narrow": [1, 2, 17, 31, 32, 33, 3, 9, 16, 15, 40, 8, 100],
             "rows64": [1, 2, 17, 31, 32, 33, 3, 9, 16, 15, 40, 8, 64],
             "rows32": [1, 2, 17, 31, 32, 3, 9, 16, 15, 8],
             "rows64_every_length": list(range(64, 0, -1)),
             "rows32_every_length": list(range(1, 33)),
             "latency_128": [128],
             "latency_ragged": [5, 97, 33],
             "latency_512": [512]}


@pytest.fixture(params=[0, 2], ids=["by_shape", "latency_form"])
def attention_form(request, torch_gpu):
    """Every exact-attention test runs with the kernel the batch's shape selects, and
    again with the latency form forced onto the same batch."""
    ae.set_attention_form(request.param)
    yield request.param
    ae.set_attention_form(0)


@pytest.mark.parametrize("lens", list(ATTN_LENS.values()), ids=list(ATTN_LENS))
def test_attention_bit_exact(torch_gpu, attention_form, lens):
    """Segment-bounded attention in the reference's scalar order: bit-exact."""
    torch = torch_gpu
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    T = int(cu[-1])
    rng = np.random.default_rng(21)
    qkv = rng.normal(0, 1.0, (T, 1152)).astype(f32)
    qkv_d, cu_d = dev(torch, qkv), dev(torch, cu)
    ctx_d = torch.zeros((T, 384), dtype=torch.float32, device="cuda")
    print("attention form", attention_form, "lens", lens, flush=True)
    ae.attention_varlen(qkv_d.data_ptr(), cu_d.data_ptr(), len(lens), T, ctx_d.data_ptr())
    torch.cuda.synchronize()
    ref = orc.attention(qkv, cu)
    assert np.array_equal(bits(ctx_d.cpu().numpy()), bits(ref))


# the latency form's choices: up to 16 segments its workgroups find their items (up to
# 42 tiles of 16 queries with eight waves, up to 80 all resident at once, else longest
# first), from 17 on the plan's; one row of up to 168 tokens, or a few short ones of
# about as many in all, have a kernel of their own (up to 128 and up to 256 keys); by the
# batch up to 1,024 tokens, or, where the longest row is over 1.5 times the mean, up to
# 9,000 with 16 segments or with a row over 400 (2,500 where the longest row is not known
# and the rows are not mostly short).  Each set takes the latency form and the 32-query tiles.
LATENCY_LENS = {"one_65": [65], "one_128": [128], "one_129": [129], "one_161": [161], "one_168": [168],
                "one_169": [169], "one_497": [497], "few_66_66": [66, 66], "few_140_16": [140, 16],
                "few_80_20_20_20": [80, 20, 20, 20], "few_129_1_30": [129, 1, 30], "few_88_90": [88, 90],
                "two": [81, 17], "tiles_42": [336, 335], "tiles_44": [337, 340],
                "resident_80_tiles": [256, 241, 255, 250, 242],
                "longest_first": [16, 257, 1, 512, 512, 15, 31, 33, 48, 512, 49, 500, 2, 64, 65],
                "segments_16": [96, 95, 97] + [15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64, 65, 1],
                "segments_17": [96, 95, 97] + [15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64, 65, 1, 2],
                "even_1024": [128] * 8, "even_1025": [128] * 7 + [129],
                "bound_2500": [130] * 18 + [160], "bound_2501": [130] * 18 + [161],
                "short_4000": [100] + [20] * 195, "short_4001": [100] + [20] * 194 + [21],
                "mixed_9000": [512] * 4 + [200] * 34 + [152], "mixed_9001": [512] * 4 + [200] * 34 + [153],
                **{k: v for k, v in ATTN_LENS.items() if k.startswith("tiled")}}


@pytest.mark.parametrize("form", [0, 1, 2], ids=["by_shape", "tiles32", "latency_form"])
@pytest.mark.parametrize("lens", list(LATENCY_LENS.values()), ids=list(LATENCY_LENS))
def test_attention_latency_form_choices(torch_gpu, form, lens):
    """Bit-exact on both sides of each of the latency form's limits, through the operator that
    finds the longest row itself and through the one that is given a bound (512 here)."""
    torch = torch_gpu
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    T = int(cu[-1])
    rng = np.random.default_rng(len(lens) + T)
    qkv = rng.normal(0, 1.0, (T, 1152)).astype(f32)
    qkv_d, cu_d = dev(torch, qkv), dev(torch, cu)
    ctx_d = torch.full((2, T, 384), float("nan"), dtype=torch.float32, device="cuda")
    print("attention form", form, "segments", len(lens), "tokens", T, flush=True)
    ae.set_attention_form(form)
    try:
        ae.attention_varlen(qkv_d.data_ptr(), cu_d.data_ptr(), len(lens), T, ctx_d[0].data_ptr())
        ae.attention_varlen_noalloc(qkv_d.data_ptr(), cu_d.data_ptr(), len(lens), T, 512, ctx_d[1].data_ptr())
        torch.cuda.synchronize()
    finally:
        ae.set_attention_form(0)
    ref = bits(orc.attention(qkv, cu))
    assert np.array_equal(bits(ctx_d[0].cpu().numpy()), ref) and np.array_equal(bits(ctx_d[1].cpu().numpy()), ref)


@pytest.mark.parametrize("lens", [[1, 2, 7, 8, 9, 15, 16, 17, 31, 32, 33], [5, 40, 97, 300, 1, 512, 63],
                                  [100] * 3, [21, 3, 500], list(range(1, 70)),
                                  [505, 506, 507, 511, 512, 497, 480, 481, 449]],
                         ids=["edges", "ragged", "uniform", "long", "every_length_to_69", "long_tails"])
def test_attention_quantized_bit_exact(torch_gpu, lens):
    """The reference's quantized (ArmSme) attention over a packed batch: int8 Q, K, V,
    exact-range int16 P (the cubic on each row's 8-aligned part, exp2f on the rest):
    bit-exact with the oracle."""
    torch = torch_gpu
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    T = int(cu[-1])
    rng = np.random.default_rng(23)
    qkv = rng.normal(0, 1.0, (T, 1152)).astype(f32)
    qkv[:, 768:] *= rng.uniform(0.1, 3.0, 384).astype(f32)  # per-column V ranges
    qkv_d, cu_d = dev(torch, qkv), dev(torch, cu)
    ctx_d = torch.zeros((T, 384), dtype=torch.float32, device="cuda")
    print("quantized attention lens", lens, flush=True)
    ae.attention_varlen_quantized(qkv_d.data_ptr(), cu_d.data_ptr(), len(lens), T, ctx_d.data_ptr())
    torch.cuda.synchronize()
    ref = orc.attention_sme(qkv, cu)
    got = ctx_d.cpu().numpy()
    assert np.array_equal(bits(got), bits(ref)), np.abs(got - ref).max()


def test_mfma_products_equal_rounded_products(torch_gpu):
    """The attention kernels take every product from v_mfma_f32_16x16x1_4b_f32 with a zero
    accumulator: each result must be the correctly rounded f32 product (numpy's), including
    denormal results, infinities and NaN; only the sign of an exact zero may differ."""
    torch = torch_gpu
    rng = np.random.default_rng(17)
    n_sets = 2048
    a = np.ldexp(rng.uniform(-1, 1, (n_sets, 64)), rng.integers(-80, 66, (n_sets, 64))).astype(f32)
    b = np.ldexp(rng.uniform(-1, 1, (n_sets, 64)), rng.integers(-80, 66, (n_sets, 64))).astype(f32)
    a[:64] = np.ldexp(rng.uniform(-1, 1, (64, 64)), -70).astype(f32)  # denormal products
    b[:64] = np.ldexp(rng.uniform(-1, 1, (64, 64)), -75).astype(f32)
    special = np.array([0.0, -0.0, np.inf, -np.inf, np.nan, 1e-45, -1e-45, 3.4e38], f32)
    a[64] = np.tile(special, 8)
    b[64] = np.repeat(special, 8)
    a_d, b_d = dev(torch, a), dev(torch, b)
    out_d = torch.empty((n_sets, 64, 16), dtype=torch.float32, device="cuda")
    ae.mfma_products(a_d.data_ptr(), b_d.data_ptr(), out_d.data_ptr(), n_sets)
    torch.cuda.synchronize()
    got = out_d.cpu().numpy()
    lane = np.arange(64)[:, None]
    r = np.arange(16)[None, :]
    blk, m, n = r // 4, 4 * (lane // 16) + r % 4, lane % 16
    with np.errstate(all="ignore"):
        ref = a[:, blk * 16 + m] * b[:, blk * 16 + n]
    nan = np.isnan(ref)
    assert np.array_equal(np.isnan(got), nan)
    same = (bits(got) == bits(ref)) | ((got == 0) & (ref == 0))
    assert same[~nan].all()
    assert np.count_nonzero((ref != 0) & (np.abs(ref) < np.finfo(f32).tiny)) > 1000  # denormals were covered


@pytest.mark.parametrize("lens", [[5, 40, 97, 300], [5, 40, 19, 33, 1, 90], [5, 40, 19, 33, 1], [5, 31, 19, 27, 1],
                                  [97, 5, 33]],
                         ids=["tiled_wide", "tiled_narrow", "rows64", "rows32", "latency"])
def test_attention_bit_exact_extreme_magnitudes(torch_gpu, attention_form, lens):
    """Scores and PV terms with denormal products, exact zeros and huge dynamic range."""
    torch = torch_gpu
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    T = int(cu[-1])
    rng = np.random.default_rng(23)
    qkv = np.ldexp(rng.uniform(-1, 1, (T, 1152)), rng.integers(-70, 4, (T, 1152))).astype(f32)
    qkv[::7, :] = 0.0
    qkv[3::11, 384:768] *= -0.0
    qkv_d, cu_d = dev(torch, qkv), dev(torch, cu)
    ctx_d = torch.zeros((T, 384), dtype=torch.float32, device="cuda")
    ae.attention_varlen(qkv_d.data_ptr(), cu_d.data_ptr(), len(lens), T, ctx_d.data_ptr())
    torch.cuda.synchronize()
    ref = orc.attention(qkv, cu)
    assert np.array_equal(bits(ctx_d.cpu().numpy()), bits(ref))


def test_workspace_attention_operators(torch_gpu, model_dir):
    """The workspace-scratch attention operators (asynchronous, no allocation or host copy per
    call) give the bits of the synchronous operators; the quantized operator refuses batches whose
    V scales would include rows outside the segments (a segment over 512 tokens, or cu_seqlens not
    ending at total_tokens) instead of cutting them."""
    torch = torch_gpu
    engine = ae.Engine.from_dir(str(model_dir))
    w = engine.workspace(4096, 16)
    lens = [1, 16, 33, 130, 512, 7, 64]
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    T = int(cu[-1])
    rng = np.random.default_rng(71)
    qkv = rng.normal(0, 1.0, (T, 1152)).astype(f32)
    qkv_d, cu_d = dev(torch, qkv), dev(torch, cu)
    for quantized in (False, True):
        a = torch.zeros((T, 384), dtype=torch.float32, device="cuda")
        b = torch.zeros((T, 384), dtype=torch.float32, device="cuda")
        (ae.attention_varlen_quantized if quantized else ae.attention_varlen)(
            qkv_d.data_ptr(), cu_d.data_ptr(), len(lens), T, a.data_ptr())
        for _ in range(2):
            w.attention_varlen(qkv_d.data_ptr(), cu_d.data_ptr(), len(lens), T, max(lens), b.data_ptr(),
                               quantized=quantized)
        w.synchronize()
        assert np.array_equal(bits(a.cpu().numpy()), bits(b.cpu().numpy())), quantized
    ctx = torch.zeros((T, 384), dtype=torch.float32, device="cuda")
    for bad in ([0, 600, 700], [0, 16, 40]):  # 600 > 512; cu ends below total_tokens = 48
        c = dev(torch, np.array(bad, np.int32))
        with pytest.raises(ae.AeError) as e:
            ae.attention_varlen_quantized(qkv_d.data_ptr(), c.data_ptr(), 2, bad[-1] if bad[-1] > 48 else 48,
                                          ctx.data_ptr())
        assert e.value.code == ae.AE_ERR_INVALID_ARG
    with pytest.raises(ae.AeError) as e:  # more sequences than the workspace holds
        w.attention_varlen(qkv_d.data_ptr(), cu_d.data_ptr(), 17, T, 512, ctx.data_ptr())
    assert e.value.code == ae.AE_ERR_CAPACITY
    w.close()
    engine.close()
