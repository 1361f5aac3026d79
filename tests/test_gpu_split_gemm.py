"""f32 contraction on the bf16 matrix cores (split_gemm.h): f32 operands in three exact bf16 parts.

The parts reproduce every f32 operand exactly and at most three products of parts (2^-25 of a term
each) are left out, so the outputs keep the f32 accumulation bound the other paths are held to:
2^-22 |y| + 1e-5 * sum_k |term_k| of the f64 value (bf16 outputs: one bf16 ulp, 2^-8 |y|, for the
relative part).  Shapes sit on the edges: rows, columns and k past the last whole tile, K of one
slice and of many, operands at the ends of f32's range."""
import dataclasses

import numpy as np
import pytest

import compute_amd as ca
from oracle import oracle as O
from tests.qd_helpers import QDenseRun

pytestmark = pytest.mark.gpu

F32, BF16 = O.DT_FLOAT32, O.DT_BFLOAT16


def check(p, y):
    truth, scale = O.qdense_f64(p), O.qdense_f64(p, absolute=True)
    got = (O.bf16_to_f32(y) if p.x_dtype == BF16 else y).astype(np.float64)
    rel = 2.0 ** -8 if p.x_dtype == BF16 else 2.0 ** -22
    bad = np.abs(got - truth) > rel * np.abs(truth) + 1e-5 * scale
    assert not bad.any(), f"{bad.sum()} outputs outside the bound; worst at {np.argwhere(bad)[0]}"


def dot_general(backend, x, w, transposed):
    """x [M, K] . w [K, N] through DotGeneral, w passed as it is or transposed."""
    bld = backend.Builder("dot")
    f = bld.Main()
    vals = [x, w.T if transposed else w]
    shapes = [ca.Shape(ca.Float32, *v.shape) for v in vals]
    a, b = (f.Parameter(n, s) for n, s in zip("ab", shapes))
    f.Return([f.DotGeneral(a, [1], [], b, [1 if transposed else 0], [])])
    bufs = [backend.BufferFromFlatData(0, np.ascontiguousarray(v).ravel(), s) for v, s in zip(vals, shapes)]
    return bld.Compile().Execute(bufs)[0].ToFlatData().reshape(x.shape[0], w.shape[1])


def ggml_dense(backend, t, x, w):
    """x [M, K] . GGML rows w, through mx_qdense."""
    (M, K), N = x.shape, w.shape[0]
    up = lambda v, s: backend.BufferFromFlatData(0, np.ascontiguousarray(v).ravel(), s)
    out = up(np.zeros(M * N, np.float32), ca.Shape(ca.Float32, M, N))
    bufs = [up(x, ca.Shape(ca.Float32, M, K)), up(w, ca.Shape(ca.Uint8, *w.shape))]
    a = ca._lib.mx_qdense_args()
    a.x, a.w, a.out = bufs[0].DevicePtr(), bufs[1].DevicePtr(), out.DevicePtr()
    a.M, a.K, a.N, a.x_dtype, a.scheme, a.ggml_type = M, K, N, F32, int(ca.QuantGGML), int(t)
    assert backend.QDensePlan(a) == "ggml_dequant_f32_mfma"
    backend.QDense(a)
    return out.ToFlatData().reshape(M, N)


# (x, axis, B, zero point, NF4): the row form (B a multiple of 128, or one block; no zero points), the
# column form (one scale per column) and the weight form (everything else).
FORMS = [(F32, 1, 128, False, False), (F32, 1, 128, True, False), (BF16, 1, 4096, True, False), (F32, 0, None, False, False),
         (F32, 0, 96, True, False), (BF16, 0, 96, False, False), (F32, 1, 4, True, False), (BF16, 1, 7, True, False),
         (F32, 1, 7, False, False), (F32, 1, 128, False, True)]


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("w_dtype", [O.DT_INT8, O.DT_UINT4])
@pytest.mark.parametrize("M,K,N", [(131, 1048, 144), (257, 2088, 400)])
def test_forms_at_ragged_edges(backend, form, w_dtype, M, K, N):
    x_dtype, axis, B, zp, nf4 = form
    p = O.make_problem(M, K, N, w_dtype=w_dtype, x_dtype=x_dtype, scale_dtype=x_dtype, block_axis=axis,
                       block_size=K if B is None else B, zp=zp, scheme=O.QUANT_NF4 if nf4 else O.QUANT_LINEAR, bias=True,
                       seed=M + K + w_dtype)
    r = QDenseRun(backend, p)
    assert r.plan() == "qdense_refgemm_f32_mfma"
    y = r.run()
    check(p, y)
    assert np.array_equal(y, r.run()), "not deterministic"


@pytest.mark.parametrize("form", [FORMS[0], FORMS[6]])
@pytest.mark.parametrize("M,K,N", [(65, 16388, 16), (129, 8196, 1040), (640, 1028, 2064)])
def test_k_slices_with_and_without_allocation(backend, form, M, K, N):
    """One tile in many K slices, tiles in a few, and (85 tiles) none; the allocation-free entry
    point takes the same slices, so its result is the same bits."""
    x_dtype, axis, B, zp, _ = form
    p = O.make_problem(M, K, N, w_dtype=O.DT_INT4, x_dtype=x_dtype, scale_dtype=F32, block_axis=axis, block_size=B, zp=zp,
                       bias=False, seed=K)
    r = QDenseRun(backend, p)
    assert r.plan() == "qdense_refgemm_f32_mfma"
    y = r.run()
    check(p, y)
    out = backend.BufferFromFlatData(0, np.zeros(M * N, np.float32), ca.Shape(ca.Float32, M, N))
    backend.QDenseNoAlloc(r.args(out))
    assert np.array_equal(out.ToFlatData().reshape(M, N).view(np.uint32), y.view(np.uint32))


# A product's error without its smallest parts is up to 2^-17 of it; with them it is a few roundings,
# 2^-24 each: of x * s or w * s, of each of up to four sums, and the three products left out.
ONE_PRODUCT = 2.0 ** -21


def one_term_rows(M, K, magnitude, rng):
    """x with one value of 24 significant bits in each row, at k from 0 to K - 1."""
    x = np.zeros((M, K), np.float32)
    k = np.linspace(0, K - 1, M).round().astype(int)
    x[np.arange(M), k] = rng.uniform(0.5, 2.0, M).astype(np.float32) * np.float32(magnitude)
    return x


@pytest.mark.parametrize("axis,B,zp,nf4", [(1, 128, False, False), (1, 272, False, False), (0, None, False, False), (1, 64, False, False),
                                           (1, 7, True, False), (0, 96, True, False), (1, 128, True, False), (1, 128, False, True)])
@pytest.mark.parametrize("magnitude,s", [(1.0, 0.01), (1e-37, 0.01), (1e-3, 1e-34), (1.0, 1e-37)])
@pytest.mark.parametrize("M,K", [(131, 1048), (70, 8196)])
def test_every_part_of_every_product(backend, axis, B, zp, nf4, magnitude, s, M, K):
    """Outputs of a single product each, over every k (K slices and the last part of a block among
    them), with operands down to the smallest normals: each holds all of its operands' bits.  Against
    the reference's own roundings, so that w * s + zp has no error of its own."""
    N = 272
    p = O.make_problem(M, K, N, w_dtype=O.DT_INT4 if nf4 or B == 64 else O.DT_INT8, x_dtype=F32, scale_dtype=F32, block_axis=axis,
                       block_size=K if B is None else B, zp=zp, scheme=O.QUANT_NF4 if nf4 else O.QUANT_LINEAR, bias=False,
                       scale_range=(0.5 * s, 2 * s), seed=M + K)
    p = dataclasses.replace(p, x=one_term_rows(M, K, magnitude, np.random.default_rng(K)), zp=p.zp * np.float32(20 * s) if zp else None)
    r = QDenseRun(backend, p)
    assert r.plan() == "qdense_refgemm_f32_mfma"
    y, want = r.run().astype(np.float64), O.qdense_f32(p).astype(np.float64)
    # Results below the smallest normal keep its step, and (x*w)*s may pass through that range before.
    assert np.all(np.abs(y - want) <= ONE_PRODUCT * np.abs(want) + 2.0 ** -147)
    assert np.count_nonzero(y) > 0.8 * y.size


@pytest.mark.parametrize("t", [ca.GGMLQ4_0, ca.GGMLQ8_0, ca.GGMLIQ4NL, ca.GGMLQ4_K, ca.GGMLQ6_K])
@pytest.mark.parametrize("magnitude", [1.0, 1e-34])
def test_every_part_of_every_ggml_product(backend, t, magnitude):
    rng = np.random.default_rng(int(t))
    M, K, N = 70, 2048, 260
    w, x = O.ggml_random_rows(int(t), N, K, rng), one_term_rows(M, K, magnitude, rng)
    y, (exact, _) = ggml_dense(backend, t, x, w), O.ggml_dense_f64(x, w, int(t), None)
    assert np.all(np.abs(y.astype(np.float64) - exact) <= ONE_PRODUCT * np.abs(exact) + 2.0 ** -147)


@pytest.mark.parametrize("transposed", [True, False])
@pytest.mark.parametrize("mx,mw", [(1.0, 1.0), (1e-37, 1.0), (1.0, 1e-37)])
def test_every_part_of_every_dot_general_product(backend, transposed, mx, mw):
    M, K, N = 1037, 1028, 1036
    rng = np.random.default_rng(3)
    x, w = one_term_rows(M, K, mx, rng), (rng.standard_normal((K, N)) * mw).astype(np.float32)
    y, want = dot_general(backend, x, w, transposed).astype(np.float64), x.astype(np.float64) @ w.astype(np.float64)
    assert np.all(np.abs(y - want) <= ONE_PRODUCT * np.abs(want) + 2.0 ** -147)


@pytest.mark.parametrize("B", [128, 32])
@pytest.mark.parametrize("magnitude", [1e-36, 1e30])
def test_operands_at_the_ends_of_the_range(backend, B, magnitude):
    """x near f32's smallest normals (its lower parts are subnormal) and large."""
    p = O.make_problem(96, 1024, 256, w_dtype=O.DT_INT4, x_dtype=F32, scale_dtype=F32, block_axis=1, block_size=B, bias=False,
                       scale_range=(0.5, 2.0), seed=3)
    p = dataclasses.replace(p, x=(p.x * np.float32(magnitude)).astype(np.float32))
    check(p, QDenseRun(backend, p).run())


@pytest.mark.parametrize("B,K", [(128, 1024), (32, 1024), (128, 16384)])
def test_infinite_and_nan_operands(backend, B, K):
    """A tile that holds an operand with no split (infinite, or past the largest bf16) is summed by
    f32 FMAs: infinities keep their sign, NaN stays in its row or column, the rest is as close as
    ever.  Codes are positive, so that no infinities of both signs meet."""
    p = O.make_problem(260, K, 256, w_dtype=O.DT_UINT8, x_dtype=F32, scale_dtype=F32, block_axis=1, block_size=B, bias=True,
                       scale_range=(0.001, 0.0039), seed=4)  # codes * scales < 1: no finite x makes an infinite term
    w = np.maximum(p.w, 1)
    x, s = p.x.copy(), p.scale.copy()
    x[3, 17], x[140, 5], x[141, 9] = np.inf, -np.inf, np.nan
    x[200, 1023] = 3.4e38  # rounds past bf16's largest value
    s[33, 0] = np.inf      # the first block's columns, every row
    x[:, 33] = np.abs(x[:, 33]) + 0.5
    p = dataclasses.replace(p, w=w, x=x, scale=s)
    y = QDenseRun(backend, p).run().astype(np.float64)
    with np.errstate(invalid="ignore", over="ignore"):
        truth, scale = O.qdense_f64(p), O.qdense_f64(p, absolute=True)
    assert np.array_equal(np.isnan(y), np.isnan(truth))
    inf = np.isinf(truth)
    assert np.array_equal(y[inf], truth[inf])
    fin = np.isfinite(truth)
    assert fin.any() and inf.any()
    assert np.all(np.abs(y[fin] - truth[fin]) <= 2.0 ** -22 * np.abs(truth[fin]) + 1e-5 * scale[fin])


@pytest.mark.parametrize("K", [1024, 1000])
@pytest.mark.parametrize("axis,B,zp,nf4", [(1, 64, False, False), (1, 128, False, True), (0, 96, True, False), (1, 7, True, False)])
def test_infinite_and_nan_bf16_x(backend, axis, B, zp, nf4, K):
    """bf16 x is one part and meets three parts of each weight factor: an infinity keeps its sign."""
    p = O.make_problem(260, K, 256, w_dtype=O.DT_UINT4, x_dtype=BF16, scale_dtype=BF16, block_axis=axis, block_size=B, zp=zp,
                       scheme=O.QUANT_NF4 if nf4 else O.QUANT_LINEAR, bias=True, seed=K + B)
    x = p.x.copy()
    x[3, 17], x[140, 5], x[141, 9], x[259, K - 1] = 0x7F80, 0xFF80, 0x7FC0, 0x7F80
    p = dataclasses.replace(p, x=x)
    r = QDenseRun(backend, p)
    assert r.plan() == "qdense_refgemm_f32_mfma"
    y = O.bf16_to_f32(r.run()).astype(np.float64)
    with np.errstate(invalid="ignore", over="ignore"):
        truth, scale = O.qdense_f64(p), O.qdense_f64(p, absolute=True)
    assert np.array_equal(np.isnan(y), np.isnan(truth)) and np.isnan(truth[141]).all()
    inf = np.isinf(truth)
    assert inf[3].any() and inf[140].any() and inf[259].any() and np.array_equal(y[inf], truth[inf])
    fin = np.isfinite(truth)
    assert np.all(np.abs(y[fin] - truth[fin]) <= 2.0 ** -8 * np.abs(truth[fin]) + 1e-5 * scale[fin])


@pytest.mark.parametrize("axis,B,K,s", [(1, 64, 1024, 1e14), (1, 64, 16388, 1e14), (0, 96, 1024, 1e14), (0, None, 1024, 1e14), (1, 128, 1024, 1e14)])
def test_finite_operands_that_overflow(backend, axis, B, K, s):
    """Products of finite operands past f32's range are infinities, not NaN; rows beside them are as
    close as ever.  (The sums of one row have one sign, so that no infinities cancel.)"""
    p = O.make_problem(130, K, 144, w_dtype=O.DT_UINT8, x_dtype=F32, scale_dtype=F32, block_axis=axis, block_size=K if B is None else B,
                       bias=True, scale_range=(0.5 * s, s), seed=K)
    x = np.abs(p.x) + np.float32(0.1)
    x[1] *= np.float32(1e25)
    x[2] *= np.float32(-1e25)
    p = dataclasses.replace(p, x=x, w=np.maximum(p.w, 1))
    y = QDenseRun(backend, p).run()
    assert np.all(np.isposinf(y[1])) and np.all(np.isneginf(y[2]))
    rest = np.r_[0, 3:130]
    truth, scale = O.qdense_f64(p, rest), O.qdense_f64(p, rest, absolute=True)
    assert np.all(np.abs(y[rest].astype(np.float64) - truth) <= 2.0 ** -22 * np.abs(truth) + 1e-5 * scale)


def test_column_sums_past_the_range_before_their_scale(backend):
    """One scale per column, applied to the sums: sums of x * w past f32's range whose scaled terms and
    result are in range."""
    p = O.make_problem(130, 1024, 144, w_dtype=O.DT_UINT8, x_dtype=F32, scale_dtype=F32, block_axis=0, block_size=1024, bias=True,
                       scale_range=(1e-6, 1e-5), seed=8)
    x = np.abs(p.x)
    x[5] = np.float32(1.2e36)
    p = dataclasses.replace(p, x=x)
    r = QDenseRun(backend, p)
    assert r.plan() == "qdense_refgemm_f32_mfma"
    check(p, r.run())


@pytest.mark.parametrize("M,K,N,B", [(130, 1024, 272, 128), (130, 1028, 272, 272), (24, 4096, 256, 128)])
def test_zero_points_that_cancel_the_codes(backend, M, K, N, B):
    """Asymmetric weights, zp = -z * s with codes at and next to z: the terms are x * ((w - z) * s), and
    the bound is of these, not of x * w * s and x * zp.  (64 bits: z = 8, so that z * s is exact; the
    sums' chains are at most 8 + K / 256 + 2 additions, each 2^-24 of the terms' sum.)  A column whose
    codes are all z is the bias, to the bit."""
    for z in (8, 7):
        p = O.make_problem(M, K, N, w_dtype=O.DT_UINT4, x_dtype=F32, scale_dtype=F32, block_axis=1, block_size=B, zp=True, bias=True, seed=K)
        codes = np.random.default_rng(K).integers(z - 1, z + 2, (K, N))
        codes[:, ::5] = z
        p = dataclasses.replace(p, w=O.pack_int4(codes.ravel()), zp=(-np.float32(z) * p.scale).astype(np.float32))
        r = QDenseRun(backend, p)
        assert r.plan() == "qdense_refgemm_f32_mfma"
        y = r.run()
        assert np.array_equal(y[:, ::5], np.broadcast_to(p.bias[::5], (M, len(range(0, N, 5)))))
        if z == 8:
            truth, scale = O.qdense_f64(p), O.qdense_f64(p, absolute=True)
            assert np.all(np.abs(y - truth) <= 2.0 ** -22 * np.abs(truth) + (10 + K / 256) * 2.0 ** -24 * scale)


@pytest.mark.parametrize("x_dtype,act", [(F32, O.ACT_NONE), (BF16, O.ACT_RELU)])
def test_output_aligned_to_its_elements_only(backend, x_dtype, act):
    """An output array that starts one element past a 16-byte boundary."""
    p = O.make_problem(70, 1024, 272, w_dtype=O.DT_INT8, x_dtype=x_dtype, scale_dtype=F32, block_axis=1, block_size=64, bias=True,
                       act=act, seed=9)
    r = QDenseRun(backend, p)
    want = r.run()
    dt, st = (ca.Float32, np.float32) if x_dtype == F32 else (ca.BFloat16, np.uint16)
    out = backend.BufferFromFlatData(0, np.zeros(p.M * p.N + 1, st), ca.Shape(dt, p.M * p.N + 1))
    a = r.args(out)
    a.out = out.DevicePtr() + np.dtype(st).itemsize
    backend.QDense(a)
    got = out.ToFlatData()
    assert got[0] == 0 and np.array_equal(got[1:].reshape(p.M, p.N), want)


@pytest.mark.parametrize("M,N", [(300, 11008), (1100, 7296)])
def test_tail_tiles_in_slices(backend, M, N):
    """Tiles past whole rounds of resident workgroups: 258 tiles of the weight form (256 + 2), 513 of
    the row form (512 + 1), the last ones in K slices; rows of the first and of the last tiles."""
    p = O.make_problem(M, 512, N, w_dtype=O.DT_INT8, x_dtype=F32, scale_dtype=F32, block_axis=1, block_size=64 if M == 300 else 128,
                       bias=True, seed=M)
    r = QDenseRun(backend, p)
    y = r.run()
    rows = np.r_[0:4, M - 44:M]
    truth, scale = O.qdense_f64(p, rows), O.qdense_f64(p, rows, absolute=True)
    assert np.all(np.abs(y[rows].astype(np.float64) - truth) <= 2.0 ** -22 * np.abs(truth) + 1e-5 * scale)
    assert np.array_equal(y, r.run())


@pytest.mark.parametrize("t", [ca.GGMLQ4_0, ca.GGMLQ8_0, ca.GGMLIQ4NL, ca.GGMLQ4_K, ca.GGMLQ6_K])
@pytest.mark.parametrize("M,K,N", [(17, 1024, 1031), (129, 2048, 130)])
def test_ggml_rows_at_ragged_edges(backend, t, M, K, N):
    """GGML rows past 16 rows: odd output widths (scalar stores) and one row past a tile."""
    rng = np.random.default_rng(M + int(t))
    w = O.ggml_random_rows(int(t), N, K, rng)
    x = rng.standard_normal((M, K)).astype(np.float32)
    up = lambda v, s: backend.BufferFromFlatData(0, np.ascontiguousarray(v).ravel(), s)
    out = up(np.zeros(M * N, np.float32), ca.Shape(ca.Float32, M, N))
    bufs = [up(x, ca.Shape(ca.Float32, M, K)), up(w, ca.Shape(ca.Uint8, *w.shape))]
    a = ca._lib.mx_qdense_args()
    a.x, a.w, a.out = bufs[0].DevicePtr(), bufs[1].DevicePtr(), out.DevicePtr()
    a.M, a.K, a.N, a.x_dtype, a.scheme, a.ggml_type = M, K, N, F32, int(ca.QuantGGML), int(t)
    assert backend.QDensePlan(a) == "ggml_dequant_f32_mfma"
    backend.QDense(a)
    exact, ab = O.ggml_dense_f64(x, w, int(t), None)
    assert np.all(np.abs(out.ToFlatData().reshape(M, N).astype(np.float64) - exact) <= 1e-5 * ab + 1e-30)


@pytest.mark.parametrize("M,K,N,axis,B,zp", [(17, 2048, 1040, 1, 128, False), (64, 2048, 528, 1, 32, True), (33, 4128, 272, 0, 96, False)])
def test_few_rows(backend, M, K, N, axis, B, zp):
    """The fewest rows of the reference layout and of scales along K that leave the GEMV: held to a
    third of the bound, which the GEMV's sums kept too."""
    p = O.make_problem(M, K, N, w_dtype=O.DT_INT8, x_dtype=F32, scale_dtype=F32, block_axis=axis, block_size=B, zp=zp, bias=True, seed=M)
    r = QDenseRun(backend, p)
    assert r.plan() == "qdense_refgemm_f32_mfma"
    y = r.run().astype(np.float64)
    truth, scale = O.qdense_f64(p), O.qdense_f64(p, absolute=True)
    assert np.all(np.abs(y - truth) <= 2.0 ** -22 * np.abs(truth) + 3e-6 * scale)


@pytest.mark.parametrize("transposed", [True, False])
@pytest.mark.parametrize("M,K,N", [(96, 115004, 100), (1037, 1028, 1036), (2049, 548, 1000)])
def test_dot_general_f32(backend, transposed, M, K, N):
    """f32 DotGeneral from 2^30 multiply-adds: one tile in many K slices, ragged tiles, K past the last
    block of 32; one infinity, in a row (and so a tile) of its own."""
    assert M * K * N >= 1 << 30
    rng = np.random.default_rng(K)
    x, w = rng.standard_normal((M, K)).astype(np.float32), rng.standard_normal((K, N)).astype(np.float32)
    x[M - 1, K - 1] = np.inf
    w[K - 1] = np.abs(w[K - 1]) + 0.5
    bld = backend.Builder("dot")
    f = bld.Main()
    shapes = [ca.Shape(ca.Float32, M, K), ca.Shape(ca.Float32, *((N, K) if transposed else (K, N)))]
    a, b = (f.Parameter(n, s) for n, s in zip("ab", shapes))
    f.Return([f.DotGeneral(a, [1], [], b, [1 if transposed else 0], [])])
    bufs = [backend.BufferFromFlatData(0, np.ascontiguousarray(v).ravel(), s) for v, s in zip((x, w.T if transposed else w), shapes)]
    exe = bld.Compile()
    y = exe.Execute(bufs)[0].ToFlatData().reshape(M, N)
    assert np.all(np.isposinf(y[M - 1]))
    truth, scale = x[:-1].astype(np.float64) @ w.astype(np.float64), np.abs(x[:-1]).astype(np.float64) @ np.abs(w).astype(np.float64)
    assert np.all(np.abs(y[:-1] - truth) <= 2.0 ** -22 * np.abs(truth) + 3e-6 * scale)


@pytest.mark.parametrize("transposed", [True, False])
def test_dot_general_f32_overflow(backend, transposed):
    """Rows of x whose products with the right-hand side pass f32's range: infinities, not NaN."""
    M, K, N = 1024, 1024, 1024
    rng = np.random.default_rng(7)
    x, w = np.abs(rng.standard_normal((2, M, K)).astype(np.float32)) + np.float32(0.1)
    w *= np.float32(1e25)
    x[1], x[2] = x[1] * np.float32(1e25), x[2] * np.float32(-1e25)
    y = dot_general(backend, x, w, transposed)
    assert np.all(np.isposinf(y[1])) and np.all(np.isneginf(y[2]))
    truth = x.astype(np.float64) @ w.astype(np.float64)
    rest = np.r_[0, 3:M]
    assert np.all(np.abs(y[rest] - truth[rest]) <= (2.0 ** -22 + 3e-6) * truth[rest])


@pytest.mark.parametrize("axis,B", [(1, 128), (0, None)])
def test_few_rows_of_a_wide_head(backend, axis, B):
    """256 tiles of 33 rows (a vocabulary head): as close to 64 bits as the GEMV was (1.4e-7 to 3.2e-7
    of the result's norm), which one chain of sums over K is not."""
    M, K, N = 33, 4096, 32768
    p = O.make_problem(M, K, N, w_dtype=O.DT_INT8, x_dtype=F32, scale_dtype=F32, block_axis=axis, block_size=K if B is None else B,
                       bias=False, seed=1)
    r = QDenseRun(backend, p)
    assert r.plan() == "qdense_refgemm_f32_mfma"
    rows = np.array([0, 32])
    y, truth = r.run()[rows].astype(np.float64), O.qdense_f64(p, rows)
    err = np.linalg.norm(y - truth) / np.linalg.norm(truth)
    assert err <= 1.6e-7, err


@pytest.mark.parametrize("form,K", [(f, K) for f in FORMS for K in (8, 12, 24, 28) if f[0] == F32 or K % 8 == 0])
@pytest.mark.parametrize("w_dtype", [O.DT_INT8, O.DT_UINT4])
def test_fewer_rows_of_weights_than_a_block(backend, form, K, w_dtype):
    """K below one block of 32 (a low-rank factor), with f32 x also where 4 values of a run of 8 remain
    (bf16 rows of K % 8 != 0 take the reference-order kernel)."""
    x_dtype, axis, B, zp, nf4 = form
    M, N = 2061, 1040
    p = O.make_problem(M, K, N, w_dtype=w_dtype, x_dtype=x_dtype, scale_dtype=x_dtype, block_axis=axis,
                       block_size=K if B is None else B, zp=zp, scheme=O.QUANT_NF4 if nf4 else O.QUANT_LINEAR, bias=True, seed=K)
    r = QDenseRun(backend, p)
    assert r.plan() == "qdense_refgemm_f32_mfma"
    y = r.run()
    check(p, y)
    if x_dtype == F32 and not zp:
        truth, scale = O.qdense_f64(p), O.qdense_f64(p, absolute=True)
        assert np.all(np.abs(y - truth) <= 2.0 ** -20 * scale)


@pytest.mark.parametrize("x_dtype,B,zp,nf4", [(F32, 6, True, False), (F32, 7, False, False), (BF16, 1, True, False), (BF16, 37, False, True),
                                              (F32, 1043, True, False), (F32, 4, True, False)])
@pytest.mark.parametrize("scale_dtype", [F32, BF16])
def test_groups_of_any_number_of_rows(backend, x_dtype, B, zp, nf4, scale_dtype):
    """Scales along K in groups that are no multiple of 4 rows (a scale row looked up for each row of
    weights) and the smallest that is (one for every four rows)."""
    p = O.make_problem(300, 1048, 272, w_dtype=O.DT_UINT4 if nf4 else O.DT_INT8, x_dtype=x_dtype, scale_dtype=scale_dtype, block_axis=0,
                       block_size=B, zp=zp, scheme=O.QUANT_NF4 if nf4 else O.QUANT_LINEAR, bias=True, seed=B)
    r = QDenseRun(backend, p)
    assert r.plan() == "qdense_refgemm_f32_mfma"
    y = r.run()
    check(p, y)
    assert np.array_equal(y, r.run())


@pytest.mark.parametrize("M,B,K", [(260, 64, 1024), (97, 128, 4100), (97, 64, 9000)])
def test_nan_and_infinite_scales(backend, M, B, K):
    """Columns with a NaN scale stay NaN and those with an infinite one infinite in every row, beside
    rows of x with an infinity (the last row of x among them) and sums past f32's range."""
    p = O.make_problem(M, K, 272, w_dtype=O.DT_UINT8, x_dtype=F32, scale_dtype=F32, block_axis=1, block_size=B, bias=True,
                       scale_range=(0.001, 0.0039), seed=M + K)
    w, x, s = np.maximum(p.w, 1), np.abs(p.x) + np.float32(0.1), p.scale.copy()
    s[K // 2, 1], s[K - 1, 2] = np.nan, np.inf
    x[M - 1, 5], x[8, K - 1] = np.inf, -np.inf
    x[9, :] = 3e38
    p = dataclasses.replace(p, w=w, x=x, scale=s)
    y = QDenseRun(backend, p).run().astype(np.float64)
    with np.errstate(invalid="ignore", over="ignore"):
        truth, scale = O.qdense_f64(p), O.qdense_f64(p, absolute=True)
        truth = np.where(np.abs(truth) > 3.4028235e38, np.copysign(np.inf, truth), truth)
    assert np.array_equal(np.isnan(y), np.isnan(truth)) and np.isnan(truth[:, B:2 * B]).all()
    inf = np.isinf(truth)
    assert inf[:, 2 * B:].any() and inf[M - 1].any() and inf[8].any() and inf[9].any() and np.array_equal(y[inf], truth[inf])
    fin = np.isfinite(truth)
    assert fin.any() and np.all(np.abs(y[fin] - truth[fin]) <= 2.0 ** -22 * np.abs(truth[fin]) + 1e-5 * scale[fin])

