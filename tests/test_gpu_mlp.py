"""The quantized MLP (workload C5) built through the Builder API and executed on the
GPU, checked op by op against the CPU oracle on the GPU's own intermediate values:
  - h = bf16(RMSNorm(x)) computed in f32: within one bf16 ulp of the oracle's restatement of the
    reference graph (sequential f32 ReduceSum, Rsqrt through f64; oracle.rmsnorm_chain, pinned by
    closed forms in test_oracle).  The GPU adds each row's squares in another order (strided
    partial sums and an LDS tree), so the f32 mean square may differ in its last bits;
  - gate = SiLU(FusedQuantizedDense(h)), up and down = FusedQuantizedDense(...): within
    rel 1e-2 / abs 1e-3 of the reference loop (the oracle) on the same inputs;
  - gate*up and the residual add: bit-exact bf16 products / sums of the GPU's operands.
Checked op by op because the composition rounds to bf16 six times: an intermediate that rounds
to the neighbouring bf16 value (another summation order) carries that ulp on, so an end-to-end
comparison against an independently rounded chain has no fixed relative bound.  The graph the
benchmark runs (one output) must give the same bits as the instrumented one.
"""
import numpy as np
import pytest

from compute_amd import backend as B
from compute_amd import workloads
from compute_amd.dtypes import BFloat16, Float32, Shape
from oracle import oracle as O
from tests.qd_helpers import assert_bf16_close

pytestmark = pytest.mark.gpu


def build_instrumented(backend, wl):
    bld = backend.Builder("mlp_instrumented")
    f = bld.Main()
    names = ["x", "w_gate", "s_gate", "w_up", "s_up", "w_down", "s_down"]
    p = [f.Parameter(n, sh) for n, sh in zip(names, wl.shapes())]
    x = p[0]
    xf = f.ConvertDType(x, Float32)
    ms = f.Mul(f.ReduceSum(f.Mul(xf, xf), 1), f.Constant(np.full(wl.M, 1.0 / wl.D, np.float32)))
    inv = f.Rsqrt(f.Add(ms, f.Constant(np.full(wl.M, wl.eps, np.float32))))
    h = f.ConvertDType(f.Mul(xf, f.BroadcastInDim(inv, Shape(Float32, wl.M, wl.D), [0])), BFloat16)

    def qd(v, w, sc, act):
        return f.FusedQuantizedDense(v, w, None, B.Quantization(B.QuantLinear, sc, None, 0, wl.G), B.ActivationType(act))

    g = qd(h, p[1], p[2], B.ActivationSilu)
    u = qd(h, p[3], p[4], B.ActivationNone)
    gu = f.Mul(g, u)
    d = qd(gu, p[5], p[6], B.ActivationNone)
    f.Return([h, g, u, gu, d, f.Add(d, x)])
    return bld.Compile()


def qd_ref(wl, xbits, w, sc, K, N, act):
    p = O.QDenseProblem(M=xbits.shape[0], K=K, N=N, x=xbits, x_dtype=O.DT_BFLOAT16, w=w, w_dtype=O.DT_INT4, scale=sc,
                        scale_dtype=O.DT_BFLOAT16, scale_shape=sc.shape, block_axis=0, block_size=wl.G, act=act)
    return O.qdense_f32(p, threads=8)


def test_mlp_graph_c5(backend):
    wl = workloads.make("C5")
    bufs = wl.upload(backend)
    H, G, U, GU, D, Y = [o.ToFlatData().reshape(wl.M, -1) for o in build_instrumented(backend, wl).Execute(bufs)]
    x = O.bf16_to_f32(wl.x).astype(np.float32)
    h_ref = O.rmsnorm_chain(wl.x, wl.eps)
    same_sign = (H >> 15) == (h_ref >> 15)
    ulps = np.abs(H.astype(np.int32) - h_ref.astype(np.int32))  # adjacent bf16 values differ by 1
    assert np.all(same_sign & (ulps <= 1)), "RMSNorm beyond one bf16 ulp"
    assert np.mean(ulps == 0) > 0.99, "RMSNorm: more than 1% of elements off by an ulp"
    (wg, sg, K1, N1), (wu, su, _, _), (wd, sd, K3, N3) = wl.weights
    assert_bf16_close(G, qd_ref(wl, H, wg, sg, K1, N1, O.ACT_SILU), what="gate")
    assert_bf16_close(U, qd_ref(wl, H, wu, su, K1, N1, O.ACT_NONE), what="up")
    assert np.array_equal(GU, O.bf16_round(O.bf16_to_f32(G) * O.bf16_to_f32(U))), "gate*up"
    assert_bf16_close(D, qd_ref(wl, GU, wd, sd, K3, N3, O.ACT_NONE), what="down")
    assert np.array_equal(Y, O.bf16_round(O.bf16_to_f32(D) + x)), "residual"
    # The benchmark's graph: same kernels, same bits; resident inputs give the same bits again.
    exe = wl.compile(backend)
    y1 = exe.Execute(bufs)[0].ToFlatData().reshape(wl.M, wl.D)
    y2 = exe.Execute(bufs)[0].ToFlatData().reshape(wl.M, wl.D)
    assert np.array_equal(y1, Y) and np.array_equal(y1, y2)
