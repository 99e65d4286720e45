"""GPU parity of the generic epilogue's runs of 8 columns: rows of an odd number of elements (every second one
misaligned), a bias of another type than the output, C stored beside linearRes, beta, and the element-wise rest of a row,
on each kernel that has the epilogue, against the oracle."""
import numpy as np
import pytest

import kudnn_amd as K
import oracle as O
from support import Case, compare, from_device, zeros_device

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    K.lib()


# kernel: forced configuration, K slices
KERNELS = {"pingpong": ("4", "0"), "slices": ("4", "2"), "four_wave": ("3", None), "f32": ("11", None)}


@pytest.mark.parametrize("kernel", list(KERNELS))
@pytest.mark.parametrize("M,N", [(70, 267), (257, 264), (33, 7), (256, 129)])
@pytest.mark.parametrize("op", ["bias_f32", "beta", "res", "gelu_odd", "mish"])
def test_generic_runs(monkeypatch, kernel, M, N, op):
    cfg, slices = KERNELS[kernel]
    monkeypatch.setenv("KUDNN_HIP_FORCE_CFG", cfg)
    if slices is not None:
        monkeypatch.setenv("KUDNN_HIP_FORCE_KSLICES", slices)
    dt, Kd = (O.F32, 64) if kernel == "f32" else (O.F16 if kernel == "four_wave" else O.BF16, 128)
    x = Case([M, Kd], dt, seed=820, dist="normal", lo=0.0, hi=1.0)
    w = Case([Kd, N], dt, "BA", seed=821, dist="normal", lo=0.0, hi=0.1)
    b = Case([1, N], O.F32 if op == "bias_f32" else dt, seed=822, lo=-0.2, hi=0.2)
    y = Case([M, N], dt, seed=823, lo=-1.0, hi=1.0) if op == "beta" else Case([M, N], dt, zero=True)
    s = Case([M, N], dt, seed=824, lo=-1.0, hi=1.0)
    dy = y.device()
    ref = O.Tensor(y.t.dims, y.t.strides, dt, y.t.buf.copy())
    if op in ("bias_f32", "beta"):
        alpha, beta = (0.5, 0.25) if op == "beta" else (1.0, 0.0)
        plan = K.Gemm(x.desc, w.desc, y.desc, b.desc)
        plan.run(x.device(), w.device(), dy, b.device(), alpha=alpha, beta=beta)
        O.gemm(x.t, w.t, ref, b.t, alpha, beta)
    elif op == "res":
        lr = Case([M, N], dt, zero=True)
        plan = K.LinearRes(x.desc, w.desc, y.desc, b.desc, s.desc, lr.desc, 1.0, 0.0, 0.3, O.RES_EXT)
        dlr, rlr = zeros_device(lr), lr.clone_empty()
        plan.run(x.device(), w.device(), dy, b.device(), s.device(), dlr, 0.3)
        O.linear_res(x.t, w.t, ref, b.t, s.t, rlr, O.RES_EXT, 0.3)
        torch.cuda.synchronize()
        compare(from_device(dlr, dt), rlr.buf, dt, f"linearRes {plan.describe()}")
    else:
        act = K.ACT_MISH if op == "mish" else K.ACT_GELU_TANH
        plan = K.LinearPostOps(x.desc, w.desc, y.desc, b.desc, act=act, binary=K.BIN_MUL, src=s.desc)
        plan.run(x.device(), w.device(), dy, b.device(), s.device())
        O.linear_postops(x.t, w.t, ref, b.t, act, 0.0, O.BIN_MUL, s.t)
    torch.cuda.synchronize()
    compare(from_device(dy, dt), ref.buf, dt, f"{op} {plan.describe()}")


@pytest.mark.parametrize("M,N,Kd", [(40, 72, 128), (40, 67, 130), (300, 264, 256)])
@pytest.mark.parametrize("adt,bdt", [(O.S8, O.S8), (O.U8, O.S8), (O.U8, O.U8)])
@pytest.mark.parametrize("bias", ["1N", "M1", "MN", None])
def test_integer_runs(M, N, Kd, adt, bdt, bias):
    # the integer epilogue's vector adds (bias along n and the shift's terms) and its element-wise ones, bit for bit
    x = Case([M, Kd], adt, seed=830, lo=0 if adt == O.U8 else -128, hi=255 if adt == O.U8 else 127)
    w = Case([Kd, N], bdt, "BA", seed=831, lo=0 if bdt == O.U8 else -128, hi=255 if bdt == O.U8 else 127)
    b = Case({"1N": [1, N], "M1": [M, 1], "MN": [M, N]}[bias], O.S32, seed=832, lo=-65536, hi=65536) if bias else None
    c = Case([M, N], O.S32, zero=True)
    plan = K.Gemm(x.desc, w.desc, c.desc, b.desc if b else None)
    dc = zeros_device(c)
    plan.run(x.device(), w.device(), dc, b.device() if b else None)
    torch.cuda.synchronize()
    ref = c.clone_empty()
    O.gemm(x.t, w.t, ref, b.t if b else None)
    assert np.array_equal(from_device(dc, O.S32), ref.buf), plan.describe()


@pytest.mark.parametrize("kernel", list(KERNELS))
@pytest.mark.parametrize("M,N", [(257, 1), (70, 2), (300, 9), (65, 33), (257, 264)])
@pytest.mark.parametrize("ylayout", ["AB", "BA"])
def test_few_columns_and_transposed(monkeypatch, kernel, M, N, ylayout):
    # the element-wise loop alone (no run of 8 columns fits, or the output's columns are not contiguous) and after the runs,
    # with strips of a wave's tile past the matrix
    cfg, slices = KERNELS[kernel]
    monkeypatch.setenv("KUDNN_HIP_FORCE_CFG", cfg)
    if slices is not None:
        monkeypatch.setenv("KUDNN_HIP_FORCE_KSLICES", slices)
    dt, Kd = (O.F32, 64) if kernel == "f32" else (O.F16 if kernel == "four_wave" else O.BF16, 128)
    x = Case([M, Kd], dt, seed=840, dist="normal", lo=0.0, hi=1.0)
    w = Case([Kd, N], dt, "BA", seed=841, dist="normal", lo=0.0, hi=0.1)
    b = Case([1, N], O.F32, seed=842, lo=-0.2, hi=0.2)
    y = Case([M, N], dt, ylayout, zero=True)
    plan = K.Gemm(x.desc, w.desc, y.desc, b.desc)
    dy = zeros_device(y)
    plan.run(x.device(), w.device(), dy, b.device(), alpha=0.5)
    torch.cuda.synchronize()
    ref = y.clone_empty()
    O.gemm(x.t, w.t, ref, b.t, 0.5)
    compare(from_device(dy, dt), ref.buf, dt, plan.describe())


def test_one_column_is_not_slower_than_a_tile():
    # 20480 x N x 128 takes the same 80 tiles for N = 1 and N = 128. Walking every strip and column of a tile for one
    # column made N = 1 2.2 times as long as N = 128 (33.7 against 15.4 us); half of it is left as the margin
    M, Kd, us = 20480, 128, {}
    x = torch.randn(M, Kd, device="cuda").bfloat16()
    for N in (1, 128):
        w, y = torch.randn(N, Kd, device="cuda").bfloat16(), torch.empty(M, N, device="cuda", dtype=torch.bfloat16)
        plan = K.Gemm(K.desc([M, Kd], K.BF16), K.desc([Kd, N], K.BF16, "BA"), K.desc([M, N], K.BF16))
        assert "pingpong" in plan.describe() and "pack" not in plan.describe(), plan.describe()
        plan.run(x, w, y)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            for _ in range(20):
                plan.run(x, w, y, stream=torch.cuda.current_stream())
        t = []
        for _ in range(8):
            e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            e0.record()
            graph.replay()
            e1.record()
            torch.cuda.synchronize()
            t.append(e0.elapsed_time(e1) * 1000 / 20)
        us[N] = min(t)
    assert us[1] < 1.6 * us[128], us
