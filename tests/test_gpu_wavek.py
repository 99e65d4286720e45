"""The wave-K kernel (small tiles whose K is dealt to the workgroup's waves): every tile at the edges of M, N and K, both
weight layouts, batches, graph replay and the planner's choices, against the oracle. Integer-valued inputs make the f32
sums exact in any order, so the comparisons are bit for bit."""
import ctypes

import numpy as np
import pytest

import kudnn_amd as K
import oracle as O
from support import Case, compare, explainer, from_device, zeros_device
from test_gpu_layouts import T, run_gemm

torch = pytest.importorskip("torch")

TILES = {"28": "16x16_w8", "29": "16x32_w8", "30": "32x16_w8", "31": "32x32_w8", "32": "32x64_w6", "33": "64x32_w6", "34": "64x64 ", "35": "64x64_2percu",
         "36": "64x128_w4"}
LOWP = dict(list(TILES.items())[2:], **{"37": "64x64_w1"})  # the tiles of 16-bit operands
WIDE = ("32", "34", "35", "36", "37")  # the tiles that read a [K][N] weight in place
ROWS = ("28", "29", "31", "32", "33", "35")  # the tiles that read unaligned rows (from 4 MB of weight on)


@pytest.fixture
def gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    K.lib()


# K: one chunk, one k-tile, a k-tile and a chunk, fewer k-tiles than waves, one each, one more; odd (packed)
@pytest.mark.gpu
@pytest.mark.parametrize("cfg", list(LOWP))
@pytest.mark.parametrize("M,N,Kd", [(17, 16, 8), (32, 33, 64), (33, 130, 72), (64, 128, 320), (65, 264, 512), (70, 40, 584),
                                    (255, 7, 1000), (40, 72, 131)])
@pytest.mark.parametrize("dt", [O.BF16, O.F16])
def test_tiles_exact(gpu, monkeypatch, cfg, M, N, Kd, dt):
    monkeypatch.setenv("KUDNN_HIP_FORCE_CFG", cfg)
    d, _ = run_gemm(T([M, Kd], dt), T([Kd, N], dt, "BA"), T([M, N], dt), T([1, N], O.F32), seed=850, int_valued=True)
    assert LOWP[cfg] in d and ("pack" in d) == (Kd % 8 != 0), d


@pytest.mark.gpu
@pytest.mark.parametrize("cfg", list(LOWP))
@pytest.mark.parametrize("M,N,Kd", [(17, 8, 64), (64, 128, 448), (70, 200, 512), (130, 264, 64), (33, 72, 200), (33, 70, 128)])
def test_kmajor_weight_exact(gpu, monkeypatch, cfg, M, N, Kd):
    # [K][N]: in place by the wide tiles when N is a multiple of 8 and K of 64, packed otherwise
    monkeypatch.setenv("KUDNN_HIP_FORCE_CFG", cfg)
    d, _ = run_gemm(T([M, Kd], O.BF16), T([Kd, N], O.BF16, "AB"), T([M, N], O.F32), None, seed=851, int_valued=True)
    assert ("kmajorB" in d) == (cfg in WIDE and N % 8 == 0 and Kd % 64 == 0), d


# 8-bit weights: K of one chunk, one k-tile (128), a k-tile and a chunk, k-tiles for every wave and more; K = 200 is no
# whole number of chunks, so the operands are packed
@pytest.mark.gpu
@pytest.mark.parametrize("cfg", list(TILES))
@pytest.mark.parametrize("M,N,Kd", [(1, 16, 16), (16, 33, 128), (17, 130, 144), (64, 128, 1040), (70, 40, 1168), (130, 264, 200)])
@pytest.mark.parametrize("adt,bdt,cdt", [(O.F16, O.S8, O.F32), (O.F16, O.U8, O.F32), (O.S8, O.S8, O.S32), (O.U8, O.S8, O.S32)])
def test_8bit_weights_exact(gpu, monkeypatch, cfg, M, N, Kd, adt, bdt, cdt):
    monkeypatch.setenv("KUDNN_HIP_FORCE_CFG", cfg)
    bias = T([1, N], O.S32 if cdt == O.S32 else O.F32)
    d, _ = run_gemm(T([M, Kd], adt), T([Kd, N], bdt, "BA"), T([M, N], cdt), bias, seed=855, int_valued=True)
    assert TILES[cfg] in d and ("pack" in d) == (Kd % 16 != 0), d


@pytest.mark.gpu
@pytest.mark.parametrize("adt,bdt,cdt", [(O.F16, O.S8, O.F16), (O.U8, O.S8, O.S32)])
def test_8bit_unaligned_base(gpu, adt, bdt, cdt):
    # operands that start off a 16-byte boundary are packed at run time, whatever the plan found in their strides
    M, N, Kd = 20, 96, 1024
    a, b = Case([M, Kd], adt, seed=856, lo=-1.0 if adt == O.F16 else 0, hi=1.0 if adt == O.F16 else 255), \
        Case([Kd, N], bdt, "BA", seed=857, lo=-128, hi=127)
    c = Case([M, N], cdt, zero=True)
    plan = K.Gemm(a.desc, b.desc, c.desc)
    assert "wavek" in plan.describe() and "pack" not in plan.describe(), plan.describe()
    ref = c.clone_empty()
    O.gemm(a.t, b.t, ref)
    for off_a, off_b in ((0, 0), (1, 0), (0, 1), (1, 1)):
        da, db = a.device(), b.device()
        pa = torch.zeros(da.numel() + 8, dtype=da.dtype, device="cuda")[off_a:off_a + da.numel()].copy_(da)
        pb = torch.zeros(db.numel() + 16, dtype=db.dtype, device="cuda")[off_b:off_b + db.numel()].copy_(db)
        dc = zeros_device(c)
        plan.run(pa, pb, dc)
        torch.cuda.synchronize()
        compare(from_device(dc, cdt), ref.buf, cdt, f"{off_a} {off_b} {plan.describe()}")


# rows of any alignment, read through registers: K ends 1, 3, 4, 7 elements into a 16-byte chunk (f32: 1, 3)
@pytest.mark.gpu
@pytest.mark.parametrize("cfg", ROWS)
@pytest.mark.parametrize("M,N,Kd", [(5, 4200, 1009), (33, 8500, 523), (70, 1041, 4103), (16, 4099, 1028)])
@pytest.mark.parametrize("adt,bdt,cdt", [(O.BF16, O.BF16, O.F32), (O.F16, O.F16, O.F32), (O.F16, O.S8, O.F32), (O.F16, O.U8, O.F32),
                                         (O.S8, O.S8, O.S32), (O.U8, O.S8, O.S32), (O.F32, O.F32, O.F32)])
def test_unaligned_rows_exact(gpu, monkeypatch, cfg, M, N, Kd, adt, bdt, cdt):
    monkeypatch.setenv("KUDNN_HIP_FORCE_CFG", cfg)
    if adt == O.F16 and bdt != O.F16 and Kd > 4000:
        Kd = 4099  # 16 x 255 x 4099 stays below 2^24
    d, _ = run_gemm(T([M, Kd], adt), T([Kd, N], bdt, "BA"), T([M, N], cdt), None, seed=858, int_valued=True)
    assert TILES[cfg].split("_")[0] in d and "pack" not in d, d


@pytest.mark.gpu
@pytest.mark.parametrize("cfg", list(TILES))
@pytest.mark.parametrize("M,N,Kd", [(17, 16, 4), (32, 33, 32), (33, 130, 72), (64, 128, 320), (255, 7, 1000), (70, 264, 256)])
def test_f32_tiles_exact(gpu, monkeypatch, cfg, M, N, Kd):
    monkeypatch.setenv("KUDNN_HIP_FORCE_CFG", cfg)
    d, _ = run_gemm(T([M, Kd], O.F32), T([Kd, N], O.F32, "BA"), T([M, N], O.F32), T([1, N], O.F32), seed=859, int_valued=True)
    assert d.startswith("mfma_f32_wavek_" + TILES[cfg].strip()) and "pack" not in d, d


@pytest.mark.gpu
@pytest.mark.parametrize("cfg", WIDE)
@pytest.mark.parametrize("M,N,Kd", [(33, 2104, 1009), (64, 4200, 520)])
def test_kmajor_weight_ragged_k_exact(gpu, monkeypatch, cfg, M, N, Kd):
    # [K][N] with K off the k-tile, in place from 4 MB on; the source's rows are packed unless they are whole chunks
    monkeypatch.setenv("KUDNN_HIP_FORCE_CFG", cfg)
    d, _ = run_gemm(T([M, Kd], O.BF16), T([Kd, N], O.BF16, "AB"), T([M, N], O.F32), None, seed=857, int_valued=True)
    assert "kmajorB" in d and ("packA" in d) == (Kd % 8 != 0) and "packB" not in d, d


# fp32 shapes the planner gives to the wave-K tiles, and the configuration of the kernel they replace there: the k-slice
# kernel (rows off the chunk, whole rows, its 4-wave form) and the 64 x 64 kernel
@pytest.mark.gpu
@pytest.mark.parametrize("M,N,Kd,cfg", [(100, 640, 3140, "12"), (64, 2000, 2000, "12"), (120, 1000, 2560, "12"),
                                        (500, 3000, 3000, "11"), (900, 1500, 2002, "11")])
def test_f32_planner_against_float64(gpu, monkeypatch, M, N, Kd, cfg):
    # the planner's choice is no further from 64 bits than the kernel it replaces, on the same inputs (0.36 to 0.72 of it)
    descs = K.desc([M, Kd], K.F32), K.desc([Kd, N], K.F32, "BA"), K.desc([M, N], K.F32)
    chosen = K.Gemm(*descs)
    monkeypatch.setenv("KUDNN_HIP_FORCE_CFG", cfg)
    replaced = K.Gemm(*descs)
    assert chosen.describe().startswith("mfma_f32_wavek_"), chosen.describe()
    assert replaced.describe().startswith({"11": "mfma_f32_64x64 ", "12": "mfma_f32_kslice_16x32 "}[cfg]), replaced.describe()
    err = [0.0, 0.0]
    for seed in range(3):
        g = torch.Generator(device="cuda").manual_seed(870 + seed)
        x, w = (torch.randn(*s, device="cuda", generator=g) for s in ((M, Kd), (N, Kd)))
        ref = x.double() @ w.double().t()
        for i, plan in enumerate((chosen, replaced)):
            y = torch.empty(M, N, device="cuda")
            plan.run(x, w, y)
            torch.cuda.synchronize()
            err[i] += float((y.double() - ref).norm() / ref.norm()) / 3
    assert err[0] <= err[1], err
    # K products rounded and added in f32: a random walk of at most K roundings of 2^-24
    assert err[0] < 2.0 ** -24 * Kd ** 0.5, err


@pytest.mark.gpu
@pytest.mark.parametrize("cfg", ["30", "35", "37"])
def test_batches_and_pitches_exact(gpu, monkeypatch, cfg):
    monkeypatch.setenv("KUDNN_HIP_FORCE_CFG", cfg)
    run_gemm(T([3, 40, 136], O.BF16, "ABC", [40 * 144, 144, 1]), T([3, 136, 72], O.BF16, "ACB"), T([3, 40, 72], O.BF16),
             T([3, 1, 72], O.F32), alpha=0.5, beta=0.5, seed=852, int_valued=True)
    run_gemm(T([2, 3, 40, 128], O.F16), T([2, 1, 128, 72], O.F16), T([2, 3, 40, 72], O.F16), None, seed=853, int_valued=True)


@pytest.mark.gpu
def test_rows_past_k_stay_out(gpu, monkeypatch):
    # the 16-byte chunks past K hold Inf and NaN (the next elements of a longer row): none may reach the sums
    monkeypatch.setenv("KUDNN_HIP_FORCE_CFG", "34")
    M, N, Kd, P = 40, 72, 200, 256
    x = torch.full((M, P), float("nan"), device="cuda", dtype=torch.bfloat16)
    w = torch.full((N, P), float("inf"), device="cuda", dtype=torch.bfloat16)
    x[:, :Kd] = 1.0
    w[:, :Kd] = 0.5
    y = torch.zeros(M, N, device="cuda", dtype=torch.float32)
    plan = K.Gemm(K.desc([M, Kd], K.BF16, "AB", [P, 1]), K.desc([Kd, N], K.BF16, "BA", [1, P]), K.desc([M, N], K.F32))
    assert "wavek" in plan.describe() and "pack" not in plan.describe(), plan.describe()
    plan.run(x, w, y)
    torch.cuda.synchronize()
    assert bool((y == 0.5 * Kd).all())


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,Kd,wl", [(64, 1024, 2048, "BA"), (100, 600, 1096, "BA"), (64, 1024, 2048, "AB")])
def test_planner_plans_and_graph_replays(gpu, M, N, Kd, wl):
    dt = O.BF16
    x = Case([M, Kd], dt, seed=860, dist="normal", lo=0.0, hi=1.0)
    w = Case([Kd, N], dt, wl, seed=861, dist="normal", lo=0.0, hi=0.05)
    s = Case([M, N], dt, seed=862, lo=-1.0, hi=1.0)
    y = Case([M, N], dt, zero=True)
    plan = K.LinearPostOps(x.desc, w.desc, y.desc, None, act=K.ACT_GELU_TANH, binary=K.BIN_ADD, src=s.desc)
    assert "wavek" in plan.describe(), plan.describe()
    dx, dw, ds, dy = x.device(), w.device(), s.device(), zeros_device(y)
    plan.run(dx, dw, dy, None, ds)
    torch.cuda.synchronize()
    ref = y.clone_empty()
    O.linear_postops(x.t, w.t, ref, None, O.ACT_GELU_TANH, 0.0, O.BIN_ADD, s.t)
    eager = from_device(dy, dt)
    why = explainer(dt, x.t, w.t, None, (M, N), act=K.ACT_GELU_TANH, binary=K.BIN_ADD, src=s.t)
    compare(eager, ref.buf, dt, plan.describe(), explain=why)
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        plan.run(dx, dw, dy, None, ds, stream=torch.cuda.current_stream())
    for _ in range(3):
        dy.zero_()
        torch.randn(1 << 16, device="cuda").sum()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert np.array_equal(from_device(dy, dt), eager)


# batches by the planner: a wave a tile, four waves a tile; M, N and K off the tile, both weight layouts
@pytest.mark.gpu
@pytest.mark.parametrize("B,M,N,Kd,wl,name", [(20, 300, 1000, 80, "ACB", "64x64_w1"), (20, 300, 1000, 128, "ABC", "64x64_w1"),
                                              (9, 130, 129, 96, "ACB", "64x64_2percu"), (9, 130, 136, 72, "ABC", "64x64_2percu")])
def test_short_k_batches_exact(gpu, B, M, N, Kd, wl, name):
    d, _ = run_gemm(T([B, M, Kd], O.F16), T([B, Kd, N], O.F16, wl), T([B, M, N], O.F16), T([B, 1, N], O.F32), seed=854,
                    int_valued=True)
    assert name in d and "pack" not in d, d


def test_planner_rule():
    def plan(M, Kd, N, wl="BA", dt=K.BF16):
        return K.LinearPostOps(K.desc([M, Kd], dt), K.desc([Kd, N], dt, wl), K.desc([M, N], dt)).describe()
    assert plan(17, 4096, 4096).startswith("mfma_bf16_wavek_32x16")
    assert plan(64, 4096, 4096, dt=K.F16).startswith("mfma_f16_wavek_32x32")
    assert plan(64, 4096, 11008).startswith("mfma_bf16_wavek_64x64")
    assert "kmajorB" in plan(64, 4096, 4096, "AB") and "kmajorB" in plan(64, 1000, 4096, "AB")
    assert "packA packB" in plan(64, 1000, 1024, "AB")
    assert "pack" not in plan(100, 1000, 4096) and "pack" not in plan(100, 1001, 4096)
    assert "packA packB" in plan(100, 1001, 1024)  # under 4 MB of weight
    assert plan(16, 4096, 4096).startswith("skinny") and "wavek" not in plan(256, 4096, 4096)
    assert "wavek" not in plan(16, 4096, 4096) and plan(16, 4097, 4096).startswith("mfma_bf16_wavek_16x")
    assert "wavek" not in plan(255, 4096, 14336) and "wavek" not in plan(40, 128, 4096)
    def planb(B, M, Kd, N, wl="ACB"):
        return K.Gemm(K.desc([B, M, Kd], K.BF16), K.desc([B, Kd, N], K.BF16, wl), K.desc([B, M, N], K.BF16)).describe()
    assert planb(63, 192, 80, 376).startswith("mfma_bf16_wavek_64x64_w1") and "kmajorB" in planb(63, 192, 80, 376, "ABC")
    assert planb(32, 256, 96, 256).startswith("mfma_bf16_wavek_64x64_2percu")
    assert "wavek" not in planb(32, 1024, 128, 1024) and "wavek" not in planb(16, 512, 512, 512)
    assert "skinny" in planb(8, 8, 64, 256) and "wavek_64x64_w1" in planb(16, 128, 128, 2048)
    # 8-bit weights: from M = 1, K of at least 4 k-tiles of 128 (the last may be partial) in whole 16-byte chunks

    def plan8(M, Kd, N, adt, bdt, cdt):
        return K.Gemm(K.desc([M, Kd], adt), K.desc([Kd, N], bdt, "BA"), K.desc([M, N], cdt)).describe()
    assert plan8(4, 4096, 4096, K.F16, K.S8, K.F16).startswith("mfma_f16_wavek_16x16")
    assert "pack" not in plan8(64, 1040, 4096, K.F16, K.U8, K.F16)
    assert "pack" not in plan8(4, 1001, 8192, K.F16, K.S8, K.F16) and "packB" in plan8(4, 1001, 2048, K.F16, K.S8, K.F16)
    assert "packB" in plan8(4, 384, 4096, K.F16, K.S8, K.F16)
    assert plan8(64, 4096, 4096, K.S8, K.S8, K.S32).startswith("mfma_s8_wavek")
    assert "pack" not in plan8(64, 4096, 4096, K.U8, K.S8, K.S32)
    assert "wavek" not in plan8(64, 4096, 4096, K.S8, K.U8, K.S32) and "wavek" not in plan8(1024, 4096, 4096, K.S8, K.S8, K.S32)
    assert "wavek" in plan8(1024, 4096, 4096, K.U8, K.S8, K.S32) and "wavek" not in plan8(2048, 4096, 11008, K.U8, K.S8, K.S32)
    assert "wavek" in plan(400, 4096, 4096) and "wavek" not in plan(512, 4096, 4096) and "wavek" not in plan(1000, 4096, 11008)
    def plan32(M, Kd, N):
        return K.Gemm(K.desc([M, Kd], K.F32), K.desc([Kd, N], K.F32, "BA"), K.desc([M, N], K.F32)).describe()
    # f32: chains of sums half as long as the k-slice kernel's or the split grid's leave 32 x 16 tiles, rows of whole chunks
    assert plan32(64, 2000, 2000).startswith("mfma_f32_wavek_32x16_w8") and "kslice_16x32 " in plan32(200, 1023, 1400)
    assert "wavek_64x128_w4" in plan32(500, 3000, 3000)
    # s8: 64 tiles of 256 x 256 and 128 k-tiles or more keep the tail split, fewer tiles and u8 sources do not
    assert "pingpong" in plan8(1024, 16384, 4096, K.S8, K.S8, K.S32) and "wavek" in plan8(768, 16384, 4096, K.S8, K.S8, K.S32)
    assert "wavek" in plan8(1024, 16384, 4096, K.U8, K.S8, K.S32)
    assert plan32(107, 2176, 1984).startswith("mfma_f32_wavek_32x") and "kslice_16x32 " in plan32(240, 1298, 1400)
    assert plan32(128, 1024, 1024).startswith("mfma_f32_kslice_16x32 ") and plan32(2048, 4096, 4096).startswith("mfma_f32_128x128")


def test_planner_leaves_what_the_other_kernels_do_faster():
    # products that the estimates without outputs, batches and unaligned copies had moved to the wave-K tiles, measured (us)
    # on those tiles and on the other kernel
    def batch(B, M, Kd, N, wl="ACB", bin=K.BIN_NONE):
        dy = K.desc([B, M, N], K.BF16)
        return K.LinearPostOps(K.desc([B, M, Kd], K.BF16), K.desc([B, Kd, N], K.BF16, wl), dy, binary=bin,
                               src=dy if bin else None).describe()

    def one(M, Kd, N, adt=K.BF16, bdt=None, wl="BA", xl="AB", ydt=None):
        return K.Gemm(K.desc([M, Kd], adt, xl), K.desc([Kd, N], bdt or adt, wl), K.desc([M, N], ydt or adt)).describe()
    other = [batch(64, 128, 2048, 512, "ABC"),      # 72, 51
             batch(64, 128, 2048, 512),             # 71, 54
             batch(32, 300, 512, 512),              # 28, 21
             batch(64, 128, 512, 512),              # 30, 24
             batch(13, 640, 64, 256),               # 10.2, 7.9
             batch(39, 256, 64, 576, "ABC", K.BIN_ADD),  # 19.5, 14.8
             batch(35, 256, 128, 256),              # 11.4, 8.9
             batch(50, 512, 128, 541, bin=K.BIN_ADD),  # 100, 71
             one(742, 256, 7968, wl="AB"),          # 34, 22
             one(4096, 512, 1024, K.F16, K.S8),     # 26, 23
             one(10925, 376, 2304, K.F32),          # 304, 223
             one(88640, 264, 256, K.F16, xl="BA"),  # 124, 95
             one(2048, 2676, 1408),                 # 86, 70
             one(693, 1222, 4936),                  # 55, 48
             one(1, 16384, 4, K.F16, K.S8),         # 9.8, 7.6
             one(5748, 15168, 1152, K.U8, K.S8, ydt=K.S32),   # 262, 191
             one(1792, 11712, 4096, K.U8, K.S8, ydt=K.S32)]   # 201, 148
    for d in other:
        assert "wavek" not in d, d
    wavek = [batch(16, 32, 4096, 1024, "ABC"),      # 33, 91
             batch(16, 17, 2048, 4096),             # 61, 80
             batch(8, 17, 512, 2048),               # 7.3, 11.3
             batch(57, 192, 128, 192, "ABC"),       # 11.7, 14.3 with the weight's pack
             batch(39, 145, 128, 312, "ABC"),       # 12.3, 16.2
             batch(8, 185, 64, 1487),               # 14.5, 21.7: rows of no whole 16-byte runs
             one(1216, 689, 3412, K.F16, wl="AB"),  # 35, 54
             one(17, 4096, 3264, wl="AB"),          # 17.5, 30
             one(1024, 4096, 4096, K.U8, K.S8, ydt=K.S32),    # 41, 83
             one(1, 9600, 64, K.F16, K.S8)]         # 6.9, 12
    for d in wavek:
        assert "wavek" in d, d


def test_planner_sixty_five_to_seventy_nine_tiles():
    # one round of 128 x 128 tiles beats two K slices of 256 x 256 ones; two rounds do not. A weight stored [K][N] is read in
    # place by the sliced kernel
    def plan(M, Kd, N, wl="BA"):
        return K.LinearPostOps(K.desc([M, Kd], K.BF16), K.desc([Kd, N], K.BF16, wl), K.desc([M, N], K.BF16)).describe()
    assert plan(384, 4224, 8832).startswith("mfma_bf16_128x128 ")    # 49 us against 60
    assert plan(800, 2688, 4352).startswith("mfma_bf16_128x128 ")    # 37 against 47
    assert " kslices=2" in plan(738, 10112, 5896) and " kslices=2" in plan(800, 2688, 4352, "AB")


def test_planner_keeps_the_fixed_scratch_calls():
    # plans of the allocation-free entry point: where the other kernel, the faster one, needs more than its scratch for packs
    # and sums and the wave-K tiles do not, these keep the product; the other entry points go by time alone
    for M, Kd, N, dt in ((448, 9898, 3808, K.F16), (744, 7776, 5888, K.BF16), (144, 9833, 8448, K.BF16)):
        d = K.desc([M, Kd], dt), K.desc([Kd, N], dt, "BA"), K.desc([M, N], dt)
        post, gemm = K.LinearPostOps(*d).describe(), K.Gemm(*d).describe()
        assert "wavek" in post and "pack" not in post, post
        assert "pingpong" in gemm and "packA packB kslices=" in gemm, gemm


@pytest.mark.gpu
def test_fixed_scratch_call_beside_a_large_pack(gpu):
    M, Kd, N = 448, 9898, 3808
    x, w = torch.randn(M, Kd, device="cuda").half(), (torch.randn(N, Kd, device="cuda") * 0.02).half()
    y, z = (torch.zeros(M, N, device="cuda", dtype=torch.float16) for _ in range(2))
    p = K.LinearPostOps(K.desc([M, Kd], K.F16), K.desc([Kd, N], K.F16, "BA"), K.desc([M, N], K.F16))
    p.run(x, w, y)
    st = K.lib().kudnn_linear_postops_run_noalloc(p.handle, x.data_ptr(), w.data_ptr(), z.data_ptr(), None, None,
                                                  ctypes.c_float(1.0), torch.cuda.current_stream().cuda_stream)
    assert st == K.SUCCESS, K.last_error()
    torch.cuda.synchronize()
    assert torch.equal(y, z)
