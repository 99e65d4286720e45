"""GPU parity of operands that are packed before the GEMM: rows of odd length, pitches and base addresses that are no
multiple of 16 bytes, both contiguous directions, and every type pair the planner converts. The inputs are small
integers, so every f32 sum is exact and the outputs are compared with the oracle bit for bit."""
import numpy as np
import pytest

import kudnn_amd as K
import oracle as O
from support import from_device
from test_gpu_layouts import T, run_gemm

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    K.lib()


# source type, weight type, output type: a copy of each size, and each conversion (f16 from 8-bit integers, f32 from all)
PAIRS = [(O.BF16, O.BF16, O.F32), (O.F16, O.F16, O.F32), (O.F16, O.S8, O.F32), (O.F16, O.U8, O.F32), (O.F32, O.F32, O.F32),
         (O.F32, O.BF16, O.F32), (O.F16, O.F32, O.F32), (O.S8, O.S8, O.S32), (O.U8, O.S8, O.S32), (O.S8, O.U8, O.F32)]


@pytest.mark.parametrize("adt,bdt,cdt", PAIRS)
@pytest.mark.parametrize("mnk", [(70, 67, 131), (17, 64, 65), (129, 200, 1023)])
@pytest.mark.parametrize("xl,wl", [("AB", "BA"), ("BA", "AB")])
def test_packed_operands_exact(adt, bdt, cdt, mnk, xl, wl):
    M, N, Kd = mnk
    # the integer types draw from their own range: products beyond f32's exact integers stay within s32's arithmetic
    if cdt == O.F32 and (adt in (O.S8, O.U8) or bdt in (O.S8, O.U8)) and Kd > 200:
        Kd = 199  # 200 terms of at most 16 x 255 or 125 x 255: below 2^24
    d, _ = run_gemm(T([M, Kd], adt, xl), T([Kd, N], bdt, wl), T([M, N], cdt), None, seed=800, int_valued=True)
    assert "pack" in d, d


@pytest.mark.parametrize("M,N,Kd", [(40, 72, 128), (3, 72, 128), (300, 264, 256)])
@pytest.mark.parametrize("shift", [1, 3])
def test_unaligned_base_pointers(M, N, Kd, shift):
    # operands that lie `shift` elements into their buffers are packed whatever their shape
    rng = np.random.default_rng(810)
    xv, wv = (rng.integers(-8, 9, size=n).astype(np.float32) for n in (M * Kd, N * Kd))
    x = torch.zeros(M * Kd + shift, device="cuda", dtype=torch.bfloat16)
    w = torch.zeros(N * Kd + shift, device="cuda", dtype=torch.bfloat16)
    x[shift:] = torch.from_numpy(xv).cuda()
    w[shift:] = torch.from_numpy(wv).cuda()
    y = torch.zeros(M * N, device="cuda", dtype=torch.float32)
    plan = K.Gemm(K.desc([M, Kd], K.BF16), K.desc([Kd, N], K.BF16, "BA"), K.desc([M, N], K.F32))
    plan.run(x[shift:], w[shift:], y)
    torch.cuda.synchronize()
    ref = O.empty((M, N), (N, 1), O.F32)
    O.gemm(O.Tensor((M, Kd), (Kd, 1), O.BF16, O.from_f32_rne(xv, O.BF16)),
           O.Tensor((Kd, N), (1, Kd), O.BF16, O.from_f32_rne(wv, O.BF16)), ref)
    assert np.array_equal(from_device(y, O.F32), ref.buf), plan.describe()


# packed rows of 1 to 5 k-tiles (8, 16, 24, 32 and 40 chunks of 16 bytes: 8 to 64 lanes to a row), rows off a workgroup's
@pytest.mark.parametrize("adt,bdt,cdt", [(O.BF16, O.BF16, O.F32), (O.F16, O.S8, O.F32), (O.U8, O.S8, O.S32), (O.BF16, O.F32, O.F32)])
@pytest.mark.parametrize("rows", [1, 15, 129, 515])
@pytest.mark.parametrize("tiles", [1, 2, 3, 4, 5])
def test_narrow_rows_exact(adt, bdt, cdt, rows, tiles):
    step = 32 if O.F32 in (adt, bdt) else (128 if cdt == O.S32 else 64)
    for Kd in (tiles * step - 1, (tiles - 1) * step + 3):
        if bdt == O.S8 and cdt == O.F32:
            Kd = min(Kd, 199)  # terms of at most 16 x 125: below 2^24
        d, _ = run_gemm(T([rows, Kd], adt), T([Kd, 24], bdt, "BA"), T([rows, 24], cdt), None, seed=805, int_valued=True)
        assert "pack" in d, d
