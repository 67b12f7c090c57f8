"""The autotuner times each kernel once: variants that run the same code are one
candidate."""
import ctypes

import pytest

from jet_amd import _native as nat

pytestmark = pytest.mark.gpu

F32 = 2


@pytest.mark.parametrize("m,n,k,variants", [
    (16, 16, 16, [1]), (64, 100, 300, [1]), (5, 64, 64, [1]),   # BF16 products
    (15, 64, 12, [1, 2, 3]), (64, 64, 12, [1, 2, 3])])          # FP32 MFMA tiles
def test_fp32_variants(m, n, k, variants):
    cap = 32
    ks, vs = (ctypes.c_int32 * cap)(), (ctypes.c_int32 * cap)()
    ms, cnt = (ctypes.c_float * cap)(), ctypes.c_int()
    nat.check(nat.lib().jet_hip_autotune_gemm(nat.default_context().handle, nat.C64,
                                              nat.PREC_FP32, m, n, k, 1, 1, cap, ks, vs, ms,
                                              ctypes.byref(cnt)))
    assert sorted(vs[i] for i in range(cnt.value) if ks[i] == F32) == variants
