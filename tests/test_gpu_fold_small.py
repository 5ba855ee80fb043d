"""Folds of short arrays in one launch (up to 10 shares of 4096 elements) and
the first sizes past them, at share and vector remainders, on aligned and
unaligned input, against the oracle: integers and max exact, the compensated
sum within 1e-12 of the sum of magnitudes (a partial's correction term is
itself a rounded FP32 sum of at most some 30 terms: 30 * 2^-48 = 1.1e-13)."""
import ctypes as C

import numpy as np
import pytest

from muesli4_amd import hip
from muesli4_amd.hip import DeviceArray, call
from oracle import refcpu as R

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 3, 4, 255, 4095, 4096, 4097, 8193, 16385, 40959, 40960, 40961, 45057]


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("shift", [0, 1])
def test_short_folds(n, shift):
    print(f"[case] short folds n={n} shift={shift}", flush=True)
    hip.init(0)
    rng = np.random.default_rng(n)
    f = rng.uniform(-100.0, 255.0, n + shift).astype(np.float32)
    i = rng.integers(-(1 << 31), 1 << 31, n + shift).astype(np.int32)
    df, di = DeviceArray.from_host(f), DeviceArray.from_host(i)
    f, i, pf, pi = f[shift:], i[shift:], df.ptr + 4 * shift, di.ptr + 4 * shift
    s64, s32, top, u, s = C.c_double(), C.c_float(), C.c_float(), C.c_uint32(), C.c_int64()
    call("msl_fold_sum_f32_host", pf, n, C.byref(s64), C.byref(s32))
    ref = R.fold_sum_f64(f)
    assert abs(s64.value - ref) <= 1e-12 * np.abs(f).astype(np.float64).sum()
    assert s32.value == np.float32(s64.value)
    dev = DeviceArray(1, np.float64)
    call("msl_fold_sum_f32", pf, n, dev.ptr)
    assert dev.to_host()[0] == s64.value  # device and host forms: the same kernels
    call("msl_fold_max_f32_host", pf, n, C.byref(top))
    assert top.value == f.max()
    call("msl_fold_sum_u32_host", pi, n, C.byref(u))
    assert u.value == int(i.astype(np.int64).sum()) & 0xFFFFFFFF
    call("msl_fold_sum_i32_host", pi, n, C.byref(s))
    assert s.value == int(i.astype(np.int64).sum())


@pytest.mark.parametrize("n", [5, 5000, 45057])
def test_short_folds_of_special_values(n):
    """Max of lowest values, infinities and NaN (which a comparison drops);
    the empty integer and float sums."""
    print(f"[case] short folds, special values n={n}", flush=True)
    hip.init(0)
    top, s64, s = C.c_float(), C.c_double(), C.c_int64()
    for values, want in (([np.finfo(np.float32).min], np.finfo(np.float32).min), ([-np.inf], -np.inf),
                         ([np.nan, -3.0], -3.0), ([np.inf, np.nan, 1.0], np.inf)):
        f = np.resize(np.array(values, np.float32), n)
        d = DeviceArray.from_host(f)
        call("msl_fold_max_f32_host", d.ptr, n, C.byref(top))
        assert top.value == want, (values, top.value)
    call("msl_fold_sum_f32_host", d.ptr, 0, C.byref(s64), None)
    call("msl_fold_sum_i32_host", d.ptr, 0, C.byref(s))
    assert s64.value == 0.0 and s.value == 0
