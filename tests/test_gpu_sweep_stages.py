"""The fused sweeps' form of each stage (device_math.hpp: shared reciprocals, lengths and impedances
handed over, minima and maxima as instructions) against the plain form that the per-stage kernels
run, on the device, bit for bit, over physical states, vanishing differences, subnormals, zeros of
both signs, infinities and NaN (two NaNs count as equal), for cell sizes that are powers of two and
others (armon_selftest_stages in armon-kokkos_amd/csrc/selftest_division.hip)."""
import ctypes
import os

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "armon-kokkos_amd", "lib", "libarmon_selftest.so")


@pytest.mark.gpu
@pytest.mark.parametrize("seed", [5, 90210])
def test_sweep_stages_have_the_bits_of_the_plain_stages(seed):
    fn = ctypes.CDLL(LIB).armon_selftest_stages
    fn.argtypes = [ctypes.c_uint64, ctypes.c_int64, ctypes.POINTER(ctypes.c_uint64),
                   ctypes.POINTER(ctypes.c_uint64), ctypes.POINTER(ctypes.c_double)]
    fn.restype = ctypes.c_int
    n = 1 << 29
    bad, shared = ctypes.c_uint64(0), ctypes.c_uint64(0)
    first = (ctypes.c_double * 2)()
    rc = fn(seed, n, ctypes.byref(bad), ctypes.byref(shared), first)
    assert rc == 0, f"HIP error {rc}"
    print(f"mismatches {bad.value}, samples through the shared reciprocals {shared.value}", flush=True)
    assert bad.value == 0, f"{bad.value} samples differ; one of them: {first[0]:.0f}, stages {first[1]:.0f}"
    assert 0.3 * n < shared.value < 0.95 * n   # both ways ran
