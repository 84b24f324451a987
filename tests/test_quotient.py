"""The encoders' quotient, compiled from the kernel's own source for the CPU: all mantissas."""
import ctypes
import os
import re
import subprocess
from concurrent.futures import ThreadPoolExecutor

from blockgtq_amd.build import CSRC

_LOOP = """
#include <stdint.h>
#define __device__
#define __forceinline__ static inline
typedef struct { float x, y; } float2;
%s
/* how many quotients of the 11-bit numerators 1024 .. 2047 by the divisors first .. last - 1 (24 bits) are not the rounded ones */
int64_t wrong(uint32_t first, uint32_t last, uint32_t step) {
    int64_t n = 0;
    for (uint32_t d0 = first; d0 < last; d0 += 512 * step) {
        float d[512], y[512];
        for (int i = 0; i < 512; i++) { d[i] = (float)(d0 + i * step < last ? d0 + i * step : first); y[i] = 1.0f / d[i]; }
        for (int x = 1024; x < 2048; x++) {
            int32_t bad = 0;
            for (int i = 0; i < 512; i++) { const float2 dy = {d[i], y[i]}; bad += div_by((float)x, dy) != (float)x / d[i]; }
            n += bad;
        }
    }
    return n;
}
"""


def test_one_residual_step_rounds_every_quotient_of_an_11_bit_numerator(tmp_path):
    """Powers of two change nothing (the kernel's operands and quotients are normal), so mantissas are all there is."""
    text = open(os.path.join(CSRC, "bgtq_encode.hip")).read()
    body, = re.findall(r"^__device__ __forceinline__ float div_by\(float x, float2 dy\) \{.*?^\}", text, re.S | re.M)
    fma = " fma " in open("/proc/cpuinfo").read()
    src, lib = tmp_path / "quotient.c", tmp_path / "quotient.so"
    src.write_text(_LOOP % body)
    subprocess.run(["gcc", "-O3", "-ffp-contract=off", "-shared", "-fPIC", str(src), "-o", str(lib), "-lm"] +
                   (["-mavx2", "-mfma"] if fma else []), check=True)
    fn = ctypes.CDLL(str(lib)).wrong
    fn.restype, fn.argtypes = ctypes.c_int64, [ctypes.c_uint32] * 3
    step = 1 if fma else 211                             # (without the instruction every multiply-add is a library call)
    with ThreadPoolExecutor(min(os.cpu_count(), 16)) as pool:
        assert sum(pool.map(lambda i: fn((1 << 23) + (i << 17), (1 << 23) + ((i + 1) << 17), step), range(64))) == 0
