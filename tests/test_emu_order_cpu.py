"""The emulation's order of threads: a missing barrier between a writer and a
reader shows, whichever of the two has the lower thread number."""
import os
import subprocess

import pytest

EMU = os.path.join(os.path.dirname(os.path.abspath(__file__)), "emu")

SRC = r"""
#include "hip_emu.hpp"
// Thread t publishes t + 1 and reads the word of thread t + STEP, or its own at the ends.
static uint32_t source(uint32_t t, int step) {
    const int s = (int)t + step;
    return s >= 0 && s < 256 ? (uint32_t)s : t;
}
template <int STEP, bool BARRIER>
static void kernel(uint32_t* out) {
    __shared__ uint32_t s[256];
    const uint32_t t = threadIdx.x;
    s[t] = 0;
    __syncthreads();
    s[t] = t + 1;
    if (BARRIER) __syncthreads();
    out[blockIdx.x * 256 + t] = s[source(t, STEP)];
}
template <int STEP, bool BARRIER>
static int wrong() {  // words that differ from what a barrier gives
    static uint32_t out[2 * 256];
    hipLaunchKernelGGL((kernel<STEP, BARRIER>), dim3(2), dim3(256), 0, nullptr, out);
    int bad = 0;
    for (uint32_t i = 0; i < 512; ++i) bad += out[i] != source(i % 256, STEP) + 1;
    return bad;
}
int main() {
    for (int rep = 0; rep < 2; ++rep) {
        if (wrong<1, true>() || wrong<-1, true>() || wrong<64, true>() || wrong<-64, true>()) return 1;
        if (!wrong<1, false>() || !wrong<-1, false>()) return 2;    // neighbours in a wave
        if (!wrong<64, false>() || !wrong<-64, false>()) return 3;  // the next wave and the one before
    }
    return 0;
}
"""


@pytest.mark.parametrize("opt", ["-O1"])
def test_missing_barriers_show(tmp_path, opt):
    src = tmp_path / "order.cpp"
    src.write_text(SRC)
    exe = tmp_path / "order"
    subprocess.run(["g++", opt, "-std=c++20", "-DGMS_HOST_EMULATION", "-I", EMU, "-pthread", str(src),
                    os.path.join(EMU, "hip_emu.cpp"), "-o", str(exe)], check=True)
    assert subprocess.run([str(exe)]).returncode == 0
