"""The dropout mask's short cuts of csrc/philox.h against its element-by-element form, on the host."""
import os
import shutil
import subprocess

import pytest

HEADER = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "slapo_amd",
                      "csrc", "philox.h")
SOURCE = r"""
#include "%s"
#include <cstdio>
#include <random>
using namespace slapo;
std::mt19937_64 rnd(7);

DropoutState any_state() {
    DropoutState s{};
    s.key0 = rnd(), s.key1 = rnd();
    s.base_counter = rnd() %% 3 ? rnd() %% 1000 : rnd();
    const uint64_t threads[] = {524288, 256, 256 * (1 + rnd() %% 2048), 256 * (1 + rnd() %% 7)};
    s.total_threads = threads[rnd() %% 4];
    const uint32_t vecs[] = {4, 4, 4, 2, 1, 8, 16};
    s.vec = vecs[rnd() %% 7];
    s.calls_per_iter = s.vec < 4 ? 1 : s.vec / 4;
    s.t_shift = -1;
    for (int i = 0; i < 40; ++i)
        if ((1ull << i) == s.total_threads) s.t_shift = i;
    s.g_shift = s.vec == 4 ? 0 : s.vec == 8 ? 1 : s.vec == 16 ? 2 : -1;
    s.keep_max = rnd() %% 2 ? 3865470566u : (uint32_t)rnd();
    s.keep_none = rnd() %% 50 == 0;
    return s;
}
template <int kN, bool kAligned>
int runs() {
    int bad = 0;
    for (int it = 0; it < 5000; ++it) {
        const DropoutState s = any_state();
        uint64_t e = rnd() %% 3 ? rnd() %% 100000 : rnd() %% (1ull << 36);
        if (kAligned) e &= ~3ull;
        if (rnd() %% 4 == 0) e = 4 * s.total_threads * (1 + rnd() %% 5) - (kAligned ? 8 : rnd() %% 40);
        uint32_t want = 0;
        for (int i = 0; i < kN; ++i) want |= (dropout_keep1(s, e + i) ? 1u : 0u) << i;
        bad += dropout_keep_run<kN, kAligned>(s, e) != want;
    }
    return bad;
}
int main() {
    int bad = runs<32, false>() + runs<32, true>() + runs<8, false>() + runs<4, false>();
    for (int it = 0; it < 20000; ++it) {
        const uint64_t c = rnd();
        const uint32_t t = rnd(), k0 = rnd(), k1 = rnd();
        const u32x4 a = philox4x32_10((uint32_t)c, (uint32_t)(c >> 32), t, 0, k0, k1);
        const u32x4 b = philox_block(philox_call(c, k0, k1), t);
        bad += a.x != b.x || a.y != b.y || a.z != b.z || a.w != b.w;
    }
    std::printf("%%d\n", bad);
    return bad != 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs a host compiler")
def test_runs_and_shared_rounds_equal_the_single_elements(tmp_path):
    """Runs of keep bits for every vec, thread count, alignment and wrap; blocks whose first rounds are
    shared by a call."""
    source = tmp_path / "philox.cpp"
    source.write_text(SOURCE % HEADER)
    exe = tmp_path / "philox"
    subprocess.run(["g++", "-O2", "-std=c++17", str(source), "-o", str(exe)], check=True, timeout=120)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0 and out.stdout.strip() == "0", out.stdout + out.stderr
