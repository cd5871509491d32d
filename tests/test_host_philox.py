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


def _compile_and_run(tmp_path, text):
    source = tmp_path / "philox.cpp"
    source.write_text(text)
    exe = tmp_path / "philox"
    subprocess.run(["g++", "-O2", "-std=c++17", str(source), "-o", str(exe)], check=True, timeout=120)
    return subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs a host compiler")
def test_runs_and_shared_rounds_equal_the_single_elements(tmp_path):
    """Runs of keep bits for every vec, thread count, alignment and wrap; blocks whose first rounds are
    shared by a call."""
    out = _compile_and_run(tmp_path, SOURCE % HEADER)
    assert out.returncode == 0 and out.stdout.strip() == "0", out.stdout + out.stderr


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs a host compiler")
@pytest.mark.parametrize("vec", [8, 16])
@pytest.mark.parametrize("threads", [524288, 256 * 7])
def test_wide_plans_draw_a_block_per_four_elements(tmp_path, vec, threads):
    """A run of 32 elements under the plan of a one- or two-byte tensor: eight blocks, nine where it
    does not start at a multiple of four."""
    with open(HEADER, encoding="utf-8") as f:
        header = f.read()
    start = "uint32_t k1) {\n#pragma unroll\n"  # of philox4x32_10
    assert header.count(start) == 1
    counted = tmp_path / "philox_counted.h"
    counted.write_text(header.replace("SLAPO_HD u32x4 philox4x32_10(",
                                      "static int blocks;\nSLAPO_HD u32x4 philox4x32_10(")
                       .replace(start, "uint32_t k1) {\n++blocks;\n"))
    out = _compile_and_run(tmp_path, f"""
#include "{counted}"
#include <cstdio>
using namespace slapo;
int main() {{
    DropoutState s{{}};
    s.total_threads = {threads}, s.vec = {vec}, s.calls_per_iter = {vec // 4};
    s.keep_max = 3865470566u, s.t_shift = {threads.bit_length() - 1 if threads == 524288 else -1};
    s.g_shift = {1 if vec == 8 else 2};
    dropout_keep_run<32, true>(s, 1024);
    const int aligned = blocks;
    dropout_keep_run<32, false>(s, 1023);
    std::printf("%d %d\\n", aligned, blocks - aligned);
}}
""")
    assert out.stdout.split() == ["8", "9"], out.stdout + out.stderr
