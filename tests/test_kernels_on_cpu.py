"""Device code of the PCG path compiled with g++ and run on the CPU, one thread
after the other, under AddressSanitizer: its accesses against buffers of
exactly their size.  The functions are cut out of the sources by name."""
import os
import re
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "help_amd", "csrc")

SHIM = """
#include <algorithm>
#include <cstdint>
#include <cstdio>
#include <vector>
#define __global__
#define __device__
#define __host__
#define __launch_bounds__(x)
using std::min;
using std::max;
struct Dim { int x = 0, y = 0; };
static Dim blockIdx, threadIdx, gridDim;
"""


def _cut(name, pattern):
    """The definition in file `name` that starts at `pattern`, to its closing brace."""
    text = open(os.path.join(CSRC, name)).read()
    at = re.search(pattern, text, re.M).start()
    depth, end = 0, text.index("{", at)
    while True:
        depth += {"{": 1, "}": -1}.get(text[end], 0)
        end += 1
        if depth == 0:
            break
    return text[at:end] + (";" if text[at:].startswith("struct") else "") + "\n"


def _run(tmp_path, source):
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(SHIM + source)
    b = subprocess.run(["g++", "-std=c++17", "-O0", "-g", "-w", "-fsanitize=address,undefined",
                        "-fno-sanitize-recover=all", str(src), "-o", str(exe)], capture_output=True, text=True)
    assert b.returncode == 0, b.stderr[-4000:]
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, (r.stdout + r.stderr)[-4000:]


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
@pytest.mark.parametrize("K,k0", [(1, 0), (2, 0), (3, 0), (4, 0), (5, 4), (17, 3), (17, 16), (30, 29)])
def test_block_sums_stay_inside_the_factor(tmp_path, K, k0):
    """k_pc_block reads finished columns of an m x K factor only, and leaves the
    four chains of every candidate's sum over the first k0 - k0 % 4 of them (in
    the kernel's order, so equal)."""
    _run(tmp_path, """
constexpr int kB = 256, kPcBlk = 16;
""" + _cut("pcg.h", r"^struct PcState \{") + _cut("kernels_pcg.hip", r"^__global__ .*void k_pc_block\(") + f"""
int main() {{
    const int m = 300, K = {K}, k0 = {k0}, kb = k0 & ~3;
    std::vector<double> L((size_t)m * K), wb((size_t)K * kPcBlk), acc((size_t)4 * kPcBlk * m, -1.0);
    for (size_t i = 0; i < L.size(); ++i) L[i] = (double)(i * 37 % 101) - 50;
    for (size_t i = 0; i < wb.size(); ++i) wb[i] = (double)(i * 53 % 97) - 48;
    std::vector<int32_t> pos(m);
    for (int j = 0; j < m; ++j) pos[j] = (j + 7) % m;
    std::vector<PcState> st(1);
    st[0] = PcState{{}};
    st[0].k = st[0].k0 = k0;
    for (blockIdx.x = 0; blockIdx.x < 2; ++blockIdx.x)
        for (threadIdx.x = 0; threadIdx.x < kB; ++threadIdx.x)
            k_pc_block(m, st.data(), pos.data(), wb.data(), L.data(), acc.data());
    for (int j = 0; j < m; ++j)
        for (int c = 0; c < kPcBlk; ++c)
            for (int q = 0; q < 4; ++q) {{
                double s = 0.0;
                for (int r = q; r < kb; r += 4) s += L[(size_t)r * m + j] * wb[r * kPcBlk + c];
                if (acc[(size_t)(4 * c + q) * m + j] != (pos[j] < k0 ? -1.0 : s)) return 1;
            }}
    return 0;
}}
""")


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_column_chunk_places_far_columns(tmp_path):
    """k_csc_ts takes a column's part of a chunk of nonzeros between two places in
    it: both inside the chunk, also for a column that begins or ends more than
    2^31 nonzeros from it."""
    text = open(os.path.join(CSRC, "kernels_pcg.hip")).read()
    assert re.search(r"lo = chunk_place\(b, c0\), hi = chunk_place\(e, c0\);", text)
    _run(tmp_path, "constexpr int kCscChunk = 1024;\n" + _cut("kernels_pcg.hip", r"^__device__ inline int chunk_place\(") + """
int main() {
    const int64_t far[] = {0, 1, 1023, 1024, 1025, 2147483647ll, 2147483648ll, 2147484672ll, 4294967296ll, 4294967297ll,
                           1ll << 40};
    for (int64_t c0 : {0ll, 1024ll, 5000000000ll})
        for (int64_t d : far)
            for (int64_t p : {c0 + d, c0 - d}) {
                const int64_t want = p < c0 ? 0 : p > c0 + kCscChunk ? kCscChunk : p - c0;
                if (chunk_place(p, c0) != want) return 1;
            }
    return 0;
}
""")
