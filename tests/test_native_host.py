"""Host-side checks of the native code's own rules: small C++ programs over its headers, built with g++."""
import os
import subprocess


ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "tribit_amd", "csrc")
ROCM = ["-D__HIP_PLATFORM_AMD__", "-isystem", "/opt/rocm/include"]


def run_cpp(tmp_path, source, includes=()):
    """Builds `source` against the library's headers, runs it and returns its output lines."""
    src, exe = tmp_path / "check.cpp", tmp_path / "check"
    src.write_text(source)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", *includes, "-I", CSRC, str(src), "-o", str(exe)], check=True,
                   timeout=300)
    return subprocess.run([str(exe)], check=True, timeout=300, capture_output=True, text=True).stdout.split("\n")


ENDS = r"""
#include "ends.hpp"
#include <cstdio>
int main() {
  const uint32_t ends[] = {0u, 1u, (1u << 17) - 1, 1u << 17, (1u << 17) + 1, 1u << 31, 4294901760u, 4292870145u, 0xFFFFFFFEu, 0xFFFFFFFFu};
  for (const uint64_t m : {1ull << 18, 16384001ull, 2147450880ull, 0x7FFFFFFFull}) {
    const uint32_t chunk = tb::end_chunk(m, 256);
    for (const uint32_t e : ends) std::printf("%u %u %u\n", e, chunk, tb::end_chunks(e, chunk));
  }
}
"""


def test_counting_tasks_cover_every_endpoint(tmp_path):
    """Chunks of a group's endpoints up to the most that 2^31 - 1 edges have (the complete graph on 65,536 ids among
    them): as many as whole numbers give, none lost to 32 bits."""
    rows = [list(map(int, line.split())) for line in run_cpp(tmp_path, ENDS, ROCM) if line]
    assert len(rows) == 40
    for ends, chunk, got in rows:
        assert 1 << 17 <= chunk <= 1 << 21
        assert got == -(-ends // chunk), (ends, chunk)
