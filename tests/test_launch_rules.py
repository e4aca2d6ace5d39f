"""The dispatch rules and the job lists' ring (launch_rules.h), which need no device, evaluated by host programs."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "provenloop_amd", "csrc")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    """program(body of main) -> the integers it prints."""

    def run(body):
        d = tmp_path_factory.mktemp("rules")
        src, exe = d / "rules.cpp", d / "rules"
        src.write_text('#include "launch_rules.h"\n#include <stdio.h>\n#include <utility>\n#include <vector>\n'
                       "int main() {\n" + body + "}\n")
        subprocess.run(["g++", "-std=c++20", "-Wall", "-Werror", "-I", CSRC, str(src), "-o", str(exe)], check=True)
        return [int(v) for v in subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout.split()]

    return run


@pytest.fixture(scope="module")
def evaluate(program):
    """evaluate(["expression", ...]) -> their values, as integers."""
    return lambda exprs: program("".join(f'  printf("%lld\\n", (long long)({e}));\n' for e in exprs))


def test_small_downloads_wait_in_the_runtime(evaluate):
    """Copies the runtime makes with a kernel (up to 16 KiB) are not polled; the decryptions' 32 KiB to 128 KiB are."""
    sizes = [0, 4, 8, 256, 16 << 10, (16 << 10) + 1, 32 << 10, 64 << 10, 128 << 10, 256 << 10, (256 << 10) + 1]
    got = evaluate([f"th::poll_download({b})" for b in sizes])
    assert got == [0, 0, 0, 0, 0, 1, 1, 1, 1, 1, 0]


def test_decodes_are_cut_into_at_most_one_part_per_cu(evaluate):
    """Parts of 4096 values (8192 at N = 32768, whose parts of 4096 leave a CU one small workgroup), more only while
    the batch has no more parts than the GPU has CUs; every part fits a workgroup of 8 values a thread."""
    cases = [(logn, jobs) for logn in range(10, 16) for jobs in (1, 8, 15, 16, 17, 32, 33, 64, 65, 128, 129, 256, 257, 5000)]
    got = dict(zip(cases, evaluate([f"th::decode_parts_log({n}, {j})" for n, j in cases])))
    base = {10: 0, 11: 0, 12: 0, 13: 1, 14: 2, 15: 2}
    for (logn, jobs), lp in got.items():
        assert base[logn] <= lp <= 4 and 1 << logn >> lp <= 8192
        assert lp == base[logn] or (jobs << lp <= 256 and logn - lp >= 10)
        if lp < 4 and logn - lp > 10:
            assert jobs << (lp + 1) > 256
    assert [got[15, j] for j in (16, 17, 32, 33, 64, 256)] == [4, 3, 3, 2, 2, 2]


def test_decode_threads(evaluate):
    """At most 8 values a thread (dit_stages_reg), at most 1024 threads, a quarter of the values where a CU has room."""
    cases = [(logn, jobs) for logn in range(10, 16) for jobs in (1, 16, 17, 33, 64, 65, 128, 129, 256, 257, 5000)]
    lps = evaluate([f"th::decode_parts_log({n}, {j})" for n, j in cases])
    threads = evaluate([f"th::decode_threads({n}, th::decode_parts_log({n}, {j}), {j})" for n, j in cases])
    for (logn, jobs), lp, t in zip(cases, lps, threads):
        m = 1 << logn >> lp
        assert 64 <= t <= 1024 and t % 64 == 0 and m <= 8 * t
        assert (t == min(1024, m // 4)) == (m <= 2048 or m == 8192 or (lp < 3 and jobs << lp <= 256))


def test_encodes_fill_two_workgroups_per_cu(evaluate):
    cases = [(13, 1), (13, 64), (13, 255), (13, 256), (14, 28), (14, 64), (14, 128), (14, 672), (15, 28), (15, 64), (10, 1)]
    assert evaluate([f"th::encode_parts_log({n}, {j})" for n, j in cases]) == [3, 3, 2, 1, 4, 3, 2, 2, 4, 3, 0]


def test_job_lists_are_not_rewritten_before_a_drain(program):
    """Every place handed out is clear of all the places handed out since the last drain, at the library's capacity
    and at small ones, with lists of mixed sizes; and laps do come round."""
    overlaps, laps = program("""
  long long overlaps = 0, laps = 0;
  unsigned x = 1;
  for (size_t cap : {size_t(512), size_t(768), size_t(4096), size_t(1) << 20}) {
    th::SlotRing ring(cap);
    std::vector<std::pair<size_t, size_t>> queued;  // what kernels may still read
    for (int i = 0; i < 20000; ++i) {
      x = x * 1664525u + 1013904223u;
      const size_t bytes = 1 + (x >> 8) % 512;
      const size_t at = ring.place(bytes, [&] { queued.clear(); ++laps; });
      if (at + bytes > cap || at % 256) ++overlaps;
      if (i < 9000 || cap < 5000)
        for (auto& q : queued) overlaps += at < q.first + q.second && q.first < at + bytes;
      queued.push_back({at, bytes});
    }
  }
  printf("%lld %lld\\n", overlaps, laps);
""")
    assert overlaps == 0 and laps > 1000
