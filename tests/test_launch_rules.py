"""The dispatch rules that need no device (launch_rules.h), evaluated by a host program at the lines they draw."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "provenloop_amd", "csrc")


@pytest.fixture(scope="module")
def evaluate(tmp_path_factory):
    """evaluate(["expression", ...]) -> their values, as integers."""

    def run(exprs):
        d = tmp_path_factory.mktemp("rules")
        src, exe = d / "rules.cpp", d / "rules"
        src.write_text('#include "launch_rules.h"\n#include <stdio.h>\nint main() {\n'
                       + "".join(f'  printf("%lld\\n", (long long)({e}));\n' for e in exprs) + "}\n")
        subprocess.run(["g++", "-std=c++20", "-Wall", "-Werror", "-I", CSRC, str(src), "-o", str(exe)], check=True)
        return [int(v) for v in subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout.split()]

    return run


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


def test_encodes_fill_two_workgroups_per_cu(evaluate):
    cases = [(13, 1), (13, 64), (13, 255), (13, 256), (14, 28), (14, 64), (14, 128), (14, 672), (15, 28), (15, 64), (10, 1)]
    assert evaluate([f"th::encode_parts_log({n}, {j})" for n, j in cases]) == [3, 3, 2, 1, 4, 3, 2, 2, 4, 3, 0]
