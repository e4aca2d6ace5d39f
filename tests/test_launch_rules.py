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
