"""The pause after a resident launch that gave up (csrc/backoff.hpp), on the CPU."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def probe(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("backoff") / "probe")
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror",
                    "-I" + os.path.join(ROOT, "insilico_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "backoff_probe.cpp"), "-o", exe], check=True)

    def skips(what):
        """uses that went without before each one that was tried"""
        r = subprocess.run([exe, what], capture_output=True, text=True, check=True, timeout=60)
        return [int(v) for v in r.stdout.split()]
    return skips


@pytest.mark.parametrize("what,want", [
    ("+++", [0, 0, 0]),                               # never gave up: always tried
    ("-+", [0, 16]),                                  # one give-up: 16 uses without
    ("----+", [0, 16, 32, 64, 128]),                  # they go on: the pause doubles
    ("--+-+", [0, 16, 32, 0, 32]),                    # a good end halves it, 32 -> 16 -> 32
    ("--++++-+", [0, 16, 32, 0, 0, 0, 0, 4]),         # 32 -> 2, and 4 after that
    ("-" * 12, [0] + [min(16 << k, 4096) for k in range(11)]),   # up to its most
    ("-+++++-+", [0, 16, 0, 0, 0, 0, 0, 16]),         # forgotten after five good ends
])
def test_pause_after_give_ups(probe, what, want):
    assert probe(what) == want
