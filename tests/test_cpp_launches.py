"""What the C API launches, over a stand-in for the HIP runtime (tests/cpp/launch_trace.cpp): grids,
workgroups and LDS of every launch, and what a call returns when one of them fails."""
import os
import subprocess

import pytest

from anime4kcpp_amd import _native

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


@pytest.fixture(scope="module")
def trace(tmp_path_factory):
    """trace(commands): [(return code, [(kernel, grid x, grid y, block x, LDS bytes), ...]), ...]"""
    exe = str(tmp_path_factory.mktemp("trace") / "launch_trace")
    libdir = os.path.dirname(_native.LIB_PATH)
    subprocess.run(["g++", "-std=c++17", "-O1", "-rdynamic", "-I" + os.path.join(ROOT, "include"), "-I/opt/rocm/include",
                    os.path.join(HERE, "cpp", "launch_trace.cpp"), "-L" + libdir, "-lac_hip", "-Wl,-rpath," + libdir, "-o", exe],
                   check=True, capture_output=True, text=True)

    def run(commands):
        r = subprocess.run([exe], input="\n".join(commands), capture_output=True, text=True, timeout=120)
        assert r.returncode == 0, r.stderr
        answers = []
        for line in r.stdout.splitlines():
            f = line.split()
            if f[0] == "rc":
                answers.append((int(f[1]), []))
            elif f[0] != "end":
                answers[-1][1].append((f[0],) + tuple(int(v) for v in f[1:]))
        return answers
    return run


PASSES = ["layers 1 1920 1080", "layers 1 128 96", "net8 8 0 1 1920 1080", "net8 7 0 1 200 100", "net8 18 1 1 640 480",
          "net8 4 2 1 640 480", "art 16 4 1 640 480", "art 32 3 516 200 100", "fsr 8 4 1 640 480", "fsr 8 3 2 640 480",
          "fsr 16 4 514 640 480", "batch_layers 5 200 100", "batch 1 0 5 200 100", "legacy 1 -1 1 200 100"]


@pytest.mark.parametrize("command", PASSES)
def test_failed_launch_is_reported(trace, command):
    """A pass whose k-th launch fails returns an error, for every k."""
    (rc, launches), = trace([command])
    assert rc == 0 and launches
    for k in range(len(launches)):
        (rc, _), = trace([f"fail {k}", command])
        assert rc == -5, f"launch {k} of {len(launches)} failed unnoticed"


RING, IMG = 6 * 80 * 16, 6 * 84 * 4   # LDS bytes of a layer's ring of six rows and of the source rows


@pytest.mark.parametrize("blocks", range(1, 65))
def test_acnet8_streamed_lds(trace, blocks):
    """The 16-bit ACNet<8> launches own every LDS byte they read.  The rings start 16 bytes in; the last
    layer of a launch of n reads 16-pixel segments whole, five of them below 8 layers and four from
    there on: the last lane's patch ends at pixel n - 1 + 15 + 16 (segments - 1) + 2 of a row of 80."""
    for precision in (1, 2):
        (rc, launches), = trace([f"net8 {blocks} {precision} 1 300 200"])
        assert rc == 0
        done = 0
        for k, (_, _, _, _, lds) in enumerate(launches):
            take = -(-(blocks - done) // (len(launches) - k))
            n, done = take + (k == len(launches) - 1), done + take
            segments = 5 if 80 - 2 * n > 64 else 4
            last_row = 16 + (n - 1) * RING + 5 * 80 * 16
            assert last_row + (n - 1 + 15 + 16 * (segments - 1) + 2 + 1) * 16 <= lds, (k, n)
            assert 16 + n * RING + 16 + (IMG if k == 0 else 0) <= lds, (k, n)
        assert done == blocks


WIDE = [f"{c} {w} {h}" for w, h in [(360000000, 1), (400000000, 2), (1 << 29, 1)]
        for c in ["net8 8 1 1", "net8 18 2 1", "net8 64 1 1", "net8 4 0 1", "net8 8 0 1", "net8 18 0 516"]]
WIDE += ["legacy 1 -1 1 360000000 1", "legacy 2 0 516 500000000 1", "layers 1 536870912 1", "batch_layers 3 268435456 1"]


@pytest.mark.parametrize("command", WIDE)
def test_very_wide_images(trace, command):
    """Images of more columns than 2^32 threads make in strips: accepted, in a grid whose dimensions each
    hold fewer than 2^32 threads (the stand-in refuses others, as the runtime does)."""
    (rc, launches), = trace([command])
    assert rc == 0 and launches
