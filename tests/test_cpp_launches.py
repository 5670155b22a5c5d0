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
    """trace(commands): [(return code, [(kernel, grid x, grid y, block x, LDS bytes, strips, rows), ...]), ...]"""
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
        for k, (_, _, _, _, lds, _, _) in enumerate(launches):
            take = -(-(blocks - done) // (len(launches) - k))
            n, done = take + (k == len(launches) - 1), done + take
            segments = 5 if 80 - 2 * n > 64 else 4
            last_row = 16 + (n - 1) * RING + 5 * 80 * 16
            assert last_row + (n - 1 + 15 + 16 * (segments - 1) + 2 + 1) * 16 <= lds, (k, n)
            assert 16 + n * RING + 16 + (IMG if k == 0 else 0) <= lds, (k, n)
        assert done == blocks


WIDE = [f"{c} {w} {h}" for w, h in [(360000000, 1), (400000000, 2), (1 << 29, 1)]
        for c in ["net8 8 1 1", "net8 18 2 1", "net8 64 1 1", "net8 4 0 1", "net8 8 0 1", "net8 18 0 516"]]
WIDE += ["legacy 1 -1 1 360000000 1", "legacy 2 0 516 500000000 1", "layers 1 536870912 1", "batch_layers 3 268435456 1",
         "art 32 4 1 536870912 1"]


@pytest.mark.parametrize("command", WIDE)
def test_very_wide_images(trace, command):
    """Images of more columns than 2^32 threads make in strips: accepted, in a grid whose dimensions each
    hold fewer than 2^32 threads (the stand-in refuses others, as the runtime does)."""
    (rc, launches), = trace([command])
    assert rc == 0 and launches


# Batches of u8 images (widths and heights in turn) and the us of one FP16 launch on an MI355X at heights of
# strips from 8 to 256 rows
BATCHES16 = [
    (
     "762 341 276 621 296 442 967 942 294 278 345 880 255 347 289 298 550 325 461 760 748 465 ",
     {8: 188, 12: 151, 16: 133, 20: 123, 24: 116, 32: 109, 40: 112, 48: 103, 64: 107, 80: 112, 96: 118, 128: 104, 192: 123, 256: 122}),
    (
     "474 265 148 84 1478 655 122 384 562 1088 135 151 99 378 1144 613 84 183 68 91 274 88 131 119 217 918 116 409 201 140 ",
     {8: 184, 12: 148, 16: 132, 20: 121, 24: 114, 32: 105, 40: 109, 48: 97, 64: 105, 80: 110, 96: 117, 128: 105, 192: 139, 256: 122}),
    (
     "36 174 69 468 430 83 202 148 79 123 110 136 577 299 38 97 605 327 206 232 260 55 114 78 60 264 38 58 281 485 84 429 404 "
     "54 516 56 138 44 45 245 413 47 90 209 199 51 268 47 545 247 244 529 69 62 219 486 542 361 204 99 354 225 463 322 146 233 ",
     {8: 132, 12: 108, 16: 97, 20: 94, 24: 88, 32: 85, 40: 84, 48: 87, 64: 90, 80: 76, 96: 83, 128: 99, 192: 95, 256: 118}),
]


@pytest.mark.parametrize("sizes,us", BATCHES16, ids=["11", "15", "33"])
def test_batch_strip_height(trace, sizes, us):
    """The height that the 16-bit batch takes for its strips is, by the measured times, within 12% of the
    best one (the times of one height differ by up to 4% from run to run)."""
    (rc, launches), = trace(["images 1 " + sizes])
    assert rc == 0
    assert us[launches[0][6]] <= 1.12 * min(us.values()), launches[0][6]


# The same for achip_pass_batch_layers, by (layers per launch, rows)
BATCHES32 = [
    ("300 200 " * 48,
     {(2, 8): 406, (2, 12): 376, (2, 16): 372, (2, 20): 353, (2, 24): 371, (2, 28): 371, (2, 32): 390, (2, 40): 322, (2, 48): 373, (2, 64): 393, (2, 96): 453,
      (4, 8): 581, (4, 12): 500, (4, 16): 465, (4, 20): 439, (4, 24): 435, (4, 28): 438, (4, 32): 428, (4, 40): 410, (4, 48): 440, (4, 64): 491, (4, 96): 494}),
    (
     "339 399 732 849 242 307 977 285 667 398 657 927 594 439 394 632 639 452 495 553 356 314 582 277 609 842 878 352 456 1021 "
     "411 1138 324 896 252 680 847 563 644 1006 1146 314 541 251 430 297 304 636 270 301 240 858 347 265 632 737 642 562 551 "
     "739 386 898 709 921 969 894 538 540 ",
     {(2, 8): 1532, (2, 12): 1392, (2, 16): 1360, (2, 20): 1336, (2, 24): 1319, (2, 28): 1296, (2, 32): 1279, (2, 40): 1292, (2, 48): 1268, (2, 64): 1260, (2, 96): 1300,
      (4, 8): 2076, (4, 12): 1756, (4, 16): 1604, (4, 20): 1512, (4, 24): 1441, (4, 28): 1409, (4, 32): 1383, (4, 40): 1345, (4, 48): 1320, (4, 64): 1315, (4, 96): 1331}),
    (
     "467 599 669 909 596 871 136 337 910 494 833 162 339 214 397 422 132 201 229 861 629 178 672 171 462 167 128 784 198 200 "
     "987 785 234 945 393 524 196 906 538 955 821 238 271 181 173 147 240 449 ",
     {(2, 8): 735, (2, 12): 685, (2, 16): 669, (2, 20): 657, (2, 24): 649, (2, 28): 639, (2, 32): 634, (2, 40): 642, (2, 48): 643, (2, 64): 675, (2, 96): 689,
      (4, 8): 992, (4, 12): 843, (4, 16): 772, (4, 20): 729, (4, 24): 706, (4, 28): 696, (4, 32): 685, (4, 40): 678, (4, 48): 677, (4, 64): 676, (4, 96): 725}),
]


@pytest.mark.parametrize("sizes,us", BATCHES32, ids=["48", "34", "24"])
def test_batch_layers_strips(trace, sizes, us):
    """Layers per launch and heights: within 10% of the best measured."""
    (rc, launches), = trace(["images_layers " + sizes])
    assert rc == 0
    cut = 8 // len(launches), launches[0][6]
    assert us[cut] <= 1.1 * min(us.values()), cut


# u8 passes and their us by the height of strips, in the launches that are named (the second and third of
# FSRCNNX<8>: its two-layer ones)
HEIGHTS16 = [("legacy 1 -1 1 800 600", 0, {16: 21.8, 18: 22.4, 20: 23.0, 22: 24.2, 32: 23.7}),
             ("legacy 1 -1 1 960 540", 0, {16: 21.6, 18: 22.2, 20: 23.0, 32: 23.7, 36: 25.1}),
             ("legacy 2 -1 1 644 716", 0, {16: 22.5, 18: 23.3, 20: 24.3, 32: 23.7, 36: 25.1}),
             ("legacy 1 -1 1 1920 1080", 0, {36: 58.0, 48: 59.9, 64: 46.9, 72: 50.2, 80: 54.7}),
             ("fsr 8 4 1 640 360", 1, {4: 41.4, 6: 42.3, 8: 41.9, 10: 46.4, 16: 45.6}),
             ("fsr 8 4 1 327 641", 2, {4: 42.0, 6: 43.1, 8: 41.8, 10: 45.6, 16: 44.8}),
             ("fsr 8 4 1 500 400", 1, {4: 39.2, 6: 40.5, 8: 41.0, 10: 45.6, 16: 45.0}),
             ("net8 8 1 1 800 600", 0, {16: 33.5, 18: 34.8, 20: 36.4, 32: 33.8, 36: 35.6})]


@pytest.mark.parametrize("command,launch,us", HEIGHTS16)
def test_strip_height(trace, command, launch, us):
    """The height of a pass's strips is, by the measured times, within 5% of the best one."""
    (rc, launches), = trace([command])
    assert rc == 0
    h = int(command.split()[-1])
    got = [t for r, t in us.items() if -(-h // r) == launches[launch][2]]
    assert got and min(got) <= 1.05 * min(us.values()), launches[launch]


def test_tuned_fixed_height_within_its_class(trace):
    """A tuner's verdict for the 16-bit configuration of 128-row strips (99 against 100 us at 1900 x 1900)
    holds for that size, and elsewhere in its size class only where 128 rows cost about what the
    height for the image does; 1100 x 1100 in 128 rows would leave 94 of 256 compute units idle."""
    tuned, same, other, near = trace(["tune 1 1900 1900 100 99", "legacy 1 -1 1 1900 1900", "legacy 1 -1 1 1100 1100",
                                      "legacy 1 -1 1 2040 2040"])
    assert tuned[0] == 1
    assert same[1][0][1:3] == (30, 15)
    assert other[1][0][1:3] == (18, 28)   # 40 rows
    assert near[1][0][1:3] == (32, 16)
    assert trace(["legacy 1 -1 1 1900 1900"])[0][1][0][2] != 15   # a process that tuned nothing


@pytest.mark.parametrize("w,h", [(1920, 1080), (640, 360), (256, 256)])
def test_bench_counts_acnet8_launches(trace, w, h):
    """The launches from which bench.py derives an ACNet<8> pass's HBM bytes are the ones that run."""
    import bench
    precs = ("fp32", "fp16")
    cases = [(p, b) for p in (0, 1) for b in range(1, 25)]
    for (p, b), (rc, launches) in zip(cases, trace([f"net8 {b} {p} 1 {w} {h}" for p, b in cases])):
        assert rc == 0 and len(launches) == bench.acnet8_launches(precs[p], b, w, h), (precs[p], b)
    assert bench.acnet8_bytes("fp16", 8, 1920, 1080) == 5 * 1920 * 1080
    assert bench.acnet8_bytes("fp32", 8, 1920, 1080) == (1 + 1 + 4 + 3 * 64) * 1920 * 1080
