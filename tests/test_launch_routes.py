"""Which kernels softmax, RMSNorm and attention calls launch, asked on the host.

tests/host/launches.cpp holds the library's sources compiled for the host alone and
answers the HIP calls of a launch itself: a call's kernels and grids, without a GPU
and without memory behind the addresses.
"""

from __future__ import annotations

import os
import re
import subprocess
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

import pytest

HERE = Path(__file__).resolve().parent
REPO = HERE.parent
CSRC = REPO / "orin-cuda-operator-library_amd" / "csrc"
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


@pytest.fixture(scope="module")
def launches(tmp_path_factory):
    """launches(calls) -> per call, (kernel name, its template integers, grid) of
    each launch."""
    out = tmp_path_factory.mktemp("launches")

    def compile_host(src):
        obj = out / (src.name + ".o")
        subprocess.run([HIPCC, "-O1", "-fPIC", "-std=c++17", "--offload-arch=gfx950",
                        "--offload-host-only", "-fuse-cuid=none", "-x", "hip",
                        f"-I{REPO / 'include'}", f"-I{CSRC}", "-c", str(src), "-o", str(obj)],
                       check=True, capture_output=True, text=True, timeout=300)
        return str(obj)

    sources = [CSRC / f"{name}.hip" for name in ("softmax", "rmsnorm", "attention", "scratch")]
    with ThreadPoolExecutor(5) as pool:
        objs = list(pool.map(compile_host, [*sources, HERE / "host" / "launches.cpp"]))
    exe = out / "launches"
    # The HIP calls that no launch makes stay unresolved.
    subprocess.run(["g++", *objs, "-Wl,--unresolved-symbols=ignore-all",
                    "-Wl,--allow-multiple-definition", "-o", str(exe)],
                   check=True, capture_output=True, text=True, timeout=120)

    def ask(calls):
        text = "".join(" ".join(map(str, c)) + "\n" for c in calls)
        proc = subprocess.run([str(exe)], input=text, capture_output=True, text=True, check=True,
                              timeout=60)
        answers = []
        for line in proc.stdout.splitlines():
            status, *kernels = line.split()
            assert status == "0", line
            answers.append([(re.search(r"\d([a-z_]+_kernel)I", k).group(1),
                             [int(i) for i in re.findall(r"Li(\d+)E", k.split(":")[0])],
                             tuple(map(int, k.split(":")[1].split("x")))) for k in kernels])
        assert len(answers) == len(calls)
        return answers

    return ask


def test_few_rows_split_or_not(launches):
    """Fewer than 64 rows of 4097 to 32768 columns: one workgroup per row up to the
    width where two split launches are the faster ones, on both sides of each."""
    one, split = 1, 2
    cases = []
    for op in ("softmax", "rmsnorm"):
        for rows in (1, 4, 5, 16, 17, 63):
            for dtype in ("f16", "f32"):
                if dtype == "f16":
                    same, mixed = 32768, 16384
                elif op == "softmax":
                    same, mixed = 24576, 16384
                else:
                    same, mixed = 24576 if rows <= 4 else 16384, 16384
                for offsets, width in (((0, 0), same), ((3, 3), same), ((1, 0), mixed)):
                    cases += [((op, dtype, rows, 4097, *offsets), one),
                              ((op, dtype, rows, width, *offsets), one),
                              ((op, dtype, rows, width + 1, *offsets), split)]
        cases += [((op, "f32", 64, 32768, 0, 0), one), ((op, "f16", 64, 32768, 1, 0), one)]
    for (call, want), got in zip(cases, launches([call for call, _ in cases])):
        assert len(got) == want, (call, got)
        assert (want == split) == ("split" in got[0][0]), (call, got)


def _instances(launches, calls):
    """[D, groups, wavefronts, tile keys, computed dims, row blocks] per call."""
    got = launches([("attention", *call) for call in calls])
    assert all(len(g) == 1 and g[0][0] == "attention_dma_kernel" for g in got), got
    return [g[0][1] for g in got]


def test_attention_48_row_blocks(launches):
    """fp32 D64 with every key visible: 48 rows per wavefront only where four key
    groups walk (nearly) half the tiles of two, on both sides of each line."""
    calls = [(32, 257, False), (32, 288, False), (32, 289, True), (24, 512, False),
             (64, 192, False), (48, 193, True), (48, 256, False), (42, 256, True),
             (80, 128, False), (16, 513, True), (16, 768, True), (16, 769, False),
             (1, 8193, True), (8, 1000, False)]
    got = _instances(launches, [("f32", 1, h, s, 64, 0) for h, s, _ in calls])
    for (h, s, want), inst in zip(calls, got):
        assert (inst == [64, 4, 1, 32, 64, 3]) == want, (h, s, inst)


def test_attention_one_round_of_32_row_blocks(launches):
    """fp16: 32-row blocks on four key groups wherever their grid is one round."""
    for d, layout, dims in ((128, 128, 128), (96, 128, 96), (64, 64, 64)):
        calls = [(12, 640, 0, True), (8, 1024, 0, True), (8, 1025, 0, False),
                 (8, 1024, 1, True), (4, 1500, 1, True), (1, 8192, 0, True),
                 (1, 8193, 0, False), (12, 1024, 0, False)]
        got = _instances(launches, [("f16", 1, h, s, d, c) for h, s, c, _ in calls])
        for (h, s, c, want), inst in zip(calls, got):
            assert (inst == [layout, 4, 1, 32, dims, 2]) == want, (d, h, s, c, inst)


def test_attention_one_key_tile(launches):
    """fp16, up to 32 tokens (one key tile) on many heads: one group per block."""
    calls = [(256, 17, False), (256, 32, False), (129, 1, False), (128, 33, True),
             (12, 16, True)]
    got = _instances(launches, [("f16", 1, h, s, 128, 0) for h, s, _ in calls])
    for (h, s, want), inst in zip(calls, got):
        assert (inst == [128, 4, 1, 32, 128, 2]) == want, (h, s, inst)
        if h > 128:
            assert inst == [128, 1, 2, 32, 128, 2], (h, s, inst)
