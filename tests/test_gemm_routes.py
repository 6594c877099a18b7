"""Which kernel a GEMM call takes, asked of plan_gemm (csrc/gemm.hip) on the host.

tests/host/gemm_plan.cpp is gemm.hip compiled for the host alone: the plan of any
shape, alignment and scratch capacity, without a GPU and without memory behind
the addresses. Shapes past the kernels' 32-bit offsets are pinned to the
kernels that hold 64-bit ones.
"""

from __future__ import annotations

import os
import subprocess
from pathlib import Path

import pytest

from test_gpu_ops import FEW_TILES, KSPLIT_TILES, ONE_ROUND, SPLIT_TILES
from test_shared_stream_threads import KSPLIT_MNK, SPLIT_MNK

HERE = Path(__file__).resolve().parent
REPO = HERE.parent
CSRC = REPO / "orin-cuda-operator-library_amd" / "csrc"
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


@pytest.fixture(scope="module")
def plans(tmp_path_factory):
    """plans(cases) -> one dict per (dtype, m, n, k[, a_off, b_off, capacity])."""
    out = tmp_path_factory.mktemp("gemm_plan")
    obj, exe = out / "gemm_plan.o", out / "gemm_plan"
    subprocess.run([HIPCC, "-O1", "-fPIC", "-std=c++17", "--offload-arch=gfx950",
                    "--offload-host-only", "-fuse-cuid=none", "-x", "hip",
                    f"-I{REPO / 'include'}", f"-I{CSRC}", "-c",
                    str(HERE / "host" / "gemm_plan.cpp"), "-o", str(obj)],
                   check=True, capture_output=True, text=True, timeout=300)
    # The launches' symbols stay unresolved: a plan calls none of them.
    subprocess.run(["g++", str(obj), "-Wl,--unresolved-symbols=ignore-all", "-o", str(exe)],
                   check=True, capture_output=True, text=True, timeout=120)

    def ask(cases):
        text = "".join(" ".join(map(str, (*c, *(0, 0, 0)[len(c) - 4:]))) + "\n" for c in cases)
        proc = subprocess.run([str(exe)], input=text, capture_output=True, text=True, check=True,
                              timeout=60)
        answers = [{key: value if key == "kind" else int(value) for key, value in
                    (word.split("=") for word in line.split())}
                   for line in proc.stdout.splitlines()]
        assert len(answers) == len(cases)
        return answers

    return ask


def test_few_rows_past_the_offset_limits(plans):
    """K from 2^25 (fp16) / 2^23 (fp32) or N from 2^24 on, past the offsets of the
    wavefront-split kernel: up to 32 / 64 aligned rows stream B once on the skinny
    kernels; one row more, or rows of B off the vector, go to the narrow kernel
    where N <= 16."""
    cases, want = [], []
    for dtype, most, first, limit in (("f16", 32, 5, 1 << 25), ("f32", 64, 9, 1 << 23)):
        for m in (1, first - 1, first, 16, 17, most):
            for n, k in ((16, limit), (8, limit + 64), ((1 << 24) + 8, 72)):
                cases.append((dtype, m, n, k))
                want.append(("skinny", m >= first))
        cases += [(dtype, most + 1, 16, limit), (dtype, 20, 5, limit)]
        want += [("narrow", None)] * 2
        # just below the limits the wavefront-split kernel keeps the call
        cases += [(dtype, 20, 16, limit - 64), (dtype, most, 64, limit - 64)]
        want += [("split", None)] * 2
    for case, plan, (kind, mfma) in zip(cases, plans(cases), want):
        assert plan["kind"] == kind, (case, plan)
        if mfma is not None:
            assert plan["mfma"] == mfma, (case, plan)


def _check(plans, routes):
    """routes: (call, what its plan must hold)."""
    for (case, want), plan in zip(routes, plans([case for case, _ in routes])):
        assert {key: plan.get(key) for key in want} == want, (case, plan)


def test_eight_tiles_split_past_sixteen(plans):
    """Eight 64-column tiles on 16 splits of K leave half the CUs idle: a long K is
    split further, a shorter one is not."""
    _check(plans, [(("f16", 16, 512, 262144), dict(kind="split", fm=1, splits=54)),
                   (("f16", 3, 512, 262144), dict(kind="split", fm=1, splits=54)),
                   (("f16", 16, 576, 262144), dict(kind="split", fm=1, splits=16)),
                   (("f16", 5, 16, 1 << 20), dict(kind="split", fm=1, splits=181)),
                   (("f16", 9, 450, 6464), dict(kind="split", fm=1, splits=16)),
                   (("f16", 65, 256, 10193), dict(kind="split", fm=2, splits=16))])


def test_fp32_tile_heights(plans):
    """fp32 16-row tiles in several rounds cost more on a long K, where they do not
    run by default; 96-row tiles, which hold no total of short chains, take up to
    9216 of K each."""
    _check(plans, [(("f32", 96, 12288, 12288), dict(kind="split", fm=3, splits=1)),
                   (("f32", 64, 12288, 12288), dict(kind="split", fm=4, splits=1)),
                   (("f32", 104, 8960, 2240), dict(kind="split", fm=1, splits=1)),
                   (("f32", 2564, 1792, 12352), dict(kind="split", fm=3, splits=1)),
                   (("f32", 96, 12288, 1024), dict(kind="split", fm=6, splits=1)),
                   (("f32", 1000, 1000, 1000), dict(kind="split", fm=4, splits=1))])


def test_few_rows_from_memory(plans):
    """B past the Infinity Cache: each kernel where it draws the faster stream
    (measured times beside the rules: row_stream_ns, skinny_mfma_faster and
    skinny::applies), and the cached calls as they were."""
    _check(plans, [(("f16", 24, 8704, 12288), dict(kind="skinny", mfma=1)),
                   (("f16", 8, 12288, 12288), dict(kind="skinny", mfma=1)),
                   (("f16", 16, 50264, 4096), dict(kind="split", fm=1, splits=1)),
                   (("f32", 32, 8704, 12288), dict(kind="skinny", mfma=1)),
                   (("f16", 3, 12288, 12288), dict(kind="skinny", mfma=0)),
                   (("f16", 3, 28672, 8192), dict(kind="skinny", mfma=0)),
                   (("f16", 3, 6144, 12288), dict(kind="split", fm=1, splits=5)),
                   # B's rows no multiple of 512 bytes apart
                   (("f16", 3, 12224, 4416), dict(kind="split", fm=1)),
                   (("f16", 4, 13376, 9408), dict(kind="split", fm=1)),
                   (("f32", 32, 8640, 6133), dict(kind="split")),
                   (("f16", 9, 8096, 8192), dict(kind="split", fm=1, splits=4)),
                   (("f32", 29, 10880, 12929), dict(kind="split")),
                   (("f32", 32, 8704, 2688), dict(kind="split")),
                   (("f16", 24, 11008, 12288), dict(kind="split", fm=2, splits=1)),
                   (("f32", 24, 12288, 12288), dict(kind="split", fm=2, splits=1)),
                   (("f16", 16, 16384, 8192), dict(kind="split", fm=1, splits=1)),
                   (("f16", 16, 5120, 13824), dict(kind="split", fm=1, splits=6)),
                   (("f32", 16, 8704, 12288), dict(kind="split", fm=1, splits=3)),
                   # B off 16 bytes: ksplit_kernel at any alignment
                   (("f16", 8, 12288, 12288, 0, 1), dict(kind="split", fm=1)),
                   (("f16", 16, 11008, 4096), dict(kind="split", fm=1, splits=1)),
                   (("f16", 16, 4096, 4096), dict(kind="split", fm=1, splits=3))])


def test_one_round_tiles_keep_their_xcd_order(plans):
    """fp16 grids of one round of 128 x 256 tiles whose count is no multiple of the
    eight XCDs, where that of the 128 x 128 ones is: the latter, up to 1024 rows."""
    _check(plans, [(("f16", 386, 10981, 3904), dict(kind="dma", rows=128, one_round=None)),
                   (("f16", 771, 7168, 4224), dict(kind="dma", rows=128, one_round=None)),
                   (("f16", 768, 7168, 4224), dict(kind="dma", rows=128, one_round=1)),
                   (("f16", 2064, 3072, 7360), dict(kind="dma", rows=128, one_round=1)),
                   (("f16", 2000, 3000, 512), dict(kind="dma", rows=128, one_round=1)),
                   (("f16", 3000, 3000, 3000), dict(kind="dma", rows=192, one_round=1))])


def test_gpu_tests_reach_the_instances_they_name(plans):
    """The shapes of tests/test_gpu_ops.py that stand for an instance run it, so a
    change of an estimate cannot move one off its kernel unseen."""
    _check(plans, [((dtype, m, n, k), dict(kind="split", fm=fm, deep=deep, edge=edge))
                   for dtype, m, n, k, fm, deep, edge in KSPLIT_TILES])
    seen = {(c[0], *c[4:]) for c in KSPLIT_TILES}
    assert {("f16", fm, deep, edge) for fm in range(2, 7) for deep in (0, 1)
            for edge in (0, 1)} - {("f16", 2, 0, 0)} <= seen
    assert {("f32", fm, 0, edge) for fm in (4, 5, 6) for edge in (0, 1)} <= seen
    split_tiles = [*SPLIT_TILES, ("f16", *SPLIT_MNK)]
    for case, plan in zip(split_tiles, plans(split_tiles)):
        assert plan["kind"] == "dma" and plan["rows"] == 128 and plan["tail"] > 1, (case, plan)
    # the workspace, stream and graph tests' users of the arena
    _check(plans, [(("f16", *KSPLIT_MNK), dict(kind="split", splits=7)),
                   (("f16", 16, 4096, 4096), dict(kind="split", splits=3)),
                   (("f16", 24, 8704, 6144), dict(kind="skinny", mfma=1))])
    cases = [(dtype, *c) for c in FEW_TILES for dtype in ("f16", "f32")]
    splits = set()
    for case, plan in zip(cases, plans(cases)):
        assert plan["kind"] == "split" and plan["splits"] > 16, (case, plan)
        splits.add(plan["splits"])
    assert len(splits) >= 4, splits
    got = plans([("f16", *c) for c in ONE_ROUND])
    assert [p["rows"] * p.get("one_round", 0) for p in got] == [128] * 3 + [192] * 5 + [0, 0], got
