"""The decode launch's plan (csrc/decode_plan.h, host code without HIP),
compiled here and run on the CPU: tests/native/decode_plan_check.cpp walks
shapes, split hints and workspace sizes.  The registers and LDS the plan
counts with are compared with those of the kernels built here, and its choices
with the measured times of profiles/decode_plan_timings.csv."""

from __future__ import annotations

import os
import re
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(ROOT, "paged_tierkv_amd", "csrc")
INCLUDE = os.path.join(ROOT, "include")
OBJECT = os.path.join(ROOT, "paged_tierkv_amd", "_build", "decode_attention.hip.o")
LLVM = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin")


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    exe = tmp_path_factory.mktemp("plan") / "decode_plan_check"
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-Werror", "-I", CSRC, "-I", INCLUDE,
                    os.path.join(HERE, "native", "decode_plan_check.cpp"), "-o", str(exe)], check=True)
    return str(exe)


@pytest.fixture(scope="module")
def report(check):
    return subprocess.run([check], capture_output=True, text=True, timeout=120)


def test_plans_fit_and_deterministic_plans_follow_the_shape(report):
    assert report.returncode == 0, report.stdout + report.stderr
    assert " bad 0" in report.stdout and "(two plans 0)" not in report.stdout


def test_chosen_plans_are_near_the_fastest_measured(check):
    """Over 1,336 shapes timed with every plan: the chosen plan is within 1 %
    of the fastest on average and, against the plain rule (about 2048 waves,
    the most per workgroup), more than 3 % slower in few and never by much."""
    rows = []
    with open(os.path.join(ROOT, "profiles", "decode_plan_timings.csv")) as f:
        for line in f:
            if line[0].isdigit():
                *shape, _, _, times = line.split(",")
                rows.append((shape, {k: float(t) for k, t in (x.split("=") for x in times.split())}))
    assert len(rows) == 1336
    code = {"ref_u8": "0", "absmax_i8": "1"}
    text = "\n".join(" ".join(code.get(x, x) for x in shape) for shape, _ in rows)
    out = subprocess.run([check, "plans"], input=text, capture_output=True, text=True, check=True).stdout.split()
    loss, over = [], []
    for (shape, times), plan, plain in zip(rows, out[::2], out[1::2]):
        loss.append(times[plan] / min(times.values()))
        if plain in times:
            over.append((times[plan] / times[plain], shape, plan, plain))
    assert sum(loss) / len(loss) <= 1.010
    assert len(over) > 1300 and sum(r > 1.03 for r, *_ in over) <= 0.025 * len(over)
    assert max(over)[0] <= 1.15, max(over)


@pytest.mark.skipif(not os.path.exists(OBJECT) or not os.path.exists(os.path.join(LLVM, "llvm-readelf")),
                    reason="no build of the decode kernel here")
def test_occupancy_is_that_of_the_built_kernels(report, tmp_path):
    """Every instantiation's registers allow the waves per SIMD the plan takes
    (the least over the instantiations of a kind), and its LDS is covered."""
    fat, code = tmp_path / "fat.bin", tmp_path / "decode.co"
    subprocess.run([os.path.join(LLVM, "llvm-objcopy"), f"--dump-section=.hip_fatbin={fat}", OBJECT, os.devnull],
                   check=True)
    subprocess.run([os.path.join(LLVM, "clang-offload-bundler"), "--unbundle", "--type=o", f"--input={fat}",
                    "--targets=hipv4-amdgcn-amd-amdhsa--gfx950", f"--output={code}"], check=True)
    notes = subprocess.run([os.path.join(LLVM, "llvm-readelf"), "--notes", str(code)], check=True,
                           capture_output=True, text=True).stdout
    waves, lds, seen = {}, 0, 0
    for part in notes.split(".agpr_count:")[1:]:
        name = re.search(r"tiered_decode_kernelILi(\d+)ELi(\d+)ELb([01])E", part)
        if name is None:
            continue
        seen += 1
        regs = int(re.search(r"\.vgpr_count:\s+(\d+)", part)[1])
        lds = max(lds, int(re.search(r"\.group_segment_fixed_size:\s+(\d+)", part)[1]))
        kind = tuple(int(x) for x in name.groups())
        waves[kind] = min(waves.get(kind, 8), 512 // (-(-regs // 8) * 8))
    assert seen == 128 and len(waves) == 8
    want = {tuple(int(x) for x in m.groups()[:3]): int(m[4])
            for m in re.finditer(r"^waves (\d+) (\d+) (\d+) (\d+)$", report.stdout, re.M)}
    assert waves == want
    assert lds <= int(re.search(r"^static_lds (\d+)$", report.stdout, re.M)[1]) <= lds + 256
