"""The wide GEMM tile (csrc/gemm_wide_kernel.h) compiled for the host against tests/host/hip_on_host.h:
every lane of every workgroup runs on the CPU, and each buffer read is held against the documented range
rule (lane offset below num_records - uniform offset, unsigned) and against the operand it belongs to.
The values that rows past the weight give are never stored, so no output shows a read out of range."""
import os
import re
import subprocess

import pytest

import test_gpu_gemm_wide
from moss_tts import _build

HOST = os.path.join(os.path.dirname(os.path.abspath(__file__)), "host")
_ASM = re.compile(r"\basm( volatile)?\((?:[^()]|\([^()]*\))*\);")  # device instructions, none with an address
_SOURCES = ("common.h", "gemm_wide.h", "gemm_wide_kernel.h", "gemm_wide_w4.hip", "gemm_wide_fp8.hip", "w4g32_gemm.hip")


@pytest.fixture(scope="session")
def gemm_wide_check(tmp_path_factory):
    clang = "/opt/rocm/llvm/bin/clang++"
    if not os.path.exists(clang):
        pytest.skip("clang++ not available")
    d = tmp_path_factory.mktemp("gemm_wide")
    (d / "hip").mkdir()
    (d / "hip" / "hip_runtime.h").write_text(f'#include "{HOST}/hip_on_host.h"\n')
    for name in _SOURCES:
        with open(os.path.join(_build.CSRC, name)) as f:
            (d / name).write_text(_ASM.sub(";", f.read()))
    units = ["gemm_wide_w4.hip", "gemm_wide_fp8.hip", os.path.join(HOST, "gemm_wide_check.cpp")]
    jobs = [subprocess.Popen([clang, "-std=c++17", "-O1", "-w", "-x", "c++", "-I", str(d), "-c", u, "-o", f"{i}.o"], cwd=d,
                             stderr=subprocess.PIPE, text=True) for i, u in enumerate(units)]
    for job in jobs:
        err = job.communicate()[1]
        assert job.returncode == 0, err[-3000:]
    subprocess.run([clang, "0.o", "1.o", "2.o", "-o", "check"], cwd=d, check=True)
    return str(d / "check")


def test_reads_and_stores_stay_in_bounds(gemm_wide_check):
    r = subprocess.run([gemm_wide_check, "bounds"], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout[-3000:]
    assert "launches" in r.stdout


def _plans(check, calls):
    """(r, jt, split, any, workspace bytes) of each (format, M, K, N) call with aligned operands in the wide tile,
    (-rows, columns, split, 0, bytes) in the LDS tiles, zeros elsewhere."""
    text = "\n".join(" ".join(map(str, c)) for c in calls)
    r = subprocess.run([check, "plan"], input=text, capture_output=True, text=True, check=True)
    return [tuple(map(int, line.split())) for line in r.stdout.splitlines()]


def test_offsets_fit_32_bits(gemm_wide_check):
    # a workgroup's activations: 160 rows of 2 K bytes; its offsets into the weight start at its own rows
    last = (2 ** 32 // 320) // 256 * 256
    calls = [(f, 160, k, 4) for f in (0, 1) for k in (last, last + 256, 2 ** 24)]
    assert [p[0] > 0 for p in _plans(gemm_wide_check, calls)] == [True, False, False] * 2
    large = [(0, 33, 4096, 2 ** 20 + 4), (0, 160, 4096, 2 ** 21), (1, 160, 4096, 2 ** 20 + 4)]
    assert all(p[0] > 0 for p in _plans(gemm_wide_check, large))


def _earlier_split(m, k, n):
    """The K shares of the 128-token INT4 tile, which the sums above 64 tokens have always had."""
    tiles, steps, split = -(-m // 128) * (n // 128), k // 64, 1
    while split < 8 and tiles * split * 2 <= 256 and steps % (8 * split) == 0 and steps // (2 * split) >= 8:
        split *= 2
    return split


def test_sums_keep_their_order(gemm_wide_check):
    """Above 64 tokens the projections of the 4096 / 12288 model sum K in the shares they had, but for the down
    projection of 257 to 320 tokens, where four for two is expected to save more than 15%."""
    calls = [(0, m, k, n) for m in range(65, 1100) for k, n in ((4096, 6144), (4096, 4096), (4096, 24576), (12288, 4096))]
    other = {c[1:] for c, p in zip(calls, _plans(gemm_wide_check, calls)) if p[2] != _earlier_split(*c[1:])}
    assert other == {(m, 12288, 4096) for m in range(257, 321)}


def test_slower_calls_stay_out_of_the_wide_tile(gemm_wide_check):
    """Calls that took 1.1 to 2.2 times as long in the wide tile as in the LDS tiles or the streaming kernel, and
    neighbours of theirs that take 0.2 to 0.9 of the time in it."""
    slower = [(0, 424, 832, 11701), (0, 595, 320, 12317), (0, 1003, 320, 5991), (0, 10, 576, 1506), (0, 47, 1088, 6207),
              (0, 12, 320, 13373), (1, 53, 1536, 13434), (1, 62, 1600, 9892), (1, 60, 4096, 4096),
              (0, 6, 12288, 4096), (1, 6, 12288, 4096)]
    faster = [(0, 424, 4160, 1701), (0, 150, 4160, 1001), (0, 10, 4160, 1506), (0, 154, 6976, 83), (1, 53, 6400, 3434),
              (1, 582, 4352, 102), (1, 64, 4096, 12288), (0, 24, 12288, 4096), (1, 16, 12288, 4096), (1, 17, 4096, 6144)]
    assert all(p[0] <= 0 for p in _plans(gemm_wide_check, slower))
    assert all(p[0] > 0 for p in _plans(gemm_wide_check, faster))


def test_every_instance_has_its_gpu_case(gemm_wide_check):
    """The GPU cases run the instances that they name, and they name every compiled one but the regular splits of
    256 rows by 96 (INT4) and 128 tokens, which the dispatch picked for none of 400000 calls of up to 2900 tokens, K =
    16384 and N = 32768."""
    cases = test_gpu_gemm_wide.INSTANCES
    plans = _plans(gemm_wide_check, [(i[0], *c) for i, c in cases.items()])
    assert [(i[0], r, jt, any_, int(split > 1)) for i, (r, jt, split, any_, _) in zip(cases, plans)] == list(cases)
    tiles = [(1, jt) for jt in range(1, 6)] + [(2, 3), (2, 4)]
    regular = {(f, *t, 0, s) for f in (0, 1) for t in tiles for s in (0, 1)} | {(1, 2, 5, 0, s) for s in (0, 1)}
    any_shape = {(f, *t, 1, s) for f in (0, 1) for t in tiles if t not in ((1, 3), (2, 3)) for s in (0, 1)}
    fused = {(f, *t, 0, 0) for f in (2, 3) for t in tiles}
    assert set(cases) == regular - {(0, 2, 3, 0, 1), (0, 2, 4, 0, 1), (1, 2, 4, 0, 1)} | any_shape | fused


def test_gpu_cases_of_the_lds_tiles(gemm_wide_check):
    cases = test_gpu_gemm_wide.TILES_IN_LDS
    plans = _plans(gemm_wide_check, [(i[0], *c) for i, c in cases.items()])
    assert [(i[0], -r, bn, split) for i, (r, bn, split, *_) in zip(cases, plans)] == [i[:4] for i in cases]
