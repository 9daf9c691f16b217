"""The wide GEMM tile (csrc/gemm_wide_kernel.h) copies activations from global memory into a ring of
four LDS buffers and waits for those copies with explicit vmcnt counts before its barriers.  The
counts hold only if the generated code issues exactly the loads they count.  This test compiles the
instances for gfx950 with the library's flags and replays the vector-memory order of each (loads
complete in order): when a wave meets barrier b of the steps (0 before the first), its copies of every
step up to b + 1 must have landed, because the other waves read them before the next barrier.  The
block loop is replayed twice, so the counts are checked across its back edge too.
"""
import os
import re
import shutil
import subprocess

import pytest

from moss_tts import _build

_LOAD = re.compile(r"^(global_load|buffer_load|scratch_load|flat_load)")


def _bodies(source, tmp_path):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not available")
    out = tmp_path / (source + ".s")
    flags = [f for f in _build.CFLAGS if f not in ("-fPIC", "-fvisibility=hidden")]
    r = subprocess.run([hipcc, *flags, "-I", _build.CSRC, "-S", "--cuda-device-only",
                        os.path.join(_build.CSRC, source), "-o", str(out)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    bodies, name = {}, None
    for line in out.read_text().split("\n"):
        head = line.split(":")[0]
        if line.startswith("_Z") and "gemm_wide_kernel" in head and ":" in line:
            name = head
            bodies[name] = []
        elif name:
            bodies[name].append(line.strip())
            if line.strip().startswith("s_endpgm"):
                name = None
    return bodies


def _unrolled(body):
    """The instructions in order, the block loop (the backward branch around copies) twice."""
    labels = {t.split(":")[0]: i for i, t in enumerate(body) if t.startswith(".LBB")}
    for i, t in enumerate(body):
        m = re.match(r"s_c?branch\w*\s+(\.LBB\w+)", t)
        if m and labels.get(m.group(1), i) < i:
            loop = body[labels[m.group(1)]:i]
            if any(" lds" in u and u.startswith("buffer_load") for u in loop):
                return body[:i] + loop + body[i:]
    return body


def check_ring_waits(body, copies_per_step):
    """Barriers of the steps checked; raises AssertionError at one that a needed copy may not have
    reached."""
    pending, copies, barriers, last = [], 0, 0, 0
    body = _unrolled(body)
    for t in body:
        last += bool(re.match(r"buffer_load_dwordx4 .*lds", t))
    for t in body:
        if re.match(r"buffer_load_dwordx4 .*lds", t):
            pending.append(copies // copies_per_step)
            copies += 1
        elif _LOAD.match(t):
            pending.append(None)
        elif t.startswith("s_waitcnt") and "vmcnt" in t:
            n = int(re.search(r"vmcnt\((\d+)\)", t).group(1))
            pending = pending[max(0, len(pending) - n):] if n else []
        elif t.startswith("s_barrier"):
            late = [p for p in pending if p is not None and p <= barriers + 1]
            assert not late, f"barrier {barriers}: copies of steps {sorted(set(late))} may be in flight"
            barriers += 1
            if copies == last and not any(p is not None for p in pending):
                return barriers
    raise AssertionError("copies in flight at the end")


def test_check_rejects_a_lax_wait():
    step = "buffer_load_dwordx4 v1, s[0:3], s4 offen lds"
    body = [step, step, step, "s_waitcnt vmcnt(1)", "s_barrier", "s_waitcnt vmcnt(0)", "s_barrier"]
    assert check_ring_waits(body, 1) == 2
    body[3] = "s_waitcnt vmcnt(2)"
    with pytest.raises(AssertionError):
        check_ring_waits(body, 1)


@pytest.mark.parametrize("source,instances", [("gemm_wide_w4.hip", 38), ("gemm_wide_fp8.hip", 26)])
def test_ring_waits_cover_every_copy(tmp_path, source, instances):
    bodies = _bodies(source, tmp_path)
    assert len(bodies) == instances
    for name, body in bodies.items():
        jt = int(re.search(r"gemm_wide_kernelILi\d+ELi\d+ELi(\d+)E", name).group(1))
        # prologue, two blocks of four steps, the last block's first two
        assert check_ring_waits(body, jt) == 11, name
