"""Checks of compiled code that the kernels' correctness depends on (CPU only: hipcc cross-compiles for gfx950).

The bf16 chunked-delta scan's loading waves keep their next chunk's register requests in flight across a barrier:
before it they wait with an explicit `s_waitcnt vmcnt(N)`, which is right only if exactly N loads were issued after
the wave's last direct-to-LDS load (gfx950 counts loads in one in-order counter). A different count would let a
stage be read before its direct loads land (N too large) or wait for the requests (N too small)."""
import importlib.util
import re
import shutil
import subprocess
from pathlib import Path

import pytest

NATIVE = Path(__file__).resolve().parents[1] / "metal-inference-engine_amd" / "native"
HIPCC = "/opt/rocm/bin/hipcc"
_spec = importlib.util.spec_from_file_location("rk_build", NATIVE / "build.py")
build = importlib.util.module_from_spec(_spec)
_spec.loader.exec_module(build)


@pytest.mark.skipif(shutil.which(HIPCC) is None, reason="hipcc not installed")
def test_loader_waits_count_its_register_requests(tmp_path):
    asm = tmp_path / "cols.s"
    cmd = [HIPCC, "-x", "hip", "-S", "--offload-device-only", str(NATIVE / "chunked_delta_cols.hip"), "-o", str(asm)]
    cmd += build.FLAGS + build.SOURCE_FLAGS.get("chunked_delta_cols.hip", [])
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    lines = [ln.strip() for ln in asm.read_text().splitlines()]
    checked = 0
    for i, ln in enumerate(lines):
        m = re.match(r"s_waitcnt vmcnt\((\d+)\) lgkmcnt\(0\)$", ln)
        if not m or i + 1 >= len(lines) or lines[i + 1] != "s_barrier":
            continue
        n, j = 0, i
        while j > 0:
            j -= 1
            if lines[j].startswith("global_load_lds") or lines[j] == "s_barrier":
                break
            if lines[j].startswith("global_load"):
                n += 1
        assert lines[j].startswith("global_load_lds"), f"no direct load before the wait at line {i}"
        assert n == int(m.group(1)), f"wait at line {i}: vmcnt({m.group(1)}) but {n} loads after the last direct load"
        checked += 1
    assert checked == 4, f"expected the 4 loader waits (2 waves x prologue / loop), found {checked}"


@pytest.mark.skipif(shutil.which(HIPCC) is None, reason="hipcc not installed")
def test_gemm_waits_count_its_loads(tmp_path):
    """gemm_rows waits with `s_waitcnt vmcnt(N)` for all but the loads of its newest stages, which is right only if
    every stage between two waits is the same number L of direct loads, the start is N + 2 L of them (this stage and the
    next are waited for), and no other memory access stands between the first wait and the last."""
    asm = tmp_path / "gemm.s"
    cmd = [HIPCC, "-x", "hip", "-S", "--offload-device-only", str(NATIVE / "linear_gemm.hip"), "-o", str(asm)]
    cmd += build.FLAGS + build.SOURCE_FLAGS.get("linear_gemm.hip", [])
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    kernels = re.findall(r"^(_Z\S*gemm_rows\S*):(.*?)^\.Lfunc_end", asm.read_text(), flags=re.S | re.M)
    assert len(kernels) == 12
    for name, body in kernels:
        lines = [ln.strip() for ln in body.splitlines()]
        waits = [i for i, ln in enumerate(lines) if re.match(r"s_waitcnt vmcnt\(\d+\)$", ln) and lines[i + 1] == "s_barrier"]
        n = {int(re.search(r"\d+", lines[i][10:]).group()) for i in waits}
        assert len(waits) >= 2 and len(n) == 1, name
        loads = lambda a, b: sum(ln.startswith("global_load_lds") for ln in lines[a:b])
        last_mfma = max(i for i, ln in enumerate(lines) if ln.startswith("v_mfma"))
        per = {loads(a, b) for a, b in zip(waits, waits[1:])} | {loads(waits[-1], last_mfma)}
        assert len(per - {0}) == 1, (name, per)
        L = max(per)
        assert loads(0, waits[0]) == n.copy().pop() + 2 * L, name
        other = [ln for ln in lines[waits[0]:last_mfma]
                 if re.match(r"(global|buffer|flat|scratch)_", ln) and not ln.startswith("global_load_lds")]
        assert not other, (name, other[:3])


def test_a_failed_build_leaves_the_libraries_as_they_were(tmp_path, monkeypatch):
    """rk_calls.so calls librk_path.so through prototypes compiled in: a build whose HIP part fails must not leave a new one
    beside the old library."""
    libs = [tmp_path / n for n in ("librk_path.so", "rk_calls.so")]
    for p, name in zip(libs, ("LIB", "CALLS")):
        p.write_text("old")
        monkeypatch.setattr(build, name, p)
    monkeypatch.setattr(build, "OBJ_DIR", tmp_path / "obj")

    def run(cmd, **kw):
        ok = cmd[0] == "g++"
        if ok:
            Path(cmd[cmd.index("-o") + 1]).write_text("new")
        return subprocess.CompletedProcess(cmd, 0 if ok else 1, "", "hipcc failed")
    monkeypatch.setattr(build.subprocess, "run", run)
    with pytest.raises(RuntimeError):
        build.build()
    assert [p.read_text() for p in libs] == ["old", "old"]
