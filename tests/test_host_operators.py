"""The stand-alone operators of the engine on the CPU, under AddressSanitizer and UndefinedBehaviorSanitizer: each scenario
of tests/c/operators_hosttest.cpp is one test."""

import os
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
CSRC, CDIR = ROOT / "modelexpress_amd" / "csrc", ROOT / "tests" / "c"
SOURCES = [CDIR / "operators_hosttest.cpp", CDIR / "cpu_hip" / "cpu_hip.cpp", CDIR / "cpu_hip" / "cpu_kernels.cpp",
           CSRC / "mxp_engine.cpp", CSRC / "mxp_ckpt.cpp", CSRC / "mxp_plan.cpp", CSRC / "mxp_crc32c.cpp"]
SAN = ["-fsanitize=address,undefined", "-fno-sanitize-recover=undefined", "-fno-omit-frame-pointer", "-g", "-O1"]


@pytest.fixture(scope="module")
def driver():
    out, build = CDIR / "operators_hosttest_asan", CDIR / "build"
    build.mkdir(exist_ok=True)
    headers = [*CSRC.glob("*.hpp"), *CSRC.glob("*.h"), *(ROOT / "include").glob("*.h"), CDIR / "cpu_hip" / "hip" / "hip_runtime.h", Path(__file__)]
    newest = max(p.stat().st_mtime for p in headers)
    flags = ["g++", "-std=c++17", "-Wall", f"-I{CDIR / 'cpu_hip'}", f"-I{ROOT / 'include'}", f"-I{CSRC}", *SAN]
    objects = {s: build / f"operators_{s.stem}.o" for s in SOURCES}
    running = [subprocess.Popen([*flags, "-c", str(s), "-o", str(o)], stdout=subprocess.PIPE, stderr=subprocess.PIPE, text=True)
               for s, o in objects.items() if not o.exists() or o.stat().st_mtime < max(newest, s.stat().st_mtime)]
    for proc in running:
        _o, err = proc.communicate(timeout=900)
        assert proc.returncode == 0, err[-4000:]
    if running or not out.exists():
        r = subprocess.run([*flags, *map(str, objects.values()), "-o", str(out), "-lpthread"], capture_output=True, text=True, timeout=300)
        assert r.returncode == 0, r.stderr[-4000:]
    return out


@pytest.mark.parametrize("scenario", ["copies_without_checksums", "captured_transposes", "timed_placements_with_digests",
                                      "plan_destroyed_from_another_device", "described_views", "woven_transposes", "static_checksum_in_small_tiles",
                                      "half_line_rows"])
def test_operators(driver, scenario, tmp_path):
    env = dict(os.environ, ASAN_OPTIONS="detect_leaks=1:halt_on_error=1", UBSAN_OPTIONS="print_stacktrace=1:halt_on_error=1")
    r = subprocess.run([str(driver), scenario, str(tmp_path)], capture_output=True, text=True, env=env, timeout=300)
    assert r.returncode == 0 and r.stdout == "ok\n" and "Sanitizer" not in r.stderr, (r.stdout[-2000:], r.stderr[-4000:])
