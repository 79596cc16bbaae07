"""Host-side code checked on the CPU, built with AddressSanitizer and
UndefinedBehaviorSanitizer (host code only; no GPU).

- The device-pointer scratch pool's growth rule (csrc/scratch_pool.h): a
  buffer handed to a stream is never freed or shared while the pool lives.
- The oracle (oracle/oracle.c): every function on ragged shapes.
- The library's host code (csrc/api.hip, csrc/quantize.hip): quantizers,
  descriptor checks, argument refusals.
(The library's own leak check is off: the HIP runtime it links keeps
process-lifetime allocations.)
"""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CPP = os.path.join(ROOT, "tests", "cpp")
SAN = ["-fsanitize=address,undefined", "-fno-sanitize-recover=all", "-fno-omit-frame-pointer", "-g", "-O1"]


def _run(exe):
    env = dict(os.environ, ASAN_OPTIONS="detect_leaks=1:abort_on_error=1",
               UBSAN_OPTIONS="print_stacktrace=1:halt_on_error=1")
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120, env=env)
    assert r.returncode == 0, r.stdout + r.stderr
    return r.stdout


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_scratch_pool_growth_rule_under_asan(tmp_path):
    exe = str(tmp_path / "scratch_pool_test")
    subprocess.run(["g++", "-std=c++17", *SAN, "-pthread", os.path.join(CPP, "scratch_pool_test.cpp"),
                    "-o", exe], check=True, timeout=300)
    assert "scratch pool ok" in _run(exe)


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_lease_pool_under_asan(tmp_path):
    """One holder a stream, bounds kept, buffers given back (csrc/lease_pool.h)."""
    exe = str(tmp_path / "lease_pool_test")
    subprocess.run(["g++", "-std=c++17", *SAN, "-pthread", os.path.join(CPP, "lease_pool_test.cpp"), "-o", exe],
                   check=True, timeout=300)
    assert "lease pool ok" in _run(exe)


@pytest.mark.skipif(shutil.which("gcc") is None, reason="needs gcc")
def test_oracle_under_asan(tmp_path):
    """Every oracle function on ragged shapes with exactly-sized buffers
    (tests/cpp/oracle_asan_test.c compiles oracle/oracle.c in)."""
    exe = str(tmp_path / "oracle_asan_test")
    subprocess.run(["gcc", "-std=gnu11", *SAN, "-pthread", os.path.join(CPP, "oracle_asan_test.c"), "-o", exe,
                    "-lm"], check=True, timeout=300)
    assert "oracle asan ok" in _run(exe)


HIPCC = "/opt/rocm/bin/hipcc"
# host side only: the device code is the ordinary build
HOST_SAN = ["-Xarch_host", "-fsanitize=address", "-Xarch_host", "-fsanitize=undefined",
            "-Xarch_host", "-fno-sanitize-recover=all", "-Xarch_host", "-fno-omit-frame-pointer"]


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="needs hipcc")
def test_library_host_code_under_asan(tmp_path):
    """csrc/api.hip and csrc/quantize.hip rebuilt with the sanitizers on their
    host side, linked with the library's other objects, driven on the CPU by
    tests/cpp/host_asan_test.cpp: the quantizers, descriptor checks and
    argument refusals (nothing reaches a GPU)."""
    build = os.path.join(ROOT, "sme-gemm_amd", "_build")
    others = [os.path.join(build, f + ".o") for f in ("q4_gemv", "lowbit_gemv", "gemm_mfma", "gemm_q4r",
                                                     "columns", "decode_block", "probes")]
    if not all(os.path.exists(o) for o in others):
        subprocess.run(["make", "-s", "-j8", "-C", os.path.join(ROOT, "sme-gemm_amd")], check=True, timeout=900)
    flags = ["--offload-arch=gfx950", "-O1", "-g", "-std=c++17", "-fPIC", "-ffp-contract=off",
             "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", *HOST_SAN]
    objs = []
    for src in ("api", "quantize"):
        o = str(tmp_path / (src + ".o"))
        subprocess.run([HIPCC, *flags, "-c", os.path.join(ROOT, "sme-gemm_amd", "csrc", src + ".hip"), "-o", o],
                       check=True, timeout=600, capture_output=True)
        objs.append(o)
    drv = str(tmp_path / "drv.o")
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O1", "-g", "-std=c++17", *HOST_SAN, "-c",
                    os.path.join(CPP, "host_asan_test.cpp"), "-o", drv], check=True, timeout=300,
                   capture_output=True)
    exe = str(tmp_path / "host_asan_test")
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-Xarch_host", "-fsanitize=address", "-Xarch_host",
                    "-fsanitize=undefined", *objs, drv, *others, "-o", exe, "-lpthread"], check=True, timeout=300,
                   capture_output=True)
    env = dict(os.environ, ASAN_OPTIONS="detect_leaks=0:abort_on_error=1",
               UBSAN_OPTIONS="print_stacktrace=1:halt_on_error=1")
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120, env=env)
    assert r.returncode == 0 and "host asan ok" in r.stdout, r.stdout + r.stderr


def _library_objects():
    """The library's objects, built if any is missing."""
    pkg = os.path.join(ROOT, "sme-gemm_amd")
    names = [f[:-4] for f in sorted(os.listdir(os.path.join(pkg, "csrc"))) if f.endswith(".hip")]
    objs = [os.path.join(pkg, "_build", f + ".o") for f in names]
    if not all(os.path.exists(o) for o in objs):
        subprocess.run(["make", "-s", "-j8", "-C", pkg], check=True, timeout=900)
    return objs


@pytest.fixture(scope="module")
def dispatch_rules(tmp_path_factory):
    """tests/cpp/dispatch_rules_test.cpp linked with the library's objects."""
    if not os.path.exists(HIPCC):
        pytest.skip("needs hipcc")
    tmp = tmp_path_factory.mktemp("dispatch")
    drv, exe = str(tmp / "drv.o"), str(tmp / "dispatch_rules_test")
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O1", "-std=c++17", "-Xclang", "-target-feature", "-Xclang",
                    "-packed-fp32-ops", "-I", os.path.join(ROOT, "sme-gemm_amd", "csrc"), "-x", "hip", "-c",
                    os.path.join(CPP, "dispatch_rules_test.cpp"), "-o", drv], check=True, timeout=300,
                   capture_output=True)
    subprocess.run([HIPCC, "--offload-arch=gfx950", *_library_objects(), drv, "-o", exe, "-lpthread"], check=True,
                   timeout=300, capture_output=True)
    return exe


def test_dispatch_rules(dispatch_rules):
    """The launch interface's rules (csrc/kernels.h) at the edges of their ranges,
    on the host alone."""
    r = subprocess.run([dispatch_rules], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and "dispatch rules ok" in r.stdout, r.stdout + r.stderr


def _tiles(exe, calls):
    """Each call's tile, at the 256 compute units the rules count without a GPU."""
    text = "".join(" ".join(map(str, c)) + "\n" for c in calls)
    r = subprocess.run([exe, "tiles"], input=text, capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr
    return [tuple(map(int, x.split())) for x in r.stdout.splitlines()]


def test_gpu_shapes_reach_every_tile(dispatch_rules):
    """The GPU tests' shapes take the tiles they are there for."""
    import test_gpu_dense as dense
    import test_gpu_lowbit_gemm as low
    import test_gpu_mopa as mopa
    assert _tiles(dispatch_rules, [("dense", *s) for s in dense.TILES]) == [
        (256, 256), (128, 256), (64, 128), (64, 64), (64, 64), (32, 64)]
    for bits in (1, 2):
        for block in (64, 128, 256):
            got = set(_tiles(dispatch_rules, [("lowbit", bits, block, *s) for s in low.SHAPES]))
            assert got >= {(16, 64), (32, 64), (64, 64), (64, 128)}, (bits, block, got)
        assert _tiles(dispatch_rules, [("lowbit", bits, 128, *s) for s in low.WIDE]) == [(32, 64), (64, 64), (64, 128)]
    got = _tiles(dispatch_rules, [("mopa", *s[:4]) for s in mopa.SHAPES])
    assert got == [(128, 256)] * 4 + [(256, 256)] * 4, got
