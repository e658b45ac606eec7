"""The kernel disk cache (the reference only hints at one: helium-kernel-generator/Cargo.toml:42-44, feature
`disk-cache`): a second process finds the first one's code object, and a file that is damaged is compiled again."""
import os
import subprocess
import sys

import pytest

from helpers import run_with_compiler

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

CHILD = r"""
import sys
sys.path.insert(0, %r)
from helium_amd import device
src = 'extern "C" __global__ void cached_probe(float* x) { x[threadIdx.x] = x[threadIdx.x] * 3.0f + 1.0f; }'
code = device.rtc_compile(src, "cached_probe")
assert code[:4] == b"\x7fELF", code[:8]
s = device.rtc_stats()
print(s["compiles"], s["disk_hits"], len(code))
""" % ROOT


def _child(cache_dir):
    env = dict(os.environ, HELIUM_HIP_CACHE_DIR=str(cache_dir))
    out = subprocess.run([sys.executable, "-c", CHILD], env=env, capture_output=True, text=True, timeout=300)
    assert out.returncode == 0, out.stderr
    compiles, disk_hits, size = (int(v) for v in out.stdout.split())
    return compiles, disk_hits, size


def test_second_process_hits_the_disk_and_damaged_files_are_recompiled(tmp_path):
    compiles, disk_hits, size = _child(tmp_path)
    assert (compiles, disk_hits) == (1, 0)
    files = [f for f in os.listdir(tmp_path) if f.endswith(".hekc")]
    assert len(files) == 1 and not [f for f in os.listdir(tmp_path) if ".tmp" in f]
    path = os.path.join(tmp_path, files[0])
    good = open(path, "rb").read()
    assert len(good) > size and good[:8] == b"HEKCACHE"

    assert _child(tmp_path) == (0, 1, size)          # found on disk, nothing compiled

    open(path, "wb").write(good[: len(good) // 2])   # truncated (an interrupted copy)
    assert _child(tmp_path) == (1, 0, size)
    assert open(path, "rb").read() == good           # and written afresh

    flipped = bytearray(good)
    flipped[-100] ^= 0x40                            # one bit of the code object
    open(path, "wb").write(bytes(flipped))
    assert _child(tmp_path) == (1, 0, size)

    open(path, "wb").write(good[32:])                # a bare code object, as an older format stored it
    assert _child(tmp_path) == (1, 0, size)
    assert _child(tmp_path) == (0, 1, size)


def test_cache_can_be_switched_off(tmp_path):
    env = dict(os.environ, HELIUM_HIP_CACHE_DIR="off")
    out = subprocess.run([sys.executable, "-c", CHILD], env=env, capture_output=True, text=True, timeout=300, cwd=tmp_path)
    assert out.returncode == 0, out.stderr
    assert out.stdout.split()[:2] == ["1", "0"] and not os.listdir(tmp_path)


def test_the_compiler_does_not_depend_on_what_the_program_imported_first(tmp_path):
    """torch carries a HIP compiler of its own; kernels come from the toolchain's all the same."""
    made = []
    for first in ("", "import torch\n"):
        d = tmp_path / ("with" if first else "without")
        out = subprocess.run([sys.executable, "-c", first + CHILD], env=dict(os.environ, HELIUM_HIP_CACHE_DIR=str(d)), capture_output=True,
                             text=True, timeout=300)
        assert out.returncode == 0, out.stderr
        made.append({f: open(os.path.join(d, f), "rb").read() for f in os.listdir(d)})
    assert len(made[0]) == 1 and made[0] == made[1]


def test_what_the_compiler_has_against_a_source_reaches_the_caller():
    code = ("import sys; sys.path.insert(0, %r)\nfrom helium_amd import device\n"
            "try:\n    device.rtc_compile('extern \"C\" __global__ void broken() { no_such_name(); }', 'broken')\n"
            "except Exception as e:\n    print(e)\n" % ROOT)
    out = subprocess.run([sys.executable, "-c", code], env=dict(os.environ, HELIUM_HIP_CACHE_DIR="off"), capture_output=True, text=True, timeout=300)
    assert out.returncode == 0 and "broken" in out.stdout and "no_such_name" in out.stdout, out.stdout + out.stderr


def _probe_with_compiler(tmp_path, script, **env):
    """Compiles one kernel with that compiler: (compiles, disk hits, bytes of code object) and the process."""
    tmp_path.mkdir(exist_ok=True)
    out = run_with_compiler(tmp_path, script, CHILD.split("\n", 3)[3], HELIUM_HIP_CACHE_DIR=str(tmp_path / "cache"), **env)
    assert out.returncode == 0, out.stderr
    return tuple(int(v) for v in out.stdout.split()), out


def test_the_compiler_runs_without_a_profilers_hooks(tmp_path):
    """What a profiler preloads and sets stays with the program; whatever else is preloaded reaches the compiler as it was."""
    seen = tmp_path / "environment"
    preload = ":".join(filter(None, [os.environ.get("LD_PRELOAD"), "/nowhere/librocprofiler-sdk-tool.so", "/nowhere/libother.so", "/nowhere/libroctx64.so"]))
    _probe_with_compiler(tmp_path, f'env > {seen}; exec "$REAL" "$@"', LD_PRELOAD=preload, ROCP_ONE="1",
                         ROCPROFILER_TWO="1", HSA_TOOLS_THREE="1", KEPT_ALL_THE_SAME="1")
    env = dict(line.split("=", 1) for line in seen.read_text().split("\n") if "=" in line)
    assert not [k for k in env if k.startswith(("ROCP", "HSA_TOOLS"))], env
    assert env["LD_PRELOAD"] == ":".join(filter(None, [os.environ.get("LD_PRELOAD"), "/nowhere/libother.so"]))
    assert env["KEPT_ALL_THE_SAME"] == "1" and "PATH" in env


def test_the_compiler_does_not_load_the_hip_runtime():
    import helium_amd

    listed = subprocess.run(["ldd", os.path.join(os.path.dirname(helium_amd.__file__), "helium_rtc")], capture_output=True, text=True).stdout
    assert "libhiprtc" in listed and "libamdhip64" not in listed and "libhsa" not in listed, listed


@pytest.mark.parametrize("script", ['"$REAL" "$@" > $0.out; head -c 1000 $0.out', '"$REAL" "$@" > $0.out; head -c 1000 $0.out; exit 2', '"$REAL" "$@"; exit 2',
                                    '"$REAL" "$@"; kill -9 $$', "exit 0", "printf o"],
                         ids=["cut_short", "cut_short_with_a_status", "whole_with_a_status", "killed", "nothing", "one_byte"])
def test_an_answer_that_is_not_whole_is_not_taken(tmp_path, script):
    """The kernel is compiled in-process instead, to the same code object."""
    whole, _ = _probe_with_compiler(tmp_path / "sound", 'exec "$REAL" "$@"')
    got, _ = _probe_with_compiler(tmp_path / "unsound", script)
    assert got == whole


SAYS_OTHER = r"""printf 'o\005\0\0\0\0\0\0\0other'"""


def test_the_cache_tells_compilers_apart(tmp_path):
    """A code object is found by the compiler that made it: not by another version, nor by either what was compiled in-process
    because the other process could not do its work."""
    sound, other = 'exec "$REAL" "$@"', 'if [ "$1" = --version ]; then %s; else exec "$REAL" "$@"; fi' % SAYS_OTHER
    broken = 'if [ "$1" = --version ]; then exec "$REAL" "$@"; else exit 2; fi'
    counts = lambda script: _probe_with_compiler(tmp_path, script)[0][:2]  # noqa: E731
    assert counts(sound) == (1, 0)
    assert counts(other) == (1, 0)    # made by another version: compiled afresh
    assert counts(broken) == (0, 1)   # nothing to compile
    for f in os.listdir(tmp_path / "cache"):
        os.unlink(tmp_path / "cache" / f)
    assert counts(broken) == (1, 0)   # compiled in-process
    assert counts(broken) == (0, 1)   # and kept for the next program in the same place
    assert counts(sound) == (1, 0)    # but not for the other compiler
    assert len(os.listdir(tmp_path / "cache")) == 2


def test_a_compiler_that_cannot_say_what_it_is_is_not_used(tmp_path):
    (compiles, hits, _), _ = _probe_with_compiler(tmp_path, f"touch {tmp_path}/asked_$1; exit 2")
    assert (compiles, hits) == (1, 0)
    assert [f for f in os.listdir(tmp_path) if f.startswith("asked_")] == ["asked_--version"]
