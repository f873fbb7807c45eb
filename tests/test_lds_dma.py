"""Wait states of the direct global -> LDS loads, read from the assembly of the kernels.

The loads are inline assembly, where the compiler inserts no wait states of its own: one is needed
between a scalar write of M0 (the LDS address) and the load, and five between a vector write of the
load's scalar base and the load."""

import concurrent.futures
import importlib.util
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_spec = importlib.util.spec_from_file_location("lbk_build", os.path.join(ROOT, "looped-blockell-tpu_amd", "build.py"))
build = importlib.util.module_from_spec(_spec)
_spec.loader.exec_module(build)

FILES = ["lbk_bwd.hip", "lbk_tile64.hip"]


def _hazards(lines):
    """(loads, instructions too close to one) of an assembly listing."""
    loads, bad, seen = 0, [], []          # seen: (wait states it gives, text) since the last label
    for line in lines:
        t = line.split(";")[0].strip()
        if not t or t.startswith("."):
            if t.endswith(":"):
                seen = []
            continue
        if t.endswith(":"):
            seen = []
            continue
        if re.match(r"(global|buffer|scratch)_load\S*_?lds", t) or re.search(r"_load_\S+ .*\blds$", t):
            loads += 1
            base = re.search(r"s\[(\d+):(\d+)\]", t)
            states = 0
            for ws, u in reversed(seen):
                if states < 1 and re.match(r"s_\S+ m0\b", u):
                    bad.append((u, t))
                w = re.match(r"v_\S+ s(?:(\d+)\b|\[(\d+):(\d+)\])", u)
                if base and w and states < 5:
                    lo, hi = int(w[1] or w[2]), int(w[1] or w[3])
                    if lo <= int(base[2]) and hi >= int(base[1]):
                        bad.append((u, t))
                states += ws
                if states >= 5:
                    break
        n = re.match(r"s_nop (\d+)", t)
        seen.append((int(n[1]) + 1 if n else 1, t))
    return loads, bad


def test_hazards_are_recognised():
    ok = ["s_mov_b32 m0, s4", "s_nop 0", "global_load_lds_dwordx4 v1, s[2:3]"]
    assert _hazards(ok) == (1, [])
    assert len(_hazards([ok[0], ok[2]])[1]) == 1
    assert len(_hazards(["v_readlane_b32 s3, v0, s1", *ok])[1]) == 1
    assert _hazards(["v_readlane_b32 s3, v0, s1", "s_nop 2", *ok]) == (1, [])
    assert _hazards(["v_readlane_b32 s5, v0, s1", *ok]) == (1, [])


def test_every_source_with_lds_loads_is_listed():
    with_loads = [f for f in sorted(os.listdir(build.CSRC))
                  if re.search(r"lds_load16\(", open(os.path.join(build.CSRC, f)).read()) and f.endswith(".hip")]
    assert with_loads == FILES
    for f in build.HIP_SOURCES:           # the instruction itself only in the shared helper
        text = re.sub(r"//[^\n]*", "", open(os.path.join(build.CSRC, f)).read())
        assert "load_lds" not in text, f


@pytest.mark.skipif(not shutil.which("hipcc") and not os.path.exists("/opt/rocm/bin/hipcc"), reason="no hipcc")
def test_lds_loads_keep_their_wait_states(tmp_path):
    def listing(f):
        out = str(tmp_path / (f + ".s"))
        cmd = [build.hipcc(), *build.HIP_FLAGS, *build.FILE_FLAGS.get(f, []), "-I" + build.INCLUDE, "-I" + build.CSRC,
               "--cuda-device-only", "-S", os.path.join(build.CSRC, f), "-o", out]
        subprocess.run(cmd, check=True, stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL)
        with open(out) as fh:
            return fh.readlines()

    with concurrent.futures.ThreadPoolExecutor() as ex:
        for f, lines in zip(FILES, ex.map(listing, FILES)):
            loads, bad = _hazards(lines)
            assert loads > 50 and not bad, (f, loads, len(bad), bad[:3])
