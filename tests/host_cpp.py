"""Runs a C++ snippet against the engine's own headers on the host: for rules that no entry point shows."""
import os
import subprocess

from emdee_amd import build

CSRC = build.CSRC


def run(tmp_path, body, headers=("device_state.h",)):
    """main() with `body`, compiled as the engine's .hip sources are; returns its output's lines."""
    src, exe = str(tmp_path / "snippet.hip"), str(tmp_path / "snippet")
    text = "".join(f'#include "{h}"\n' for h in headers) + "#include <cstdio>\nusing namespace emdee;\nint main() {\n" + body + "\n}\n"
    with open(src, "w") as f:
        f.write(text)
    flags = [f if f != "-O3" else "-O1" for f in build.HIP_FLAGS]
    r = subprocess.run([build.HIPCC] + flags + ["-I", CSRC, "-o", exe, src], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    env = dict(os.environ, HIP_VISIBLE_DEVICES="")
    r = subprocess.run([exe], capture_output=True, text=True, env=env, timeout=60)
    assert r.returncode == 0, r.stderr
    return r.stdout.splitlines()
