"""The library builds from its own sources: nothing of the test tree takes part, so that a build does not depend on which
commit's tests lie beside it."""
import os
import shutil
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CLANG = "/opt/rocm/llvm/bin/clang++"

# build() with its commands written down instead of run
DRY = """
import subprocess, __graft_entry__ as g
from analog_moe_amd import _abi
subprocess.run = lambda cmd, **kw: print("RUN", *cmd, flush=True)
_abi.bind = lambda path: None
g.build()
"""


def test_build_uses_no_file_of_the_test_tree(tmp_path):
    skip = shutil.ignore_patterns("*.so", "*.o", "build", "__pycache__")
    for name in ("analog_moe_amd", "include"):
        shutil.copytree(os.path.join(ROOT, name), tmp_path / name, ignore=skip)
    shutil.copy(os.path.join(ROOT, "__graft_entry__.py"), tmp_path)
    os.chmod(tmp_path / "analog_moe_amd" / "csrc" / "emu" / "build.sh", 0o644)       # a copy may lose the mode
    (tmp_path / "tests" / "emu" / "libamoe_emu.so").mkdir(parents=True)              # ... and its tests be untouchable
    got = subprocess.run([sys.executable, "-c", DRY], cwd=tmp_path, env={**os.environ, "MAX_JOBS": "1"},
                         capture_output=True, text=True)
    assert got.returncode == 0, got.stderr
    runs = [line.split()[1:] for line in got.stdout.splitlines() if line.startswith("RUN")]
    assert [cmd for cmd in runs if cmd[0] != "hipcc"] == [["sh", str(tmp_path / "analog_moe_amd" / "csrc" / "emu" / "build.sh")]]
    assert str(tmp_path / "tests") not in " ".join(sum(runs, []))
    # the host build's translation units find every header and declaration in the copy
    csrc = tmp_path / "analog_moe_amd" / "csrc"
    for unit in ("amoe.hip", "ffn.hip", "router.hip"):
        subprocess.run([CLANG, "-x", "c++", "-std=c++20", "-fsyntax-only", "-Wno-psabi", "-I", str(csrc / "emu"), "-I", str(tmp_path / "include"),
                        "-I", str(csrc), str(csrc / unit)], check=True)
