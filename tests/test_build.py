"""A fresh checkout, where the package cannot be imported yet, can load the build."""

import os
import shutil
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_the_build_module_loads_before_the_engine_is_built(tmp_path):
    shutil.copy(os.path.join(ROOT, "__graft_entry__.py"), tmp_path)
    shutil.copytree(os.path.join(ROOT, "rustautograd_amd"), tmp_path / "rustautograd_amd", ignore=shutil.ignore_patterns("*.so", "__pycache__"))
    code = "import __graft_entry__ as g; assert callable(g.native_build().build_all)"
    subprocess.run([sys.executable, "-c", code], cwd=tmp_path, check=True, timeout=60)
