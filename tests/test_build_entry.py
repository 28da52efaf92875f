"""build() compiles the test kernels that the tree holds, and does without
those it does not: a tree with another set of tests, or none, still builds."""
import os
import shutil
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# A recipe that notes its package's name in place of a compiler run.
RECIPE = """\
import os
def build(verbose=False):
    with open(os.environ["BUILT"], "a") as f:
        f.write(os.path.basename(os.path.dirname(os.path.abspath(__file__))) + "\\n")
"""


def _put(path, text):
    os.makedirs(os.path.dirname(path), exist_ok=True)
    with open(path, "w") as f:
        f.write(text)


@pytest.mark.parametrize("kernels", [
    (), ("dropin",), ("claims", "dropin"), ("claims", "dropin", "payload"),
    ("claims", "dropin", "some_other", "payload"),
], ids=lambda k: "+".join(k) or "none")
def test_builds_the_test_kernels_that_are_there(tmp_path, kernels):
    root = str(tmp_path / "tree")
    _put(os.path.join(root, "gallatin_amd", "__init__.py"), "def lib():\n    pass\n")
    _put(os.path.join(root, "oracle", "__init__.py"), "")
    recipes = ["gallatin_amd", "oracle"] + [os.path.join("tests", k) for k in kernels]
    for d in recipes:
        _put(os.path.join(root, d, "build.py"), RECIPE)
    if kernels:
        _put(os.path.join(root, "tests", "golden", "README.md"), "no recipe here\n")
    shutil.copy(os.path.join(ROOT, "__graft_entry__.py"), root)
    built = str(tmp_path / "built")
    r = subprocess.run([sys.executable, "__graft_entry__.py"], cwd=root, text=True,
                       capture_output=True, env=dict(os.environ, BUILT=built, PYTHONPATH=""))
    assert r.returncode == 0, r.stderr
    with open(built) as f:
        got = f.read().split()
    assert got[:2] == ["gallatin_amd", "oracle"]
    assert sorted(got[2:]) == sorted(kernels)
