"""The kernel names that the Python side asks the timers for are names that the
library launches under."""
import ast
import glob
import os
import re

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _asked(path):
    """The strings of every `for name in (...)` whose body queries the timers."""
    tree = ast.parse(open(os.path.join(ROOT, path)).read())
    names = []
    for node in ast.walk(tree):
        if isinstance(node, ast.For) and isinstance(node.iter, ast.Tuple) and "timing_query" in ast.dump(node):
            names += [e.value for e in node.iter.elts if isinstance(e, ast.Constant) and isinstance(e.value, str)]
    return names


def test_names_are_launched():
    launched = set()
    for f in glob.glob(os.path.join(ROOT, "fdf_amd", "csrc", "*.hip")):
        launched |= set(re.findall(r'"([A-Za-z0-9_]+)"', open(f).read()))
    asked = _asked("fdf_amd/mlp.py") + _asked("bench.py")
    assert len(asked) > 20
    assert [k for k in asked if k not in launched] == []
