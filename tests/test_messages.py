"""Every ``"..." % args`` of the package formats: its conversions are known ones, as
many as the arguments (a bare ``%`` in a message raises ValueError in its place)."""

from __future__ import annotations

import ast
import glob
import os
import re

PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "leanmoe-quant_amd", "lemoq")
SPEC = re.compile(r"%(?:\((?P<key>\w+)\))?[-+#0 ]*(?:\*|\d+)?(?:\.(?:\*|\d+))?(?P<conv>.)", re.S)


def test_percent_formats():
    seen = 0
    for path in sorted(glob.glob(os.path.join(PKG, "**", "*.py"), recursive=True)):
        with open(path, encoding="utf-8") as f:
            tree = ast.parse(f.read())
        for node in ast.walk(tree):
            if not (isinstance(node, ast.BinOp) and isinstance(node.op, ast.Mod) and isinstance(node.left, ast.Constant)
                    and isinstance(node.left.value, str)):
                continue
            where = "%s:%d" % (os.path.relpath(path, PKG), node.lineno)
            found = [m for m in SPEC.finditer(node.left.value) if m.group(0) != "%%"]
            assert all(m.group("conv") in "diouxXeEfFgGcrsa" for m in found), where
            if isinstance(node.right, ast.Tuple):
                assert len(found) == len(node.right.elts), where
            elif not isinstance(node.right, ast.Dict):
                assert len(found) == 1, where
            seen += 1
    assert seen > 50
