"""What a model family's own build holds (csrc/build.py: MODEL_SOURCES) against what its worker calls: every entry point that is named in code
reachable from the family's model class."""
import ast
import functools
import importlib.util
import os
import re

import pytest

from swiftllm_amd import registry
from swiftllm_amd.csrc import build


class _Module:
    def __init__(self, name):
        self.name, self.defs, self.imports, self.package = name, {}, {}, name.rpartition(".")[0]
        path = importlib.util.find_spec(name).origin
        if os.path.basename(path) == "__init__.py":
            self.package = name
        with open(path, encoding="utf-8") as f:
            tree = ast.parse(f.read())
        for node in ast.walk(tree):
            if isinstance(node, ast.ImportFrom):
                src = importlib.util.resolve_name("." * node.level + (node.module or ""), self.package) if node.level else node.module
                for a in node.names:
                    self.imports[a.asname or a.name] = (src, a.name)
        for node in tree.body:
            if isinstance(node, (ast.FunctionDef, ast.ClassDef)):
                self.defs[node.name] = node
            elif isinstance(node, ast.Assign):
                for t in node.targets:
                    if isinstance(t, ast.Name):
                        self.defs[t.id] = node


_module = functools.lru_cache(None)(_Module)


def _is_module(name):
    try:
        return importlib.util.find_spec(name) is not None
    except ModuleNotFoundError:
        return False


def _reachable_entry_points(module, name):
    found, seen, todo = set(), set(), [(module, name)]
    while todo:
        at = todo.pop()
        if at in seen or not at[0].startswith("swiftllm_amd.worker"):
            continue
        seen.add(at)
        m = _module(at[0])
        if at[1] not in m.defs:
            if at[1] in m.imports:      # (handed on by a package)
                todo.append(m.imports[at[1]])
            continue
        for node in ast.walk(m.defs[at[1]]):
            if isinstance(node, ast.Constant) and isinstance(node.value, str) and re.fullmatch(r"swl_\w+", node.value):
                found.add(node.value)
            elif isinstance(node, ast.Attribute):
                if node.attr.startswith("swl_"):
                    found.add(node.attr)
                if isinstance(node.value, ast.Name) and node.value.id in m.imports:     # a name out of an imported module
                    src, what = m.imports[node.value.id]
                    if _is_module(f"{src}.{what}"):
                        todo.append((f"{src}.{what}", node.attr))
            elif isinstance(node, ast.Name):
                todo.append((at[0], node.id) if node.id in m.defs else m.imports.get(node.id, ("", "")))
    return found


# named in a shared function on a branch that the family does not take: its heads are not mixed (window_attention with talk None)
NOT_TAKEN = {"Lorulix": {"swl_mix_attn", "swl_mix_attn_supported"}}


@pytest.mark.parametrize("family", sorted(build.MODEL_SOURCES))
def test_a_family_builds_every_entry_point_its_worker_names(family):
    module, cls = registry.MODELS[family][1].split(":")
    called = _reachable_entry_points(module, cls)
    assert len(called) > 10 and called <= set(build.entry_points(build.SOURCES))
    missing = called - NOT_TAKEN.get(family, set()) - set(build.entry_points(build.MODEL_SOURCES[family]))
    assert not missing, f"{family} calls {sorted(missing)}"
