"""The Makefile of the native library names, for every object, each of this repository's headers that its source
includes, directly or through another: an incremental build after a change to a header rebuilds what reads it."""
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "tritify_amd", "csrc")


def base(path):
    return re.sub(r".*[)/]", "", path)


def rules():
    """(target, source, named headers) of each rule that compiles one source."""
    out = []
    for line in open(os.path.join(CSRC, "Makefile")):
        m = re.match(r"(\$\(\w+\)/\S+): (\$\(HERE\)\S+\.(?:hip|cpp)) (.*)", line)
        if m:
            out.append((base(m[1]), base(m[2]), {base(p) for p in m[3].split()}))
    return out


def headers(name):
    found = set()
    todo = [name]
    while todo:
        f = todo.pop()
        path = next(p for p in (os.path.join(CSRC, f), os.path.join(ROOT, "include", f)) if os.path.exists(p))
        for h in re.findall(r'^\s*#include "([^"]+)"', open(path).read(), flags=re.M):
            if h not in found:
                found.add(h)
                todo.append(h)
    return found


@pytest.mark.parametrize("target,source,named", rules(), ids=[r[0] for r in rules()])
def test_every_included_header_is_a_prerequisite(target, source, named):
    assert headers(source) <= named, f"{target}: {sorted(headers(source) - named)}"


def test_every_source_has_a_rule():
    sources = {f for f in os.listdir(CSRC) if f.endswith((".hip", ".cpp"))}
    assert sources == {s for _, s, _ in rules()}
