"""The tracing kernels' code as the compiler's code generator gets it: no loop
may carry a per-lane boolean.  Those files are compiled with wave-uniform
branches left as they are (quadray-engine_amd/Makefile says why), under which
such a boolean comes out wrong; lane masks and whole numbers do not."""
import os
import re
import subprocess

import pytest

PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                   "quadray-engine_amd")


def functions(text):
    """(name, {block: [instruction lines]}) of every function, blocks in
    order."""
    for m in re.finditer(r"^define [^\n]*@([\w.$]+)\(.*?\n(.*?)^}", text, re.S | re.M):
        blocks, cur = {"": []}, ""
        for line in m.group(2).split("\n"):
            label = re.match(r"([\w.]+):", line)
            if label:
                cur = label.group(1)
                blocks[cur] = []
            elif line.strip():
                blocks[cur].append(line.strip())
        yield m.group(1), blocks


def loop_heads(blocks):
    """Blocks that a path from them comes back to (the targets of a depth
    first walk's back edges)."""
    succ = {b: re.findall(r"label %([\w.]+)", " ".join(
        x for x in ls if x.startswith(("br ", "switch ")) or re.match(r"i\d+ -?\d+, label", x)))
        for b, ls in blocks.items()}
    heads, state, todo = set(), {"": 1}, [("", iter(succ[""]))]
    while todo:
        b, it = todo[-1]
        nxt = next(it, None)
        if nxt is None:
            state[b] = 2
            todo.pop()
        elif state.get(nxt) == 1:
            heads.add(nxt)
        elif nxt not in state:
            state[nxt] = 1
            todo.append((nxt, iter(succ[nxt])))
    return heads


def carried_booleans(text):
    out = []
    for name, blocks in functions(text):
        for h in loop_heads(blocks):
            out += [f"{name}: {x}" for x in blocks[h] if " = phi i1 " in x]
    return out


def test_finds_a_carried_boolean():
    body = """define void @f(i1 %c) {
  br label %1

1:                                                ; preds = %1, %0
  %2 = phi i1 [ true, %0 ], [ %3, %1 ]
  %3 = xor i1 %2, %c
  br i1 %3, label %1, label %4

4:                                                ; preds = %1
  %5 = phi i1 [ %3, %1 ]
  ret void
}
"""
    assert len(carried_booleans(body)) == 1


@pytest.fixture(scope="module")
def ir(tmp_path_factory):
    out = tmp_path_factory.mktemp("ir")
    subprocess.run(["make", "-s", "-j4", "-C", PKG, "ir", f"IR_DIR={out}"], check=True)
    return {f.name: f.read_text() for f in sorted(out.iterdir())}


def test_no_loop_of_the_tracing_kernels_carries_a_boolean(ir):
    assert sorted(ir) == ["tracer.ll", "tracer_pt.ll", "tracer_wf.ll"]
    for name, text in ir.items():
        fns = list(functions(text))
        assert len(fns) >= 4 and any(len(loop_heads(b)) > 3 for _, b in fns), name
        assert carried_booleans(text) == [], name
