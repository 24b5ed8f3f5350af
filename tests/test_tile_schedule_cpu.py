"""The small-tile GEMM's LDS schedule, read from the kernel's source and run as a model: between
two workgroup barriers no stage is both read and written, and every read sees its own block."""

import re
from pathlib import Path

import pytest

SOURCE = Path(__file__).resolve().parents[1] / "animaxs_amd" / "csrc" / "linear_tile.hip"
TOKEN = re.compile(r"if \(group == ([01])\) barrier\(\)|\b(barrier|fetch_raw|store_x|store_w|store_sz|read_op)\((\w*)")


def _tokens(text):
    """(name, stage, group): LDS accesses and barriers in the order of the source."""
    out = []
    for m in TOKEN.finditer(re.sub(r"//[^\n]*", "", text)):
        out.append(("barrier", "", int(m[1])) if m[1] else (m[2], m[3], None))
    return out


def _section(src, start, end):
    a = src.index(start)
    return src[a:src.index(end, a)]


def _program():
    src = SOURCE.read_text()
    src = src[src.index("void tile_gemm_kernel"):]
    prologue = _tokens(_section(src, "u32x4 x0[S::XCH]", "auto step ="))
    # fetch_raw, the stores and read_op's first use; read_op's own definition is not a use.
    step = [t for t in _tokens(_section(src, "auto step =", "const int pairs"))
            if not (t[0] == "read_op" and t[1] == "int")]
    return prologue, step


def _events(group, nblk):
    """(interval, 'r' or 'w', array, stage, block) of one wave group."""
    prologue, step = _program()
    out, interval = [], 0
    content = {"x": lambda kb, st: kb + 1, "w": lambda kb, st: kb + 2}   # block a step's copy brings

    def run(tokens, kb):
        nonlocal interval
        cur = 0 if kb is None else kb & 1
        for name, stage, only in tokens:
            if only is not None and only != group:
                continue
            st = {"CUR": cur, "NXT": cur ^ 1}.get(stage, int(stage) if stage.isdigit() else None)
            if name == "barrier":
                interval += 1
            elif name == "read_op":
                out.append((interval, "r", "x", cur, kb))
            elif name == "fetch_raw":
                block = st if kb is None else kb + 1
                if block < nblk:
                    out.extend((interval, "r", a, st, block) for a in ("w", "sz"))
                else:   # of no block: its order still matters to the stage's next writer
                    out.extend((interval, "r", a, st, None) for a in ("w", "sz"))
            else:
                array = name[6:]
                block = st if kb is None else content["x" if array == "x" else "w"](kb, st)
                out.append((interval, "w", array, st, block))

    run(prologue, None)
    for kb in range(nblk):
        run(step, kb)
    return out


def test_the_source_still_has_the_modelled_form():
    prologue, step = _program()
    assert [t[0] for t in prologue].count("fetch_raw") == 1
    assert {t[0] for t in step} == {"barrier", "fetch_raw", "store_x", "store_w", "store_sz", "read_op"}
    assert [t[0] for t in step].count("barrier") == 2


@pytest.mark.parametrize("nblk", range(1, 8))
def test_no_stage_is_read_and_written_between_two_barriers(nblk):
    events = _events(0, nblk) + _events(1, nblk)
    written = {}
    for interval, kind, array, stage, block in events:
        if kind == "w":
            written.setdefault((array, stage), []).append((interval, block))
    for interval, kind, array, stage, block in events:
        if kind != "r":
            continue
        writes = written[array, stage]
        assert interval not in [i for i, _ in writes], (array, stage, block, interval)
        if block is not None:
            last = max(i for i, _ in writes if i < interval)
            before = {b for i, b in writes if i == last}
            assert before == {block}, (array, stage, block, interval)
