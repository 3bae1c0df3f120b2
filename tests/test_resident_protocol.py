"""The order of waits, barriers and stores in the kernels whose blocks hand
each other values while they run (k_lz_run, k_cheb_run), read from their
source.

A place that others wait on is emptied before it is used again.  Another block
may look at it once that block has awaited a value published later in the
owner's program, so the emptying must have arrived (drain_memory) before that
value is published; otherwise a late emptying lets the other block take the
place's old value for the new one.
"""
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "damascene_amd", "csrc")


def kernel_body(path, name, marker):
    """Text of the braces that follow `marker` in kernel `name`."""
    with open(os.path.join(CSRC, path)) as f:
        text = re.sub(r"//[^\n]*", "", f.read())
    at = text.index(marker, re.search(r"__launch_bounds__\([^;{]*\b" + name + r"\(", text).start())
    start = at = text.index("{", at + len(marker))
    depth = 0
    while True:
        depth += {"{": 1, "}": -1}.get(text[at], 0)
        at += 1
        if depth == 0:
            return text[start:at]


def events(body, patterns):
    """(kind, only one wave runs it) in program order."""
    rx = re.compile("|".join(f"(?P<{k}>{p})" for k, p in patterns.items()) + r"|(?P<one>if \(wave == 0\) \{)|(?P<o>\{)|(?P<c>\})")
    out, depth, one = [], 0, None
    for m in rx.finditer(body):
        k = m.lastgroup
        if k in ("one", "o"):
            if k == "one" and one is None:
                one = depth
            depth += 1
        elif k == "c":
            depth -= 1
            if one is not None and depth == one:
                one = None
        else:
            out.append((k, one is not None))
    return out


# k_lz_run: place emptied, and the awaited value after which others may look at it
LZ_EMPTIED = {"empty_a": "put_b", "empty_b": "put_a", "empty_z": "put_a"}
LZ_PATTERNS = {
    "drain": r"drain_memory\(\)",
    "barrier": r"__syncthreads\(\)",
    "empty_a": r"shared_store\(sla2 ",
    "empty_b": r"shared_store\(slb2 ",
    "put_a": r"shared_store\(sla \+",
    "put_b": r"shared_store\(slb \+",
    "put_z": r"shared_store\(at_byte\(\(unsigned\*\)zc",
    "empty_z": r"shared_store\(at_byte\(\(unsigned\*\)zp",
    "wait_a": r"sum_slots\(sla\)",
    "wait_b": r"sum_slots\(slb\)",
    "wait_z": r"load_halo\(zc\)",
}


@pytest.mark.parametrize("place", sorted(LZ_EMPTIED))
def test_lanczos_emptied_places_arrive_first(place):
    step = events(kernel_body("lanczos.hip", "k_lz_run", "for (int s = 0; s < steps; s++)"), LZ_PATTERNS)
    kinds = [k for k, _ in step]
    assert set(kinds) == set(LZ_PATTERNS), "the step no longer has the shape this test reads"
    two = step + step  # steps s and s + 1
    at = kinds.index(place)
    # the first publication that lets others look: of this step if it is still
    # ahead of the emptying, else of the next
    gate = next(i for i in range(at + 1, len(two)) if two[i][0] == LZ_EMPTIED[place])
    # the read it opens: the matching wait of the next step
    read = {"empty_a": "wait_a", "empty_b": "wait_b", "empty_z": "wait_z"}[place]
    first_read = len(step) + kinds.index(read)
    opened_by = max(i for i in range(first_read) if two[i][0] in ("put_a", "put_b"))
    assert gate <= opened_by
    drains = [i for i in range(at + 1, gate) if two[i][0] == "drain"]
    if step[at][1]:  # emptied by the publishing wave itself
        assert drains, f"{place} may still be on its way when {LZ_EMPTIED[place]} is published"
    else:  # by every wave: each drains, then a barrier, then one publishes
        assert any(not two[d][1] and any(two[b][0] == "barrier" for b in range(d + 1, gate)) for d in drains), place


def test_lanczos_emptied_after_all_have_read():
    step = [k for k, _ in events(kernel_body("lanczos.hip", "k_lz_run", "for (int s = 0; s < steps; s++)"),
                                 LZ_PATTERNS)]
    # the other set's alpha slots were read before their blocks published the
    # beta partials awaited at the end of the last step; its beta slots and the
    # old z before the alpha partials awaited in this one
    assert step.index("empty_b") > step.index("wait_a")
    assert step.index("empty_z") > step.index("wait_a")
    assert step.index("wait_b") > step.index("put_b") and step.index("wait_z") > step.index("put_z")


def test_filter_gives_up_between_barriers():
    """A wave leaves at `if (quit)` behind a barrier; nothing may set quit
    before every wave has passed that test, which the next barrier shows."""
    half = kernel_body("chebyshev.hip", "k_cheb_run", "const auto half =")
    await_frame = kernel_body("chebyshev.hip", "k_cheb_run", "const auto await_frame =")
    sets = r"\bquit = 1" + (r"|await_frame\(" if "quit" in await_frame else "")
    where = [m.start() for m in re.finditer(sets, half)]
    first_barrier, last_barrier = half.index("__syncthreads()"), half.rindex("__syncthreads()")
    assert where and all(first_barrier < i < last_barrier for i in where)
    assert half.index("if (quit) return") > last_barrier
