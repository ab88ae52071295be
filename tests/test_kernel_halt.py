"""Kernels that raise an error flag while their blocks meet at barriers are halted by a word they do not change.

Such a kernel may start a block while another one raises the flag.  If each wavefront read the flag itself
(LSD_HALT), some of a block could leave and the rest read what those were to leave in LDS; a kernel like that
reads what the launch before it found (LSD_HALT_LATCHED), which does not change while it runs.  Checked in the
source: the window is too narrow for a run to show it.
"""
import re
from pathlib import Path

import pytest

SRC = Path(__file__).resolve().parents[1] / "lsdem2.0_amd" / "csrc" / "kernels.hip"


def _functions(text):
    """Body and head of every function, struct members included, by name (overloads and templates joined)."""
    text = re.sub(r"//[^\n]*", "", text)
    text = re.sub(r"#define(?:[^\n]*\\\n)*[^\n]*", "", text)  # macros are looked for by name
    text = re.sub(r"__launch_bounds__\([^()]*\)", "", text)
    found = {}
    for m in re.finditer(r"(__device__|__global__)[^;{}]*?(\w+)\([^;{}]*\)\s*\{", text):
        depth, end = 1, m.end()
        while depth:
            depth += {"{": 1, "}": -1}.get(text[end], 0)
            end += 1
        head, body = found.get(m.group(2), ("", ""))
        found[m.group(2)] = (head + m.group(0), body + text[m.end():end])
    return found


FUNCTIONS = _functions(SRC.read_text())


def _reaches(name, word, seen=None):
    seen = set() if seen is None else seen
    if name in seen:
        return False
    seen.add(name)
    calls = set(re.findall(r"\b(\w+)\s*(?:<[^;<>()]*>)?\(", FUNCTIONS[name][1]))
    return word in calls or any(_reaches(c, word, seen) for c in calls if c in FUNCTIONS)


RAISING = [k for k, (head, _) in FUNCTIONS.items()
           if "__global__" in head and _reaches(k, "raiseFlag") and _reaches(k, "__syncthreads")]


def test_the_kernels_are_found():
    assert {"k_candidates", "k_broad_phase", "k_pairs_emit"} == set(RAISING)


@pytest.mark.parametrize("kernel", ["k_candidates", "k_broad_phase"])
def test_no_flag_of_this_launch_is_read_at_the_start(kernel):
    body = FUNCTIONS[kernel][1]
    start = body[:body.index("LSD_HALT_LATCHED(P)")]
    assert not re.search(r"LSD_HALT|LSD_GATE|devInt\[3\]|\breturn\b", start)
    if "rebuildFlagIdx" in body:  # its gate: nothing in this kernel may clear it
        assert not _reaches(kernel, "dropGates")
    # the launches before it keep what they found
    for k in ["k_pair_check"] if kernel == "k_candidates" else ["k_kick_drift", "k_reduce_drift", "k_reduce_drift_small"]:
        assert "LSD_HALT_LATCH(P)" in FUNCTIONS[k][1] and not _reaches(k, "raiseFlag")


def test_the_gated_emission_leaves_together():
    # its gate is cleared only by an overflowing list, for which every wavefront leaves before a barrier
    assert re.search(r"LSD_GATE\([^;]*;\s*if \(pairOverflow\(P\)\) \{[^{}]*return;\s*\}", FUNCTIONS["k_pairs_emit"][1])
