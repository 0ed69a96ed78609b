"""Words that decide whether a workgroup of the rounds engine goes on
(nsfps_runs.hip) are never written by the launch that tests them: workgroups
of one launch run in any order, so a wave could read such a word before the
write and its neighbour after it, and one of the two would leave ahead of a
barrier.  Read from the source, since no run shows it reliably."""

import os
import re

import pytest

from conftest import ROOT

SRC = os.path.join(ROOT, "ns_fps_amd", "csrc", "nsfps_runs.hip")


def bodies():
    """{name: body} of the file's functions, comments removed."""
    with open(SRC) as f:
        text = re.sub(r"//[^\n]*", "", f.read())
    out = {}
    for m in re.finditer(r"\b(k_\w+|record_samples|sel_replay|node_key|settle)\s*\([^;{}]*\)\s*\{", text):
        depth, at = 1, m.end()
        while depth:
            depth += {"{": 1, "}": -1}.get(text[at], 0)
            at += 1
        out[m.group(1)] = text[m.end():at]
    return out


def launches():
    """{kernel: its body with the bodies of the helpers that it calls}"""
    fns = bodies()
    return {k: b + "".join(h for n, h in fns.items() if not n.startswith("k_") and n + "(" in b)
            for k, b in fns.items() if k.startswith("k_")}


@pytest.mark.parametrize("word", [r"\*gptr\(c\.done\)", r"\brs\.fin\b"])
def test_no_launch_writes_a_word_that_it_tests(word):
    found = launches()
    assert {"k_update", "k_refine", "k_gather", "k_accept", "k_order", "k_runs_init"} <= set(found)
    writers = [k for k, b in found.items() if re.search(word + r"\s*=[^=]", b)]
    testers = [k for k, b in found.items() if re.search(word + r"(?!\s*=[^=])", b)]
    assert writers and testers
    assert not set(writers) & set(testers), (writers, testers)


def test_one_wave_reads_the_node_key_that_siblings_write():
    """The split update pass returns on the node's key ahead of a barrier
    while sibling workgroups write parts of it: wave 0 alone reads it there,
    and every wave takes its value from LDS after a barrier."""
    body = bodies()["k_update"]
    reads = [m.start() for m in re.finditer(r"node_key\(", body)]
    assert len(reads) == 1
    assert re.search(r"if \(wave == 0\) nkey = node_key\(c, gn\);", body)
    publish = re.search(r"tid == 0\) s_nkey = nkey;.*?__syncthreads\(\);\s*if \(SPLIT > 1\) nkey = uni\(s_nkey\);",
                        body, re.S)
    assert publish and reads[0] < publish.start()
    # nothing looks at the value before it is shared, but the wait for the reads
    between = re.sub(r"pin_sgpr\([^;]*;", "", body[reads[0]:publish.start()])
    assert between.count("nkey") == 0
