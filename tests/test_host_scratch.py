"""Every user of a stream's scratch holds that stream's lock (host-side, no GPU)."""

import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "lucid_amd", "csrc")
USE = re.compile(r"\b(workspace|stream_buffer|kept_buffer|call_buffer|sk_scratch)\(")
# what defines the buffers (a caller of sk_scratch holds the lock for it), and the start-up call of one thread
DEFINES = {("runtime.hip", "stream_buffer"), ("runtime.hip", "kept_buffer"), ("runtime.hip", "call_buffer"), ("runtime.hip", "workspace"),
           ("runtime.hip", "lq_init"), ("qgemm.hip", "sk_scratch")}


def _uses():
    for name in sorted(os.listdir(CSRC)):
        if not name.endswith((".hip", ".hpp")) or name == "common.hpp":
            continue
        lines = [re.sub(r"//.*", "", line) for line in open(os.path.join(CSRC, name))]
        for i, line in enumerate(lines):
            if USE.search(line):
                start = max(j for j in range(i + 1) if re.match(r"[A-Za-z].*\(", lines[j]))
                yield name, re.search(r"(\w+)\(", lines[start]).group(1), i, lines[start:i + 1]


def test_scratch_is_asked_for_under_the_streams_lock():
    """Two threads on one stream: the launches of one that pass data through the scratch must not be
    interleaved with another's, nor a buffer be outgrown and freed before it is launched on."""
    uses = [u for u in _uses() if (u[0], u[1]) not in DEFINES]
    assert len(uses) >= 12
    bad = [f"{name}:{i + 1} in {fn}" for name, fn, i, body in uses if not any("scratch_lock(" in b for b in body)]
    assert not bad, bad
