"""Every wave of a block takes the same decision on the device error word.

Another block of the launch (or a kernel on another stream) may set the word
between two waves' reads. A wave that left on its own reading would owe the
others what it should have put into LDS: a window of keys, a count, a share of a
walk that ends when all counts are zero. So a kernel that goes on to a barrier
decides through block_stops or __syncthreads_or, not wave by wave. A block of
one wave (K == 1) cannot disagree with itself.

Read from the sources: the race itself is not something to provoke on a GPU.
"""
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "gpu-nbody_amd", "csrc")
FILES = ["nb_force.hip", "nb_keys.hip", "nb_learned.hip", "nb_tree.hip"]
BARRIERS = {"__syncthreads", "__syncthreads_or"}


def _source(name):
    with open(os.path.join(CSRC, name)) as f:
        text = f.read()
    text = re.sub(r"//[^\n]*|/\*.*?\*/", "", text, flags=re.S)
    return re.sub(r"__attribute__\(\([^()]*(?:\([^()]*\))?\)\)|__launch_bounds__\([^()]*\)", "", text)


def _functions(text):
    """(name, body) of the device functions and kernels."""
    for m in re.finditer(r"__(?:global|device)__[^;{}()]*\b(\w+)\s*\(", text):
        at = text.find("{", m.end())
        if at < 0 or ";" in text[m.end():at]:
            continue
        depth, end = 1, at + 1
        while depth:
            depth += {"{": 1, "}": -1}.get(text[end], 0)
            end += 1
        yield m.group(1), text[at:end]


def _lone_exits(name):
    """Exits on the error word that each wave takes by itself, with a barrier
    after them: (function, statement)."""
    header, text = list(_functions(_source("nb_device.h"))), list(_functions(_source(name)))
    barriers = set(BARRIERS)
    while True:  # functions that reach a barrier
        more = {f for f, body in header + text if any(re.search(rf"\b{b}\b", body) for b in barriers)} - barriers
        if not more:
            break
        barriers |= more
    bad = []
    for f, body in text:
        words = [r"->\s*error"] + [rf"\b{v}\b" for v in re.findall(r"(\w+)\s*=\s*[\w.]+->\s*error\b", body)]
        for m in re.finditer(r"if\s*\(([^;{}]*)\)\s*return\b", body):
            cond = m.group(1)
            if not any(re.search(w, cond) for w in words) or re.search(r"\b(block_stops|__syncthreads_or)\b", cond):
                continue
            if re.search(r"\bK == 1\b", cond):
                continue
            if any(re.search(rf"\b{b}\b", body[m.end():]) for b in barriers):
                bad.append((f, " ".join(m.group(0).split())))
    return bad


@pytest.mark.parametrize("name", FILES)
def test_blocks_decide_together(name):
    assert _lone_exits(name) == []


def test_kernels_are_found():
    names = {f for name in FILES for f, _ in _functions(_source(name))}
    assert {"k_force", "coarse_traverse", "k_bintree", "k_bucket_sort", "k_link", "k_bbox", "k_scan_sums"} <= names
