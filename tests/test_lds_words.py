"""The decision words that a workgroup's threads share in LDS (``sh``): a word that every thread reads is
not stored to, or counted in, before the next barrier. A wave that reads late would otherwise take another
decision than the others, and its barriers no longer pair with theirs. Read from the kernels' source: such a
race shows in outputs only now and then."""

from __future__ import annotations

import re
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "vinfer_amd" / "csrc"
BARRIERS = ("lds_barrier", "__syncthreads", "block_excl_scan", "block_sum", "block_max_u64", "sort_top", "sort_cands",
            "sample_bound", "kth_key20")
TOKEN = re.compile(r"\b(?P<barrier>" + "|".join(BARRIERS) + r")\s*[<(]"
                   r"|(?P<rmw>&)?\bsh\[(?P<word>[^\]]+)\](?P<store>\s*=(?!=))?"
                   r"|(?P<guard>\bif\s*\((?:tid < kWave|tid == 0|l == i)\))"
                   r"|(?P<brace>[{}])|(?P<semi>;)")


def functions(text: str):
    """(name, body) of every function that keeps its decisions in ``sh``, comments removed."""
    text = re.sub(r"//[^\n]*", "", text)
    for m in re.finditer(r"\b(\w+)\s*\([^;{}]*\)\s*\{", text):
        if m.start() and text.rfind("\n", 0, m.start()) >= 0 and not text[text.rfind("\n", 0, m.start()) + 1].isspace():
            body = text[m.end() - 1:text.find("\n}\n", m.end()) + 2]
            if re.search(r"\bsh\[", body):
                yield m.group(1), body


def conflicts(body: str) -> list[tuple[str, int]]:
    """(word, line) of every word both read by all threads and written between two barriers."""
    found, read, written = [], {}, set()
    depth, guards, pending = 0, [], False  # guards: brace depths of blocks that one wave runs
    for m in TOKEN.finditer(body):
        line = body.count("\n", 0, m.start())
        if m["barrier"]:
            if not guards:
                read, written = {}, set()
        elif m["guard"]:
            pending = True
        elif m["brace"] == "{":
            depth += 1
            if pending:
                guards.append(depth)
                pending = False
        elif m["brace"] == "}":
            if guards and guards[-1] == depth:
                guards.pop()
            depth -= 1
        elif m["semi"]:
            pending = False
        else:
            word = m["word"]
            if m["store"] or m["rmw"]:
                written.add(word)
                found += [(word, line)] if word in read or (word == "tid" and read) else []
            elif not (guards or pending):
                read[word] = line
                found += [(word, line)] if word in written or "tid" in written else []
    return found


@pytest.mark.parametrize("name", ["sample.cuh", "logprobs.cuh"])
def test_no_shared_word_is_read_and_written_between_two_barriers(name):
    seen = dict(functions((CSRC / name).read_text()))
    assert {"sample.cuh": {"tile_row", "lowered_pass"}, "logprobs.cuh": {"lp_stream", "lp_one_pass"}}[name] <= set(seen)
    assert {f: c for f, b in seen.items() if (c := conflicts(b))} == {}


def test_the_reading_finds_a_reset_beside_a_read():
    body = "{\n  lds_barrier();\n  const int n = sh[2];\n  if (n > 3) return;\n  if (tid == 0) sh[2] = 0;\n  lds_barrier();\n}\n"
    assert conflicts(body) == [("2", 4)]
    assert conflicts(body.replace("if (tid == 0) sh[2]", "lds_barrier(); sh[2]")) == []
