"""Which kernels of the library's calls wait for other workgroups. A workgroup that polls for what
another one writes keeps its place on the device meanwhile, so a launch that polls ends only if the
device holds enough of it at once: launches overlapping on several streams, a CU mask or a partitioned
device break that. Of the calls in include/llm_amd/kernels.h only the one-pass attention waits, and its
contract says so."""
import re

from conftest import PKG_DIR, ROOT

POLLS = re.compile(r"\bop_poll\b|\bwait_gives_up\b|\w*SPIN_LIMIT\b|for \(;;\)|while \((?:true|1)\)")


def functions(text):
    """{name: body} of the function definitions of a source."""
    text = re.sub(r"//[^\n]*|/\*.*?\*/", "", text, flags=re.S)
    found = {}
    for m in re.finditer(r"(\w+)\s*\([^;{}()]*\)\s*\{", text):
        if m.group(1) in ("if", "for", "while", "switch") or text[m.start() - 1] == "]":
            continue
        depth, end = 1, m.end()
        while depth:
            depth += {"{": 1, "}": -1}.get(text[end], 0)
            end += 1
        found[m.group(1)] = text[m.end():end]
    return found


def test_only_the_one_pass_attention_waits():
    bodies = functions((PKG_DIR / "csrc" / "kernels.hip").read_text())
    kernels = {n for n in bodies if n.endswith("_kernel")}
    assert {"attn_scores_kernel", "attn_rope_scores_kernel", "attn_pv_kernel", "attn_combine_kernel",
            "attn_one_pass_kernel", "sample_sums_kernel", "argmax_stage2_kernel"} <= kernels
    waits = {n for n, body in bodies.items() if POLLS.search(body)}
    while True:  # and what calls a function that polls
        more = {n for n, body in bodies.items()
                if n not in waits and any(re.search(r"\b%s\b" % w, body) for w in waits)}
        if not more:
            break
        waits |= more
    assert waits & kernels == {"attn_one_pass_kernel"}
    contract = (ROOT / "include" / "llm_amd" / "kernels.h").read_text()
    assert re.search(r"workgroups wait for each\s+\*\s+other", contract)


def test_the_draw_keeps_nothing_in_out():
    """`out` belongs to the caller, who may give the same one to overlapping calls: no kernel of
    sample_forward reads it."""
    bodies = functions((PKG_DIR / "csrc" / "kernels.hip").read_text())
    for name in ("sample_kernel", "sample_sums_kernel"):
        uses = re.findall(r"[^;{}]*\bout\b[^;{}]*", bodies[name])
        assert uses and all(re.fullmatch(r"\s*(if \(t == 0\)\s*)?\*out = chosen", u) for u in uses), uses
