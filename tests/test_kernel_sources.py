"""Rules that the kernel sources keep, checked on the text (no GPU)."""
import re
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "hdcmamba_amd" / "csrc"
SOURCES = sorted(p for p in CSRC.iterdir() if p.suffix in (".hip", ".h"))

# Conditions around a barrier that every thread of a workgroup decides alike: sizes and options of the
# launch, the block's index, template parameters.
UNIFORM = {"(EPI == EPI_ROWLN)", "(kt + 1 < nk)", "((int)blockIdx.x < M)"}


def _strip(text):
    text = re.sub(r"/\*.*?\*/", lambda m: re.sub(r"[^\n]", " ", m.group()), text, flags=re.S)
    return re.sub(r"//[^\n]*", "", text)


def _guards(text):
    """(line, [heads of the enclosing if / else blocks]) of every workgroup barrier in ``text``; an else
    carries its if's condition."""
    text = _strip(text)
    out, stack, head, paren, closed = [], [], 0, 0, ""
    for m in re.finditer(r"[{};()]|__syncthreads\s*\(\s*\)|__builtin_amdgcn_s_barrier\s*\(\s*\)|\bplain_barrier\s*\(\s*\)", text):
        t = m.group()
        if t == "{":
            h = " ".join(text[head:m.start()].split())
            stack.append(closed + " " + h if h.startswith("else") and "if" not in h else h)
            head = m.end()
        elif t == "}":
            closed, head = stack.pop(), m.end()
        elif t == ";" and paren == 0:
            head = m.end()
        elif t in "()":
            paren += 1 if t == "(" else -1
        elif t != ";":
            own = " ".join(text[head:m.start()].split())
            out.append((text.count("\n", 0, m.start()) + 1, [h for h in [*stack, own] if re.match(r"(else\b|.*\bif\b)", h)]))
    return out


def _divergent(text):
    """Barriers under a condition that is neither a template parameter's nor in UNIFORM."""
    bad = []
    for line, heads in _guards(text):
        for h in heads:
            conds = [c.strip() for c in re.findall(r"\bif\s+(?!constexpr)(\(.*\))", h.replace("if constexpr", "if_constexpr"))]
            if any(c not in UNIFORM for c in conds):
                bad.append((line, h))
    return bad


def test_guard_parser():
    """The parser sees a barrier in either arm of a thread-dependent condition, and none of the
    others."""
    assert _divergent("void f() { if (j < 5) { g(); __syncthreads(); } }")
    assert _divergent("void f() { if (j < 5) { g(); } else { __syncthreads(); } }")
    assert _divergent("void f() { for (int i = 0; i < n; ++i) { if (w < 4) __syncthreads(); } }")
    assert not _divergent("void f() { if (j < 5) { g(); } __syncthreads(); }")
    assert not _divergent("void f() { if constexpr (A > 1) { __syncthreads(); } else { h(); __syncthreads(); } }")
    assert not _divergent("// if (x) {\nvoid f() { if (kt + 1 < nk) { __syncthreads(); } }")


@pytest.mark.parametrize("path", SOURCES, ids=lambda p: p.name)
def test_no_barrier_in_divergent_code(path):
    """A workgroup barrier that the two arms of a condition within one wave both reach (or only one
    does) is passed a different number of times by that wave than by the others: the waits of the
    workgroup no longer pair up, and what the barrier was to order is a race."""
    text = path.read_text()
    n = len(re.findall(r"__syncthreads\s*\(\s*\)|__builtin_amdgcn_s_barrier\s*\(\s*\)|\bplain_barrier\s*\(\s*\)", _strip(text)))
    assert len(_guards(text)) == n
    assert _divergent(text) == []
