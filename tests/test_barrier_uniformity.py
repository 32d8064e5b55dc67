"""Every barrier of the device code that workgroups of several waves run is reached by
all of their waves: it stands under no condition and in no loop that could differ
between two waves (each wave of an ensemble's workgroup has its own elements, of which
some may be smooth, some rough, some absent).  Read from the sources: around a
__syncthreads() only compile-time conditions and loops with compile-time bounds."""

import os
import re

import pytest

from scratch_wadge_amd import build as B

# function -> file; the kernels that call them launch more than one wave per workgroup
FUNCTIONS = {
    "vol_body": "wadges.hip", "stage_body": "wadges.hip", "surf_kernel": "wadges.hip",
    "update_kernel": "wadges.hip", "batch_stage_flat": "wadges_batch.hpp",
    "team_volume": "wadges_team.hpp", "team_vol_kernel": "wadges_team.hpp",
    "team_stage_kernel": "wadges_team.hpp", "stage_wide": "wadges_wide.hpp",
    "update_vjp_kernel": "wadges_adjoint.hpp", "update_vjp_mfma_kernel": "wadges_adjoint.hpp",
    "proj_vjp_kernel": "wadges_adjoint.hpp", "project_kernel": "wadges_adjoint.hpp",
}

CONST = r"(?:\w+::)*[A-Z][A-Z0-9_]*(?:<[^<>]*>)?"       # NQ, S::NFQ, X::Vf::STEPS
LOOP = re.compile(rf"for \(int (\w+) = [\d]+; \1 < (?:{CONST}|\w+::{CONST}); (?:\+\+\1|\1 \+= {CONST})\)$")


def source(name):
    text = open(os.path.join(B.CSRC, name)).read()
    text = re.sub(r"//[^\n]*|/\*.*?\*/", "", text, flags=re.S)
    return re.sub(r"\s+", " ", text)


def body(text, function):
    """Text between the braces of the function's definition."""
    for m in re.finditer(rf"\b{function}\(", text):
        k, depth = m.end(), 1
        while depth:
            depth += {"(": 1, ")": -1}.get(text[k], 0)
            k += 1
        if text[k:].lstrip().startswith("{"):
            start = text.index("{", k) + 1
            end, depth = start, 1
            while depth:
                depth += {"{": 1, "}": -1}.get(text[end], 0)
                end += 1
            return text[start:end - 1]
    raise AssertionError(f"no definition of {function}")


def compile_time(header):
    """Whether a statement header lets all waves of a workgroup through alike."""
    header = header.strip()
    if not re.match(r"(?:else )?(?:if|for|while|switch|do)\b|else\b", header):
        return True                                   # a block, a lambda, an expression
    if re.match(r"(?:else )?if constexpr \(", header) or header == "else constexpr":
        return True
    if LOOP.match(header):
        return True
    m = re.match(r"if \((.*)\)$", header)
    return bool(m) and not re.sub(rf"{CONST}|\b\d+\b|[-+*/%<>=!&|() ]", "", m.group(1))


def barriers(code):
    """For each __syncthreads(): the statement headers around it."""
    stack, out, start, k, paren = [], [], 0, 0, 0
    closed_constexpr = [False]                         # the block just closed was `if constexpr`
    while k < len(code):
        c = code[k]
        paren += {"(": 1, ")": -1}.get(c, 0)
        if code.startswith("__syncthreads();", k):
            own = code[start:k].strip()                # a header without braces
            out.append(stack + ([own] if own else []))
            k += len("__syncthreads();")
            start = k
            continue
        if c == "{":
            head = code[start:k].strip()
            if head == "else" and closed_constexpr[-1]:
                head = "else constexpr"
            stack.append(head)
            closed_constexpr.append(False)
            start = k + 1
        elif c == "}":
            head = stack.pop()
            closed_constexpr.pop()
            closed_constexpr[-1] = "if constexpr" in head
            start = k + 1
        elif c == ";" and paren == 0:
            start = k + 1
        k += 1
    return out


@pytest.mark.parametrize("function", sorted(FUNCTIONS))
def test_barriers_are_met_by_every_wave(function):
    found = barriers(body(source(FUNCTIONS[function]), function))
    for headers in found:
        bad = [h for h in headers if not compile_time(h)]
        assert not bad, f"{function}: barrier under {bad}"
    if function != "batch_stage_flat":                 # its barriers are stage_body's
        assert found


def test_the_reader_finds_conditional_barriers():
    """The check itself, on code with barriers that waves could miss."""
    ok = "int a = 0; for (int h = 0; h < H; ++h) { f(); if (H > 1) __syncthreads(); } __syncthreads();"
    assert all(compile_time(h) for b in barriers(ok) for h in b) and len(barriers(ok)) == 2
    ok = "if constexpr (S::A) { g(); } else { __syncthreads(); } auto p = [&](int i) { __syncthreads(); };"
    assert all(compile_time(h) for b in barriers(ok) for h in b) and len(barriers(ok)) == 2
    for bad in ("if (LAZY && !smooth) { f(); __syncthreads(); }", "if (valid) __syncthreads();",
                "for (int t = 0; t < steps; ++t) { __syncthreads(); }", "while (it < n) { __syncthreads(); }",
                "if (x) { f(); } else { __syncthreads(); }"):
        assert any(not compile_time(h) for b in barriers(bad) for h in b), bad
