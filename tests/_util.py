"""Shared helpers for the test-suite (not collected by pytest)."""

from __future__ import annotations

import ctypes
import hashlib
import json
import pathlib
import re

import numpy as np
import torch

GOLDEN = pathlib.Path(__file__).resolve().parent / "golden"

ULP_BF16 = 2.0 ** -8  # spacing of bf16 values in [1, 2)


def load_npz(name: str) -> dict:
    with np.load(GOLDEN / name, allow_pickle=False) as z:
        return {k: z[k] for k in z.files}


def load_json(name: str) -> dict:
    return json.loads((GOLDEN / name).read_text())


def sha256_of(*tensors: torch.Tensor) -> str:
    h = hashlib.sha256()
    for t in tensors:
        h.update(t.contiguous().cpu().numpy().tobytes())
    return h.hexdigest()


def c1_inputs():
    """c1 = fp32 [4,256,32000] ~ N(0, 2^2), targets U[0,32000), CPU generator seed 0."""
    g = torch.Generator().manual_seed(0)
    logits = torch.randn(4, 256, 32000, generator=g) * 2.0
    target = torch.randint(0, 32000, (4, 256), generator=g)
    return logits, target


def header_functions() -> list[str]:
    """Names of the functions declared in include/nmce.h."""
    import re
    text = (pathlib.Path(__file__).resolve().parent.parent / "include" / "nmce.h").read_text()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(nmce_\w+)\s*\(", text)))


def assert_close_rel(actual, expected, rtol, atol=0.0, what=""):
    a = np.asarray(actual, dtype=np.float64)
    e = np.asarray(expected, dtype=np.float64)
    err = np.abs(a - e)
    bound = atol + rtol * np.abs(e)
    bad = ~(err <= bound)
    if bad.any():
        i = np.flatnonzero(bad.ravel())[0]
        raise AssertionError(
            f"{what}: {int(bad.sum())} of {a.size} outside rtol={rtol} atol={atol}; first at flat "
            f"{i}: got {a.ravel()[i]!r} expected {e.ravel()[i]!r}; max abs err {err.max():.3e}")


def assert_bf16_close(actual_bf16: np.ndarray, expected: np.ndarray, what="", ulps=1.0,
                      atol=0.0):
    """bf16 values within ``ulps`` bf16 ulps (relative 2^-8) of ``expected``."""
    assert_close_rel(actual_bf16, expected, rtol=ulps * ULP_BF16, atol=atol, what=what)


def mfma_hazards(asm: str) -> tuple[int, list[str]]:
    """(MFMAs, offending instructions) of a gfx950 listing: a VALU instruction
    that writes a source of an MFMA within two wait states before it, and any
    other than an MFMA that names a register which one wrote within 16 wait
    states after it. Both are looked for along every path: through branches, to
    a loop's head from its end, and across what lies between."""
    def regs(token):
        m = re.match(r"([va])(?:\[(\d+):(\d+)\]|(\d+))$", token)
        if not m:
            return frozenset()
        lo, hi = (m[2], m[3]) if m[2] else (m[4], m[4])
        return frozenset((m[1], i) for i in range(int(lo), int(hi) + 1))

    ops, labels, pending = [], {}, []  # pending: labels of the next instruction
    for line in asm.splitlines():
        text = line.split(";")[0].strip()
        label = re.match(r"([.\w$]+):$", text)
        if label:
            pending.append(label[1])
            continue
        op, _, rest = text.partition(" ")
        if not op or op.startswith("."):
            continue
        labels.update((name, len(ops)) for name in pending)
        pending = []
        tokens = [t.strip() for t in re.split(r",(?![^\[]*\])", rest)]
        ops.append((op, tokens, text, int(tokens[0], 0) + 1 if op == "s_nop" else 1))
    after = [[] for _ in ops]
    before = [[] for _ in ops]
    for i, (op, tokens, text, _) in enumerate(ops):
        if op in ("s_setpc_b64", "s_swappc_b64"):
            raise AssertionError(f"a call or computed branch: {text}")
        to = [labels[tokens[0]]] if op.startswith(("s_branch", "s_cbranch")) else []
        if not op.startswith(("s_branch", "s_endpgm")) and i + 1 < len(ops):
            to.append(i + 1)
        after[i] = to
        for j in to:
            before[j].append(i)

    def writes(o):
        if not o[0].startswith("v_") or o[0].startswith("v_mfma"):
            return frozenset()
        return frozenset().union(*map(regs, o[1][:2 if "swap" in o[0] else 1]))

    def walk(start, edges, limit, bad):
        """Instructions reached from `start` before `limit` wait states pass."""
        found, seen, todo = [], {}, [(j, 0) for j in edges[start]]
        while todo:
            j, waited = todo.pop()
            if waited >= limit or seen.get(j, limit) <= waited:
                continue
            seen[j] = waited
            if bad(ops[j]):
                found.append(f"{ops[j][2]}  against  {ops[start][2]}")
            todo += [(k, waited + ops[j][3]) for k in edges[j]]
        return found

    mfmas, offenders = 0, []
    for i, (op, tokens, _, _) in enumerate(ops):
        if not op.startswith("v_mfma"):
            continue
        mfmas += 1
        sources, written = frozenset().union(*map(regs, tokens[1:4])), regs(tokens[0])
        offenders += walk(i, before, 2, lambda o: writes(o) & sources)
        offenders += walk(i, after, 16, lambda o: not o[0].startswith("v_mfma") and
                          any(regs(t) & written for t in o[1]))
    return mfmas, offenders
