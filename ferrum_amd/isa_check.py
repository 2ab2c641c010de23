"""Build-time check of the hand-scheduled loads in this library's own kernels.

The sources in ``CHECKED_SOURCES`` and ``COUNTED_SOURCES`` issue memory instructions through
``asm volatile`` that the compiler cannot see the timing of:

* LDS-direct loads (``s_mov_b32 m0, <lds address>``, ``s_nop 0``,
  ``global_load_lds_dwordx4``): the statement writes M0, which an asm statement cannot
  name as a clobber on this target.  The invariant is that the compiler keeps nothing of
  its own in M0 inside these kernels: every mention of M0 in a kernel's code must be one
  of these statements.  A load into LDS may not be the next instruction behind the one that writes its M0: the
  compiler puts a wait state between the two, and so must the statement.
* register loads (``global_load_dwordx2/x4 vDST, vADDR, off`` in gemv_stream.hip): the
  destination registers hold the data only after the hand-placed ``s_waitcnt vmcnt(n)``
  that follows.  The invariant is that nothing between the load and that wait reads or
  writes the destination registers (no copy, no spill), and that the kernel has no
  scratch at all, so that no spill code can exist.
* ``s_waitcnt vmcnt(n)`` counts are the author's: they are right only if the compiler
  has put no vector-memory load of its own between the counted loads and the
  wait.  The check counts the vector-memory instructions outside asm statements between
  a hand-issued load and the hand-placed wait that covers it; there must be none, except
  stores behind LDS-direct loads, which can only lengthen the wait.

A second kind of kernel (``COUNTED_SOURCES``) leaves its register loads to the compiler, which orders and counts them,
and only says when its LDS-direct loads have landed: ``s_waitcnt vmcnt(n)``, n being the register loads the source issues behind them.
The invariant is that the generated code has at least n of them there
(``counted_violations``): with fewer, n outstanding loads could include one that the wait
is for.  In ``HAND_ISSUED_SOURCES`` all LDS-direct loads are asm statements: M0 and scratch are checked as above (``m0_violations``).
In the others the first ones are and the compiler issues the rest: M0 then belongs to the statements and to the compiler's own
LDS-direct loads, each of which finds the M0 that the compiler wrote for it.  Scratch may be there: no register is
loaded by a statement, and a spill between a load and its wait only lengthens the wait.

The check reads the assembly hipcc writes with ``-S`` for this library's own sources
(text, before it becomes a code object) and returns every violation it finds.  It is a
linear scan in program-text order, which is the order these straight-line stretches are
laid out in, and for counted loads also follows branches back over them.  ``ferrum_amd.build.build`` runs it and refuses to produce a library when
it fails; the hipcc release the kernels were validated with is recorded in
``VALIDATED_HIPCC`` and any other release is reported.
"""
from __future__ import annotations

import re

# `hipcc --version` of the toolchain every kernel here was validated with on gfx950
VALIDATED_HIPCC = "7.2.26015"

CHECKED_SOURCES = ("gemm.hip", "gemm_decoded.hip", "gemv_stream.hip", "gemm_skinny.hip", "probe.hip")
COUNTED_SOURCES = ("gemm_pairs.hip", "gemm_rows_q4_k.hip", "gemm_rows_q5_k.hip", "gemm_rows_q6_k.hip", "gemm_rows_iq4_xs.hip",
                   "gemm_rows_q8_0.hip")
HAND_ISSUED_SOURCES = ("gemm_pairs.hip",)   # counted, and all their LDS-direct loads are asm statements

_KERNEL_LABEL = re.compile(r"^(_Z\w+|\w+):\s*(;.*)?$")
_VREG_RANGE = re.compile(r"\bv\[(\d+):(\d+)\]")
_VREG_ONE = re.compile(r"\bv(\d+)\b")
_REG_LOAD = re.compile(r"^global_load_dwordx[234]\s+(v\[\d+:\d+\]|v\d+)\s*,")
_VMEM = re.compile(r"^(global_|buffer_|flat_|scratch_)(load|store|atomic)")
_LDS_LOAD = re.compile(r"^(global_load_lds_|buffer_load_\w+ .*\blds$)")
_STORE = re.compile(r"^(global_|buffer_|flat_)store")


def _no_wait_state(where: str, number: int, name: str) -> str:
    return f"{where}{number}: {name}: no wait state between M0 and the LDS-direct load that uses it"


def _vregs(text: str) -> set[int]:
    regs: set[int] = set()
    for lo, hi in _VREG_RANGE.findall(text):
        regs.update(range(int(lo), int(hi) + 1))
    for one in _VREG_ONE.findall(_VREG_RANGE.sub(" ", text)):
        regs.add(int(one))
    return regs


def _functions(asm: str, labels: bool = False):
    """Yields (name, [(line number, instruction text, inside an asm statement)]) per function; with `labels`
    the local labels are among the texts."""
    name, body, in_asm = None, [], False
    for number, raw in enumerate(asm.splitlines(), 1):
        line = raw.strip()
        if "#ASMSTART" in line:
            in_asm = True
            continue
        if "#ASMEND" in line:
            in_asm = False
            continue
        if not line or line.startswith(";") or line.startswith("//"):
            continue
        if line.startswith(".Lfunc_end"):
            if name is not None:
                yield name, body
            name, body = None, []
            continue
        if line.startswith("."):
            if labels and name is not None and line.startswith(".LBB") and line.split(";")[0].strip().endswith(":"):
                body.append((number, line.split(";")[0].strip(), False))
            continue
        label = _KERNEL_LABEL.match(line)
        if label and not line.startswith(".L"):
            name, body, in_asm = label.group(1), [], False
            continue
        if name is not None:
            body.append((number, line.split(";")[0].strip(), in_asm))


def violations(asm: str, source: str = "", counted: bool = False) -> list[str]:
    """Every break of the invariants in the module docstring found in `asm` (the text
    `hipcc -S --offload-device-only` writes for one source)."""
    found: list[str] = []
    where = (source + ":") if source else ""
    scratch = {}
    current = None
    for raw in asm.splitlines():
        line = raw.strip()
        if line.startswith(".amdhsa_kernel"):
            current = line.split()[1]
        elif line.startswith(".amdhsa_private_segment_fixed_size") and current:
            scratch[current] = int(line.split()[1])
    for name, body in _functions(asm):
        hand_loads = False
        for at, (number, text, in_asm) in enumerate(body):
            if not text:
                continue
            mentions_m0 = re.search(r"\bm0\b", text) is not None
            if mentions_m0:
                nxt = body[at + 1][1] if at + 1 < len(body) else ""
                nxt2 = body[at + 2][1] if at + 2 < len(body) else ""
                ours = in_asm and text.startswith("s_mov_b32 m0,") and (
                    nxt.startswith("global_load_lds_") or (nxt.startswith("s_nop") and nxt2.startswith("global_load_lds_")))
                if not ours:
                    found.append(f"{where}{number}: {name}: M0 is used outside an LDS-direct load statement: {text}")
                elif not nxt.startswith("s_nop"):
                    found.append(_no_wait_state(where, number, name))
            if in_asm and text.startswith("global_load_lds_"):
                hand_loads = True
                if not counted:
                    found.extend(_scan_to_wait(body, at, set(), name, where))
            match = _REG_LOAD.match(text) if in_asm else None
            if match:
                hand_loads = True
                found.extend(_scan_to_wait(body, at, _vregs(match.group(1)), name, where))
        if hand_loads and scratch.get(name, 0) != 0:
            found.append(f"{where}{name}: a kernel with hand-scheduled loads uses {scratch[name]} bytes of scratch")
    return found


def counted_violations(asm: str, source: str = "") -> list[str]:
    """Kernels that wait for LDS-direct loads by counting the register loads behind them.  Behind every run of the former,
    up to the next hand-placed wait, the next run or the function's end, there must be at least as many of the latter as the
    hand-placed ``s_waitcnt vmcnt(n)`` leave outstanding: the largest n of the kernel where the compiler issues the runs; in
    ``HAND_ISSUED_SOURCES``, whose last rounds request nothing behind a run and wait for all, the n of the next wait, and one
    must follow.  Likewise along every branch back over a run, up to the first wait behind its target.  The compiler uses M0 for
    LDS-direct loads of its own alone and writes it for each run of them."""
    found: list[str] = []
    where = (source + ":") if source else ""
    next_wait_counts = source in HAND_ISSUED_SOURCES
    for name, body in _functions(asm, labels=True):
        at_label = {text[:-1]: at for at, (_, text, _) in enumerate(body) if text.endswith(":")}
        waits = {at: int(m.group(1)) for at, (_, text, in_asm) in enumerate(body)
                 if in_asm and (m := re.match(r"s_waitcnt vmcnt\((\d+)\)", text))}
        lds = [at for at, (_, text, _) in enumerate(body) if _LDS_LOAD.match(text)]
        theirs = True    # M0 is as the compiler last wrote it
        for at, (number, text, in_asm) in enumerate(body):
            if re.match(r"s_\w+ m0,", text):
                theirs = not in_asm
                if at + 1 < len(body) and _LDS_LOAD.match(body[at + 1][1]):
                    found.append(_no_wait_state(where, number, name))
                own = next((asm for _, t, asm in body[at + 1:] if _LDS_LOAD.match(t)), None) is False
                if not in_asm and (not own or "m0" in text.split(",", 1)[1]):
                    found.append(f"{where}{number}: {name}: M0 is used outside an LDS-direct load: {text}")
            elif re.search(r"\bm0\b", text):
                found.append(f"{where}{number}: {name}: M0 is used outside an LDS-direct load: {text}")
            elif _LDS_LOAD.match(text) and not in_asm and not theirs:
                found.append(f"{where}{number}: {name}: the compiler's LDS-direct load finds M0 as an asm statement left it")
        if lds and not waits:
            found.append(f"{where}{body[lds[0]][0]}: {name}: LDS-direct loads without a hand-placed wait")
            continue
        for at in lds:
            number = body[at][0]
            behind, needs, end = 0, [], "the function's end"
            for here in range(at + 1, len(body)):
                _, text, _ = body[here]
                if _LDS_LOAD.match(text):
                    if behind == 0:
                        end = "more of the run"
                        break
                    if not next_wait_counts:
                        end = "the next run"
                        break
                elif here in waits:
                    end = "a wait"
                    break
                elif text.startswith(("global_load_", "buffer_load_")):
                    behind += 1
                target = text.split()[-1] if text.startswith(("s_cbranch", "s_branch")) else None
                if target in at_label and at_label[target] < at:
                    needs.append((next((waits[w] for w in sorted(waits) if w >= at_label[target]), None), behind))
            if end == "more of the run":    # its last load counts
                continue
            if not next_wait_counts:
                needs.append((max(waits.values()), behind))
            else:
                needs.append((waits[here] if end == "a wait" else None, behind))
            for allowed, behind in needs:
                if allowed is None:
                    found.append(f"{where}{number}: {name}: no hand-placed wait follows this LDS-direct load")
                elif behind < allowed:
                    found.append(f"{where}{number}: {name}: {behind} register loads follow this LDS-direct load, "
                                 f"the wait for it allows {allowed} outstanding")
    return found


def m0_violations(asm: str, source: str = "") -> list[str]:
    """Of the invariants of ``violations``, those that do not depend on what else is in flight: M0 belongs to the
    LDS-direct statements alone, and a kernel with such statements has no scratch."""
    return violations(asm, source, counted=True)


def _scan_to_wait(body, at, dst: set[int], name: str, where: str) -> list[str]:
    found = []
    number0 = body[at][0]
    for number, text, in_asm in body[at + 1:]:
        if in_asm and text.startswith("s_waitcnt") and "vmcnt" in text:
            return found
        if text.startswith("s_endpgm") or text.startswith("s_setpc"):
            break
        if in_asm and (_REG_LOAD.match(text) or text.startswith("global_load_lds_") or text.startswith("s_mov_b32 m0,")
                       or text.startswith("s_nop")):
            # the following hand-issued loads of the same run; a destination may not be reused
            if dst and _REG_LOAD.match(text) and dst & _vregs(_REG_LOAD.match(text).group(1)):
                found.append(f"{where}{number}: {name}: a second load targets registers still in flight since line {number0}")
            continue
        if dst and dst & _vregs(text):
            found.append(f"{where}{number}: {name}: '{text}' touches registers loaded at line {number0} before the wait")
        # A store of the compiler's between an LDS-direct load and its wait can only lengthen the wait:
        # loads retire in order among themselves, so "at most n operations outstanding", n the later
        # loads, still means the awaited load has landed whether or not a store is among the n.
        if not dst and not in_asm and _STORE.match(text):
            continue
        if not in_asm and _VMEM.match(text):
            found.append(f"{where}{number}: {name}: the compiler's '{text.split()[0]}' sits between the load at line "
                         f"{number0} and its hand-counted wait")
    # no hand-placed wait follows: LDS-direct loads at the end of a kernel's text are waited
    # for by a later stretch the scan cannot order; register loads must always find theirs
    if dst:
        found.append(f"{where}{number0}: {name}: no hand-placed s_waitcnt vmcnt follows this register load")
    return found


def hipcc_release(version_text: str) -> str:
    match = re.search(r"HIP version:\s*([0-9.]+)", version_text)
    return match.group(1) if match else ""
