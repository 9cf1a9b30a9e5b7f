"""Loads that a kernel waits for by hand: the compiler takes a load's registers as written when its statement ends, so that a copy
of them before the wait would read what has not landed.  The listing of the built source says whether there is one: from every
load on, along every way through the kernel, nothing may touch its registers until a wait has covered it."""
import os
import re
import subprocess

import pytest

from llmopt_amd import build

KERNELS = os.path.join(os.path.dirname(build.__file__), "csrc", "kernels")
MEMORY = re.compile(r"(global|buffer|flat|scratch)_(load|store|atomic)")
LOAD = re.compile(r"(?:global|buffer|flat|scratch)_load_(?!lds)\w+ ([va]\[?[\d:]+\]?)")
REGISTER = re.compile(r"\b([va])(?:\[(\d+):(\d+)\]|(\d+)\b)")


def registers(text):
    return {(kind, r) for kind, first, last, one in REGISTER.findall(text)
            for r in (range(int(first), int(last) + 1) if first else (int(one),))}


def functions(listing):
    """Name and instructions of each, and where its labels point."""
    for name, body in re.findall(r"^(_Z\w+):[^\n]*\n(.*?)^\.Lfunc_end", listing, re.M | re.S):
        code, labels = [], {}
        for line in body.split("\n"):
            line = line.split(";")[0].strip()
            if line.endswith(":"):
                labels[line[:-1]] = len(code)
            elif line and not line.startswith("."):
                code.append(line)
        yield name, code, labels


def touched_in_flight(code, labels):
    """(load, instruction that touches its registers too early), loads return in the order of their requests."""
    after = []
    for at, line in enumerate(code):
        target = [labels[line.split()[1]]] if re.match(r"s_c?branch", line) else []
        after.append(target if re.match(r"s_(branch|endpgm)", line) and target else
                     [] if line.startswith("s_endpgm") else target + [at + 1])
    touches, memory = [registers(line) for line in code], [bool(MEMORY.match(line)) for line in code]
    waits = [int(m.group(1)) if (m := re.search(r"s_waitcnt.*vmcnt\((\d+)\)", line)) else None for line in code]
    for start, line in enumerate(code):
        load = LOAD.match(line)
        if not load or " lds" in line:
            continue
        goal, seen, way = registers(load.group(1)), set(), [(at, 0) for at in after[start]]
        while way:
            at, younger = way.pop()
            if at >= len(code) or (at, younger) in seen:
                continue
            seen.add((at, younger))
            if waits[at] is not None and waits[at] <= younger:
                continue
            if touches[at] & goal:
                yield line, code[at]
            way += [(to, min(younger + memory[at], 64)) for to in after[at]]


def test_a_copy_before_the_wait_is_found():
    code = ["global_load_dwordx4 v[4:7], v0, s[2:3]", "global_load_ushort v8, v0, s[2:3]", "v_mov_b32_e32 v9, v5",
            "s_waitcnt vmcnt(1)", "v_mov_b32_e32 v10, v6", "s_cbranch_scc1 top", "s_waitcnt vmcnt(0)", "v_mov_b32_e32 v11, v8", "s_endpgm"]
    assert list(touched_in_flight(code, {"top": 4})) == [(code[0], code[2])]
    assert list(touched_in_flight(code, {"top": 7}))[1:] == [(code[1], code[7])]


@pytest.fixture(scope="module")
def listing(tmp_path_factory):
    source, out = "w4a16_gemm.hip", str(tmp_path_factory.mktemp("listing") / "listing.s")
    subprocess.run(["hipcc", *build.COMMON, *build.PER_FILE.get(source, []), "--cuda-device-only", "-S",
                    os.path.join(KERNELS, source), "-o", out], check=True, capture_output=True)
    with open(out) as f:
        return list(functions(f.read()))


# The tiles of four phases (products and gated pairs) and of four stages.  (Those of two stages have their second step under a
# test: a way from the first to the first, which nothing takes but the listing holds.)
@pytest.mark.parametrize("kernel", ["w4a16_gemm_phased_kernelILb0E", "w4a16_gemm_phased_kernelILb1E",
                                    "w4a16_gemm_kernelILi1ELi2ELb0ELi4E", "w4a16_gemm_kernelILi1ELi2ELb1ELi4E"])
def test_nothing_touches_a_load_in_flight(listing, kernel):
    found = [(code, labels) for name, code, labels in listing if kernel in name]
    assert found
    for code, labels in found:
        assert any(LOAD.match(line) for line in code) and list(touched_in_flight(code, labels)) == []
