"""The 16x16x32 loop issues its MFMAs as inline assembly (csrc/gemm_core16.hpp), so the compiler does not know that their
results arrive late: what keeps an accumulator from being read too early is where the code that reads it ends up.  Checked
here on the listing of the built library: on no path is an AGPR that such an MFMA writes touched by anything but MFMAs that
accumulate into it within 18 wait states, what the longest of these instructions needs (an instruction counts one, s_nop n
counts n + 1; MFMAs, which take longer to issue, count one too)."""

import os
import re
import shutil
import subprocess

import pytest

from verl_amd import _abi

OBJDUMP = next((p for p in ("/opt/rocm/llvm/bin/llvm-objdump", shutil.which("llvm-objdump")) if p and os.path.exists(p)), None)
WAIT_STATES = 18

_LINE = re.compile(r"^\s+([a-z]\w+)\s*(.*?)\s*//\s*([0-9A-F]+):\s*[0-9A-F ]+(?:<(.+?)(?:\+0x([0-9a-f]+))?>)?\s*$")
_HEAD = re.compile(r"^([0-9a-f]+) <(.+)>:$")
_AGPR = re.compile(r"\ba\[(\d+):(\d+)\]|\ba(\d+)\b")


def _agprs(text):
    return {r for lo, hi, one in _AGPR.findall(text) for r in (range(int(lo), int(hi) + 1) if lo else (int(one),))}


def _kernels(listing):
    """(name, instructions) of every kernel; an instruction: mnemonic, operands, index of the branch target or None."""
    name, start, at, code = None, 0, {}, []
    for line in listing.splitlines() + ["0000000000000000 <end>:"]:
        head = _HEAD.match(line)
        if head:
            if name and any(m.startswith("v_mfma_f32_16x16x32") for m, _, _ in code):
                yield name, [(m, ops, at.get(t)) for m, ops, t in code]
            name, start, at, code = head.group(2), int(head.group(1), 16), {}, []
            continue
        got = _LINE.match(line)
        if got and name:
            mnemonic, operands, address, target, offset = got.groups()
            at[int(address, 16)] = len(code)
            code.append((mnemonic, operands, start + int(offset or "0", 16) if target == name and "branch" in mnemonic else None))


def too_early(code, wait_states=WAIT_STATES):
    """The first access to an accumulator that is too close behind the MFMA that writes it, or None; and how many MFMAs have
    been looked at."""
    looked = 0
    for i, (mnemonic, operands, _) in enumerate(code):
        if not mnemonic.startswith("v_mfma_f32_16x16x32"):
            continue
        result = _agprs(operands.split(", ")[0])
        if not result:
            continue  # (in ordinary registers: a builtin's, which the compiler knows)
        looked += 1
        seen, todo = {}, [(i + 1, wait_states)]
        while todo:
            k, left = todo.pop()
            while left > 0 and k < len(code) and seen.get(k, 0) < left:
                seen[k] = left
                m, ops, target = code[k]
                if m.startswith("v_mfma"):
                    d, a, b, c = ops.split(", ")[:4]
                    touched = result & (_agprs(a) | _agprs(b))
                    if result & _agprs(d) and _agprs(d) != result or result & _agprs(c) and _agprs(c) != result:
                        touched = result  # (part of it: not the chain that the matrix pipe orders)
                else:
                    touched = result & _agprs(ops)
                if touched:
                    return f"{code[i][0]} {code[i][1]}, then {m} {ops} within {wait_states - left + 1} wait states", looked
                if m == "s_endpgm":
                    break
                left -= int(ops, 0) + 1 if m == "s_nop" else 1
                if target is not None:
                    todo.append((target, left))
                if m == "s_branch":
                    break
                k += 1
    return None, looked


def test_the_check_sees_what_it_is_for():
    mfma = ("v_mfma_f32_16x16x32_bf16", "a[0:3], v[0:3], v[4:7], a[0:3]", None)
    filler = [("v_mov_b32_e32", "v9, v8", None)]
    read = ("v_accvgpr_read_b32", "v1, a2", None)
    end = ("s_endpgm", "", None)
    assert too_early([mfma, mfma, *filler * 17, read, end])[0]
    assert too_early([mfma, mfma, *filler * 18, read, end]) == (None, 2)
    assert too_early([mfma, ("s_nop", "15", None), ("s_nop", "1", None), read, end]) == (None, 1)
    assert too_early([mfma, ("s_nop", "15", None), ("s_nop", "0", None), read, end])[0]
    assert too_early([mfma, ("s_cbranch_scc1", "3", 20), *filler * 18, ("s_branch", "1", 21), read, end])[0]  # (at the branch's target)
    assert too_early([mfma, ("ds_write_b128", "v1, a[0:3]", None), end])[0]
    assert too_early([mfma, ("v_mfma_f32_16x16x32_bf16", "a[4:7], a[0:3], v[4:7], a[4:7]", None), end])[0]


@pytest.mark.skipif(OBJDUMP is None, reason="no llvm-objdump")
def test_no_accumulator_is_read_before_it_is_there(tmp_path):
    lib = shutil.copy(_abi.LIB_PATH, tmp_path)
    subprocess.run([OBJDUMP, "--offloading", lib], check=True, capture_output=True, cwd=tmp_path, timeout=120)
    looked, kernels = 0, 0
    for f in sorted(os.listdir(tmp_path)):
        if not f.endswith("amdgcn-amd-amdhsa--gfx950"):
            continue
        listing = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", str(tmp_path / f)], check=True, capture_output=True, text=True, timeout=120).stdout
        for name, code in _kernels(listing):
            wrong, n = too_early(code)
            assert wrong is None, f"{name}: {wrong}"
            looked, kernels = looked + n, kernels + (n > 0)
    assert kernels >= 12 and looked >= 12 * 64, (kernels, looked)  # (forward, d_logits and gradient GEMMs of three element types)


@pytest.mark.skipif(OBJDUMP is None, reason="no llvm-objdump")
def test_no_kernel_of_the_loop_uses_scratch_memory(tmp_path):
    """A reload from scratch memory waits for every load and store issued before it, the next tile's among them."""
    lib = shutil.copy(_abi.LIB_PATH, tmp_path)
    subprocess.run([OBJDUMP, "--offloading", lib], check=True, capture_output=True, cwd=tmp_path, timeout=120)
    readelf = os.path.join(os.path.dirname(OBJDUMP), "llvm-readelf")
    seen = set()
    for f in sorted(os.listdir(tmp_path)):
        if not f.endswith("amdgcn-amd-amdhsa--gfx950"):
            continue
        notes = subprocess.run([readelf, "--notes", str(tmp_path / f)], check=True, capture_output=True, text=True, timeout=120).stdout
        for name, rest in re.findall(r"\.name:\s+(\S*GemmCfg16\S*)(.*?)\.wavefront_size", notes, re.S):
            assert re.search(r"\.private_segment_fixed_size:\s+(\d+)", rest).group(1) == "0", name
            seen.add(name)
    assert len(seen) >= 16, seen
