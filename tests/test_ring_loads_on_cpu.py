"""The waits of the 16x16x32 loop (csrc/gemm_core16.hpp) are counts of vector-memory operations in flight, and the counter
behind them has six bits.  Checked here on the listing of the built library for the forward, which may store a finished
tile's logits ahead of the next tile's first loads: on no path are more than 63 operations in flight when a load into
the ring has been issued."""

import os
import re
import shutil
import subprocess

import pytest

from test_mfma_distance_on_cpu import OBJDUMP, _kernels
from verl_amd import _abi

MOST = 63  # what s_waitcnt's vmcnt can tell apart

_VMCNT = re.compile(r"vmcnt\((\d+)\)")


def in_flight(code):
    """The largest number of vector-memory operations in flight behind a load into LDS, over all paths; and the number of such
    loads.  Counted up to 200, where a loop that stores without waiting ends up."""
    most, seen, todo = 0, {}, [(0, 0)]
    while todo:
        k, n = todo.pop()
        while k < len(code) and seen.get(k, -1) < n:
            seen[k] = n
            mnemonic, operands, target = code[k]
            if mnemonic == "s_waitcnt":
                wait = _VMCNT.search(operands)
                n = min(n, int(wait.group(1))) if wait else n
            elif mnemonic.startswith(("global_", "buffer_", "flat_", "scratch_")) and "inv" not in mnemonic and "wb" not in mnemonic:
                n = min(n + 1, 200)
                if "_lds" in mnemonic:
                    most = max(most, n)
            if mnemonic == "s_endpgm":
                break
            if target is not None:
                todo.append((target, n))
            if mnemonic == "s_branch":
                break
            k += 1
    return most, sum("_lds" in m for m, _, _ in code)


def test_the_count_sees_what_it_is_for():
    store, load, end = ("buffer_store_dwordx4", "v[0:3], v4, s[0:3], 0 offen", None), ("global_load_lds_dwordx4", "v[0:1], off", None), ("s_endpgm", "", None)
    wait = [("s_waitcnt", "vmcnt(24)", None)]
    assert in_flight([*[store] * 40, load, end]) == (41, 1)
    assert in_flight([*[store] * 40, *wait, load, load, end]) == (26, 2)
    assert in_flight([*[store] * 40, ("s_waitcnt", "lgkmcnt(0)", None), load, end])[0] == 41
    assert in_flight([*[store] * 8, ("s_cbranch_scc1", "3", 11), *wait * 2, load, end])[0] == 9  # (the branch skips the wait: 8 are fewer)
    assert in_flight([*[store] * 30, ("s_cbranch_scc1", "2", 32), *wait, load, end])[0] == 31
    assert in_flight([load, ("s_cbranch_scc0", "-2", 0), end])[0] == 200  # (a loop without a wait)


@pytest.mark.skipif(OBJDUMP is None, reason="no llvm-objdump")
def test_no_load_into_the_ring_overruns_the_counter(tmp_path):
    lib = shutil.copy(_abi.LIB_PATH, tmp_path)
    subprocess.run([OBJDUMP, "--offloading", lib], check=True, capture_output=True, cwd=tmp_path, timeout=120)
    kernels = {}
    for f in sorted(os.listdir(tmp_path)):
        if not f.endswith("amdgcn-amd-amdhsa--gfx950"):
            continue
        listing = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", str(tmp_path / f)], check=True, capture_output=True, text=True, timeout=120).stdout
        for name, code in _kernels(listing):
            if "lce_fwd16_kernel" in name:
                kernels[name] = in_flight(code)
    wrong = {name: most for name, (most, loads) in kernels.items() if most > MOST}
    assert not wrong, wrong
    assert len(kernels) >= 12 and all(loads >= 32 for _, loads in kernels.values()), kernels
    assert any(most > 32 for most, _ in kernels.values()), kernels  # (stores ahead of the loads are among what is counted)
