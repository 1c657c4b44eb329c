"""What the library is built of: the large kernel instances are there once each, and none that no call reaches."""

import os
import re
import shutil
import subprocess

import pytest

from test_mfma_distance_on_cpu import OBJDUMP
from verl_amd import _abi

# (names are mangled: types and template arguments as the compiler writes them)
_LARGE = re.compile(r"^_ZN3lce\d+(lce_(?:fwd|fwd16|fwd_few|bwd_chunk|bwd_chunk16|dh16|dw16|bwd_ds)_kernel)I(\S+?)EEEvNS_")


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    if OBJDUMP is None:
        pytest.skip("no llvm-objdump")
    where = tmp_path_factory.mktemp("objects")
    subprocess.run([OBJDUMP, "--offloading", shutil.copy(_abi.LIB_PATH, where)], check=True, capture_output=True, cwd=where, timeout=120)
    names = []
    for f in sorted(os.listdir(where)):
        if not f.endswith("amdgcn-amd-amdhsa--gfx950"):
            continue
        readelf = os.path.join(os.path.dirname(OBJDUMP), "llvm-readelf")
        table = subprocess.run([readelf, "-sW", str(where / f)], check=True, capture_output=True, text=True, timeout=120).stdout
        symbols = {line.split()[-1] for line in table.splitlines() if " FUNC " in line}
        names += [m.groups() for m in map(_LARGE.match, symbols) if m]
    assert len(names) >= 40
    return names


def test_no_kernel_is_there_twice(kernels):
    assert sorted(kernels) == sorted(set(kernels)), sorted(k for k in set(kernels) if kernels.count(k) > 1)


def test_only_tiles_that_a_call_reaches_keep_the_logits(kernels):
    """Of the 32x32x16 loop's forwards the 128-token tile of the two 16-bit types, with W marked as read once; the others belong to
    forced variants and to fp32, for which nothing is kept."""
    keep = [args for kernel, args in kernels if kernel == "lce_fwd_kernel" and args.endswith("Lb1")]
    assert len(keep) == 2 and all("Li256ELi128E" in args and args.endswith("Li1EEELb1") for args in keep), keep
