"""Compiled load order of ragged_kernel: the checks of test_isa_order.py on the
kernel that runs the same pipeline over batches of several context lengths."""
import os
import re
import shutil
import subprocess

import pytest

import test_isa_order as isa

INSTANCES = [(d, hh, tt) for d, hh, vs, tt in isa.INSTANCES if not vs]
NAME = re.compile(r"^_ZN12_GLOBAL__N_113ragged_kernelILi(\d+)ELi(\d)ELi(\d+)E\S*:")


@pytest.fixture(scope="module")
def kernels():
    if not os.path.exists("/opt/rocm/bin/hipcc") and not shutil.which("hipcc"):
        pytest.skip("hipcc not available")
    subprocess.run(["make", "-s", "-C", isa.PKG, "asm"], check=True)
    lines = open(isa.ASM).read().splitlines()
    out = {}
    for i, ln in enumerate(lines):
        m = NAME.match(ln)
        if m:
            end = next(k for k in range(i, len(lines)) if lines[k].startswith(".Lfunc_end"))
            out[tuple(int(x) for x in m.groups())] = lines[i + 1:end]
    return out


def test_every_instantiation_found(kernels):
    assert set(kernels) == set(INSTANCES)


@pytest.mark.parametrize("d,hh,tt", INSTANCES)
def test_groups_and_waits(kernels, d, hh, tt):
    gpd = d // 64
    n_scale, n_v, n_reg = max(4 * tt * gpd * 4, 1024) // 1024, tt * 32 * gpd // 1024, tt // 16 * gpd
    body = kernels[(d, hh, tt)]
    with_loads = [(lb, tk) for lb, tk in isa.blocks(body) if tk]
    # prologue: the 4-byte prime load of a V slot and the first scale load
    # come first (the first explicit wait needs exactly those two)
    assert with_loads[0][1].startswith("DD"), with_loads[0]
    loop = with_loads[1:]
    assert loop
    group = "D" * (n_v + n_scale) + "g" * n_reg
    for lb, tk in loop:
        assert re.fullmatch("(%s)+" % group, tk), (lb, tk, group)
    loop = [(lb, tk) for lb, tk in isa.tokens(body) if any(t in ("D", "g") for t in tk)][1:]
    assert isa.check_waits(loop, n_v, n_scale, n_reg) >= 1


def test_no_scratch(kernels):
    metas = open(isa.ASM).read().split("  - .agpr_count:")[1:]
    seen = 0
    for m in metas:
        if "ragged_kernel" not in re.search(r"\.name:\s+(\S+)", m).group(1):
            continue
        seen += 1
        for key in ("private_segment_fixed_size", "vgpr_spill_count", "sgpr_spill_count"):
            assert int(re.search(r"\.%s:\s+(\d+)" % key, m).group(1)) == 0, m[:200]
    assert seen == len(INSTANCES)
