"""Registers, LDS and scratch of launches that count on so many workgroups a compute unit or on no spilled registers, read from the built libraries' own
kernel metadata."""
import os
import re
import subprocess

import pytest

from nanollama_amd import _lib

LLVM = "/opt/rocm/llvm/bin/"

# kernel<template arguments>, wavefronts of a workgroup, workgroups on a compute unit (512 registers a SIMD lane over four SIMDs, 160 KB of LDS)
RESIDENT = [("pgemm_kernel<2, 4, 1, 1, 0, 0>", 4, 3), ("pgemm_kernel<2, 4, 1, 1, 1, 0>", 4, 3), ("pgemm_kernel<2, 4, 1, 1, 2, 0>", 4, 3)]
# decode attention of heads of 32 at four wavefronts: as many workgroups as LDS holds, eight; seven where the rotation comes with it
RESIDENT += [(f"attn_kernel<32, {g}, {fin}, {rope}, 256>", 4, 7 if rope == "true" else 8)
             for g in (1, 2) for fin, rope in (("false", "false"), ("false", "true"), ("true", "true"))]

# kernel<template arguments>, bytes of scratch a lane at most
SPILLED = [("pgemm_kernel<2, 4, 1, 1, 0, 0>", 20), ("pgemm_kernel<2, 8, 2, 1, 2, 0>", 0),
           ("gla_seg_kernel<float, 4, 2, 8, true, 4>", 0), ("gla_seg_kernel<float, 4, 4, 8, true, 4>", 0), ("gla_seg_kernel<float, 8, 4, 8, true, 1>", 0),
           ("gla_seg_kernel<float, 4, 2, 16, true, 1>", 0), ("gla_seg_kernel<float, 8, 4, 16, true, 1>", 0), ("gla_seg_kernel<float, 16, 4, 16, true, 1>", 92),
           ("gla_seg_kernel<float, 16, 4, 16, false, 1>", 0)]


def _kernels(lib, d):
    if not os.path.exists(LLVM + "clang-offload-bundler"):
        pytest.skip("no LLVM tools")
    run = lambda *a: subprocess.run(a, check=True, capture_output=True, text=True).stdout
    run(LLVM + "llvm-objcopy", "--dump-section", f".hip_fatbin={d}/fat", lib, "/dev/null")
    run(LLVM + "clang-offload-bundler", "--unbundle", "--type=o", "--targets=hipv4-amdgcn-amd-amdhsa--gfx950", f"--input={d}/fat", f"--output={d}/co")
    out, cur = {}, {}
    for line in run(LLVM + "llvm-readelf", "--notes", f"{d}/co").splitlines():
        m = re.match(r" +(?:- )?\.(symbol|vgpr_count|private_segment_fixed_size|group_segment_fixed_size|max_flat_workgroup_size): +(\S+)", line)
        if m:
            cur[m[1]] = m[2].strip("'")
        if ".wavefront_size" in line:
            out[cur.pop("symbol")] = cur
            cur = {}
    names = subprocess.run(["c++filt"], input="\n".join(n.removesuffix(".kd") for n in out), capture_output=True, text=True, check=True).stdout.splitlines()
    return dict(zip(names, out.values()))


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    _lib.lib()                                     # (builds it where nothing is built)
    return _kernels(_lib.LIB_PATH, tmp_path_factory.mktemp("co"))


@pytest.fixture(scope="module")
def stack_kernels(tmp_path_factory):
    _lib.stack_lib()
    return _kernels(_lib.STACK_LIB_PATH, tmp_path_factory.mktemp("co"))


@pytest.mark.parametrize("name,waves,groups", RESIDENT)
def test_workgroups_a_compute_unit(kernels, name, waves, groups):
    k, = [v for n, v in kernels.items() if name in n]
    assert int(k["max_flat_workgroup_size"]) == waves * 64
    registers = -(-int(k["vgpr_count"]) // 8) * 8
    assert 4 * (512 // registers) // waves >= groups and 160 * 1024 // int(k["group_segment_fixed_size"]) >= groups, k


@pytest.mark.parametrize("name,most", SPILLED)
def test_scratch(kernels, stack_kernels, name, most):
    k, = [v for n, v in {**kernels, **stack_kernels}.items() if name in n]
    assert int(k["private_segment_fixed_size"]) <= most, k


def test_float32_products_hold_no_residual_rows(stack_kernels):
    # ST_RESID takes the registers of ST_F32: rows requested in front of its loop were sixteen more
    plain, resid = ([int(v["vgpr_count"]) for n, v in stack_kernels.items() if f"direct_kernel<float, {epi}, 1, 1, 4, 4, 4>" in n] for epi in (0, 1))
    assert len(plain) == len(resid) == 1 and resid <= plain
