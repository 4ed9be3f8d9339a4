"""Registers and scratch of the built kernels, as the compiler records them in the library's code objects:
what the resident wavefronts of a kernel hang on, and what no result shows."""
import os
import re
import shutil
import struct
import subprocess

import pytest

from horses2d_amd import gpu

READELF = shutil.which("llvm-readelf", path=os.environ.get("PATH", "") + ":/opt/rocm/llvm/bin:/opt/rocm/lib/llvm/bin")


def _code_objects(data):
    """The gfx code objects of the offload bundles in a shared library."""
    magic, at = b"__CLANG_OFFLOAD_BUNDLE__", 0
    while (at := data.find(magic, at)) >= 0:
        count, p = struct.unpack_from("<Q", data, at + 24)[0], at + 32
        for _ in range(count if count < 16 else 0):
            offset, size, length = struct.unpack_from("<QQQ", data, p)
            if b"gfx" in data[p + 24:p + 24 + length] and size:
                yield data[at + offset:at + offset + size]
            p += 24 + length
        at += 24


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """name (with template arguments) -> (VGPRs, scratch bytes per lane)."""
    if READELF is None or not os.path.exists(gpu.LIB_PATH):
        pytest.skip("needs the built library and llvm-readelf")
    with open(gpu.LIB_PATH, "rb") as f:
        data = f.read()
    path, out = tmp_path_factory.mktemp("co") / "co.o", {}
    for co in _code_objects(data):
        path.write_bytes(co)
        notes = subprocess.run([READELF, "--notes", str(path)], capture_output=True, text=True, check=True).stdout
        for block in re.split(r"\n  - ", notes):
            field = {k: v for k, v in re.findall(r"\.(symbol|vgpr_count|private_segment_fixed_size):\s+(\S+)", block)}
            if field.get("symbol", "").endswith(".kd"):
                out[field["symbol"][:-3]] = (int(field["vgpr_count"]), int(field["private_segment_fixed_size"]))
    names = subprocess.run(["c++filt"], input="\n".join(out), capture_output=True, text=True, check=True).stdout
    found = {re.sub(r"^void |hg::", "", n).split("(")[0]: r for n, r in zip(names.splitlines(), out.values())}
    assert any(n.startswith("k_stage<") for n in found)
    return found


def _select(kernels, pattern, least):
    hits = {n: r for n, r in kernels.items() if re.fullmatch(pattern, n)}
    assert len(hits) >= least, (pattern, len(hits))
    return hits


def test_interior_penalty_gradient_with_boundary_kinds_keeps_five_wavefronts(kernels):
    """96 registers, five wavefronts per SIMD, at every order and tile: the gradient that runs each stage
    of the FP64 interior penalty with artificial viscosity."""
    for pattern, least in ((r"k_gradient<\d+, \d+, false, double, double, true>", 20),
                           (r"k_batch_gradient_p<\d+, [01], false, double, double>", 20)):
        for name, (vgprs, scratch) in _select(kernels, pattern, least).items():
            assert vgprs <= 96 and scratch == 0, (name, vgprs, scratch)


def test_exact_solver_keeps_its_wavefronts(kernels):
    """FP64 Navier-Stokes with the exact solver, and interior penalty with the solver chosen at run time:
    three wavefronts per SIMD (168 registers), without scratch at the low orders, where it does not pay;
    Euler: four in FP64 (128) and seven in FP32 (72), but at P = 8."""
    ns = _select(kernels, r"k_stage<\d+, \d+, true, (true|false), 2, double, double, (true|false)>", 48)
    ns.update(_select(kernels, r"k_stage<\d+, \d+, true, true, -1, double, double, false>", 12))
    for name, (vgprs, _) in ns.items():
        assert vgprs <= 168, (name, vgprs)
    for pattern in (r"k_stage<[2-7], \d+, true, true, 2, double, double, false>",
                    r"k_stage<[234], \d+, true, false, 2, double, double, false>"):
        for name, (_, scratch) in _select(kernels, pattern, 6).items():
            assert scratch == 0, (name, scratch)
    for name, (vgprs, _) in _select(kernels, r"k_stage<\d+, \d+, false, false, 2, double, double, (true|false)>", 24).items():
        assert vgprs <= 128, (name, vgprs)
    for name, (vgprs, _) in _select(kernels, r"k_stage<\d+, \d+, false, false, 2, float, float, false>", 20).items():
        assert vgprs <= 72 or name.startswith("k_stage<8,"), (name, vgprs)


def test_batched_br1_keeps_four_wavefronts(kernels):
    """FP64 BR1 in the batched stage kernels (which meshes of several orders run too): 128 registers, four
    wavefronts per SIMD, without scratch, with every solver but the exact one."""
    hits = _select(kernels, r"k_batch_stage<[01], true, false, [013], double, double>", 6)
    hits.update(_select(kernels, r"k_batch_stage_p<\d+, [01], true, false, [013], double, double>", 60))
    for name, (vgprs, scratch) in hits.items():
        assert vgprs <= 128 and scratch == 0, (name, vgprs, scratch)
