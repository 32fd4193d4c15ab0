"""The C-ABI library loads and exports every symbol the header declares (CPU)."""

import ctypes
import re
from pathlib import Path

import pytest
import torch

import jigsaw_amd
from jigsaw_amd import _lib

ROOT = Path(__file__).resolve().parents[1]
HEADER = ROOT / "include" / "jigsaw_hip.h"


def declared_symbols() -> list[str]:
    text = HEADER.read_text()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(jg_[a-z0-9_]+)\s*\(", text)))


def test_header_declares_entry_points():
    syms = declared_symbols()
    assert "jg_last_error" in syms and "jg_halo_assemble_3d" in syms
    assert len(syms) >= 10


def test_library_is_built_in_tree():
    assert jigsaw_amd.lib_path().exists(), "run `python -m jigsaw_amd.build` first"
    assert ROOT in jigsaw_amd.lib_path().parents


def test_every_declared_symbol_is_exported():
    lib = ctypes.CDLL(str(jigsaw_amd.lib_path()))
    missing = [s for s in declared_symbols() if not hasattr(lib, s)]
    assert not missing, f"declared in the header but not exported: {missing}"


def test_binding_table_matches_header():
    assert sorted(_lib.SIGNATURES) == declared_symbols()


def test_the_interface_holds_no_entry_points_of_the_tests():
    """What only tests call is bound apart from the header's entry points."""
    declared = declared_symbols()
    assert not [s for s in declared if s.endswith("_polls")]
    assert set(_lib._NOT_IN_THE_HEADER) == {"jg_gn_forward_polls", "jg_gn_backward_polls"} and not set(_lib._NOT_IN_THE_HEADER) & set(declared)


def test_abi_version_and_error_string():
    assert jigsaw_amd.abi_version() >= 1
    assert isinstance(jigsaw_amd.load().jg_last_error(), bytes)


def test_bad_arguments_are_rejected_without_a_gpu():
    """Argument validation happens on the host before any launch."""
    lib = jigsaw_amd.load()
    g = _lib.HaloGeom()
    g.planes = 1
    for a in range(3):
        g.size[a], g.lo[a], g.hi[a] = 4, 0, 0
    g.lo[2] = 9  # wider than the tile
    tab = _lib.VoidP27()
    rc = lib.jg_halo_assemble_3d(ctypes.c_void_p(16), tab, g, 2, None)
    assert rc == -1
    assert b"wider than the tile" in lib.jg_last_error()
    with pytest.raises(ValueError):
        _lib.check(rc, "jg_halo_assemble_3d")


@pytest.mark.parametrize("d", [64, 96])
@pytest.mark.parametrize("which", ["q", "out", "k", "dk"])
def test_misaligned_chunks_are_refused_without_a_gpu(which, d):
    """jg_attn_fwd_chunks / jg_attn_bwd_chunks move 16 bytes per lane: a tensor that starts off a 16-byte boundary is
    JG_ERR_UNSUPPORTED before anything is launched, at any length and head size."""
    lib = jigsaw_amd.load()
    at = {n: 0x1000 * (i + 1) + (2 if n == which else 0) for i, n in enumerate(("q", "out", "k", "v", "dq", "dk", "dv", "dout", "lse", "ws"))}
    p = {n: ctypes.c_void_p(v) for n, v in at.items()}
    one = lambda n: (ctypes.c_void_p * 1)(at[n])  # noqa: E731
    bf16 = _lib.dtype_code(torch.bfloat16)
    for sq, sk in ((100, 1000), (256, 128)):
        if which != "dk":
            rc = lib.jg_attn_fwd_chunks(p["out"], p["lse"], p["q"], one("k"), one("v"), 1, 2, sq, sk, d, 0.125, bf16, None)
            assert rc == -2 and b"aligned" in lib.jg_last_error()
        rc = lib.jg_attn_bwd_chunks(p["dq"], one("dk"), one("dv"), p["dout"], p["q"], one("k"), one("v"), 1, p["out"], p["lse"], 2,
                                    sq, sk, d, 0.125, bf16, p["ws"], 1 << 20, None)
        assert rc == -2 and b"aligned" in lib.jg_last_error()


class _ConvReduction(ctypes.Structure):
    _fields_ = ([(n, ctypes.c_int32) for n in ("kind", "dtype")] + [(n, ctypes.c_void_p) for n in ("part", "bias_part", "gw", "gb")]
                + [(n, ctypes.c_int32) for n in ("runs", "sub", "slots", "npairs", "pairs", "rows", "cols", "ci_step", "ci_blocks", "KD",
                                                 "cin", "cout", "bias_cout", "bias_parts")])


@pytest.mark.parametrize("wrong", [
    {"kind": 3}, {"kind": -1}, {"dtype": 7}, {"kind": 2}, {"part": None}, {"gw": None}, {"bias_part": None}, {"runs": 0}, {"runs": 35}, {"sub": 3},
    {"slots": 0}, {"npairs": 2}, {"pairs": 0}, {"rows": 0}, {"cols": -1}, {"ci_step": 0}, {"ci_blocks": 0}, {"KD": 0}, {"cin": 0}, {"cout": 0},
    {"bias_cout": 0}, {"bias_parts": 4}, {"kind": 2, "dtype": 0, "rows": 1, "cols": 1},
], ids=str)
def test_sums_that_no_weight_gradient_left_are_refused_without_a_gpu(wrong):
    """jg_conv_reduce and jg_halo_fold_border_reduce_3d take a descriptor that the weight gradient has filled, and none else."""
    lib, at = jigsaw_amd.load(), 0x1000
    good = dict(kind=1, dtype=1, part=at, bias_part=at, gw=at, gb=at, runs=36, sub=2, slots=4, npairs=1, pairs=1, rows=32, cols=1, ci_step=32,
                ci_blocks=1, KD=1, cin=8, cout=8, bias_cout=8, bias_parts=1)
    geom = _lib.HaloGeom()
    geom.planes = 8
    for a, (size, halo) in enumerate(((1, 0), (8, 1), (8, 1))):
        geom.size[a], geom.lo[a], geom.hi[a] = size, halo, halo
    left = _ConvReduction(**{**good, **wrong})
    strips = _lib.VoidP27()
    assert lib.jg_conv_reduce(ctypes.byref(left), None) == -1 and b"jg_conv_reduce" in lib.jg_last_error()
    rc = lib.jg_halo_fold_border_reduce_3d(ctypes.c_void_p(at), strips, geom, left.dtype if wrong.get("dtype") != 7 else 1, ctypes.byref(left), None)
    assert rc == -1 and b"sums" in lib.jg_last_error()
    none = _ConvReduction()
    assert lib.jg_conv_reduce(ctypes.byref(none), None) == 0  # nothing left


def test_weight_gradient_of_large_operands_keeps_its_kernel_without_a_gpu():
    """jg_proj_tn on bf16 operands of 2^32 bytes and more: the matrix-core kernel, which asks for its workspace (the
    one-product-at-a-time kernel needs none)."""
    lib = jigsaw_amd.load()
    bf16, at = _lib.dtype_code(torch.bfloat16), ctypes.c_void_p(0x1000)
    for rows, n, c in ((1 << 20, 2048, 64), (1 << 20, 64, 2048), (1 << 22, 1536, 512), (1 << 32, 8, 8)):
        assert lib.jg_proj_tn_workspace(rows, n, c) > 0
        rc = lib.jg_proj_tn(at, at, at, at, bf16, bf16, rows, n, c, 0, 0, 1, 1, 1, 1, None, 0, None)
        assert rc == -4 and b"workspace" in lib.jg_last_error(), (rc, rows, n, c)
