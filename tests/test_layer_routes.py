"""Which kernels a layer call takes, on the CPU: csrc/layer.c linked with
stand-ins for the launchers that log their names (tests/support/stub_launches.c).

Tensors off a 16-byte boundary must not reach kernels that load 16 bytes per
lane without a look at the address: the tiled path and the resident decode
kernels. Resident calls take the separate operators then, whose projections
fall back to scalar loads; FP8 calls the row dots, a decode token without the
launch it otherwise shares with its attention blocks, which load the caches that
way.
"""
import ctypes
import os
import subprocess

import numpy as np
import pytest

import lunelette_amd as lh
from lunelette_amd import build

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
TENSORS = ("qkv", "o", "gate", "up", "down", "input_norm", "post_norm", "x", "keys", "values")

FUSED = "qkv_rope:%d attention matvec:%d gateup_silu:%d matvec:%d"
FP8_ROWS = FUSED % (0, 0, 0, 0)
F32_ROWS = FUSED % (2, 2, 2, 2)
F32_OPERATORS = ("rmsnorm matvec:2 matvec:2 matvec:2 rope_append attention matvec:2 rmsnorm "
                 "matvec:2 matvec:2 silu_mul matvec:2")
TILES = ("norm_tile qkv_tile:%d attention_tiles residual_tile:%d norm_tile gateup_tile:%d "
         "residual_tile:%d")


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("routes") / "liblayer_stub.so")
    subprocess.run(["gcc", "-shared", "-Werror"] + build.C_FLAGS +
                   ["-I" + os.path.join(ROOT, "include"), "-I" + build.CSRC,
                    os.path.join(build.CSRC, "layer.c"),
                    os.path.join(ROOT, "tests", "support", "stub_launches.c"), "-o", out],
                   check=True)
    stub = ctypes.CDLL(out)
    for name in ("lh_workspace_create", "lh_workspace_destroy", "lh_workspace_set_tokens",
                 "lh_layer_forward"):
        entry, product = getattr(stub, name), getattr(lh.lib(), name)
        entry.argtypes, entry.restype = product.argtypes, product.restype
    return stub


def route(stub, path, count, moved=None, length=70, chained=0):
    """The launches of one layer call whose tensor `moved` lies 4 bytes past a
    16-byte boundary."""
    at = {name: 0x10000 * (i + 1) + (4 if name == moved else 0) for i, name in enumerate(TENSORS)}
    weights = lh.LayerWeights()
    for name in TENSORS[:5]:
        setattr(weights, ("f32_" if path == lh.PATH_RESIDENT else "") + name, at[name])
    weights.input_norm, weights.post_norm = at["input_norm"], at["post_norm"]
    ctypes.c_int.in_dll(stub, "stub_chained").value = chained
    log = (ctypes.c_char * 4096).in_dll(stub, "stub_log")
    ws = stub.lh_workspace_create(256, 16)
    assert ws
    try:
        ids = np.zeros(count, np.int64)
        assert stub.lh_workspace_set_tokens(ws, ids.ctypes.data_as(lh.c_int64_p), length, count,
                                            None) == 0
        log.value = b""
        assert stub.lh_layer_forward(ctypes.byref(weights), at["x"], at["keys"], at["values"], ws,
                                     path, None) == 0
        return log.value.decode()
    finally:
        stub.lh_workspace_destroy(ws)


def test_aligned_routes(stub):
    assert route(stub, lh.PATH_FUSED, 4) == FP8_ROWS
    assert route(stub, lh.PATH_FUSED, 5) == TILES % (0, 0, 0, 0)
    assert route(stub, lh.PATH_LOOKUP, 5) == TILES % (0, 0, 0, 0)
    assert route(stub, lh.PATH_RESIDENT, 1) == F32_ROWS
    assert route(stub, lh.PATH_RESIDENT, 2) == TILES % (1, 1, 1, 1)


@pytest.mark.parametrize("moved", TENSORS)
def test_unaligned_resident_tensor(stub, moved):
    for count in (1, 2, 9):
        assert route(stub, lh.PATH_RESIDENT, count, moved) == F32_OPERATORS


@pytest.mark.parametrize("moved", TENSORS)
def test_unaligned_fp8_tensor(stub, moved):
    for count in (4, 9):
        assert route(stub, lh.PATH_FUSED, count, moved) == FP8_ROWS


def test_unaligned_cache_is_not_chained(stub):
    chained = "qkv_attention:%d matvec:0 gateup_silu:%d matvec:0"
    for path, lookup in ((lh.PATH_FUSED, 0), (lh.PATH_LOOKUP, 1)):
        assert route(stub, path, 1, chained=1) == chained % (lookup, lookup)
        for moved in ("keys", "values"):
            assert route(stub, path, 1, moved, chained=1) == FUSED % (lookup, 0, lookup, 0)
