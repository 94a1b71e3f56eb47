"""The workspace's layout (csrc/speedy_workspace.hpp) and the tags by which a block of the
single launch knows a word of its own call.

A workspace serves calls on several grids, so a tagged word of one grid must not lie
where another grid's call writes anything else: a level set, a chunk word or an integer
of an argument block there could carry the tag of a later call, whose sums would then
take it for a partial.  (Before, the places went with the grid: last_s of 300 members
covered the tagged partials of the first nine blocks of a 128 x 64 adjoint.)"""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from jcm_amd import _native

HERE = os.path.dirname(os.path.abspath(__file__))
GRIDS = [(64, 32, 1), (96, 48, 1), (128, 64, 1), (256, 128, 1), (256, 128, 4), (16, 16, 62), (16, 16, 512),
         (17, 16, 63), (33, 19, 3), (1280, 640, 1), (640, 320, 3), (512, 256, 3), (96, 48, 300), (96, 48, 64),
         (8, 8, 300), (4, 2, 1), (1, 1, 4095), (5, 7, 333), (16, 17, 4000), (1, 256, 2000)]
REGIONS = ("last_s", "partial", "prm", "bud", "desc", "total")


@pytest.fixture(scope="module")
def ws(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("ws") / "libws.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-o", so,
                    os.path.join(HERE, "host_column", "workspace_host.cpp")], check=True)
    lib = ctypes.CDLL(so)
    for f in (lib.ws_call_tag, lib.ws_next_generation):
        f.restype, f.argtypes = ctypes.c_uint32, [ctypes.c_uint32]
    lib.ws_tagged_word.restype, lib.ws_tagged_word.argtypes = ctypes.c_uint64, [ctypes.c_uint32] * 2
    lib.ws_grid.argtypes = [ctypes.c_int64, ctypes.c_int64, ctypes.c_int32, ctypes.c_uint64, ctypes.c_uint64,
                            ctypes.POINTER(ctypes.c_uint64)]
    return lib


def _constants(ws):
    c = (ctypes.c_uint64 * 9)()
    ws.ws_constants(c)
    return dict(zip(("header", "words", "tags", "blocks", "block", "params", "budgets", "arrived", "merged"), c))


def _grid(ws, grid, desc=2048, tags=None):
    out = (ctypes.c_uint64 * 9)()
    ws.ws_grid(*grid, desc, _constants(ws)["tags"] if tags is None else tags, out)
    return dict(zip(("nblk", "ls_blocks", "jmax") + REGIONS, out))


@pytest.mark.parametrize("grid", GRIDS)
def test_only_tagged_words_lie_among_the_tagged_words(ws, grid):
    k, g = _constants(ws), _grid(ws, grid)
    nlon, nlat, nmember = grid
    assert 4 * (k["arrived"] + k["merged"]) <= k["header"]
    begin, end = k["header"], k["header"] + k["tags"]
    # both kinds of tagged words, at places that do not go with the grid
    if g["nblk"] <= k["blocks"] and nlon * nlat >= k["block"]:
        last = g["nblk"] - 1
        assert begin + 8 * (2 * last + 1) + 8 <= begin + k["words"]
        assert begin + k["words"] + 8 * ((2 * last + 1) * k["params"] + k["params"] - 1) + 8 <= end
    # everything else of every grid lies past them, each region where the one before ends
    sizes = {"last_s": 4 * nmember, "partial": 4 * g["ls_blocks"] * g["jmax"]}
    wide = nlon * nlat >= k["block"]
    sizes["prm"] = 4 * k["params"] * (2 * g["nblk"] if wide else nlon * nlat * nmember)
    sizes["bud"] = 8 * k["budgets"] * (g["nblk"] + nmember if wide else nlon * nlat * nmember)
    sizes["desc"] = 2048
    for name, after in zip(REGIONS, REGIONS[1:]):
        assert g[name] >= end and g[name] % 256 == 0
        assert g[name] + sizes[name] <= g[after], name
    assert _grid(ws, grid, tags=0)["total"] == g["total"] - k["tags"]


def test_layout_is_the_library_s(ws):
    lib = _native.load()
    desc = {lib.speedy_workspace_bytes(*g) - _grid(ws, g, desc=0)["total"] for g in GRIDS}
    assert len(desc) == 1 and 512 <= desc.pop() <= 8192   # the argument block


@pytest.mark.parametrize("grid", [g for g in GRIDS if g[0] * g[1] >= 256])
def test_budget_partials_have_places_of_their_own(ws, grid):
    k, g = _constants(ws), _grid(ws, grid)
    ncol, ntot = grid[0] * grid[1], grid[0] * grid[1] * grid[2]
    b = np.arange(g["nblk"])
    first, last = b * k["block"] // ncol, (np.minimum((b + 1) * k["block"], ntot) - 1) // ncol
    assert (last - first).max() <= 1
    places = np.concatenate([b + first, (b + last)[last > first]])
    assert len(np.unique(places)) == len(places) and places.max() < g["nblk"] + grid[2]


def test_tags_return_only_after_every_other(ws):
    """No tag is that of a zeroed word, and the tag of a call is not met again within the
    2^32 - 1 calls that follow (15-bit tags came back after 32768)."""
    assert ws.ws_call_tag(0) != 0
    for gen in (0, 1, 32767, 32768, (1 << 31) - 1, (1 << 32) - 3):
        assert ws.ws_next_generation(gen) == gen + 1
        assert ws.ws_call_tag(gen) == gen + 1
    assert ws.ws_next_generation((1 << 32) - 2) == 0 and ws.ws_call_tag((1 << 32) - 2) == (1 << 32) - 1
    for tag, bits in ((1, 0xFFFF), (0x8001, 0xFC), ((1 << 32) - 1, 0)):
        w = ws.ws_tagged_word(tag, bits)
        assert w >> 32 == tag and w & 0xFFFFFFFF == bits


def test_a_wait_ends(ws):
    """A wait for a word that does not come gives up, and the waits after it look only
    once: a launch always ends."""
    ws.ws_await.argtypes = [ctypes.c_uint32, ctypes.c_uint32, ctypes.c_uint64, ctypes.POINTER(ctypes.c_uint64)]
    limit = ws.ws_spin_limit()
    assert limit * 4e-6 < 120.0     # seconds: 4 us a poll

    def wait(left, polls):
        out = (ctypes.c_uint64 * 4)()
        ws.ws_await(9, left, polls, out)
        return tuple(out)

    assert wait(limit, 0) == (1, 1, 0, limit)
    assert wait(limit, 3) == (1, 4, 3, limit - 3)
    assert wait(limit, 1 << 40) == (0, limit + 1, 256, 0)
    assert wait(0, 1 << 40) == (0, 1, 0, 0)
    assert wait(0, 0) == (1, 1, 0, 0)
