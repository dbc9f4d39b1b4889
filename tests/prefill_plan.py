"""The prefill launches' plan (vapi_amd/csrc/prefill_plan.hpp), built for the
CPU by tests/cpp/build.py."""
import ctypes
import importlib.util
from dataclasses import dataclass
from functools import lru_cache
from pathlib import Path

ANY_BYTES = (1 << 64) - 1
LIST_ORDER, LIST_PARTS, SEQUENCES, PARTS, BY_CLASS = range(5)  # PfOrder


@lru_cache(maxsize=None)
def _lib():
    spec = importlib.util.spec_from_file_location("cpp_tests_build",
                                                  Path(__file__).parent / "cpp" / "build.py")
    b = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(b)
    if not b.plan_is_current():
        b.build_plan()
    return ctypes.CDLL(str(b.PLAN))


@dataclass
class Route:
    items: int
    qtiles: int
    n_split: int
    ranges: int
    range_bytes: int
    order: int
    rows: int


def route(f32, n_seqs, heads, kvh, max_q, max_k, head_dim, split_ok=True, ws_bytes=ANY_BYTES,
          pool_dim=None):
    """How a prefill launch over n_seqs listed sequences runs. `head_dim`: the
    kernel's (64, 128 or 256); `pool_dim`: the pool's, where it is another."""
    out = (ctypes.c_uint64 * 6)()
    fn = _lib().plan_route_f32 if f32 else _lib().plan_route16
    u32 = ctypes.c_uint32
    fn(u32(n_seqs), u32(kvh), u32(heads // kvh), u32(max_q), u32(max_k), u32(head_dim),
       u32((pool_dim or head_dim) * (4 if f32 else 2)), int(split_ok), ctypes.c_uint64(ws_bytes), out)
    rows = 128 if f32 or head_dim == 256 else 256
    return Route(out[0], out[1], out[2], out[3], out[4], out[5], rows)


def check_walk(r, lens_q, lens_k, heads, kvh, wl=-1, wr=0):
    """0, or the number of the check that the route's ranges fail."""
    n = len(lens_q)
    a = (ctypes.c_uint32 * n)(*lens_q)
    b = (ctypes.c_uint32 * n)(*lens_k)
    return _lib().plan_check_walk(ctypes.c_uint32(n), a, b, ctypes.c_uint32(kvh),
                                  ctypes.c_uint32(heads // kvh), ctypes.c_uint32(r.rows),
                                  ctypes.c_uint32(r.qtiles), ctypes.c_int32(wl),
                                  ctypes.c_int32(wr), ctypes.c_uint32(r.ranges))


def tile_order(lens_k, tiles, step):
    """The (sequence, tile) pairs of a launch by classes, in its order."""
    n, total = len(lens_k), sum(tiles)
    out = (ctypes.c_uint32 * (2 * total))()
    bad = _lib().plan_order(ctypes.c_uint32(n), (ctypes.c_uint32 * n)(*lens_k),
                            (ctypes.c_uint32 * n)(*tiles), ctypes.c_uint32(step), out)
    assert bad == 0, bad
    return [(out[2 * i], out[2 * i + 1]) for i in range(total)]


def item_order(n_seqs, qtiles, kvh):
    """The (list entry, kv head, tile) of every item of a launch in LIST_PARTS."""
    out = (ctypes.c_uint32 * (3 * n_seqs * qtiles * kvh))()
    _lib().plan_list_parts(ctypes.c_uint32(n_seqs), ctypes.c_uint32(kvh), ctypes.c_uint32(qtiles),
                           out)
    return [tuple(out[3 * i:3 * i + 3]) for i in range(n_seqs * qtiles * kvh)]
