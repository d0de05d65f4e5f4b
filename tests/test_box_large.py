"""Outputs beyond 4 GiB in box kernels: the planes of an untiled dimension
lie further apart than a 32-bit byte offset reaches.  One workgroup of the
kernel runs on the emulator, over arrays whose pages exist only where it
touches them."""
import ctypes
import mmap

import numpy as np
import pytest

import kernel_emu
from polymage_amd.constructs import Parameter, Variable, Interval, Image, Function, Int, Float, Double, Short
from polymage_amd.hip_emit import plan_pipeline

from helpers import build

PLANES, TILE = 16, (16, 32)


def _sparse(shape, dt):
    """A zeroed array whose untouched pages take no memory."""
    n = int(np.prod(shape, dtype=np.int64)) * np.dtype(dt).itemsize
    m = mmap.mmap(-1, n, flags=mmap.MAP_PRIVATE | mmap.MAP_ANONYMOUS | 0x4000)     # MAP_NORESERVE
    return np.frombuffer(m, dt).reshape(shape)


@pytest.mark.parametrize("typ,n", [(Float, 10000), (Double, 11000), (Short, 11000), (Float, 64)])
def test_planes_beyond_4_gib(typ, n):
    from polymage_amd.box_plan import BoxPlan
    R, C = Parameter(Int, 'R'), Parameter(Int, 'C')
    x, y, c = Variable(Int, 'x'), Variable(Int, 'y'), Variable(Int, 'c')
    img = Image(Float, 'img', [R, C])
    a = Function(([x, y], [Interval(Int, 0, R - 2), Interval(Int, 0, C - 1)]), Float, 'a')
    a.defn = [img(x, y) + img(x + 1, y)]
    out = Function(([c, x, y], [Interval(Int, 0, PLANES - 1), Interval(Int, 0, R - 3), Interval(Int, 0, C - 2)]),
                   typ, 'out')
    out.defn = [(a(x, y) + a(x + 1, y)) * (c + 1)]
    pipe = build(out, {'R': R, 'C': C}, {'R': 96, 'C': 144}, 'boxlarge', list(TILE))
    plan = plan_pipeline(pipe)[0]
    box = BoxPlan.of(plan)
    assert box is not None and box.anchor.cnt[0] > 1
    lib = kernel_emu.build(pipe).lib
    fn = ctypes.c_void_p()
    assert lib.pmx_module_function(None, b'pmx_boxlarge_g0', ctypes.byref(fn)) == 0
    i, o = _sparse((n, n), np.float32), _sparse((PLANES, n - 2, n - 1), typ.np_dtype())
    assert o.size < 2 ** 31
    top = np.arange(18 * 40, dtype=np.float32).reshape(18, 40) % 97
    i[:18, :40] = top
    err = (ctypes.c_int * 16)()
    vals = [ctypes.cast(err, ctypes.c_void_p), ctypes.c_void_p(i.ctypes.data), ctypes.c_void_p(o.ctypes.data),
            ctypes.c_int(n), ctypes.c_int(n)]         # C, R
    args = (ctypes.c_void_p * len(vals))(*[ctypes.addressof(v) for v in vals])
    threads = int(box.opts.get('threads', 256))
    assert lib.pmx_launch(fn, 1, 1, 1, threads, 1, 1, 0, None, args) == 0
    want = (top[:-2] + 2 * top[1:-1] + top[2:])[:, :32] * np.arange(1, PLANES + 1)[:, None, None]
    assert np.array_equal(o[:, :TILE[0], :TILE[1]], want.astype(typ.np_dtype()))
    if n < 100:
        # nothing else was stored
        o[:, :TILE[0], :TILE[1]] = 0
        assert not o.any()
