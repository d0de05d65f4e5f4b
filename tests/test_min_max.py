"""Min, Max and Selects that are one of them, for every element type, against
the oracle's conditionals: the same bits, with equal values, signed zeros,
infinities and NaN, with the sides of the condition exchanged, non-strict
comparisons, sides wider than their type, and nested."""
import numpy as np
import pytest

from oracle import cemit
from polymage_amd.constructs import (Parameter, Variable, Interval, Image, Function, Condition, Select, Cast,
                                     Max, Min, Int, Float, Double, Short, UShort, UChar)

from helpers import build, bits_equal, gpu_build, emulating

TYPES = {'uchar': UChar, 'short': Short, 'ushort': UShort, 'int': Int, 'float': Float, 'double': Double}


def _case(name, opts=None):
    n, m = 21, 150
    typ = TYPES[name]
    R, C = Parameter(Int, 'R'), Parameter(Int, 'C')
    x, y, c = Variable(Int, 'x'), Variable(Int, 'y'), Variable(Int, 'c')
    img = Image(typ, 'img', [R, C])
    dom = ([x, y], [Interval(Int, 1, R - 2), Interval(Int, 1, C - 2)])
    a, b, d, e = img(x, y - 1), img(x, y + 1), img(x - 1, y), img(x + 1, y)
    sel = lambda op, t, f: Select(Condition(a, op, b), t, f)
    exprs = [Min(Max(img(x, y), Min(Min(a, b), Min(d, e))), Max(Max(a, b), Max(d, e))),
             Max(a, b), Min(b, a), sel('<', b, a), sel('>', b, a), sel('<=', a, b), sel('>=', a, b),
             sel('<=', b, a), sel('>=', b, a),
             Max(Cast(typ, a - b), Cast(typ, b - a)), Min(a + b, d + e), Max(a * 3, b * 2)]
    n_ex = len(exprs)
    out = Function(([c, x, y], [Interval(Int, 0, n_ex - 1)] + dom[1]), typ, 'out')
    v = Cast(typ, exprs[0])
    for i in range(1, n_ex):
        v = Select(Condition(c, '==', i), Cast(typ, exprs[i]), v)
    out.defn = [v]
    dt = typ.np_dtype()
    g = np.random.default_rng(5)
    if np.dtype(dt).kind == 'f':
        pool = np.array([0.0, -0.0, 1.5, -1.5, np.inf, -np.inf, np.nan, 3.25], dt)
    else:
        i = np.iinfo(dt)
        # int values stay where sums and products do not overflow
        lim = (i.min, i.max) if i.bits < 32 else (-10 ** 6, 10 ** 6)
        pool = np.array([lim[0], lim[0] + 1, 0, 1, 2, 100, lim[1] - 1, lim[1]], dt)
    vals = {'R': n, 'C': m, 'img': pool[g.integers(0, len(pool), (n, m))]}
    pipe = build(out, {'R': R, 'C': C}, {'R': 64, 'C': 192}, 'minmax_' + name, [8, 32], group_size=20, gpu_options=opts)
    return out, pipe, vals, (n_ex, n - 2, m - 2)


def _check(out, run, vals, shape):
    o = np.zeros(shape, out.typ.np_dtype())
    g = o.copy()
    run(dict(vals, **{out.name: g}))
    cemit.build([out], 'minmax_o')(dict(vals, **{out.name: o}))
    nan = o != o
    assert (nan == (g != g)).all() and bits_equal(np.where(nan, 0, g), np.where(nan, 0, o))


@pytest.mark.parametrize("opts", [None, {'no_box': 1}])
@pytest.mark.parametrize("name", sorted(TYPES))
def test_min_max_on_the_emulator(name, opts):
    import kernel_emu
    out, pipe, vals, shape = _case(name, opts)
    _check(out, kernel_emu.build(pipe).run_host, vals, shape)


@pytest.mark.gpu
@pytest.mark.parametrize("name", sorted(TYPES))
def test_min_max_bitexact(gpu, name):
    if emulating():
        pytest.skip("covered by the emulator test")
    print("case minmax", name, flush=True)
    out, pipe, vals, shape = _case(name)
    _check(out, gpu_build(pipe).run_host, vals, shape)
