"""Constants that box kernels fold: selects with a branch of typed integer
constants, literals that C holds in a long, and planes whose variable is not an Int, against the general
kernels' path and the oracle."""
import numpy as np
import pytest

from oracle import cemit
from polymage_amd.constructs import (Parameter, Variable, Interval, Image, Function, Condition, Select, Cast,
                                     Int, UInt, Float)
from polymage_amd.expr_ast import Value

from helpers import build, bits_equal, gpu_build, emulating

N, M = 45, 70


def _case(form, opts=None):
    R, C = Parameter(Int, 'R'), Parameter(Int, 'C')
    x, y, c = Variable(Int, 'x'), Variable(Int, 'y'), Variable(UInt, 'c')
    img = Image(Float, 'img', [R, C])
    a = Function(([x, y], [Interval(Int, 0, R - 1), Interval(Int, 0, C - 1)]), Float, 'a')
    a.defn = [img(x, y) * 2.0]
    dom = ([x, y], [Interval(Int, 1, R - 2), Interval(Int, 1, C - 2)])
    shape = (N - 2, M - 2)
    if form == 'plane':
        dom, shape = ([c] + dom[0], [Interval(UInt, 0, 2)] + dom[1]), (3,) + shape
    out = Function(dom, Float, 'out')
    bright = Condition(img(x, y), '>', 0.5)
    out.defn = [{'minus': lambda: Select(bright, -Value(1, Float), a(x - 1, y + 1)),
                 'sum': lambda: Select(bright, a(x - 1, y + 1), Value(1, Float) + Value(2, Float)),
                 # (an int would overflow)
                 'long': lambda: a(x - 1, y) + Cast(Float, (Value(2 ** 31 + 5, Int) - Value(2 ** 31, Int)) *
                                                   (x * 40000000)),
                 'plane': lambda: a(x - 1, y) + Select(Condition(x, '>', 7), c, Value(3, UInt))}[form]()]
    pipe = build(out, {'R': R, 'C': C}, {'R': 96, 'C': 144}, 'boxconst_' + form, [16, 32], gpu_options=opts)
    img_ = np.random.default_rng(3).random((N, M)).astype(np.float32)
    return out, pipe, {'R': N, 'C': M, 'img': img_}, shape


FORMS = ['minus', 'sum', 'long', 'plane']


def _check(out, run, vals, shape):
    o = np.full(shape, 7, np.float32)
    g = o.copy()
    run(dict(vals, out=g))
    cemit.build([out], 'boxconst')(dict(vals, out=o))
    assert bits_equal(g, o)


@pytest.mark.parametrize("opts", [None, {'no_box': 1}])
@pytest.mark.parametrize("form", FORMS)
def test_constants_on_the_emulator(form, opts):
    import kernel_emu
    from polymage_amd.box_plan import BoxPlan
    from polymage_amd.hip_emit import plan_pipeline
    out, pipe, vals, shape = _case(form, opts)
    assert all((BoxPlan.of(p) is None) == bool(opts) for p in plan_pipeline(pipe))
    _check(out, kernel_emu.build(pipe).run_host, vals, shape)


@pytest.mark.gpu
@pytest.mark.parametrize("form", FORMS)
def test_constants_bitexact(gpu, form):
    if emulating():
        pytest.skip("covered by the emulator test")
    print("case constant", form, flush=True)
    out, pipe, vals, shape = _case(form)
    _check(out, gpu_build(pipe).run_host, vals, shape)
