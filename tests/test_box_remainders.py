"""Remainders in box kernels, with C's sign, against the general kernels'
path and the oracle: a shift below zero, a remainder used as a value,
domains that start below zero, a relabelling stage read at a shift (its
remainder moves to the reader's point), Cases that begin where the left
side is no longer negative, and left sides that never are."""
import numpy as np
import pytest

from oracle import cemit
from polymage_amd.constructs import (Parameter, Variable, Interval, Image, Function, Case, Condition,
                                     Select, Cast, Int, Float)

from helpers import build, bits_equal, gpu_build, emulating

N, M = 45, 70


def _case(form, opts=None):
    R, C = Parameter(Int, 'R'), Parameter(Int, 'C')
    x, y = Variable(Int, 'x'), Variable(Int, 'y')
    img = Image(Float, 'img', [R, C])
    whole = [Interval(Int, 0, R - 1), Interval(Int, 0, C - 1)]
    inner = [Interval(Int, 1, R - 2), Interval(Int, 1, C - 2)]

    def func(name, dom, *defn):
        f = Function(([x, y], dom), Float, name)
        f.defn = list(defn)
        return f
    a = func('a', whole, img(x, y) * 2.0)
    sel = lambda c: Select(c, a(x - 1, y), a(x, y + 1))
    shape = (N - 2, M - 2)
    if form == 'equal':
        out = func('out', inner, sel(Condition((x - 5) % 2, '==', 1)))
    elif form == 'less':
        out = func('out', inner, sel(Condition((x - 5) % 4, '<', 2)))
    elif form == 'value':
        b = func('b', whole, Select(Condition((x - 1) % 2, '==', 1), img(x, y), img(x, y) * 0.5) +
                 Cast(Float, (y - 3) % 4))
        out = func('out', inner, b(x - 1, y) + b(x + 1, y + 1))
    elif form == 'stage':
        b = func('b', [Interval(Int, -3, R - 4), whole[1]], Select(
            Condition(x % 2, '==', 1), img(x + 3, y), img(x + 3, y) * 0.5))
        out = func('out', [Interval(Int, -2, R - 5), inner[1]], b(x - 1, y) + b(x, y + 1))
    elif form == 'output':
        out = func('out', [Interval(Int, -4, R - 5), Interval(Int, -4, C - 5)], Select(
            Condition(y % 2, '==', 1), img(x + 4, y + 4), img(x + 4, y + 4) * 0.5))
        shape = (N, M)
    elif form == 'relabel':
        b = func('b', [Interval(Int, -3, R - 4), whole[1]], Select(
            Condition(x % 2, '==', 1), a(x + 3, y), img(x + 3, y)))
        out = func('out', [Interval(Int, -1, R - 4), inner[1]], b(x - 2, y) + 0.5 * b(x, y - 1))
    elif form == 'case':
        rem = Select(Condition((x - 5) % 2, '==', 1), a(x - 1, y), a(x, y + 1))
        out = func('out', inner, Case(Condition(x, '<', 5), rem), Case(Condition(x, '>=', 5), rem * 3.0))
    else:
        out = func('out', inner, sel(Condition((x + 3) % 2, '==', 1) & Condition((y - 1) % 4, '!=', 2)))
    pipe = build(out, {'R': R, 'C': C}, {'R': 96, 'C': 144}, 'boxrem_' + form, [16, 32], gpu_options=opts)
    img_ = np.random.default_rng(1).random((N, M)).astype(np.float32)
    return out, pipe, {'R': N, 'C': M, 'img': img_}, shape


FORMS = ['equal', 'less', 'value', 'stage', 'output', 'relabel', 'case', 'known']


def _check(out, run, vals, shape):
    o = np.full(shape, 7, np.float32)
    g = o.copy()
    run(dict(vals, out=g))
    cemit.build([out], 'boxrem')(dict(vals, out=o))
    assert bits_equal(g, o)


@pytest.mark.parametrize("opts", [None, {'no_box': 1}])
@pytest.mark.parametrize("form", FORMS)
def test_remainders_on_the_emulator(form, opts):
    import kernel_emu
    from polymage_amd.box_plan import BoxPlan
    from polymage_amd.hip_emit import plan_pipeline
    out, pipe, vals, shape = _case(form, opts)
    assert all((BoxPlan.of(p) is None) == bool(opts) for p in plan_pipeline(pipe))
    _check(out, kernel_emu.build(pipe).run_host, vals, shape)


def test_known_remainders_fold():
    """Where the left side is nowhere negative the remainder is gone from
    the kernel; where it is, it stays."""
    for form, stays in (('known', False), ('equal', True)):
        src = _case(form)[1].generate_code().hip_src
        kernel = src[src.index('_body('):]
        assert ('% 2)' in kernel[kernel.index('phase 0'):]) == stays


@pytest.mark.gpu
@pytest.mark.parametrize("form", FORMS)
def test_remainders_bitexact(gpu, form):
    if emulating():
        pytest.skip("covered by the emulator test")
    print("case remainder", form, flush=True)
    out, pipe, vals, shape = _case(form)
    _check(out, gpu_build(pipe).run_host, vals, shape)
