"""Owner-cell reductions with their bins in registers, against the owner
kernel with LDS accumulators and the oracle: whole and cut cells, domains
smaller than a cell, bins clamped at both ends, every operator, float and
integer accumulators, constant and pixel values, one and two planes."""
import numpy as np
import pytest

from oracle import cemit
from polymage_amd.constructs import (Parameter, Variable, Interval, Image, Reduction, Reduce, Op, Case,
                                     Condition, Cast, Int, Float)
from polymage_amd.hip_emit import plan_pipeline

from helpers import build, bits_equal, gpu_build, emulating


def _case(form, R, C, opts=None):
    rows, cols = Parameter(Int, 'rows'), Parameter(Int, 'cols')
    x, y, z, c = (Variable(Int, n) for n in 'xyzc')
    img = Image(Float, 'img', [rows, cols])
    r, q = Interval(Int, 0, rows - 1), Interval(Int, 0, cols - 1)
    op = {'sum': Op.Sum, 'mul': Op.Mul, 'min': Op.Min, 'max': Op.Max}.get(form, Op.Sum)
    if form in ('grid', 'ints'):
        # values and their count, as in the bilateral grid
        T = Float if form == 'grid' else Int
        g = Reduction(([c, x, y, z], [Interval(Int, 0, 1), Interval(Int, 0, rows / 8 + 3),
                                      Interval(Int, 0, cols / 8 + 3), Interval(Int, 0, 6)]),
                      ([x, y], [r, q]), T, 'grid')
        b = 1 + Cast(Int, img(x, y) * 4)
        v = img(x, y) if form == 'grid' else Cast(Int, img(x, y) * 100)
        g.defn = [Case(Condition(c, '==', 0), Reduce(g(0, 2 + x / 8, 2 + y / 8, b), v, Op.Sum)),
                  Case(Condition(c, '==', 1), Reduce(g(1, 2 + x / 8, 2 + y / 8, b), 1, Op.Sum))]
        shape = (2, R // 8 + 4, C // 8 + 4, 7)
        g.default = 0
    else:
        g = Reduction(([x, y, z], [Interval(Int, 0, rows / 4), Interval(Int, 0, cols / 2),
                                   Interval(Int, -1, 4)]), ([x, y], [r, q]), Float, 'grid')
        g.defn = [Reduce(g(x / 4, y / 2, Cast(Int, img(x, y) * 3)), img(x, y) + 0.5, op)]
        shape = (R // 4 + 1, C // 2 + 1, 6)
        g.default = 1 if form == 'mul' else 0
    pipe = build(g, {'rows': rows, 'cols': cols}, {'rows': 64, 'cols': 64}, 'binned', [16, 16], gpu_options=opts)
    a = np.random.default_rng(R + C).uniform(-0.7, 1.9, (R, C)).astype(np.float32)
    return g, pipe, {'rows': R, 'cols': C, 'img': a}, shape


CASES = [('grid', 64, 64), ('grid', 67, 43), ('grid', 5, 7), ('grid', 130, 8), ('ints', 41, 70),
         ('sum', 33, 35), ('mul', 16, 18), ('min', 3, 1), ('max', 29, 66)]


def _run(g, run, vals, shape):
    d = np.full(shape, 7, g.typ.np_dtype())
    run(dict(vals, grid=d))
    return d


def _check(g, run, vals, shape):
    """On values whose bins all lie in the grid (an index outside it has no
    meaning to the oracle)."""
    vals = dict(vals, img=np.clip(vals['img'], np.float32(-0.49), np.float32(1.49)))
    o = np.full(shape, 7, g.typ.np_dtype())
    cemit.build([g], 'binned_oracle')(dict(vals, grid=o))
    assert bits_equal(_run(g, run, vals, shape), o)


@pytest.mark.parametrize("form,R,C", CASES)
def test_binned_and_lds_kernels_on_the_emulator(form, R, C):
    import kernel_emu
    clamped = []
    for opts in (None, {'no_bins': 1}):
        g, pipe, vals, shape = _case(form, R, C, opts)
        plan = plan_pipeline(pipe)[0]
        assert plan.owner and (plan.bin_dim is None) == bool(opts)
        run = kernel_emu.build(pipe).run_host
        _check(g, run, vals, shape)
        clamped.append(_run(g, run, vals, shape))
    assert bits_equal(*clamped)     # bins outside the grid: clamped alike


@pytest.mark.gpu
@pytest.mark.parametrize("form,R,C", CASES)
def test_binned_reduction_bitexact(gpu, form, R, C):
    if emulating():
        pytest.skip("covered by the emulator test")
    print("case binned", form, R, C, flush=True)
    g, pipe, vals, shape = _case(form, R, C)
    _check(g, gpu_build(pipe).run_host, vals, shape)
