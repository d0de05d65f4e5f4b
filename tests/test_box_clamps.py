"""Clamped reads of one image that share their unclamped index in box
kernels: different bounds, bounds inside the image beside an unclamped read,
and in the columns; against the general kernels' path and the oracle."""
import numpy as np
import pytest

from oracle import cemit
from polymage_amd.constructs import Parameter, Variable, Interval, Image, Function, Max, Min, Int, Float

from helpers import build, bits_equal, gpu_build, emulating

FORMS = ['rows', 'plain', 'columns', 'shifted']
SIZES = [(45, 70), (96, 140)]


def _case(form, R_, C_, opts=None):
    R, C = Parameter(Int, 'R'), Parameter(Int, 'C')
    x, y = Variable(Int, 'x'), Variable(Int, 'y')
    img = Image(Float, 'img', [R, C])
    clamp = lambda e, lo, hi: Min(Max(e, lo), hi)
    rows, cols = Interval(Int, -3, R + 1), Interval(Int, 0, C - 3)
    if form == 'rows':
        e = img(clamp(x, 0, R - 1), y) * 2.0 - img(clamp(x, 2, R - 4), y)
    elif form == 'plain':
        rows = Interval(Int, 0, R - 1)
        e = img(clamp(x, 3, R - 3), y) * 2.0 - img(x, y)
    elif form == 'columns':
        rows, cols = Interval(Int, 0, R - 1), Interval(Int, -2, C + 2)
        e = img(x, clamp(y, 0, C - 1)) * 2.0 - img(x, clamp(y, 5, C - 7))
    else:
        # the same element at different points of a block
        e = img(clamp(x - 1, 0, R - 1), y) * 2.0 - img(clamp(x - 1, 1, R - 4), y + 2)
    out = Function(([x, y], [rows, cols]), Float, 'out')
    out.defn = [e]
    shape = (R_ + (5 if form in ('rows', 'shifted') else 0), C_ + (5 if form == 'columns' else -2))
    pipe = build(out, {'R': R, 'C': C}, {'R': 96, 'C': 140}, 'boxclamp_' + form, [16, 32], gpu_options=opts)
    img_ = np.random.default_rng(R_).random((R_, C_)).astype(np.float32)
    return out, pipe, {'R': R_, 'C': C_, 'img': img_}, shape


def _check(out, run, vals, shape):
    o = np.full(shape, 7, np.float32)
    g = o.copy()
    run(dict(vals, out=g))
    cemit.build([out], 'boxclamp')(dict(vals, out=o))
    assert bits_equal(g, o)


@pytest.mark.parametrize("opts", [None, {'no_box': 1}])
@pytest.mark.parametrize("form", FORMS)
def test_clamps_on_the_emulator(form, opts):
    import kernel_emu
    from polymage_amd.box_plan import BoxPlan
    from polymage_amd.hip_emit import plan_pipeline
    for R, C in SIZES:
        out, pipe, vals, shape = _case(form, R, C, opts)
        assert all((BoxPlan.of(p) is None) == bool(opts) for p in plan_pipeline(pipe))
        _check(out, kernel_emu.build(pipe).run_host, vals, shape)


@pytest.mark.gpu
@pytest.mark.parametrize("form", FORMS)
def test_clamps_bitexact(gpu, form):
    if emulating():
        pytest.skip("covered by the emulator test")
    for R, C in SIZES:
        print("case clamp", form, R, C, flush=True)
        out, pipe, vals, shape = _case(form, R, C)
        _check(out, gpu_build(pipe).run_host, vals, shape)
