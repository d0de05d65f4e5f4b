"""Box kernels with indices computed per point: thirds of an in-group stage
and of an image, beside halves, and every third point; selects between two
such reads (their indices are selected, one read is left), by 3, by 8 and of
halves in blocks that do not know the parity; against the general kernels'
path and the oracle.  Tiles that are and are not multiples of the scale."""
import numpy as np
import pytest

from oracle import cemit
from polymage_amd.constructs import Parameter, Variable, Interval, Image, Function, Condition, Select, Int, Float

from helpers import build, bits_equal, gpu_build, emulating

FORMS = ['stage', 'image', 'halves', 'sixths', 'every_third', 'select3', 'select8', 'parity']
BOXES = ('stage', 'image', 'every_third', 'select3', 'parity')      # (an axis read at two scales has no constant box)


def _case(form, R_, C_, tiles, opts=None):
    R, C = Parameter(Int, 'R'), Parameter(Int, 'C')
    x, y = Variable(Int, 'x'), Variable(Int, 'y')
    img = Image(Float, 'img', [R, C])
    a = Function(([x, y], [Interval(Int, 0, R - 1), Interval(Int, 0, C - 1)]), Float, 'a')
    a.defn = [img(x, y) * 2.0]
    dom, shape = [Interval(Int, 0, R - 2), Interval(Int, 0, C - 2)], (R_ - 1, C_ - 1)
    if form == 'every_third':
        dom, shape = [Interval(Int, 0, R / 3 - 1), Interval(Int, 0, C / 3 - 1)], (R_ // 3, C_ // 3)
    out = Function(([x, y], dom), Float, 'out')
    out.defn = [{'stage': lambda: a(x / 3, y / 3) + img(x, y),
                 'image': lambda: img(x / 3, y / 3) - a(x + 1, y),
                 'halves': lambda: a(x / 3, y / 2) + a(x / 2, y / 3) * img(x / 2, (y + 1) / 2),
                 'sixths': lambda: a(x / 2 / 3, (y + 1) / 3 / 2) + a(x / 4, y / 3),
                 'select3': lambda: Select(Condition(x % 3, '==', 0), a(x / 3, y / 3), a(x / 3 + 1, y / 3)),
                 'select8': lambda: Select(Condition(x % 8, '<', 4), a(x / 8, y / 8), a(x / 8 + 1, y / 8)),
                 'parity': lambda: Select(Condition(x % 2, '==', 0), a(x / 2, y / 2), a(x / 2 + 1, y / 2)) +
                 Select(Condition(y % 2, '==', 0), a(x / 2, y / 2), a(x / 2, y / 2 + 1)),
                 'every_third': lambda: a(3 * x + 1, 3 * y) + a(3 * x, 3 * y + 2)}[form]()]
    if form == 'parity' and not (opts or {}).get('no_box'):
        opts = dict(opts or {}, box_blocks={'out': [1, 1]})
    pipe = build(out, {'R': R, 'C': C}, {'R': 320, 'C': 440}, 'boxscale_' + form, tiles, gpu_options=opts)
    img_ = np.random.default_rng(R_).random((R_, C_)).astype(np.float32)
    return out, pipe, {'R': R_, 'C': C_, 'img': img_}, shape


CASES = [(form, R, C, tiles) for form in FORMS for (R, C, tiles) in ((100, 150, [24, 48]), (49, 97, [12, 48]),
                                                                     (70, 67, [16, 32]))]


def _check(out, run, vals, shape):
    o = np.full(shape, 7, np.float32)
    g = o.copy()
    run(dict(vals, out=g))
    cemit.build([out], 'boxscale')(dict(vals, out=o))
    assert bits_equal(g, o)


@pytest.mark.parametrize("opts", [None, {'no_box': 1}])
@pytest.mark.parametrize("form,R,C,tiles", CASES)
def test_scales_on_the_emulator(form, R, C, tiles, opts):
    import kernel_emu
    from polymage_amd.box_plan import BoxPlan
    from polymage_amd.hip_emit import plan_pipeline
    out, pipe, vals, shape = _case(form, R, C, tiles, opts)
    if opts is None and tiles != [16, 32] and form in BOXES:
        assert all(BoxPlan.of(p) is not None for p in plan_pipeline(pipe))
    _check(out, kernel_emu.build(pipe).run_host, vals, shape)


@pytest.mark.gpu
@pytest.mark.parametrize("form,R,C,tiles", CASES)
def test_scales_bitexact(gpu, form, R, C, tiles):
    if emulating():
        pytest.skip("covered by the emulator test")
    print("case scale", form, R, C, tiles, flush=True)
    out, pipe, vals, shape = _case(form, R, C, tiles)
    _check(out, gpu_build(pipe).run_host, vals, shape)
