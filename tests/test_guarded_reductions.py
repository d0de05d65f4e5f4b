"""Reductions whose Cases or Selects keep reads inside their arrays: the
value, the bin or both read a neighbour that exists only where the condition
holds.  Run on the emulator under AddressSanitizer (the arrays there are
separate allocations), against the oracle, in every form of the kernel."""
import os
import subprocess
import sys

import numpy as np
import pytest

import kernel_emu
from oracle import cemit
from polymage_amd.constructs import (Parameter, Variable, Interval, Image, Reduction, Reduce, Op, Case,
                                     Condition, Select, Cast, Int, Float)
from polymage_amd.hip_emit import plan_pipeline

from helpers import build, bits_equal, gpu_build, emulating

HERE = os.path.dirname(os.path.abspath(__file__))


def _case(form, R, C, opts=None):
    rows, cols = Parameter(Int, 'rows'), Parameter(Int, 'cols')
    x, y, z, c = (Variable(Int, n) for n in 'xyzc')
    img = Image(Float, 'img', [rows, cols])
    dom = ([x, y], [Interval(Int, 0, rows - 1), Interval(Int, 0, cols - 1)])
    b = lambda e: 1 + Cast(Int, e * 4)
    typ = Float
    if form == 'atomic':
        g = Reduction(([z], [Interval(Int, 0, 5)]), dom, Int, 'grid')
        at, typ, shape = (lambda e: g(b(e))), Int, (6,)
    else:
        g = Reduction(([x, y, z], [Interval(Int, 0, rows / 4), Interval(Int, 0, cols / 4), Interval(Int, 0, 5)]),
                      dom, Float, 'grid')
        at, shape = (lambda e: g(x / 4, y / 4, b(e))), (R // 4 + 1, C // 4 + 1, 6)
    inner, last = Condition(x, '>=', 1), Condition(x, '<', rows - 1)
    if form in ('value', 'bin', 'plane'):
        # planes decided by their constant index, with and without a guard
        # too (the kernel with bins in registers serves guarded cases of more
        # than 16 accumulators)
        g = Reduction(([c, x, y, z], [Interval(Int, 0, 1), Interval(Int, 0, rows / 4), Interval(Int, 0, cols / 4),
                                      Interval(Int, 0, 9)]), dom, Float, 'grid')
        at, shape = (lambda k, e: g(k, x / 4, y / 4, b(e))), (2, R // 4 + 1, C // 4 + 1, 10)
    if form == 'value':
        g.defn = [Case(inner, Reduce(at(0, img(x, y)), img(x, y) - img(x - 1, y), Op.Sum)),
                  Case(last, Reduce(at(1, img(x, y)), img(x, y) * img(x + 1, y), Op.Max))]
    elif form == 'select':
        g.defn = [Reduce(at(img(x, y)), Select(inner, img(x - 1, y), img(x, y)) + Select(last, img(x + 1, y), img(x, y)),
                         Op.Sum)]
    elif form == 'and':
        # the right side of && reads only where the left one holds
        g.defn = [Reduce(at(img(x, y)), Select(inner & Condition(img(x - 1, y), '>', 0.5), img(x, y), img(x, y) * 2.0),
                         Op.Max)]
    elif form == 'or':
        g.defn = [Reduce(at(img(x, y)), img(x, y) * Select(Condition(x, '<', 1) | Condition(img(x - 1, y), '>', 0.5),
                                                          img(x, y), img(x, y) + 2.0), Op.Sum)]
    elif form == 'bin':
        g.defn = [Case(inner, Reduce(at(0, img(x - 1, y)), img(x, y), Op.Sum)),
                  Case(Condition(x, '<', 1), Reduce(at(1, img(x, y)), img(x + 1, y), Op.Sum))]
    elif form == 'plane':
        g.defn = [Case(Condition(c, '==', 0) & inner, Reduce(at(0, img(x, y)), img(x - 1, y), Op.Sum)),
                  Case(Condition(c, '==', 1), Reduce(at(1, img(x, y)), 1, Op.Sum)),
                  Case(Condition(c, '==', 0), Reduce(at(1, img(x, y)), 5, Op.Sum))]
    else:
        g.defn = [Case(inner, Reduce(at(img(x - 1, y)), Cast(Int, img(x - 1, y) * 100), Op.Sum))]
    g.default = 0
    pipe = build(g, {'rows': rows, 'cols': cols}, {'rows': 64, 'cols': 64}, 'guarded_' + form, [16, 16],
                 gpu_options=opts)
    a = np.random.default_rng(R + C).random((R + 4, C)).astype(np.float32)
    # (the oracle evaluates both branches of a Select: rows around the image)
    return g, pipe, {'rows': R, 'cols': C, 'img': a[2:R + 2]}, shape, typ


BINNED = ['value', 'select', 'and', 'or', 'bin', 'plane']
SIZES = [(32, 64), (33, 70)]


def _check(form, R, C, opts):
    g, pipe, vals, shape, typ = _case(form, R, C, opts)
    plan = plan_pipeline(pipe)[0]
    assert (plan.owner and plan.bin_dim is not None) == (form != 'atomic' and not opts)
    assert plan.atomic == (form == 'atomic')
    d = np.full(shape, 7, typ.np_dtype())
    o = d.copy()
    cemit.build([g], 'guarded_oracle')(dict(vals, grid=o))
    gpu_build(pipe).run_host(dict(vals, grid=d))
    assert bits_equal(d, o)


def _under_asan(forms, opts):
    """The forms in a child process that preloads the sanitizer."""
    env = dict(os.environ, PMX_EMULATE='asan', ASAN_OPTIONS='detect_leaks=0', LD_PRELOAD=kernel_emu.asan_runtime())
    code = ('import sys; sys.path[:0] = [%r, %r]; import test_guarded_reductions as t\n'
            'for f in %r:\n  for R, C in t.SIZES:\n    print("case", f, R, C, flush=True); t._check(f, R, C, %r)\n'
            'print("guarded ok")' % (HERE, os.path.dirname(HERE), forms, opts))
    r = subprocess.run([sys.executable, '-c', code], env=env, stdout=subprocess.PIPE, stderr=subprocess.STDOUT,
                       timeout=900, cwd=os.path.dirname(HERE))
    txt = r.stdout.decode(errors='replace')
    assert r.returncode == 0 and 'guarded ok' in txt, txt[-3000:]


@pytest.mark.parametrize("form", BINNED + ['atomic'])
def test_guarded_reads_under_asan(form):
    _under_asan([form], {'no_bins': 1} if form != 'atomic' else None)


def test_binned_guarded_reads_under_asan():
    _under_asan(BINNED, None)


@pytest.mark.parametrize("cell,bins,planes,guard,binned", [
    ((8, 8), 14, 2, False, True), ((8, 8), 8, 1, False, True), ((8, 8), 32, 1, False, False),
    ((2, 2), 8, 1, False, False), ((2, 2), 12, 1, False, True), ((4, 2), 6, 1, False, True),
    ((8, 8), 14, 2, True, False), ((4, 4), 8, 2, True, False), ((4, 4), 10, 2, True, True)])
def test_where_bins_go_to_registers(cell, bins, planes, guard, binned):
    rows, cols = Parameter(Int, 'rows'), Parameter(Int, 'cols')
    x, y, z, c = (Variable(Int, n) for n in 'xyzc')
    img = Image(Float, 'img', [rows, cols])
    g = Reduction(([c, x, y, z], [Interval(Int, 0, planes - 1), Interval(Int, 0, rows / cell[0]),
                                  Interval(Int, 0, cols / cell[1]), Interval(Int, 0, bins - 1)]),
                  ([x, y], [Interval(Int, 0, rows - 1), Interval(Int, 0, cols - 1)]), Float, 'grid')
    red = [Reduce(g(k, x / cell[0], y / cell[1], Cast(Int, img(x, y) * 3)), img(x, y), Op.Sum) for k in range(planes)]
    g.defn = [Case(Condition(x, '>=', 1), r) if guard else r for r in red]
    g.default = 0
    pipe = build(g, {'rows': rows, 'cols': cols}, {'rows': 64, 'cols': 64}, 'where_bins', [16, 16])
    assert (plan_pipeline(pipe)[0].bin_dim is not None) == binned


@pytest.mark.gpu
@pytest.mark.parametrize("opts", [None, {'no_bins': 1}])
@pytest.mark.parametrize("form", BINNED + ['atomic'])
def test_guarded_reductions_bitexact(gpu, form, opts):
    if emulating():
        pytest.skip("covered by the emulator tests")
    for R, C in SIZES:
        print("case guarded", form, R, C, opts, flush=True)
        _check(form, R, C, opts)
