"""General kernels with inlined stages that only a Case or a Select's branch
reads, outside whose domain their reads leave the image or the tile's LDS,
and with a Case's loads that a later sweep reads again: AddressSanitizer on
the emulator, and the oracle's bits."""
import os
import subprocess
import sys

import numpy as np
import pytest

import kernel_emu
from oracle import cemit
from polymage_amd.constructs import (Parameter, Variable, Interval, Image, Function, Case, Condition, Select, Int,
                                     Float)

from helpers import build, bits_equal, gpu_build, emulating

HERE = os.path.dirname(os.path.abspath(__file__))
FORMS = ['case', 'select', 'chain', 'rows', 'forward']
R_, C_ = 70, 100


def _check(form):
    R, C = Parameter(Int, 'R'), Parameter(Int, 'C')
    x, y = Variable(Int, 'x'), Variable(Int, 'y')
    img = Image(Float, 'img', [R, C])
    cols = Interval(Int, 0, C - 1)
    here = Condition(x, '>=', 30)

    def func(name, lo, *defn):
        f = Function(([x, y], [Interval(Int, lo, R - 1), cols]), Float, name)
        f.defn = list(defn)
        return f
    t = func('t', 30, img(x - 30, y) * 2.0 + img(x - 29, y))
    if form == 'case':
        out = func('out', 0, Case(here, t(x, y)), Case(Condition(x, '<', 30), img(x, y)))
    elif form == 'select':
        out = func('out', 0, Select(here, t(x, y), img(x, y)))
    elif form == 'chain':
        u = func('u', 30, t(x, y) * 0.5)
        out = func('out', 0, Select(here, u(x, y), img(x, y)))
    elif form == 'forward':
        a = func('a', 0, Case(here, img(x - 30, y) * 0.5 + img(x, y)), Case(Condition(x, '<', 30), img(x, y) * 2.0))
        cols = Interval(Int, 1, C - 2)
        two = a(x, y - 1) + a(x, y + 1) + img(x, y)
        out = func('out', 0, Case(here, two + img(x - 30, y)), Case(Condition(x, '<', 30), two))
    else:
        # a stage in LDS of which a tile below row 30 computes nothing
        a = func('a', 30, img(x - 30, y) + img(x - 29, y))
        b = func('b', 31, a(x, y) + a(x - 1, y) * 0.5)
        out = func('out', 0, Case(Condition(x, '>=', 40), b(x, y)), Case(Condition(x, '<', 40), img(x, y)))
    opts, tiles, c0 = {'no_box': 1}, [16, 16], C_
    if form == 'forward':
        opts, tiles, c0 = {'no_box': 1, 'threads': 128, 'block': (8, 1)}, [16, 60], C_ - 2
    pipe = build(out, {'R': R, 'C': C}, {'R': 96, 'C': 128}, 'inlguard_' + form, tiles, gpu_options=opts)
    # (the oracle evaluates both branches of a Select: rows around the image)
    big = np.random.default_rng(4).random((R_ + 70, C_)).astype(np.float32)
    vals = {'R': R_, 'C': C_, 'img': big[35:35 + R_].copy()}
    g = np.full((R_, c0), 7, np.float32)
    o = g.copy()
    gpu_build(pipe).run_host(dict(vals, out=g))
    cemit.build([out], 'inlguard')(dict(vals, img=big[35:35 + R_], out=o))
    assert bits_equal(g, o)


@pytest.mark.parametrize("form", FORMS)
def test_inlined_reads_under_asan(form):
    env = dict(os.environ, PMX_EMULATE='asan', ASAN_OPTIONS='detect_leaks=0', LD_PRELOAD=kernel_emu.asan_runtime())
    code = ('import sys; sys.path[:0] = [%r, %r]; import test_inline_guards as t\n'
            't._check(%r)\nprint("inline ok")' % (HERE, os.path.dirname(HERE), form))
    r = subprocess.run([sys.executable, '-c', code], env=env, stdout=subprocess.PIPE, stderr=subprocess.STDOUT,
                       timeout=900, cwd=os.path.dirname(HERE))
    txt = r.stdout.decode(errors='replace')
    assert r.returncode == 0 and 'inline ok' in txt, txt[-3000:]


@pytest.mark.gpu
@pytest.mark.parametrize("form", FORMS)
def test_inlined_reads_bitexact(gpu, form):
    if emulating():
        pytest.skip("covered by the emulator test")
    print("case inline", form, flush=True)
    _check(form)
