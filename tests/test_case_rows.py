"""General kernels whose blocks read LDS rows that only a border Case reads:
in tiles without border points those rows are not computed, and the block
must not load them (AddressSanitizer on the emulator); the oracle's bits."""
import os
import subprocess
import sys

import numpy as np
import pytest

import kernel_emu
from oracle import cemit
from polymage_amd.constructs import Parameter, Variable, Interval, Image, Function, Case, Condition, Int, Float

from helpers import build, bits_equal, gpu_build, emulating

HERE = os.path.dirname(os.path.abspath(__file__))
SIZES = [(70, 100), (97, 131)]


def _check(R_, C_):
    R, C = Parameter(Int, 'R'), Parameter(Int, 'C')
    x, y = Variable(Int, 'x'), Variable(Int, 'y')
    img = Image(Float, 'img', [R, C])
    a = Function(([x, y], [Interval(Int, 0, R - 2), Interval(Int, 0, C - 1)]), Float, 'a')
    a.defn = [img(x, y) + img(x + 1, y)]
    out = Function(([x, y], [Interval(Int, 1, R - 3), Interval(Int, 1, C - 2)]), Float, 'out')
    inner = Condition(x, '>=', 2) & Condition(x, '<=', R - 4) & Condition(y, '>=', 2) & Condition(y, '<=', C - 3)
    edge = Condition(x, '<', 2) | Condition(x, '>', R - 4) | Condition(y, '<', 2) | Condition(y, '>', C - 3)
    out.defn = [Case(inner, img(x, y) * 2.0), Case(edge, sum(a(x + i, y + j) * (0.5 + i) for i in (-1, 0, 1) for j in (-1, 0, 1)))]
    pipe = build(out, {'R': R, 'C': C}, {'R': 96, 'C': 128}, 'caserows', [16, 16], gpu_options={'vlds': 1, 'block': (2, 4)})
    src = pipe.generate_code().hip_src
    assert 'pmx_ld4<float4>' in src[src.index('_body('):]
    img_ = np.random.default_rng(R_).random((R_, C_)).astype(np.float32)
    g = np.full((R_ - 3, C_ - 2), 7, np.float32)
    o = g.copy()
    gpu_build(pipe).run_host({'R': R_, 'C': C_, 'img': img_, 'out': g})
    cemit.build([out], 'caserows')({'R': R_, 'C': C_, 'img': img_, 'out': o})
    assert bits_equal(g, o)


def test_rows_of_a_border_case_under_asan():
    env = dict(os.environ, PMX_EMULATE='asan', ASAN_OPTIONS='detect_leaks=0', LD_PRELOAD=kernel_emu.asan_runtime())
    code = ('import sys; sys.path[:0] = [%r, %r]; import test_case_rows as t\n'
            'for s in t.SIZES: t._check(*s)\nprint("rows ok")' % (HERE, os.path.dirname(HERE)))
    r = subprocess.run([sys.executable, '-c', code], env=env, stdout=subprocess.PIPE, stderr=subprocess.STDOUT,
                       timeout=900, cwd=os.path.dirname(HERE))
    txt = r.stdout.decode(errors='replace')
    assert r.returncode == 0 and 'rows ok' in txt, txt[-3000:]


@pytest.mark.gpu
@pytest.mark.parametrize("R,C", SIZES)
def test_rows_of_a_border_case_bitexact(gpu, R, C):
    if emulating():
        pytest.skip("covered by the emulator test")
    print("case rows", R, C, flush=True)
    _check(R, C)
