"""Box kernels (constant tile shapes) against the general kernels' path and
the oracle.

Every case runs on the CPU emulator under both kernels and on the GPU under
the default; results are the oracle's bits.  Sizes: one tile and less, tiles
cut in both directions, a last tile of one row or column, and a size at
which inner tiles exist; accesses: shifts, downsampling, upsampling by
parity, interleaving, edge replication, constant planes, Cases that meet
inside a tile, odd grid origins."""
import numpy as np
import pytest

from oracle import cemit
from polymage_amd.apps import inputs
from polymage_amd.constructs import (Parameter, Variable, Interval, Image, Function, Case, Condition,
                                     Select, Cast, Max, Min, Int, Float, Short, UChar)

from helpers import build, bits_equal, gpu_build, emulating


def _shapes(n, dt):
    """A pipeline of every access form: [n, m] image of type dt."""
    R, C = Parameter(Int, 'R'), Parameter(Int, 'C')
    x, y, c = Variable(Int, 'x'), Variable(Int, 'y'), Variable(Int, 'c')
    typ = {'f': Float, 's': Short, 'b': UChar}[dt]
    img = Image(typ, 'img', [R, C])
    rows, cols = Interval(Int, 0, R - 1), Interval(Int, 0, C - 1)
    cx = Min(Max(x - 3, 0), R - 1)
    pad = Function(([x, y], [Interval(Int, 0, R + 4), cols]), typ, 'pad')
    pad.defn = [Cast(typ, img(cx, y))]                          # edge replication
    half = Function(([x, y], [Interval(Int, 1, R / 2 - 2), Interval(Int, 1, C / 2 - 2)]), Float, 'half')
    half.defn = [(pad(2 * x - 1, 2 * y) + 3.0 * pad(2 * x, 2 * y) + pad(2 * x + 1, 2 * y + 1)) * 0.2]
    lo, hr, hc = 5, R - 12, C - 12
    up = Function(([x, y], [Interval(Int, lo, hr), Interval(Int, lo, hc)]), Float, 'up')
    up.defn = [Select(Condition(x % 2, '==', 0),
                      0.25 * half(x / 2 - 1, y / 2) + 0.75 * half(x / 2, (y + 1) / 2),
                      0.25 * half(x / 2 + 1, y / 2) + 0.75 * half(x / 2, (y + 1) / 2))]
    mix = Function(([x, y], [Interval(Int, lo, hr), Interval(Int, lo, hc)]), Float, 'mix')
    mix.defn = [Select(Condition(y % 2, '==', 0), up(x, y), half(x / 2, y / 2))]     # interleaving
    two = Function(([c, x, y], [Interval(Int, 0, 1), Interval(Int, lo, hr), Interval(Int, lo, hc)]),
                   Float, 'two')
    two.defn = [Case(Condition(c, '==', 0), mix(x, y) * 0.5), Case(Condition(c, '==', 1), mix(x, y) + pad(x, y))]
    box = Condition(x, '>=', lo + 1) & Condition(x, '<=', hr - 1) & Condition(y, '>=', lo + 1) & \
        Condition(y, '<=', hc - 1)
    edge = Condition(x, '<', lo + 1) | Condition(x, '>', hr - 1) | Condition(y, '<', lo + 1) | \
        Condition(y, '>', hc - 1)
    out = Function(([c, x, y], [Interval(Int, 0, 1), Interval(Int, lo, hr), Interval(Int, lo, hc)]),
                   Float, 'out')
    out.defn = [Case(box, two(c, x - 1, y) + two(c, x + 1, y) - two(1, x, y) * two(c, x, y - 1)),
                Case(edge, two(c, x, y) - 1.0)]
    return out, {'R': R, 'C': C}


def _forms(R, C, tiles, dt, opts):
    out, pd = _shapes(R, dt)
    pipe = build(out, pd, {'R': 96, 'C': 150}, 'boxforms', tiles, group_size=20, gpu_options=opts)
    g = np.random.default_rng(R * 3 + C)
    img = g.random((R, C)).astype(np.float32) if dt == 'f' else \
        g.integers(-900, 900, (R, C)).astype(np.int16) if dt == 's' else \
        g.integers(0, 256, (R, C)).astype(np.uint8)
    return out, pipe, {'R': R, 'C': C, 'img': img}, (2, R - 16, C - 16)


def _app(app, R, C, tiles, opts):
    pd = {}
    g = np.random.default_rng(R + 7 * C)
    if app == 'harris':
        from polymage_amd.apps.harris import harris_pipe
        out = harris_pipe(pd)
        vals, shape, gs = {'R': R - 2, 'C': C - 2, 'img': g.random((R, C)).astype(np.float32)}, (R, C), 11
        sizes = {'R': 126, 'C': 158}
    elif app == 'campipe':
        from polymage_amd.apps.campipe import camera_pipe, MATRIX_3200, MATRIX_7000
        out = camera_pipe(pd, variant='batch')
        vals = {'R': R, 'C': C, 'colour_temp': 3700.0, 'gamma': 2.2, 'contrast': 50.0,
                'img': g.integers(0, 1024, (R, C)).astype(np.uint16),
                'matrix_3200': np.array(MATRIX_3200, np.float32),
                'matrix_7000': np.array(MATRIX_7000, np.float32)}
        shape, gs, sizes = (3, R - 48, C - 64), 40, {'R': 160, 'C': 256}
    else:
        from polymage_amd.apps.bilateral import bilateral_grid_full
        out = bilateral_grid_full(pd)
        vals = {'rows': R, 'cols': C, 'input': inputs.smooth_field(g, R, C, 1)[0]}
        shape, gs, sizes = (1, R, C), 5, {'rows': 160, 'cols': 128}
    return out, build(out, pd, sizes, app, tiles, group_size=gs, gpu_options=opts), vals, shape


CASES = [('forms', R, C, tiles, dt) for (R, C, tiles, dt) in (
             (96, 150, [16, 32], 'f'), (33, 49, [16, 32], 's'), (34, 81, [8, 16], 'f'),
             (50, 40, [32, 64], 'f'), (67, 97, [16, 16], 'b'))] + \
        [('harris', 130, 290, [16, 64], 'f'), ('harris', 37, 66, [32, 64], 'f'), ('harris', 67, 131, [16, 30], 'f'),
         ('campipe', 128, 192, [16, 32], 's'), ('campipe', 114, 162, [32, 32], 's'),
         ('campipe', 210, 268, [32, 64], 's'), ('bilateral', 131, 97, [32, 32], 'f'),
         ('bilateral', 40, 72, [64, 16], 'f')]


def _case(app, R, C, tiles, dt, opts=None):
    return _forms(R, C, tiles, dt, opts) if app == 'forms' else _app(app, R, C, tiles, opts)


def _check(out, run, vals, shape):
    o = np.full(shape, 7, out.typ.np_dtype())
    g = o.copy()
    run(dict(vals, **{out.name: g}))
    cemit.build([out], 'box_%s' % out.name)(dict(vals, **{out.name: o}))
    assert bits_equal(g, o)


@pytest.mark.parametrize("app,R,C,tiles,dt", CASES)
def test_box_and_general_kernels_on_the_emulator(app, R, C, tiles, dt):
    import kernel_emu
    from polymage_amd.box_plan import BoxPlan
    from polymage_amd.group_plan import GroupPlan
    from polymage_amd.hip_emit import plan_pipeline
    out, pipe, vals, shape = _case(app, R, C, tiles, dt)
    plans = [p for p in plan_pipeline(pipe) if isinstance(p, GroupPlan)]
    assert plans and all(BoxPlan.of(p) is not None for p in plans)
    _check(out, kernel_emu.build(pipe).run_host, vals, shape)
    out, pipe, vals, shape = _case(app, R, C, tiles, dt, {'no_box': 1})
    assert all(BoxPlan.of(p) is None for p in plan_pipeline(pipe) if isinstance(p, GroupPlan))
    _check(out, kernel_emu.build(pipe).run_host, vals, shape)


@pytest.mark.gpu
@pytest.mark.parametrize("app,R,C,tiles,dt", CASES)
def test_box_kernels_bitexact(gpu, app, R, C, tiles, dt):
    if emulating():
        pytest.skip("covered by the emulator test")
    print("case box", app, R, C, tiles, dt, flush=True)
    out, pipe, vals, shape = _case(app, R, C, tiles, dt)
    _check(out, gpu_build(pipe).run_host, vals, shape)


def _small_frames(n):
    """n Harris frames of uneven sizes (some of one tile) and their outputs."""
    from polymage_amd.apps.harris import harris_pipe
    pd = {}
    out = harris_pipe(pd)
    pipe = build(out, pd, {'R': 62, 'C': 94}, 'harris', [16, 32])
    orc = cemit.build([out], 'box_harris')
    g = np.random.default_rng(n)
    recs, refs = [], []
    for k in range(n):
        R, C = 5 + (7 * k) % 40, 6 + (11 * k) % 60
        vals = {'R': R, 'C': C, 'img': g.random((R + 2, C + 2)).astype(np.float32)}
        o = np.full((R + 2, C + 2), -7.0, np.float32)
        orc(dict(vals, harris=o))
        refs.append(o)
        recs.append(dict(vals, harris=np.full_like(o, -7.0)))
    return pipe, recs, refs


def test_batch_of_many_frames_on_the_emulator():
    import kernel_emu
    pipe, recs, refs = _small_frames(5)
    kernel_emu.build(pipe).run_batch(recs, 'persistent')
    assert all(bits_equal(rec['harris'], r) for rec, r in zip(recs, refs))


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 63, 64, 65, 130])
def test_batch_of_many_frames(gpu, n):
    """A work item's frame is found 64 frames a step."""
    if emulating():
        pytest.skip("device tensors are not emulated")
    import torch
    print("case batch frames", n, flush=True)
    pipe, recs, refs = _small_frames(n)
    bp = gpu_build(pipe)
    dev = [dict(rec, img=torch.from_numpy(rec['img']).cuda(), harris=torch.from_numpy(rec['harris']).cuda())
           for rec in recs]
    h = bp.batch_create(dev)
    try:
        for mode in ('persistent', 'graph', 'graph'):
            for d in dev:
                d['harris'].fill_(-7.0)
            bp.batch_run(h, torch.cuda.current_stream().cuda_stream, mode)
            torch.cuda.synchronize()
            assert all(bits_equal(d['harris'].cpu().numpy(), r) for d, r in zip(dev, refs))
    finally:
        bp.batch_destroy(h)


def test_merged_launches_keep_dependences():
    """Every kernel is launched once, after what it reads, and never beside a
    kernel that writes what it reads; merged members have equal workgroups."""
    from polymage_amd.apps import workloads
    from polymage_amd.hip_emit import plan_launches
    for app in ('blend', 'laplacian', 'interpolate', 'bilateral'):
        w = workloads.tuned(app, 'learned', with_data=False)
        kernels = w.pipe.generate_code().kernels
        launches = plan_launches(w.pipe, kernels, w.pipe.sorted_parameters())[1]
        written = dict((f, k) for k in kernels for f in k.writes)
        done = []
        for l in launches:
            members = l.members or [l]
            assert len(set(m.threads for m in members)) == 1
            for m in members:
                for f in m.reads:
                    assert f not in written or written[f] in done
            done += members
        assert len(done) == len(kernels) and set(done) == set(kernels)
        if app in ('blend', 'laplacian'):
            assert len(launches) < len(kernels)


def _blend(opts):
    from polymage_amd.apps.pyramid_blend import pyramid_blend
    pd = {}
    out = pyramid_blend(pd)
    R, C = 130, 203
    g = np.random.default_rng(3)
    pipe = build(out, pd, {'R': R, 'C': C}, 'blend', [8, 64], group_size=6, gpu_options=opts)
    return out, pipe, {'R': R, 'C': C, 'img1': g.random((3, R, C)).astype(np.float32),
                       'img2': g.random((3, R, C)).astype(np.float32),
                       'mask': g.random((R, C)).astype(np.float32)}, (3, R - 60, C - 60)


@pytest.mark.gpu
@pytest.mark.parametrize("opts", [None, {'no_merge': 1}])
def test_merged_launches_bitexact(gpu, opts):
    if emulating():
        pytest.skip("the emulator's blend tests run merged launches")
    print("case merged", opts, flush=True)
    out, pipe, vals, shape = _blend(opts)
    _check(out, gpu_build(pipe).run_host, vals, shape)


@pytest.mark.parametrize("opts", [{'batch_tiles': [16, 48]}, {'batch_tiles': [32, 64], 'batch_threads': 128},
                                  {'batch_tiles': [512, 512]}])
def test_batch_tiles_on_the_emulator(opts):
    """Batch kernels on tiles of their own (the last do not fit LDS: the
    plain kernels' tiles serve the batch) give the plain call's output."""
    import kernel_emu
    sizes = [(114, 162), (128, 192), (98, 130)]
    recs, refs = [], []
    for (R, C) in sizes:
        out, pipe, vals, shape = _app('campipe', R, C, [16, 32], opts)
        o = np.full(shape, 7, np.uint8)
        cemit.build([out], 'box_process')(dict(vals, process=o))
        refs.append(o)
        recs.append(dict(vals, process=np.full(shape, 7, np.uint8)))
    ep = kernel_emu.build(pipe)
    ep.run_batch(recs, 'persistent')
    assert all(bits_equal(rec['process'], r) for rec, r in zip(recs, refs))
    g = np.full(shape, 7, np.uint8)
    ep.run_host(dict(vals, process=g))
    assert bits_equal(g, refs[-1])
