"""Blocks of box kernels whose padded LDS rows would halve the workgroups
of a compute unit: fewer rows a block, the residency of the general kernel,
the same bits."""
import numpy as np
import pytest

from oracle import cemit
from polymage_amd.apps.harris import harris_pipe
from polymage_amd.box_plan import BoxPlan, resident
from polymage_amd.hip_emit import plan_pipeline

from helpers import build, bits_equal, gpu_build, emulating


def _pipe(tiles, threads):
    pd = {}
    out = harris_pipe(pd)
    return out, build(out, pd, {'R': 2046, 'C': 2046}, 'harris', tiles, gpu_options={'threads': threads})


@pytest.mark.parametrize("tiles,threads,rows", [([16, 512], 512, 2), ([32, 288], 512, 2), ([32, 256], 512, 4),
                                                ([16, 340], 256, 4), ([14, 62], 128, 4)])
def test_blocks_keep_residency(tiles, threads, rows):
    plan = plan_pipeline(_pipe(tiles, threads)[1])[0]
    box = BoxPlan.of(plan)
    assert box.sweeps[0][1][0].blk[0] == rows
    assert 2 * resident(threads, box.lds_bytes) > resident(threads, plan.lds_bytes)


def _check(run, out, R, C):
    img = np.random.default_rng(R).random((R + 2, C + 2)).astype(np.float32)
    g = np.full((R + 2, C + 2), -7.0, np.float32)
    o = g.copy()
    run({'R': R, 'C': C, 'img': img, 'harris': g})
    cemit.build([out], 'harris_oracle_double')({'R': R, 'C': C, 'img': img, 'harris': o})
    assert bits_equal(g, o)


@pytest.mark.parametrize("R,C", [(20, 520), (50, 1600)])
def test_smaller_blocks_on_the_emulator(R, C):
    import kernel_emu
    out, pipe = _pipe([16, 512], 512)
    _check(kernel_emu.build(pipe).run_host, out, R, C)


@pytest.mark.gpu
@pytest.mark.parametrize("R,C", [(20, 520), (50, 1600), (1001, 2100)])
def test_smaller_blocks_bitexact(gpu, R, C):
    if emulating():
        pytest.skip("covered by the emulator test")
    print("case residency", R, C, flush=True)
    out, pipe = _pipe([16, 512], 512)
    _check(gpu_build(pipe).run_host, out, R, C)
