"""The search for a batch item's frame, 64 lanes at a step: its result and
the number of its steps, with a wavefront of 64 host threads; frames without
work items, the first and last item of a frame, and batches of one frame to
several thousand."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from polymage_amd.cprint import DEVICE_PRELUDE
from helpers import gpu_build, bits_equal, emulating
from test_box_kernels import _small_frames

HARNESS = r'''
#include <pthread.h>
#include <cstring>
static thread_local struct { unsigned x; } threadIdx;
static pthread_barrier_t bar;
static unsigned char bits[64];
static int steps;
static unsigned long long __ballot(bool p) {
  bits[threadIdx.x] = p;
  pthread_barrier_wait(&bar);
  unsigned long long m = 0;
  for (int i = 0; i < 64; ++i) m |= (unsigned long long)bits[i] << i;
  if (threadIdx.x == 0) ++steps;
  pthread_barrier_wait(&bar);
  return m;
}
#define __device__
#define __forceinline__ inline
#define __popcll __builtin_popcountll
#define __builtin_amdgcn_readfirstlane(v) (v)
#define PMX_DEVICE_AS 1
%s
struct Arg { const long long* first; int n; const long long* t; int nt; int* out; unsigned lane; };
static void* lane(void* p) {
  Arg* a = (Arg*)p;
  threadIdx.x = a->lane;
  for (int k = 0; k < a->nt; ++k) {
    const int r = pmx_find_frame64(a->first, a->n, a->t[k]);
    if (a->lane == k %% 64) a->out[k] = r;
  }
  return nullptr;
}
extern "C" int search(const long long* first, int n, const long long* t, int nt, int* out) {
  steps = 0;
  pthread_barrier_init(&bar, nullptr, 64);
  pthread_t th[64];
  Arg a[64];
  for (unsigned i = 0; i < 64; ++i) { a[i] = Arg{first, n, t, nt, out, i}; pthread_create(&th[i], nullptr, lane, &a[i]); }
  for (unsigned i = 0; i < 64; ++i) pthread_join(th[i], nullptr);
  pthread_barrier_destroy(&bar);
  return steps;
}
'''


@pytest.fixture(scope="module")
def search(tmp_path_factory):
    d = tmp_path_factory.mktemp('search')
    a = DEVICE_PRELUDE.index('__device__ __forceinline__ int pmx_find_frame(')
    b = DEVICE_PRELUDE.index('#ifndef PMX_LD4', a)
    (d / 's.cpp').write_text(HARNESS % DEVICE_PRELUDE[a:b])
    so = str(d / 's.so')
    subprocess.check_call(['g++', '-O1', '-shared', '-fPIC', '-pthread', '-o', so, str(d / 's.cpp')])
    return ctypes.CDLL(so).search


@pytest.mark.parametrize("n", [1, 2, 48, 63, 64, 65, 130, 4095, 4096, 4097, 6000])
def test_frame_of_an_item(search, n):
    g = np.random.default_rng(n)
    items = g.integers(0, 4, n)         # a quarter of the frames has none
    items[0] = 1
    first = np.concatenate([[0], np.cumsum(items)[:-1]]).astype(np.int64)
    total = int(items.sum())
    t = np.unique(np.concatenate([[0, total - 1], g.integers(0, total, 20)])).astype(np.int64)
    out = np.full(len(t), -1, np.int32)
    p = lambda a: ctypes.c_void_p(a.ctypes.data)
    steps = search(p(first), n, p(t), len(t), p(out))
    assert np.array_equal(out, np.searchsorted(first, t, side='right') - 1)
    assert steps == len(t) * (1 if n <= 64 else 2 if n <= 4096 else 3)


@pytest.mark.gpu
def test_batch_of_thousands_of_frames(gpu):
    """4200 frames: three steps of the search."""
    if emulating():
        pytest.skip("device tensors are not emulated")
    import torch
    n = 4200
    print("case batch frames", n, flush=True)
    pipe, recs, refs = _small_frames(60)
    bp = gpu_build(pipe)
    recs = [dict(recs[i % 60]) for i in range(n)]
    imgs = [torch.from_numpy(recs[i]['img']).cuda() for i in range(60)]
    dev = [dict(rec, img=imgs[i % 60], harris=torch.full(rec['harris'].shape, -7.0, device='cuda'))
           for i, rec in enumerate(recs)]
    h = bp.batch_create(dev)
    try:
        bp.batch_run(h, torch.cuda.current_stream().cuda_stream, 'persistent')
        torch.cuda.synchronize()
        assert all(bits_equal(d['harris'].cpu().numpy(), refs[i % 60]) for i, d in enumerate(dev))
    finally:
        bp.batch_destroy(h)
