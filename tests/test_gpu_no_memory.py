"""Device allocations that fail while a plan is built: the build ends with
an error or with a working plan, and does without a schedule that it
only would have timed.

A second copy of the library is loaded behind a shim of hipMalloc that fails
one call, by number; nothing is really short of memory."""
import ctypes
import os
import shutil
import subprocess

import numpy as np
import pytest

from helpers import residual
from rbsptrsv import LIB_PATH, SCHED_AUTO, SCHED_BLOCKED, _lib, gen

pytestmark = pytest.mark.gpu

SHIM = r"""
#include <dlfcn.h>
#include <stddef.h>
static int calls, bad;
static int (*real)(void **, size_t);
int shim_fail(void *f, int at) { real = f; calls = 0; bad = at; return 0; }
int shim_calls(void) { return calls; }
int hipMalloc(void **p, size_t n) {
    if (++calls == bad) { *p = NULL; return 2; }  /* hipErrorOutOfMemory */
    return real(p, n);
}
"""


@pytest.fixture(scope="module")
def shim(tmp_path_factory):
    import torch
    assert torch.cuda.is_available()
    real = ctypes.cast(_lib.lib().hipMalloc, ctypes.c_void_p)  # of the loaded runtime
    d = tmp_path_factory.mktemp("shim")
    (d / "shim.c").write_text(SHIM)
    subprocess.run(["gcc", "-shared", "-fPIC", str(d / "shim.c"), "-o", str(d / "shim.so")],
                   check=True)
    S = ctypes.CDLL(str(d / "shim.so"), mode=os.RTLD_GLOBAL)
    S.shim_fail.argtypes = [ctypes.c_void_p, ctypes.c_int]
    copy = str(d / "copy.so")
    shutil.copy(LIB_PATH, copy)
    L = ctypes.CDLL(copy)
    vp, i = ctypes.c_void_p, ctypes.c_int
    L.rb_plan_create.argtypes = [vp, vp, vp, i, i, i, i, i, vp, vp, ctypes.POINTER(vp)]
    L.rb_solve.argtypes = [vp, vp, i, vp, i, i, vp]
    L.rb_plan_destroy.argtypes = [vp]
    L.rb_plan_schedule.argtypes = [vp]
    return torch, S, L, real


def _failures(shim, f, schedule):
    """(statuses of builds whose k-th allocation fails, schedules kept)"""
    torch, S, L, real = shim
    dev = [torch.as_tensor(a, device="cuda") for a in (f.colptr, f.rowidx, f.val)]
    rng = np.random.default_rng(1)
    b = torch.as_tensor(rng.uniform(-1, 1, f.n), device="cuda")
    x = torch.empty_like(b)
    opts = _lib.rb_opts()
    opts.schedule = schedule
    status, kept, k = [], set(), 0
    while True:
        k += 1
        S.shim_fail(real, k)
        h = ctypes.c_void_p()
        st = L.rb_plan_create(dev[0].data_ptr(), dev[1].data_ptr(), dev[2].data_ptr(), f.n, f.n,
                              int(f.colptr[-1]), f.substitution, -1, ctypes.byref(opts), None,
                              ctypes.byref(h))
        calls = S.shim_calls()
        assert st in (0, 6, 7), (k, st)
        S.shim_fail(real, 0)
        if st == 0:
            kept.add(L.rb_plan_schedule(h))
            assert L.rb_solve(h, b.data_ptr(), f.n, x.data_ptr(), f.n, 1, None) == 0
            torch.cuda.synchronize()
            assert residual(f, x.cpu().numpy(), b.cpu().numpy()) < 1e-12, k
            L.rb_plan_destroy(h)
        if k > calls:
            return status, kept
        status.append(st)


@pytest.mark.parametrize("make", [lambda: gen.powerlaw(30000, seed=1),
                                  lambda: gen.banded(20000, seed=1)], ids=["wide", "deep"])
def test_build_does_without_what_it_only_would_time(shim, make):
    f = make()
    alone, _ = _failures(shim, f, SCHED_BLOCKED)
    status, kept = _failures(shim, f, SCHED_AUTO)
    print(f.name, "allocations", len(alone), len(status), "failed", sum(s != 0 for s in alone),
          sum(s != 0 for s in status), "kept", kept, flush=True)
    assert len(alone) > 4 and len(status) > len(alone) and len(kept) > 1
    # two more: the right-hand side and solution that schedules are timed on
    assert sum(s != 0 for s in status) <= sum(s != 0 for s in alone) + 2
