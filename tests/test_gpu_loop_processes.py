"""One-launch loops of two processes on one device: a process that has none of the
device's places runs step by step meanwhile, with the same results, and neither
ever waits for workgroups that do not fit."""
import ast
import fcntl
import glob
import os
import subprocess
import sys
import textwrap

import numpy as np
import pytest

import test_gpu_patch_step as PS
from flexshell import _lib, explicit, femm as FM
from flexshell.material import MatDeforElastIso

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _job(ctx, nx, ny):
    _, xyz, conn, d = PS._grid(3, nx, ny)
    f = FM.make(conn, MatDeforElastIso(70e9, 0.33, 2700.0), thickness=0.02, ctx=ctx)
    f.associategeometry(xyz)
    f.stiffness(FM.SysmatAssemblerHIP(_lib.FS_BLOCK_FF), xyz, None, None, d)
    f.mass(FM.SysmatAssemblerHIP(_lib.FS_BLOCK_FF), xyz, d)
    z, V0 = np.zeros(d.nfreedofs), np.random.default_rng(4).normal(0, 1e-3, d.nfreedofs)

    def run(nsteps):
        r = explicit.run(f._model, 0.0, z, V0, 1e-8, nsteps, z, np.zeros(nsteps + 1))
        return f._model.cd_form(), r["U"]

    return f, run


def test_lock_of_another_process(ctx):
    print("[gpu] loop places, lock held", flush=True)
    f, run = _job(ctx, 40, 30)
    form, U = run(100)
    assert form == _lib.FS_CD_ONE_LAUNCH
    files = glob.glob("/dev/shm/flexshell-loops-*")
    assert files
    # a lock through a file description of its own, as another process has it
    held = [open(p) for p in files]
    for h in held:
        fcntl.flock(h, fcntl.LOCK_EX | fcntl.LOCK_NB)  # free between loops
    form, V = run(100)
    assert form == _lib.FS_CD_PATCHES and np.array_equal(U, V)
    for h in held:
        h.close()
    form, V = run(100)
    assert form == _lib.FS_CD_ONE_LAUNCH and np.array_equal(U, V)
    f._model.close()


def test_two_processes(ctx):
    """Two processes with 450 patches each (a device has 512 places): loops side by side
    for a second."""
    print("[gpu] loops of two processes", flush=True)
    script = textwrap.dedent("""
        import sys, time
        sys.path[:0] = [sys.argv[1], sys.argv[1] + "/finetoolsflexstructures.jl_amd", sys.argv[1] + "/tests"]
        import test_gpu_loop_processes as T
        from flexshell import _lib
        f, run = T._job(_lib.Context(0), 140, 130)
        run(100)
        print("ready", flush=True)
        sys.stdin.readline()
        end, forms, U = time.time() + 1.0, set(), None
        while time.time() < end:
            form, V = run(2000)
            assert U is None or (U == V).all()
            U = V
            forms.add(form)
        print(sorted(forms), flush=True)
    """)
    p = subprocess.Popen([sys.executable, "-u", "-c", script, ROOT], stdin=subprocess.PIPE, stdout=subprocess.PIPE,
                         stderr=subprocess.STDOUT, text=True)
    try:
        f, run = _job(ctx, 140, 130)
        form, U = run(2000)
        assert form == _lib.FS_CD_ONE_LAUNCH
        for line in p.stdout:
            if line.strip() == "ready":
                break
        else:
            raise AssertionError("the other process did not start")
        p.stdin.write("\n")
        p.stdin.flush()
        forms = set()
        while p.poll() is None:
            form, V = run(2000)
            forms.add(form)
            assert np.array_equal(U, V)
        theirs = p.stdout.read().strip()
    finally:
        p.kill()
        p.wait()
    both = {_lib.FS_CD_PATCHES, _lib.FS_CD_ONE_LAUNCH}
    assert p.returncode == 0 and forms and forms <= both, (forms, theirs)
    assert set(ast.literal_eval(theirs.splitlines()[-1])) <= both, theirs
    f._model.close()
