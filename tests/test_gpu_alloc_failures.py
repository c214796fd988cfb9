"""Calls during which an allocation fails, forced from the host: a child process
loads a library that stands before the runtime's allocation entry points and
turns chosen calls into ones that the runtime refuses (an impossible size)."""
import ctypes as C
import os
import subprocess
import sys

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))

SHIM = r"""
#include <dlfcn.h>
#include <stddef.h>
static long left = -1, calls = 0;
static int keep = 0, no_pinned = 0;
extern "C" void shim_no_pinned(int on) { no_pinned = on; }
extern "C" int hipHostMalloc(void **p, size_t n, unsigned flags)
{
    static int (*real)(void **, size_t, unsigned) = (int (*)(void **, size_t, unsigned))dlsym(RTLD_NEXT, "hipHostMalloc");
    if (no_pinned) {
        no_pinned++;
        n = (size_t)1 << 60;
    }
    return real(p, n, flags);
}
extern "C" int shim_pinned_refused() { return no_pinned - 1; }
extern "C" void shim_malloc(long after, int stay) { left = after; keep = stay; }
extern "C" long shim_calls() { return calls; }
extern "C" int hipMalloc(void **p, size_t n)
{
    static int (*real)(void **, size_t) = (int (*)(void **, size_t))dlsym(RTLD_NEXT, "hipMalloc");
    calls++;
    if (left == 0) {
        if (!keep) left = -1;
        n = (size_t)1 << 60;
    } else if (left > 0) {
        left--;
    }
    return real(p, n);
}
"""


@pytest.fixture(scope="module")
def shim(tmp_path_factory):
    d = tmp_path_factory.mktemp("shim")
    src, lib = d / "shim.cpp", d / "libshim.so"
    src.write_text(SHIM)
    subprocess.run(["g++", "-O1", "-shared", "-fPIC", str(src), "-o", str(lib), "-L/opt/rocm/lib", "-Wl,-rpath,/opt/rocm/lib",
                    "-Wl,--no-as-needed", "-lamdhip64", "-ldl"], check=True)
    return str(lib)


def child(shim, name):
    r = subprocess.run([sys.executable, os.path.abspath(__file__), shim, name], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-4000:]


@pytest.mark.gpu
def test_failed_adjoint_setup_is_not_taken_for_whole(shim):
    child(shim, "adjoint_setup")


@pytest.mark.gpu
def test_without_memory_for_the_fused_pass(shim):
    child(shim, "weight_rows")


@pytest.mark.gpu
def test_transfers_without_pinned_memory(shim):
    child(shim, "pinned")


# ---------------------------------------------------------------------------
# in the child
# ---------------------------------------------------------------------------
class Failures:
    def __init__(self, path):
        self.lib = C.CDLL(path, mode=C.RTLD_GLOBAL)
        self.lib.shim_calls.restype = C.c_long
        self.lib.shim_malloc.argtypes = [C.c_long, C.c_int]

    def calls(self):
        return self.lib.shim_calls()

    def after(self, n, keep=False):
        """Fail the (n + 1)-th allocation from now on, and with keep all that follow."""
        self.lib.shim_malloc(n, 1 if keep else 0)

    def off(self):
        self.lib.shim_malloc(-1, 0)


def small_solver():
    import cases
    from lbfs_amd import abi
    mesh = cases.channel_mesh(24, 16, 16, seed=8)
    s = abi.Solver(mesh, abi.make_params(visc=1.0 / 6.0, dt=0.25, body_force=(2e-5, 0.0, 0.0)))
    s.set_state(*cases.smooth_state(mesh, seed=8, amp=0.005))
    x, t = abi.rbc(4, 8.0, center=(12.0, 8.0, 8.0))
    s.add_membranes([abi.Membrane(x, t, **dict(abi.RBC_PARAMS, volume_ratio=0.95))])
    return s


def refused(call, *args):
    from lbfs_amd import abi
    try:
        call(*args)
    except abi.LbfsError:
        return True
    return False


def adjoint_setup(fail):
    """A gradient whose set-up failed fails again while memory is short, and
    succeeds in full afterwards."""
    rng = np.random.default_rng(3)

    def gradient(s):
        s.adjoint_forward(9, 4)
        lam = rng0.standard_normal((s.n_mem_nodes, 3))
        g = s.adjoint_backward(lam_nodes=lam, lam_state=rng0.standard_normal((s.n, 4)))
        return [s.membrane_nodes()[0], g["body_force"], g["moduli"], g["state0"], g["nodes0"]]

    s = small_solver()
    assert fail.calls() > 0  # the allocations do pass through the library
    c0 = fail.calls()
    rng0 = np.random.default_rng(3)
    want = gradient(s)
    n = fail.calls() - c0
    s.close()
    for k in sorted(set([0, 1, n - 1] + list(rng.integers(0, n, 8)))):
        print("set-up of %d allocations, failing at %d" % (n, k), flush=True)
        s = small_solver()
        fail.after(int(k), keep=True)
        assert refused(s.adjoint_forward, 9, 4)
        assert refused(s.adjoint_forward, 9, 4)
        fail.off()
        assert refused(s.adjoint_rewind)
        rng0 = np.random.default_rng(3)
        got = gradient(s)
        for a, b in zip(want, got):
            assert np.all(np.isfinite(a)) and np.array_equal(a, b)
        s.close()


def weight_rows(fail):
    """A solver whose fused pass's weight rows find no memory runs the two passes,
    and gives the rows back where a later allocation needs them: the same bits."""
    import cases
    from lbfs_amd import abi
    mesh = cases.channel_mesh(24, 16, 16, seed=8)
    x, t = abi.rbc(4, 8.0, center=(12.0, 8.0, 8.0))

    def create():
        return abi.Solver(mesh, abi.make_params(visc=1.0 / 6.0, dt=0.25, body_force=(2e-5, 0.0, 0.0)))

    def run(s, membranes_fail=None, gradient_fail=None):
        rng = np.random.default_rng(3)
        s.set_state(*cases.smooth_state(mesh, seed=8, amp=0.005))
        s.step(5)
        if membranes_fail is not None:
            fail.after(membranes_fail)
        c = fail.calls()
        s.add_membranes([abi.Membrane(x, t, **dict(abi.RBC_PARAMS, volume_ratio=0.95))])
        c_mem = fail.calls() - c
        s.step(5)
        if gradient_fail is not None:
            fail.after(gradient_fail)
        c = fail.calls()
        s.adjoint_forward(9, 4)
        c_adj = fail.calls() - c
        g = s.adjoint_backward(lam_nodes=rng.standard_normal((s.n_mem_nodes, 3)),
                               lam_state=rng.standard_normal((s.n, 4)))
        out = list(s.get_state()) + list(s.membrane_nodes()) + [g[k] for k in sorted(g)]
        return out, c_mem, c_adj

    def equal(a, b):
        return all(np.all(np.isfinite(p)) and np.array_equal(p, q) for p, q in zip(a, b))

    c = fail.calls()
    s = create()
    n = fail.calls() - c
    s.set_fused(True)
    want, n_mem, n_adj = run(s)
    s.close()
    created = []
    for k in range(n):
        print("creation of %d allocations, failing at %d" % (n, k), flush=True)
        fail.after(k)
        try:
            s = create()
        except abi.LbfsError:
            fail.off()
            continue
        fail.off()
        created.append(k)
        assert refused(s.set_fused, True)
        assert equal(want, run(s)[0])
        s.close()
    assert created == [n - 1]
    for kw in [dict(membranes_fail=k) for k in (0, n_mem // 2, n_mem - 1)] + \
              [dict(gradient_fail=k) for k in (0, n_adj // 2, n_adj - 1)]:
        print(kw, flush=True)
        s = create()
        assert equal(want, run(s, **kw)[0])
        assert refused(s.set_fused, True)
        s.close()


def pinned(fail):
    """Readbacks and adjoint seeds without pinned memory: the same values, on a
    small solver and on one whose arrays move in three staged chunks."""
    import cases
    from lbfs_amd import abi
    rng = np.random.default_rng(5)
    lam_nodes = lam_state = None
    mesh = abi.HexMesh(96, 80, 72, periodic=(1, 0, 0), jitter=0.1, seed=2)
    large_state, large_seed = cases.smooth_state(mesh, seed=1), rng.standard_normal((mesh.n_cells, 4))

    def run_large():
        s = abi.Solver(mesh, abi.make_params(visc=1.0 / 6.0, dt=0.25))
        s.set_state(*large_state)
        s.adjoint_forward(1, 1)
        g = s.adjoint_backward(lam_state=large_seed)
        out = [g["state0"], g["body_force"]] + list(s.get_state())
        s.close()
        return out

    def run():
        nonlocal lam_nodes, lam_state
        s = small_solver()
        s.step(3)
        out = list(s.get_state()) + list(s.membrane_nodes())
        s.adjoint_forward(5, 3)
        if lam_nodes is None:
            lam_nodes, lam_state = rng.standard_normal((s.n_mem_nodes, 3)), rng.standard_normal((s.n, 4))
        g = s.adjoint_backward(lam_nodes=lam_nodes, lam_state=lam_state)
        s.step(2)
        out += [g[k] for k in sorted(g)] + list(s.get_state())
        s.close()
        return out

    want = run() + run_large()
    fail.lib.shim_no_pinned(1)
    got = run() + run_large()
    assert fail.lib.shim_pinned_refused() > 0
    for a, b in zip(want, got):
        assert np.all(np.isfinite(a)) and np.array_equal(a, b)


if __name__ == "__main__":
    sys.path[:0] = [HERE, os.path.dirname(HERE), os.path.join(os.path.dirname(HERE), "lbfs-ibm-ade-sp_amd")]
    globals()[sys.argv[2]](Failures(sys.argv[1]))
