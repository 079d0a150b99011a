"""Host side of libofx.so without a GPU: failed allocations, retries, and the
order of what is launched, on a stand-in for the HIP runtime (fake_hip.cpp;
kernels do not run).  Each scenario runs in a process of its own, which loads
the stand-in before the library."""
import ctypes
import shutil
import subprocess
import sys
from pathlib import Path

import numpy as np
import pytest

HERE = Path(__file__).resolve().parent
if str(HERE.parent) not in sys.path:
    sys.path.insert(0, str(HERE.parent))

SCENARIOS = {}


def scenario(f):
    SCENARIOS[f.__name__] = f
    return f


# ---- what the scenarios share

def mesh(name):
    from oneflow_amd import meshgen
    if name == "chain":  # one cell per level: pipelined sweeps
        return meshgen.box2d(300, 1)
    g = meshgen.box2d(40, 30)  # coloured: a launch per level
    return meshgen.renumber(g, meshgen.multicolor_order(g))


def config(**kw):
    from oneflow_amd.config import CaseConfig
    return CaseConfig(**{**dict(dim=2, ischeme=1, ilim=-1, vismodel=3, mach_ref=0.5, reynolds=1e4), **kw})


def upload(L, h, g):
    """The return code of a mesh upload."""
    from oneflow_amd.solver import _dp, _ip
    x, y, z = (np.ascontiguousarray(a, np.float64) for a in (g.x, g.y, g.z))
    n, f, lc, rc, bc = (np.ascontiguousarray(a, np.int32) for a in (g.face_node_count, g.face_nodes, g.lc, g.rc, g.bc_type))
    return L.ofx_mesh_upload(h, g.dim, g.n_nodes, _dp(x), _dp(y), _dp(z), g.n_faces, g.n_cells, g.n_bfaces, _ip(n),
                             _ip(f), _ip(lc), _ip(rc), _ip(bc))


def context(fake):
    from oneflow_amd.solver import load_library
    L, h = load_library(), ctypes.c_void_p()
    assert L.ofx_ctx_create(ctypes.byref(h), 0) == 0
    return L, h


def zones_set(L, h, n, cells, faces):
    """The return code of declaring n zones of `cells` cells and `faces` boundary faces each."""
    from oneflow_amd.config import OfxConfig
    cfgs = (OfxConfig * n)()
    for z in range(n):
        cfgs[z] = config().to_c()
    start = lambda k: (ctypes.c_int * (n + 1))(*[k * z for z in range(n)], k * n)
    return L.ofx_zones_set(h, n, start(cells), start(faces), cfgs)


def lines(fake, word):
    return [s for s in fake.fake_log().decode().splitlines() if s.startswith(word)]


def sweep_kernels(fake, L, h):
    """Kernels of one NS and one SA sweep pair."""
    c = config().to_c()
    assert L.ofx_config_set(h, ctypes.byref(c)) == 0
    fake.fake_clear()
    assert L.ofx_lusgs_ns(h) == 0 and L.ofx_lusgs_sa(h) == 0
    return lines(fake, "launch")


# ---- scenarios

@scenario
def retried_upload(fake):
    """An upload that fails after the sweeps' schedule is built, then another
    mesh: its sweeps are its own."""
    L, h = context(fake)
    assert upload(L, h, mesh("chain")) == 0
    calls = {b"hipMalloc": len(lines(fake, "hipMalloc")), b"hipStreamSynchronize": len(lines(fake, "sync"))}
    assert any("k_sweep_pipe" in k for k in sweep_kernels(fake, L, h))
    for other in ("coloured", "chain"):
        for fn, k in [(fn, n - i) for fn, n in calls.items() for i in range(4)]:  # the upload's last calls
            L, h = context(fake)
            fake.fake_fail(fn, k)
            if upload(L, h, mesh("chain")) == 0:
                continue
            assert upload(L, h, mesh(other)) == 0
            piped = [s for s in sweep_kernels(fake, L, h) if "k_sweep_pipe" in s]
            assert bool(piped) == (other == "chain"), (other, fn, k, piped)


@scenario
def sweeps_without_memory(fake):
    """A mesh that fits without the pipelined sweeps' streams is accepted and swept
    level by level, whichever of their allocations fails; streams that are there
    give way to a later allocation."""
    L, h = context(fake)
    assert upload(L, h, mesh("chain")) == 0
    n, full = len(lines(fake, "hipMalloc")), fake.fake_held()
    L.ofx_ctx_destroy(h)
    assert fake.fake_held() == 0
    fake.fake_capacity(full - 1)
    L, h = context(fake)
    assert upload(L, h, mesh("chain")) == 0, L.ofx_last_error()
    need = fake.fake_held()  # without the streams
    assert need < full
    kernels = sweep_kernels(fake, L, h)
    assert kernels and not any("k_sweep_pipe" in k for k in kernels)
    L.ofx_ctx_destroy(h)
    fake.fake_capacity(need)
    L, h = context(fake)
    assert upload(L, h, mesh("chain")) == 0, L.ofx_last_error()
    L.ofx_ctx_destroy(h)
    fake.fake_capacity(2 * full)
    piped = []
    for k in range(1, n + 1):
        L, h = context(fake)
        fake.fake_fail(b"hipMalloc", k)
        if upload(L, h, mesh("chain")) == 0:
            piped.append(any("k_sweep_pipe" in s for s in sweep_kernels(fake, L, h)))
        fake.fake_fail(b"hipMalloc", 0)
        L.ofx_ctx_destroy(h)
        assert fake.fake_held() == 0
    assert len(piped) > 10 and not any(piped)
    # zones declared later: their arrays take the streams' place, and the sweeps go level by level
    L, h = context(fake)
    assert upload(L, h, mesh("chain")) == 0
    assert any("k_sweep_pipe" in k for k in sweep_kernels(fake, L, h))
    fake.fake_capacity(full)
    cfg, start = config().to_c(), (ctypes.c_int * 2)
    assert L.ofx_zones_set(h, 1, start(0, 300), start(0, 602), ctypes.byref(cfg)) == 0, L.ofx_last_error()
    assert not any("k_sweep_pipe" in k for k in sweep_kernels(fake, L, h))
    L.ofx_ctx_destroy(h)
    assert fake.fake_held() == 0


@scenario
def network_is_ready(fake):
    """Whatever ofx_mlp_create launches on the network's stream is finished when it
    returns: a forward pass may follow on any other stream."""
    from oneflow_amd.mlp import Mlp
    m = Mlp(seed=3)
    work = [s for s in fake.fake_log().decode().splitlines() if s.split()[0] in ("launch", "copy", "sync")]
    assert any("k_frag" in s for s in work)
    streams = {s.split()[1] for s in work}
    for st in streams:
        assert [s for s in work if s.split()[1] == st][-1] == "sync " + st, (st, work[-8:])
    del m


@scenario
def network_buffers_overlap(fake):
    """Outputs that overwrite inputs: every input is read before the first output
    is written, on the host (one upload, then one download) and on the device (the
    forward kernel reads a copy)."""
    from oneflow_amd.mlp import NIN, NOUT, Mlp, _fp
    m, n = Mlp(seed=3), 1 << 19
    buf = np.zeros((NIN + 2 * NOUT) * n, np.float32)
    x = buf[NOUT * n: (NOUT + NIN) * n]
    for at, apart in ((0, True), (1, False), (NOUT * n, False), ((NOUT + NIN) * n - 1, False), ((NOUT + NIN) * n, True)):
        fake.fake_clear()
        assert m._L.ofx_mlp_forward(m.h, _fp(x), n, _fp(buf[at:])) == 0
        assert (len(lines(fake, "copy")) > 2) == apart, at
    n = 1024
    x = buf[NOUT * n: (NOUT + NIN) * n]
    dev = lambda a: ctypes.c_void_p(a.ctypes.data)
    for at, apart in ((0, True), (1, False), (NOUT * n, False), ((NOUT + NIN) * n - 1, False), ((NOUT + NIN) * n, True)):
        fake.fake_clear()
        assert m._L.ofx_mlp_forward_noalloc(m.h, dev(x), n, dev(buf[at:]), None) == 0
        kernels = lines(fake, "launch")
        assert len(kernels) == (1 if apart else 2) and "k_mlp_forward" in kernels[-1], (at, kernels)
    del m


@scenario
def zones_refused(fake):
    """ofx_zones_set that fails, at whichever allocation, leaves the context with the
    zones and the result memory it had: norms and forces still go somewhere."""
    from oneflow_amd import meshgen
    from oneflow_amd.solver import OfxNorms
    parts = 140
    one = meshgen.box2d(3, 2)
    g = meshgen.concat_grids([one] * parts)[0]
    cells, faces = one.n_cells, one.n_bfaces
    for kernel, arg in (("k_norm_partial", 2), ("k_norm_final", 1), ("k_norm_final", 2), ("k_aero", 3)):
        fake.fake_watch(kernel.encode(), arg)
    out, forces = (OfxNorms * parts)(), (ctypes.c_double * (4 * parts))()
    for before in (1, 2, 70):  # zones when the refused call comes
        n = {"hipMalloc": 0, "hipHostMalloc": 0}
        for fn in n:
            k = 0
            while True:
                L, h = context(fake)
                c = config().to_c()
                assert upload(L, h, g) == 0 and L.ofx_config_set(h, ctypes.byref(c)) == 0
                if before > 1:
                    assert zones_set(L, h, before, cells * parts // before, faces * parts // before) == 0
                k += 1
                fake.fake_fail(fn.encode(), k)
                rc = zones_set(L, h, parts, cells, faces)
                fake.fake_fail(fn.encode(), 0)
                fake.fake_clear()
                assert L.ofx_zones_norms(h, out) == 0 and L.ofx_zones_aero(h, forces) == 0
                assert L.ofx_init_freestream(h) == 0
                now = parts if rc == 0 else before
                sizes = [int(s.split()[1]) for s in lines(fake, "arg")]
                want = [6 * 512 * 8 * now, 6 * 512 * 8 * now, 6 * 8 * now, 6 * 8 * now]
                assert len(sizes) == 4 and all(a >= b for a, b in zip(sizes, want)), (before, fn, k, rc, sizes, want)
                L.ofx_ctx_destroy(h)
                assert fake.fake_held() == 0
                if rc == 0:
                    break
                n[fn] += 1
        assert n["hipMalloc"] >= 7 and n["hipHostMalloc"] == 1, n


@scenario
def piped_forward_fails(fake):
    """The piped forward pass without a second stream, or with a copy that fails
    midway: it falls back, or reports the error with nothing left in flight to the
    caller's outputs, and the next call succeeds."""
    from oneflow_amd.mlp import NIN, NOUT, Mlp, _fp
    n = 1 << 19
    x, y = np.zeros((n, NIN), np.float32), np.zeros((n, NOUT), np.float32)
    m = Mlp(seed=3)
    fake.fake_fail(b"hipStreamCreateWithFlags", 1)
    assert m._L.ofx_mlp_forward(m.h, _fp(x), n, _fp(y)) == 0, m._L.ofx_last_error()
    for k in range(1, 10):
        fake.fake_clear()
        fake.fake_fail(b"hipMemcpyAsync", k)
        rc = m._L.ofx_mlp_forward(m.h, _fp(x), n, _fp(y))
        fake.fake_fail(b"hipMemcpyAsync", 0)
        work = [s for s in fake.fake_log().decode().splitlines() if s.split()[0] in ("copy", "sync")]
        assert (rc != 0) == (k <= 8), (k, rc)
        for st in {s.split()[1] for s in work}:
            assert [s for s in work if s.split()[1] == st][-1] == "sync " + st, (k, st, work)
        assert m._L.ofx_mlp_forward(m.h, _fp(x), n, _fp(y)) == 0, (k, m._L.ofx_last_error())
    del m


@scenario
def autotune_keeps_the_fused_gradients(fake):
    """Gradient kernels timed one by one, the form by face id a little faster: a full
    LU-SGS step keeps the form that evaluates both gradients in one kernel, which no
    such timing covers; a multi-stage run, which has no such kernel, takes the
    faster ones."""
    for k in (b"k_ns_gradILi2ELi4ELin1ELb0", b"k_ns_gradILi2ELi4ELi0ELb0", b"k_sa_gradILi2ELi4ELb0"):
        fake.fake_cost(k, 1.0)
    for k in (b"k_ns_grad", b"k_sa_grad"):
        fake.fake_cost(k, 1.01)
    for kw, fused in ((dict(), True), (dict(time_integral=1, rk_stage=3), False), (dict(vismodel=1), False)):
        L, h = context(fake)
        c = config(**kw).to_c()
        assert upload(L, h, mesh("coloured")) == 0 and L.ofx_config_set(h, ctypes.byref(c)) == 0
        assert L.ofx_autotune(h, 1, None) == 0
        v = [ctypes.c_int() for _ in range(2)]
        for x, kernel in zip(v, (0, 5)):
            assert L.ofx_get_kernel_variant(h, kernel, ctypes.byref(x)) == 0
        sa = kw.get("vismodel", 3) == 3
        assert [x.value for x in v] == [int(fused), int(fused or not sa)], (kw, [x.value for x in v])
        fake.fake_clear()
        assert L.ofx_iterate(h, 1, 1, None) == 0
        assert any("k_sa_grad_boundary" in s for s in lines(fake, "launch")) == fused
        L.ofx_ctx_destroy(h)


@pytest.mark.parametrize("name", list(SCENARIOS))
def test_host_path(name, tmp_path):
    if not shutil.which("g++"):
        pytest.skip("g++ not available")
    if not (HERE.parent / "oneflow_amd" / "libofx.so").exists():
        pytest.skip("libofx.so not built in this checkout")
    so = tmp_path / "libfake_hip.so"
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-pthread", str(HERE / "fake_hip.cpp"), "-o", str(so)],
                   check=True)
    r = subprocess.run([sys.executable, str(HERE / "test_host_paths.py"), str(so), name], capture_output=True, text=True,
                       timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr


if __name__ == "__main__":
    lib = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)  # before libofx.so: its symbols come first
    lib.fake_log.restype = ctypes.c_char_p
    lib.fake_held.restype = ctypes.c_size_t
    lib.fake_capacity.argtypes = [ctypes.c_size_t]
    lib.fake_cost.argtypes = [ctypes.c_char_p, ctypes.c_double]
    SCENARIOS[sys.argv[2]](lib)
