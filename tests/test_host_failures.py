"""Host code of libvpbs when a HIP call fails, on the CPU: the library runs on a HIP runtime without a GPU
(``fake_hip.c``: device memory in host memory, kernels counted and not run), in a process of its own."""
import ctypes
import json
import math
import pathlib
import subprocess
import sys
from types import SimpleNamespace

import numpy as np
import pytest

HERE = pathlib.Path(__file__).resolve().parent
TWO_PI = 2 * math.pi


@pytest.fixture(scope="module")
def fake_hip(tmp_path_factory):
    lib = tmp_path_factory.mktemp("fake_hip") / "libfakehip.so"
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-o", str(lib), str(HERE / "fake_hip.c")], check=True)
    return lib


def run(fake_hip, scenario, *args):
    r = subprocess.run([sys.executable, __file__, str(fake_hip), scenario, *map(str, args)], capture_output=True,
                       text=True, timeout=100)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-4000:]
    return json.loads(r.stdout.splitlines()[-1])


@pytest.mark.parametrize("work", ["points", "advance", "learned", "gradient"])
def test_out_of_memory_while_growing(fake_hip, work):
    """Buffers grow for a larger call and one allocation after the other fails: that call says so or does without, no
    call after it takes the freed buffers for valid ones, and a smaller call then has every buffer that it has in a new
    context."""
    out = run(fake_hip, work)
    assert out["allocations"] >= 3
    for k, after in enumerate(out["after"], 1):
        assert after["refused"] or after["grid"], f"allocation {k}: the larger call did not fail"
        assert not after["stale"], f"allocation {k}: {after['stale']} took freed buffers"
        assert not after["again"], f"allocation {k}: the smaller call: {after['again']}"
        assert len(after["blocks"]) == len(out["fresh"]), f"allocation {k}: buffers missing"
        assert all(a >= b for a, b in zip(after["blocks"], out["fresh"])), f"allocation {k}: buffers too small"


def test_interpolation_without_memory_for_slabs(fake_hip):
    """The six buffers of the interpolation fused with the inverse x transform: without one of them a call interpolates
    from the real grid, which took less memory all along, and with memory again the next one is fused again."""
    out = run(fake_hip, "points")
    assert [a["grid"] for a in out["after"]].count(True) == 6
    assert all(a["fused_again"] for a in out["after"])


@pytest.mark.parametrize("call", ["hipHostGetDevicePointer", "hipLaunchKernel"])
def test_filaments_are_there_once_their_kernels_ran(fake_hip, call):
    """An upload that fails before its kernels ran leaves no filaments to step: the filament of each node, which the
    step's kernels index with, comes from them."""
    assert run(fake_hip, "upload", call) == {"upload": True, "advance": True, "again": ""}


# --------------------------------------------------------------------------- #
# In the process of its own


def points(n, seed=1):
    rng = np.random.default_rng(seed)
    one = rng.normal(size=(3, n))
    return SimpleNamespace(nodes=rng.random((3, n)) * TWO_PI, node_idx_prev=np.roll(np.arange(n, dtype=np.int32), 1),
                           sp=one, spp=one, dlm=np.full(n, 0.1), dlp=np.full(n, 0.1),
                           points=rng.random((3, n)) * TWO_PI, charges=one)


class Work:
    """One kind of calls: ``start`` makes what they need, ``call(state, n)`` is one of size n, ``stale`` are calls that
    need what the failed one replaced."""

    def __init__(self, vp, kind):
        self.vp, self.kind = vp, kind
        spl = vp.GaussianSplitting.create(Ls=TWO_PI, β=2.5 if kind == "learned" else 3.0, Ns=(40, 42, 44))
        self.p = vp.ParamsBiotSavart.build(np.float64, Γ=1.0, a=1e-6, Δ=0.25, splitting=spl,
                                           quadrature=vp.GaussLegendre(1))

    def start(self):
        if self.kind == "gradient":
            net = self.vp._lib.MLP(32, 32, 2, 3)
            net.set_params(np.zeros(net.nparams), np.zeros(32), np.ones(32), np.ones(3))
            return net
        ctx = self.vp._lib.Context(self.p)
        if self.kind == "learned":
            ctx.net = self.vp._lib.MLP(128, 128, 3, 3)
            ctx.net.set_params(np.zeros(ctx.net.nparams), np.zeros(128), np.ones(128), np.ones(3))
            ctx.learned_setup(ctx.net, 0.7 * self.p.α, 1.3 * self.p.rcut, 0.5 * self.p.rcut, sample_fraction=0.5)
        return ctx

    def call(self, s, n):
        F = self.vp._lib
        if self.kind == "gradient":
            X, T = np.zeros((n, 32), np.float32), np.zeros((n, 3), np.float32)
            g, loss = np.empty(s.nparams, np.float32), ctypes.c_double()
            rc = s._L.vpbs_mlp_gradient(s.handle, n, X.ctypes.data, T.ctypes.data, ctypes.byref(loss), g.ctypes.data)
            return s._check(rc, "vpbs_mlp_gradient")
        if self.kind == "points":
            s.set_points(points(n))
            s.compute(F.VELOCITY | F.STREAMFUNCTION | F.KEEP_UHAT | F.NEIGHBOUR_STATS)
            return s.energy_spectrum(max(n // 10, 1), 1.0)
        self.upload(s, n)
        if self.kind == "learned":
            s.compute_learned()
        else:
            s.advance(1e-3, 1)

    def upload(self, s, n):
        t = TWO_PI * np.arange(n) / n
        X = np.stack([1 + np.cos(t), 2 + np.sin(t), 3 + 0.1 * np.sin(3 * t)], axis=1)
        s.set_filaments(self.vp.FilamentBatch([self.vp.ClosedFilament(X, np.zeros(3))]), self.p)

    def stale(self, s):
        """Calls on what the failed one replaced, of which none may find anything."""
        if self.kind == "gradient":
            return []
        calls = {"get_points": s.get_points, "neighbour_stats": s.neighbour_stats, "advance": lambda: s.advance(1e-3),
                 "compute": lambda: s.compute(self.vp._lib.VELOCITY)}
        took = []
        for name, f in calls.items():
            try:
                f()
                took.append(name)
            except self.vp._lib.VpbsError:
                pass
        return took


def grow_and_fail(vp, fake, kind):
    small, large = (60, 200) if kind != "gradient" else (512, 2048)
    w = Work(vp, kind)

    def blocks():
        b = (ctypes.c_size_t * 4096)()
        return sorted(b[: fake.fake_blocks(b, 4096)])

    s = w.start()
    w.call(s, small)
    fresh = blocks()
    before, grids = fake.fake_mallocs(), fake.fake_launches(b"spec_x_inverse")
    w.call(s, large)
    count, ordinary = fake.fake_mallocs() - before, fake.fake_launches(b"spec_x_inverse") - grids
    s.close()
    if hasattr(s, "net"):
        s.net.close()
    out = {"allocations": count, "fresh": fresh, "after": []}
    assert not blocks()
    for k in range(1, count + 1):
        s = w.start()
        w.call(s, small)
        fake.fake_fail_malloc(k)
        grids = fake.fake_launches(b"spec_x_inverse")
        try:
            w.call(s, large)
            refused = False
        except vp._lib.VpbsError as e:
            refused = "out of memory" in str(e)
        fake.fake_fail_malloc(0)
        grid = not refused and fake.fake_launches(b"spec_x_inverse") - grids > ordinary
        # what a failed set_points or set_filaments leaves; later stages may fail with the points in place
        pts = ctypes.c_int(s._L.vpbs_get_points(s._h, *([None] * 8))).value == 0 if kind != "gradient" else True
        stale = [] if pts else w.stale(s)
        again, slabs = "", fake.fake_launches(b"x_inverse_interp")
        try:
            w.call(s, small)
        except vp._lib.VpbsError as e:
            again = str(e)
        out["after"].append({"refused": refused, "grid": grid, "stale": stale, "again": again, "blocks": blocks(),
                             "fused_again": fake.fake_launches(b"x_inverse_interp") > slabs})
        s.close()
        if hasattr(s, "net"):
            s.net.close()
    return out


def upload_and_fail(vp, fake, call):
    w = Work(vp, "advance")
    s = w.start()
    out = {}

    def refused(f):
        try:
            f()
        except vp._lib.VpbsError as e:
            return str(e)
        return ""

    fake.fake_fail_call(call.encode())
    out["upload"] = "invalid value" in refused(lambda: w.upload(s, 60))
    fake.fake_fail_call(None)
    out["advance"] = "no filaments on the device" in refused(lambda: s.advance(1e-3, 1))
    out["again"] = refused(lambda: w.call(s, 60))
    s.close()
    return out


def main():
    fake = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
    fake.fake_mallocs.restype = fake.fake_launches.restype = ctypes.c_long
    fake.fake_fail_malloc.argtypes = [ctypes.c_long]
    fake.fake_fail_call.argtypes = fake.fake_launches.argtypes = [ctypes.c_char_p]
    sys.path.insert(0, str(HERE.parent))
    import __graft_entry__ as ge

    vp = ge.load_package()
    if sys.argv[2] == "upload":
        print(json.dumps(upload_and_fail(vp, fake, sys.argv[3])))
    else:
        print(json.dumps(grow_and_fail(vp, fake, sys.argv[2])))


if __name__ == "__main__":
    main()
