"""Leapfrog KDK and FP64 diagnostics on the GPU against the reference (vectors
and oracle), plus the reference's two-body orbit regression."""
import ctypes as C
import math

import numpy as np
import pytest

from nbx_testlib import Diagnostics, Particles, gravity

pytestmark = pytest.mark.gpu


def fixture_particles(golden, name):
    n = golden[f"{name}/px"].size
    return Particles(n, {k: golden[f"{name}/{k}"] for k in ("px", "py", "pz", "vx", "vy", "vz", "m")})


def test_kdk_three_steps_bit_identical_to_reference_vectors(nbx, golden):
    """integrator.c:47-85 with the scalar kernel, 3 steps, dt=1e-3, eps=0.01."""
    p = fixture_particles(golden, "globular1000_s3")
    with nbx.Engine(p.n) as e:
        e.upload_view(p.view)
        e.compute_force("hip_direct_fp64", eps=0.01)
        e.advance("hip_direct_fp64", dt=1e-3, steps=3, eps=0.01)
        out = e.download()
        d = e.diagnostics(eps=0.01, potential=True)
    for k, col in (("px", 0), ("py", 1), ("pz", 2)):
        assert np.array_equal(out["pos"][:, col], golden[f"globular1000_s3/kdk3/{k}"])
    for k, col in (("vx", 0), ("vy", 1), ("vz", 2)):
        assert np.array_equal(out["vel"][:, col], golden[f"globular1000_s3/kdk3/{k}"])
    assert np.array_equal(out["acc"], golden["globular1000_s3/kdk3/acc"])
    ref = golden["globular1000_s3/kdk3/diagnostics"]
    names = [f for f, _ in Diagnostics._fields_]
    for k, name in enumerate(names):
        # FP64 tree reduction vs the reference's sequential sum: 1e-12 relative
        scale = max(abs(ref[k]), 1e-12 if "momentum" in name or "center" in name else 1e-300)
        assert abs(d[name] - ref[k]) <= 1e-12 * scale + 1e-15, name
    u = golden["globular1000_s3/kdk3/potential"][0]
    assert abs(d["potential_energy"] - u) <= 1e-12 * abs(u)


def test_diagnostics_closed_forms(nbx):
    p = Particles(2, {"px": [1, 4], "py": [2, 5], "pz": [3, 6], "vx": [1, 0], "vy": [0, 1],
                      "vz": [0, 0], "m": [2.0, 3.0]})
    with nbx.Engine(2) as e:
        e.upload_view(p.view)
        d = e.diagnostics(eps=0.0, potential=False)
    assert d["kinetic_energy"] == 2.5
    assert (d["total_momentum_x"], d["total_momentum_y"], d["total_momentum_z"]) == (2, 3, 0)
    assert (d["total_angular_momentum_x"], d["total_angular_momentum_y"],
            d["total_angular_momentum_z"]) == (-18, 6, 8)
    assert d["center_of_mass_x"] == pytest.approx(14 / 5, abs=1e-15)
    pair = Particles(2, {"px": [-0.5, 0.5], "py": [0, 0], "pz": [0, 0], "m": [1.0, 1.0]})
    with nbx.Engine(2) as e:
        e.upload_view(pair.view)
        assert e.diagnostics(eps=0.0)["potential_energy"] == pytest.approx(-1.0, abs=1e-15)


@pytest.mark.parametrize("n,capacity", [(1, 1), (255, 300), (257, 257), (32768, 32768),
                                        (32769, 40000)])
def test_transfers_bring_every_array(nbx, n, capacity):
    """Ten arrays up to 32768 particles go through the pinned block, more by
    copy commands; arrays that a view leaves out keep their values."""
    rng = np.random.default_rng(n)
    names = ("px", "py", "pz", "vx", "vy", "vz", "ax", "ay", "az", "m")
    a = {k: rng.normal(size=n) for k in names}
    b = {k: np.full(n, np.nan) for k in names}
    with nbx.Engine(capacity) as e:
        e.upload_view(nbx.make_view(n, **a))
        e.download_view(nbx.make_view(n, **b))
        for k in names:
            assert np.array_equal(a[k], b[k]), k
        c = {k: rng.normal(size=n) for k in ("px", "py", "pz", "m")}
        e.upload_view(nbx.make_view(n, **c))
        part = {k: np.full(n, np.nan) for k in ("vx", "az", "m")}
        e.download_view(nbx.make_view(n, **part))
        assert np.array_equal(part["vx"], a["vx"]) and np.array_equal(part["az"], a["az"])
        assert np.array_equal(part["m"], c["m"])


@pytest.mark.parametrize("n,pinned", [(1, 10), (257, 10), (32768, 7), (40001, 10), (40001, 3)])
def test_transfers_of_pinned_arrays(nbx, n, pinned):
    """Arrays in pinned memory are reached by the kernel itself, all or none:
    with a pageable one among them the other routes serve."""
    names = ("px", "py", "pz", "vx", "vy", "vz", "ax", "ay", "az", "m")
    rng = np.random.default_rng(n)
    lib = nbx.load()   # (symbols of the HIP runtime it is linked to, too)
    lib.hipHostMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t, C.c_uint]
    lib.hipHostFree.argtypes = [C.c_void_p]

    def arrays():
        block = C.c_void_p()
        assert lib.hipHostMalloc(C.byref(block), pinned * (n + 1) * 8, 0) == 0
        rows = np.ctypeslib.as_array(C.cast(block, C.POINTER(C.c_double)), (pinned, n + 1))
        rows[:] = np.nan
        columns = [r[1:] for r in rows] + [np.full(n, np.nan) for _ in range(10 - pinned)]
        return block, rows, dict(zip(names, columns))

    block_a, _, a = arrays()
    block_b, rows_b, b = arrays()
    for k in names:
        a[k][:] = rng.normal(size=n)
    with nbx.Engine(n) as e:
        e.upload_view(nbx.make_view(n, **a))
        e.download_view(nbx.make_view(n, **b))
    for k in names:
        assert np.array_equal(a[k], b[k]), k
    assert np.all(np.isnan(rows_b[:, 0]))   # nothing before the arrays was touched
    assert lib.hipHostFree(block_a) == 0 and lib.hipHostFree(block_b) == 0


@pytest.mark.parametrize("n,shift", [(1, 0), (257, 0), (257, 100), (40001, 0), (40001, 7)])
def test_download_into_pinned_arrays_that_share_memory(nbx, n, shift):
    """The view's later array stays, as with one copy after the other: vx, vy
    and vz go `shift` elements apart into one pinned block, x to another."""
    rng = np.random.default_rng(n)
    src = {k: rng.normal(size=n) for k in ("px", "py", "pz", "vx", "vy", "vz", "m")}
    lib = nbx.load()
    lib.hipHostMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t, C.c_uint]
    lib.hipHostFree.argtypes = [C.c_void_p]
    block = C.c_void_p()
    words = 2 * n + 2 * shift
    assert lib.hipHostMalloc(C.byref(block), words * 8, 0) == 0
    host = np.ctypeslib.as_array(C.cast(block, C.POINTER(C.c_double)), (words,))
    host[:] = np.nan
    want = np.full(n + 2 * shift, np.nan)
    for k, name in enumerate(("vx", "vy", "vz")):
        want[k * shift:k * shift + n] = src[name]
    at = {name: host[n + k * shift:2 * n + k * shift] for k, name in enumerate(("vx", "vy", "vz"))}
    with nbx.Engine(n) as e:
        e.upload_view(nbx.make_view(n, **src))
        e.download_view(nbx.make_view(n, px=host[:n], **at))
    assert np.array_equal(host[:n], src["px"]) and np.array_equal(host[n:], want)
    assert lib.hipHostFree(block) == 0


def test_all_pairs_advance_times_its_last_evaluation(nbx):
    p = Particles(500, {k: np.random.default_rng(7).normal(size=500) for k in ("px", "py", "pz", "m")})
    for alg, per in (("hip_direct_fp64", 56.0), ("hip_direct_fp32", 40.0)):
        with nbx.Engine(500) as e:
            e.upload_view(p.view)
            e.compute_force(alg, eps=0.05)
            e.advance(alg, dt=1e-3, steps=4, eps=0.05)
            t = e.timings()
        assert t["kernel_ms"] > 0.0 and t["integrate_ms"] > t["kernel_ms"]
        assert t["kernel_bytes"] == per * 500 and t["kernel_flops"] == 20.0 * 500 * 499


@pytest.mark.parametrize("n,eps,scale", [
    (1, 0.01, 1.0), (2, 0.01, 1.0), (16, 0.0, 1.0), (17, 0.01, 1.0), (64, 0.01, 1.0),
    (65, 0.0, 1.0), (129, 0.01, 1.0), (1000, 0.01, 1.0),
    (4099, 0.01, 1.0),     # more units than waves
    (70, 0.0, 1e-158),     # squared distances below the normal range
    (70, 0.0, 1e160),      # and past the largest number
])
def test_potential_units(nbx, n, eps, scale):
    """Edges of the potential's 64-target by 16-source units. All terms have one
    sign; each is right to 3 roundings and passes at most 16 + 24 + 8 + 8
    additions: 60 x 1.1e-16."""
    rng = np.random.default_rng(n)
    q = rng.normal(0, 1, (3, n)) * scale
    m = rng.uniform(0.5, 1.5, n)
    with np.errstate(over="ignore"):
        u = np.longdouble(0)
        for i in range(n - 1):
            d = q[:, i + 1:] - q[:, i:i + 1]
            r2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2] + eps * eps
            u += np.sum((m[i] * m[i + 1:] / np.sqrt(r2)).astype(np.longdouble))
    p = Particles(n, {"px": q[0], "py": q[1], "pz": q[2], "m": m})
    with nbx.Engine(n) as e:
        e.upload_view(p.view)
        got = e.diagnostics(eps=eps)["potential_energy"]
    assert abs(got + float(u)) <= 7e-15 * abs(float(u))


def test_potential_of_coincident_pair(nbx):
    p = Particles(40, {"px": [*range(39), 7], "py": [0] * 40, "pz": [0] * 40, "m": [1.0] * 40})
    with nbx.Engine(40) as e:
        e.upload_view(p.view)
        assert e.diagnostics(eps=0.0)["potential_energy"] == -np.inf


@pytest.mark.parametrize("integrator", [1, 2])
def test_two_body_orbit_regression(nbx, integrator):
    """two_body_test.c:57-184: 8 orbits x 500 steps, eps=0."""
    s = math.sqrt(2.0) / 2.0
    p = Particles(2, {"px": [-0.5, 0.5], "py": [0, 0], "pz": [0, 0], "vx": [0, 0],
                      "vy": [s, -s], "vz": [0, 0], "m": [1.0, 1.0]})
    period = 2.0 * math.pi / math.sqrt(2.0)
    dt = period / 500
    with nbx.Engine(2) as e:
        e.upload_view(p.view)
        e.compute_force("hip_direct_fp64", eps=0.0)
        d0 = e.diagnostics(eps=0.0)
        e.advance("hip_direct_fp64", dt=dt, steps=8 * 500, eps=0.0, integrator=integrator)
        d1 = e.diagnostics(eps=0.0)
        out = e.download()
    e0 = d0["kinetic_energy"] + d0["potential_energy"]
    e1 = d1["kinetic_energy"] + d1["potential_energy"]
    assert abs((e1 - e0) / e0) < 1e-3
    sep = np.linalg.norm(out["pos"][1] - out["pos"][0])
    assert abs(sep - 1.0) < 1e-2
    assert abs(d1["total_momentum_x"]) < 1e-12 and abs(d1["total_momentum_y"]) < 1e-12
    assert abs(d1["center_of_mass_x"]) < 1e-12 and abs(d1["center_of_mass_y"]) < 1e-12


def test_invalid_timestep_rejected(nbx):
    p = Particles(2, {"px": [-0.5, 0.5], "py": [0, 0], "pz": [0, 0], "m": [1.0, 1.0]})
    with nbx.Engine(2) as e:
        e.upload_view(p.view)
        with pytest.raises(nbx.NBXError) as ex:
            e.advance("hip_direct_fp64", dt=0.0, steps=1)
        assert ex.value.status == 1


def test_barnes_hut_kdk_conserves_momentum(nbx):
    d = nbx.two_galaxy(100_000, seed=1)
    p = Particles(len(d["m"]), {"px": d["pos"][:, 0], "py": d["pos"][:, 1], "pz": d["pos"][:, 2],
                                "vx": d["vel"][:, 0], "vy": d["vel"][:, 1], "vz": d["vel"][:, 2],
                                "m": d["m"]})
    with nbx.Engine(p.n) as e:
        e.upload_view(p.view)
        e.compute_force("hip_barnes_hut", eps=0.01)
        q0 = e.diagnostics(potential=False)
        e.advance("hip_barnes_hut", dt=1e-3, steps=3, eps=0.01)
        q1 = e.diagnostics(potential=False)
    for c in "xyz":
        assert abs(q1[f"total_momentum_{c}"] - q0[f"total_momentum_{c}"]) < 1e-5
