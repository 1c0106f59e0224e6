"""GPU: point counts around the edges of the point sort and the plane sums.

Up to 2,048 points one workgroup sorts them (64, 256 or 1,024 threads), more
go through two radix passes of 1,024-point blocks; a plane of more than 65,536
points is summed in parts.
"""
import numpy as np
import pytest

from conftest import rel_err
from oracle import oracle, sph

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ring():
    from gimic_amd import synth
    s = synth.ring12()
    ctx = s.context(screening=1e-8)
    yield s, ctx
    ctx.close()


def _points(n, seed=1):
    return np.random.default_rng(seed).uniform(-6.0, 6.0, (n, 3))


@pytest.mark.parametrize("n", [1, 2, 3, 63, 64, 65, 128, 129, 512, 513, 2047, 2048, 2049, 3072, 5000])
def test_point_counts_around_the_sort(ring, n):
    s, ctx = ring
    pts = _points(n)
    pts[n // 2] = pts[0]  # a repeated point
    print("case sort of", n, flush=True)
    J = ctx.jtensor(pts, precision="fp64")
    sub = np.unique(np.r_[0, n // 2, n - 1, np.random.default_rng(n).integers(0, n, 20)])
    ref = oracle.jtensor(s.arrays(), sph.to_cartesian(s.dens, s.shell_l), pts[sub], screening=1e-8)
    # the scale of the error floor is that of the whole set
    scale = max(np.linalg.norm(J, axis=1).max(), 1e-300)
    e = np.linalg.norm(J[sub] - ref, axis=1) / np.maximum(np.linalg.norm(ref, axis=1), 1e-3 * scale)
    assert e.max() <= 1e-10, e.max()
    assert np.array_equal(ctx.jtensor(pts, precision="fp64"), J)


def test_points_in_one_cell_and_not_a_number(ring):
    """all points in one Morton cell (equal keys keep their order), and a point
    that is not a number (it gets a cell, and only its own tensor)"""
    s, ctx = ring
    for n in (100, 3000):
        pts = np.tile([1.0, 0.5, 0.3], (n, 1))
        J = ctx.jtensor(pts, precision="fp64")
        assert np.array_equal(J, np.tile(J[0], (n, 1)))
        pts = _points(n, 3)
        J = ctx.jtensor(pts, precision="fp64")
        bad = pts.copy()
        bad[n // 3, 1] = np.nan
        K = ctx.jtensor(bad, precision="fp64")
        keep = np.arange(n) != n // 3
        assert rel_err(K[keep], J[keep]).max() <= 1e-12


@pytest.mark.parametrize("sizes", [[65535], [65536], [200000], [150000, 3, 0, 90000]])
def test_plane_sums_in_parts(ring, sizes):
    s, ctx = ring
    rng = np.random.default_rng(len(sizes))
    planes = []
    for n in sizes:
        planes.append(dict(points=rng.uniform(-5.0, 5.0, (n, 3)), weights=rng.uniform(0.0, 1.0, n),
                           normal=[0.6, 0.0, 0.8], bfield=[0.0, 0.0, 1.0], center=[0.0, 0.0, 0.0]))
    print("case plane sums", sizes, flush=True)
    flux, mod, acid, jt = ctx.flux_planes(planes, return_jt=True, modulus=True, acid=True)
    at = 0
    for k, p in enumerate(planes):
        n = sizes[k]
        T = jt[at:at + n].reshape(-1, 3, 3).transpose(0, 2, 1)
        at += n
        jv = T @ np.asarray(p["bfield"])
        v = p["weights"] * (jv @ np.asarray(p["normal"]))
        m = p["weights"] * np.sign(jv @ np.asarray(p["normal"])) * np.linalg.norm(jv, axis=1)
        for got, w in ((flux[k], v), (mod[k], m)):
            ref = np.array([w.sum(), w[w > 0].sum(), w[w <= 0].sum()])
            # rounding of sums of n terms in another order
            assert np.abs(got - ref).max() <= 1e-15 * max(n, 1) ** 0.5 * 100 * np.abs(w).sum() + 1e-300
        assert (acid[k] > 0.0) == (n > 0)
    plain = ctx.flux_planes(planes)
    assert np.array_equal(plain, flux)
    assert np.array_equal(ctx.flux_planes(planes, acid=True)[1], acid)


@pytest.fixture(scope="module")
def cage():
    from gimic_amd import synth
    s = synth.cage60()
    ctx = s.context(screening=1e-8)
    yield s, ctx
    ctx.close()


@pytest.mark.parametrize("n", [1, 5, 64, 65, 257, 4000])
def test_small_launches_split_over_k_and_all_xcds(cage, n):
    """few row tiles of a large basis: N- and K-ranges on every XCD, their sums
    added by a launch of their own"""
    s, ctx = cage
    # spread over the whole cage, so the tiles list most functions
    pts = np.random.default_rng(n).uniform(-8.0, 8.0, (n, 3))
    print("case cage60 small launch", n, flush=True)
    J = ctx.jtensor(pts, precision="fp64")
    sub = np.random.default_rng(2).integers(0, n, min(n, 16))
    ref = oracle.jtensor(s.arrays(), sph.to_cartesian(s.dens, s.shell_l), pts[sub], screening=1e-8)
    scale = np.linalg.norm(J, axis=1).max()
    e = np.linalg.norm(J[sub] - ref, axis=1) / np.maximum(np.linalg.norm(ref, axis=1), 1e-3 * scale)
    assert e.max() <= 1e-10, e.max()
    assert np.array_equal(ctx.jtensor(pts, precision="fp64"), J)
    M = ctx.jtensor(pts, precision="mixed")
    assert rel_err(M, J).max() <= 1e-5
    assert np.array_equal(ctx.jtensor(pts, precision="mixed"), M)
    # the same points in a full launch: other tiles, fewer ranges
    far = np.random.default_rng(9).uniform(-8.0, 8.0, (60000, 3))
    K = ctx.jtensor(np.concatenate([pts, far]), precision="fp64")[:n]
    assert rel_err(K, J).max() <= 1e-12


@pytest.mark.parametrize("variant,split", [(3, 4), (4, 1), (5, 4), (8, 2), (9, 1), (9, 8)])
@pytest.mark.parametrize("n", [1, 127, 129, 256, 257, 1000, 40000])
def test_mixed_tiles_with_fewer_n_tiles_than_ranges(ring, n, variant, split):
    """near and far points in one set: the row tiles list from none to all of
    the ring's functions, so N-ranges stay empty in some; the mixed path's 1e-5,
    of the largest tensor (the far ones vanish)"""
    s, _ = ring
    pts = _points(n)
    pts[::2] *= 1.0 + 12.0 * np.arange(len(pts[::2]))[:, None] / n
    print("case ring12 mixed", variant, split, n, flush=True)
    with s.context(screening=1e-8) as ctx:
        J = ctx.jtensor(pts, precision="fp64")
        ctx.set_mixed_kernel(variant, split)
        M = ctx.jtensor(pts, precision="mixed")
    assert np.abs(M - J).max() <= 1e-5 * np.abs(J).max()


@pytest.mark.parametrize("natoms", [1, 33, 65, 129, 513])
def test_fp64_lists_by_atoms(natoms):
    """FP64 lists test a tile's points with 8, 4, 2 or 1 lanes an atom, and go by
    the box alone beyond 512 atoms; a chain of hydrogen atoms, points all along it"""
    from gimic_amd import synth
    xyz = np.c_[1.7 * np.arange(natoms), np.zeros((natoms, 2))]
    s, rng = synth.build_system("chain", ["H"] * natoms, xyz, {"H": "2s1p"}, natoms)
    s.dens = synth.density_family(rng, s.nbf, max(1, s.nbf // 4))[None]
    pts = np.random.default_rng(natoms).uniform(-4.0, 4.0, (700, 3))
    pts[:, 0] = np.random.default_rng(1).uniform(-4.0, 1.7 * natoms + 4.0, 700)
    print("case chain of", natoms, flush=True)
    with s.context(screening=1e-8) as ctx:
        J = ctx.jtensor(pts, precision="fp64")
    sub = np.arange(0, 700, 35)
    ref = oracle.jtensor(s.arrays(), sph.to_cartesian(s.dens, s.shell_l), pts[sub], screening=1e-8)
    scale = np.linalg.norm(J, axis=1).max()
    e = np.linalg.norm(J[sub] - ref, axis=1) / np.maximum(np.linalg.norm(ref, axis=1), 1e-3 * scale)
    assert e.max() <= 1e-10, e.max()


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-12), ("mixed", 1e-5)])
def test_many_points_not_a_number(precision, tol):
    """no shell is screened out at such a point, those that only share a group
    with a shell in reach of its tile included: these have no columns in the
    tile's compressed rows and must not be written.  A chain of 20 hydrogen
    atoms, so that every tile lists a part of the functions only"""
    from gimic_amd import synth
    xyz = np.c_[1.7 * np.arange(20), np.zeros((20, 2))]
    s, rng = synth.build_system("chain", ["H"] * 20, xyz, {"H": "2s1p"}, 20)
    s.dens = synth.density_family(rng, s.nbf, s.nbf // 4)[None]
    n = 3000
    pts = rng.uniform(-2.0, 2.0, (n, 3))
    pts[:, 0] = rng.uniform(-2.0, 34.3, n)
    odd = pts.copy()
    odd[::7, 1] = np.nan
    keep = ~np.isnan(odd[:, 1])
    with s.context(screening=1e-8) as ctx:
        J = ctx.jtensor(pts, precision="fp64")
        print("case chain of 20, every seventh point nan", precision, flush=True)
        K = ctx.jtensor(odd, precision=precision)
    assert rel_err(K[keep], J[keep]).max() <= tol
    assert np.isnan(K[~keep]).all()


@pytest.mark.parametrize("bad", [np.nan, np.inf, -np.inf, 1e200], ids=str)
@pytest.mark.parametrize("n", [100, 3000, 20000])
@pytest.mark.parametrize("precision,tol", [("fp64", 1e-12), ("mixed", 1e-5)])
def test_point_that_is_not_finite_beside_others(sheet, n, precision, tol, bad):
    """a basis of 64 shells or more, whose basis kernel lists the shells that
    reach its rows: a coordinate that is not a number, infinite or too large to
    square costs only its own tensor (1, 4 or 32 rows a workgroup)"""
    s, ctx = sheet
    rng = np.random.default_rng(n)
    R = np.asarray(s.coords)
    pts = R[rng.integers(0, len(R), n)] + rng.uniform(-2.0, 2.0, (n, 3))
    J = ctx.jtensor(pts, precision="fp64")
    odd = pts.copy()
    for k in range(3):
        odd[(2 * k + 1) * n // 7, k] = bad
    keep = np.isfinite(odd).all(axis=1) & (np.abs(odd) < 1e100).all(axis=1)
    assert keep.sum() == n - 3
    print("case sheet30", n, "points, three", bad, precision, flush=True)
    K = ctx.jtensor(odd, precision=precision)
    assert rel_err(K[keep], J[keep]).max() <= tol
    if np.isnan(bad):
        assert np.isnan(K[~keep]).all()


@pytest.fixture(scope="module")
def sheet():
    from gimic_amd import synth
    s = synth.sheet30()
    ctx = s.context(screening=1e-8)
    yield s, ctx
    ctx.close()


def test_fp64_rows_too_wide_to_compress():
    """4,825 functions: FP64 rows wider than the basis kernel's LDS image stay
    dense (4,832 columns, 7 of them padding that must read as zero).  Two chunks
    of 256 and 44 points, then fewer points in the same buffers (other plane
    strides), and the allocation-free call, whose scratch held other data"""
    import torch
    from gimic_amd import synth
    at = np.arange(965)
    xyz = 3.0 * np.c_[at % 10, at // 10 % 10, at // 100] - 13.5
    s, rng = synth.build_system("block", ["H"] * 965, xyz, {"H": "2s1p"}, 7)
    s.dens = rng.standard_normal((1, 4, s.nbf, s.nbf))
    pts = rng.uniform(-15.0, 15.0, (300, 3))
    sub = np.r_[0:300:43, 299]
    ref = oracle.jtensor(s.arrays(), sph.to_cartesian(s.dens, s.shell_l), pts[sub], screening=1e-8)
    with s.context(screening=1e-8) as ctx:
        assert ctx.nbf == 4825
        ctx.set_chunk_bytes(256 * 4832 * 32)
        print("case block of 4825 functions, 300 points in two chunks", flush=True)
        J = ctx.jtensor(pts, precision="fp64")
        assert rel_err(J[sub], ref).max() <= 1e-10
        ctx.set_chunk_bytes(0)
        for n in (70, 300, 129):
            print("case block of 4825 functions", n, flush=True)
            K = ctx.jtensor(pts[:n], precision="fp64")
            assert rel_err(K, J[:n]).max() <= 1e-10
        print("case block of 4825 functions, mixed", flush=True)
        M = ctx.jtensor(pts, precision="mixed")
        assert rel_err(M, J).max() <= 1e-5
        d = torch.tensor(pts, device="cuda")
        ctx.jtensor_device(d[:1])
        for prec, n, tol in (("mixed", 300, 1e-5), ("fp64", 300, 1e-10), ("fp64", 70, 1e-10)):
            print("case block of 4825 functions, allocation-free", prec, n, flush=True)
            ctx.jtensor_device(d[:1], precision=prec)
            K = ctx.jtensor_device_noalloc(d[:n], precision=prec)
            torch.cuda.synchronize()
            assert rel_err(K.cpu().numpy(), J[:n]).max() <= tol


def test_call_after_one_too_large_for_the_device(ring):
    """a host batch of 2^40 points (26 TB of them alone; refused before any copy
    or launch) is an error, and none of the call that follows it"""
    from gimic_amd import lib
    s, ctx = ring
    pts = _points(100)
    J = ctx.jtensor(pts)
    out = np.zeros((1, 9))
    for call in ("points", "planes"):
        print("case 2^40", call, flush=True)
        with pytest.raises(lib.GimicError, match="out of memory"):
            if call == "points":
                lib.check(ctx._lib.gimic_jtensor_batch(ctx._h, 1 << 40, lib.ptr(pts), lib.ptr(out),
                                                       0, 0))
            else:
                offs = np.array([0, 1 << 40], dtype=np.int64)
                lib.check(ctx._lib.gimic_flux_planes(
                    ctx._h, 1, lib.ptr(offs), lib.ptr(pts), lib.ptr(pts), lib.ptr(pts),
                    lib.ptr(pts), lib.ptr(pts), lib.ptr(pts), 0, 0, lib.ptr(out), None, None, None))
        assert np.array_equal(ctx.jtensor(pts), J)
