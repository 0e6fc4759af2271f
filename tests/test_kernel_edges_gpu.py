"""Kernel variants at the sizes where their rules change, against the general path or
the oracle:

* P1 Gauss-Seidel (small sweeps in one workgroup, point pairs in registers, interleaved
  vectors in packs) against a sweep colour by colour on the oracle's matrix, and the forms
  of large levels against each other;
* P2 constant Gauss-Seidel (assembled rows) against a sweep colour by colour with the
  apply kernel;
* the P2 coarse conjugate gradients on element matrices (levels 0 to 2) and the
  launch-by-launch iteration above, against the same iteration in numpy, over more
  iterations than one launch runs;
* the halo exchange of a mesh with a face of three cells;
* P2 restriction into levels whose face points fill several wavefronts, of interleaved
  vectors, and from a lattice too wide for the point lists;
* the Stokes blocks over an odd number of interior tiles, and by each of the apply's forms.
"""
import ctypes as C

import numpy as np
import pytest

import hyteg_amd as hg
from hyteg_amd import problems
from hyteg_amd._lib import lib
from meshes import octahedron, relmax, three_on_a_face
from oracle import pyoracle as po
from test_stokes_gpu import _apply_parity

pytestmark = pytest.mark.gpu

NUMPY = {hg.F64: np.float64, hg.F32: np.float32, hg.F16: np.float16}
EPS = {hg.F64: 2.0**-53, hg.F32: 2.0**-24, hg.F16: 2.0**-11}


def _storage(ctx, name):
    return hg.PrimitiveStorage.cuboid(ctx) if name == "cube" else hg.PrimitiveStorage.from_cells(ctx, *octahedron())


def _colour_sweep(A, colour, free, x, b, relax, backward, dtype):
    """a multicolour sweep of all vectors in FP64 with the results of each colour rounded
    to the storage type"""
    d = A.diagonal()[:, None]
    for c in sorted(set(colour[free]), reverse=backward):
        r = free & (colour == c)
        new = (1.0 - relax) * x[r] + relax / d[r] * (b[r] - A[r] @ x + d[r] * x[r])
        x[r] = new.astype(NUMPY[dtype])
    return x


@pytest.mark.parametrize("dtype", [hg.F64, hg.F32, hg.F16])
@pytest.mark.parametrize("name", ["cube", "octa"])
def test_p1_sweeps_equal_the_sweep_by_colours(ctx, name, dtype):
    """levels on both sides of the one-workgroup sweep's limit (cube 4 and octahedron 4 for
    one vector, 3 for several), by vectors: one to four in a workgroup and several workgroups"""
    st = _storage(ctx, name)
    om = po.Mesh.cuboid() if name == "cube" else po.Mesh.from_arrays(*octahedron())
    for L in range(1, 6):
        A, csr = hg.P1ConstantLaplaceOperator(st, L, L), po.P1Op(om, L).csr()
        colour, _ = A.sor_colours(L)
        n = st.ndofs(L)
        for nvec in (1, 2, 4, 8):
            rng = np.random.default_rng(10 * L + nvec)
            x0, b = (rng.uniform(-1, 1, (n, nvec)).astype(np.float16).astype(np.float64) for _ in range(2))
            x, fb = (hg.P1Function("f", st, L, L, dtype, nvec=nvec) for _ in range(2))
            fb.upload(L, b.reshape(n) if nvec == 1 else b)
            for flag, relax, backward in ((hg.GMG_FLAG, 1.0, False), (hg.ALL, 1.3, True)):
                print(f"P1 sweep by colours {name} L{L} nvec {nvec} dtype {dtype} backward {backward}", flush=True)
                x.upload(L, x0.reshape(n) if nvec == 1 else x0)
                (A.smooth_sor_backwards if backward else A.smooth_sor)(x, fb, relax, L, flag)
                ref = _colour_sweep(csr, colour, (om.flags(L) & flag) != 0, x0.copy(), b, relax, backward, dtype)
                # rows of at most 30 entries, summed in FP64 or FP32 in another order, whose
                # errors later colours take in with row sums below 2; FP16: roundings that the
                # FP32 sum's error turns, at most one a colour and value
                tol = 64 * EPS[dtype] if dtype != hg.F16 else 8 * EPS[dtype]
                assert relmax(x.download(L).reshape(n, nvec), ref) <= tol, (L, nvec, backward)
            x.destroy()
            fb.destroy()


@pytest.mark.parametrize("dtype", [hg.F64, hg.F32, hg.F16])
@pytest.mark.parametrize("name,levels", [("cube", range(5, 9)), ("octa", range(5, 7))])
def test_p1_sweep_by_pairs_equals_the_interleaved_sweep(ctx, name, levels, dtype):
    """point pairs in registers (one vector) against the sweep of two interleaved vectors,
    with rows shorter and longer than a wavefront's pairs (levels above the one-workgroup
    sweep's)"""
    st = _storage(ctx, name)
    for L in levels:
        A = hg.P1ConstantLaplaceOperator(st, L, L)
        n = st.ndofs(L)
        rng = np.random.default_rng(L)
        x0, b = rng.uniform(-1, 1, (n, 2)), rng.uniform(-1, 1, (n, 2))
        xb, bb = (hg.P1Function("f", st, L, L, dtype, nvec=2) for _ in range(2))
        xs, bs = (hg.P1Function("g", st, L, L, dtype) for _ in range(2))
        bb.upload(L, b)
        for flag, relax, sweep in ((hg.GMG_FLAG, 1.0, "smooth_sor"), (hg.ALL, 1.3, "smooth_sor_backwards")):
            print(f"P1 {sweep} {name} L{L} dtype {dtype}", flush=True)
            xb.upload(L, x0)
            getattr(A, sweep)(xb, bb, relax, L, flag)
            ref = xb.download(L)
            for k in range(2):
                xs.upload(L, x0[:, k])
                bs.upload(L, b[:, k])
                getattr(A, sweep)(xs, bs, relax, L, flag)
                # rows of at most 30 entries (a boundary row adds one partial sum a cell)
                # in another order; errors of earlier colours enter with row sums below 2
                assert relmax(xs.download(L), ref[:, k]) <= 64 * EPS[dtype], (L, sweep, k)
        for f in (xb, bb, xs, bs):
            f.destroy()


@pytest.mark.parametrize("dtype", [hg.F64, hg.F32, hg.F16])
@pytest.mark.parametrize("nvec", [2, 4, 8, 64])
def test_p1_interleaved_sweep_by_vectors_a_lane(ctx, nvec, dtype):
    """every width of the interleaved sweep's packs (1, 2 or 4 vectors a lane, by the number
    of lanes) on levels above the one-workgroup sweep's limit for several vectors: each
    vector as alone (in one workgroup at level 4, in point pairs at level 5)"""
    st = hg.PrimitiveStorage.cuboid(ctx)
    for L in (4, 5):
        A = hg.P1ConstantLaplaceOperator(st, L, L)
        n = st.ndofs(L)
        rng = np.random.default_rng(nvec + L)
        x0, b = rng.uniform(-1, 1, (n, nvec)), rng.uniform(-1, 1, (n, nvec))
        xb, bb = (hg.P1Function("f", st, L, L, dtype, nvec=nvec) for _ in range(2))
        xs, bs = (hg.P1Function("g", st, L, L, dtype) for _ in range(2))
        xb.upload(L, x0)
        bb.upload(L, b)
        print(f"P1 interleaved sweep L{L} nvec {nvec} dtype {dtype}", flush=True)
        A.smooth_sor(xb, bb, 1.1, L, hg.GMG_FLAG)
        got = xb.download(L)
        for k in {0, 1, nvec // 2, nvec - 1}:
            xs.upload(L, x0[:, k])
            bs.upload(L, b[:, k])
            A.smooth_sor(xs, bs, 1.1, L, hg.GMG_FLAG)
            assert relmax(got[:, k], xs.download(L)) <= 64 * EPS[dtype], (L, k)
        for f in (xb, bb, xs, bs):
            f.destroy()


@pytest.mark.parametrize("name,L", [("cube", 4), ("cube", 5), ("cube", 6), ("octa", 4)])
def test_p2_constant_sweep_equals_the_sweep_by_colours(ctx, name, L):
    st = _storage(ctx, name)
    A = hg.P2ConstantLaplaceOperator(st, L, L)
    colour, _ = A.sor_colours(L)
    free = (st.flags(L + 1) & hg.GMG_FLAG) != 0
    n = len(colour)
    rng = np.random.default_rng(L)
    x0, b = rng.uniform(-1, 1, n), rng.uniform(-1, 1, n)
    x, fb, y = (hg.P2Function("f", st, L, L) for _ in range(3))
    A.inverse_diagonal(L, y)
    inv = y.download(L)
    fb.upload(L, b)
    for backward in (False, True):
        print(f"P2 constant sweep {name} L{L} backward {backward}", flush=True)
        ref = x0.copy()
        for c in sorted(set(colour[free]), reverse=backward):
            x.upload(L, ref)
            A.apply(x, y, L, hg.ALL)
            rows = free & (colour == c)
            ref[rows] += 1.2 * inv[rows] * (b - y.download(L))[rows]
        x.upload(L, x0)
        (A.smooth_sor_backwards if backward else A.smooth_sor)(x, fb, L, hg.GMG_FLAG, 1.2)
        assert relmax(x.download(L), ref) < 1e-12
    for f in (x, fb, y):
        f.destroy()
    A.destroy()


@pytest.mark.parametrize("jacobi", [True, False])
@pytest.mark.parametrize("name,L", [("cube", 1), ("cube", 2), ("cube", 3), ("shell", 0), ("shell", 1)])
def test_p2_cg_iterates(ctx, name, L, jacobi):
    st = hg.PrimitiveStorage.cuboid(ctx) if name == "cube" else hg.PrimitiveStorage.shell(ctx, 2, 2, 0.55, 1.0)
    A = hg.P2DivKGradOperator(st, L, L, *problems.shell_coefficient(3))
    n = st.p2_ndofs(L)
    free = (st.flags(L + 1) & hg.GMG_FLAG) != 0
    rng = np.random.default_rng(L)
    b, x0 = rng.uniform(-1, 1, n), rng.uniform(-1, 1, n)
    x, fb, y = (hg.P2Function("f", st, L, L) for _ in range(3))
    fb.upload(L, b)

    def mul(v):
        x.upload(L, v)
        A.apply(x, y, L, hg.ALL)
        return np.where(free, y.download(L), 0.0)

    d = np.where(free, 1.0, 0.0)
    if jacobi:
        A.inverse_diagonal(L, y)
        d = np.where(free, y.download(L), 0.0)
    for iterations in (1, 2, 7):
        print(f"P2 CG {name} L{L} jacobi {jacobi}: {iterations} iterations", flush=True)
        ref = x0.copy()
        r = np.where(free, b, 0.0) - mul(ref)
        p = d * r
        rz = r @ p
        for _ in range(iterations):
            ap = mul(p)
            alpha = rz / (p @ ap)
            ref += alpha * p
            r -= alpha * ap
            rz, old = r @ (d * r), rz
            p = d * r + (rz / old) * p
        x.upload(L, x0)
        hg.p2_cg_solve(A, x, fb, L, iterations, 0.0, 0.0, jacobi)
        got = x.download(L)
        assert np.array_equal(got[~free], x0[~free])
        assert relmax(got, ref) < 1e-11, (iterations, relmax(got, ref))
    for f in (x, fb, y):
        f.destroy()
    A.destroy()


def test_p2_cg_runs_on_over_several_launches(ctx):
    """1100 iterations (a launch runs 1024) of a system scaled so that r.z does not
    underflow: the residual stays at its rounding limit"""
    st = hg.PrimitiveStorage.cuboid(ctx)
    L = 2
    A = hg.P2DivKGradOperator(st, L, L, *problems.shell_coefficient(3))
    free = (st.flags(L + 1) & hg.GMG_FLAG) != 0
    b = np.where(free, 1e120 * np.random.default_rng(0).uniform(-1, 1, len(free)), 0.0)
    x, fb, y = (hg.P2Function("f", st, L, L) for _ in range(3))
    fb.upload(L, b)
    x.upload(L, 0.0 * b)
    print("P2 CG over two launches", flush=True)
    assert hg.p2_cg_solve(A, x, fb, L, 1100, 0.0, 0.0) == 1099
    A.apply(x, y, L, hg.ALL)
    r = np.where(free, b - y.download(L), 0.0)
    assert np.abs(r).max() < 1e-11 * np.abs(b).max()
    for f in (x, fb, y):
        f.destroy()
    A.destroy()


@pytest.mark.parametrize("jacobi", [True, False])
def test_p2_cg_stands_still_at_a_zero_residual(ctx, jacobi):
    """iterations after the residual is exactly zero (one free DoF, or b = 0), zero
    tolerances: the ratios 0 / 0 count as 0 and x keeps the solution"""
    st = hg.PrimitiveStorage.cuboid(ctx)
    A = hg.P2DivKGradOperator(st, 0, 0, *problems.shell_coefficient(3))
    free = (st.flags(1) & hg.GMG_FLAG) != 0
    assert free.sum() == 1
    x, fb, y = (hg.P2Function("f", st, 0, 0) for _ in range(3))
    A.inverse_diagonal(0, y)
    inv = y.download(0)[free]
    for b in (0.0, 0.7):
        fb.upload(0, np.where(free, b, 0.0))
        x.upload(0, np.zeros(len(free)))
        print(f"P2 CG from a zero residual, b {b}, jacobi {jacobi}", flush=True)
        assert hg.p2_cg_solve(A, x, fb, 0, 25, 0.0, 0.0, jacobi) == 24
        got = x.download(0)
        assert np.all(got[~free] == 0.0)
        # the diagonal: a sum of at most 24 micro-cells times 11 points, in another order
        assert abs(got[free] - b * inv) <= 512 * EPS[hg.F64] * abs(b * inv)
    for f in (x, fb, y):
        f.destroy()
    A.destroy()


@pytest.mark.parametrize("L", [0, 1, 2])
def test_an_apply_can_be_captured_after_a_cg_solve(ctx, L):
    """a solve builds what the applies of its level need (coefficient table, tile lists):
    a capture, which cannot allocate, finds them"""
    st = hg.PrimitiveStorage.cuboid(ctx)
    A = hg.P2DivKGradOperator(st, L, L, *problems.shell_coefficient(3))
    x, b, y = (hg.P2Function("f", st, L, L) for _ in range(3))
    rng = np.random.default_rng(L)
    b.upload(L, np.where(st.flags(L + 1) == hg.INNER, rng.uniform(-1, 1, st.p2_ndofs(L)), 0.0))
    print(f"P2 apply captured after a CG solve, L{L}", flush=True)
    hg.p2_cg_solve(A, x, b, L, 20)
    graph = C.c_int64()
    ctx.check(lib().hg_graph_begin_capture(ctx.h), "begin capture")
    try:
        A.apply(x, y, L, hg.ALL)
    finally:
        ctx.check(lib().hg_graph_end_capture(ctx.h, C.byref(graph)), "end capture")
    A.apply(x, b, L, hg.ALL)
    ref = b.download(L)
    for _ in range(3):
        y.interpolate(0.0, L)
        ctx.check(lib().hg_graph_launch(ctx.h, graph), "graph launch")
        # sums of the micro-cells around a DoF by atomics, in any order
        assert relmax(y.download(L), ref) <= 64 * EPS[hg.F64]
    ctx.check(lib().hg_graph_destroy(ctx.h, graph), "graph destroy")
    for f in (x, b, y):
        f.destroy()
    A.destroy()


@pytest.mark.parametrize("dtype", [hg.F64, hg.F32, hg.F16])
@pytest.mark.parametrize("name,L", [("cube", 5), ("octa", 4)])
def test_p2_restriction_into_large_levels(ctx, name, L, dtype):
    st = _storage(ctx, name)
    om = po.Mesh.cuboid() if name == "cube" else po.Mesh.from_arrays(*octahedron())
    f = hg.P2Function("f", st, L - 1, L, dtype)
    rng = np.random.default_rng(L)
    c0, fine = rng.uniform(-1, 1, om.ndofs(L)), rng.uniform(-1, 1, om.ndofs(L + 1))
    f.upload(L, fine)
    fine = f.download(L)  # rounded to the storage type
    for flag in (hg.ALL, hg.GMG_FLAG):
        print(f"P2 restriction {name} {L}->{L - 1} dtype {dtype} flag {flag}", flush=True)
        f.upload(L - 1, c0)
        ref = f.download(L - 1)
        hg.restrict(f, L, flag)
        om.p2_restrict(L, fine, ref, flag)
        # a sum of at most 125 a cell products with weights of sum 8, then one rounding
        assert relmax(f.download(L - 1), ref) < (1e-12 if dtype == hg.F64 else 256 * EPS[hg.F32] if dtype == hg.F32
                                                 else 2 * EPS[hg.F16]), flag
    f.destroy()


def test_p2_restriction_from_a_wide_lattice(ctx):
    """level 10 of one cell (2049 points an edge), beyond the lists of cell and face points:
    the restriction of 1 is a constant on each class of boundary points, so that its sums
    over the boundary are polynomials of degree 2 in the edge length, exact in FP16"""
    X, c = octahedron()
    used = np.unique(c[:1])
    lut = np.zeros(len(X), dtype=c.dtype)
    lut[used] = np.arange(len(used))
    st = hg.PrimitiveStorage.from_cells(ctx, np.ascontiguousarray(X[used]), np.ascontiguousarray(lut[c[:1]]))
    sums = {}
    for L in (3, 4, 5, 6, 10):
        f, one = hg.P2Function("f", st, L - 1, L, hg.F16), hg.P2Function("g", st, L - 1, L - 1, hg.F16)
        print(f"P2 restriction of 1 on one cell {L}->{L - 1}", flush=True)
        f.interpolate(1.0, L)
        f.interpolate(0.0, L - 1)
        one.interpolate(1.0, L - 1)
        hg.restrict(f, L, hg.ALL)
        sums[L] = np.array([f.dot(one, L - 1, hg.DIRICHLET), f.dot(f, L - 1, hg.DIRICHLET)])
        f.destroy()
        one.destroy()
    edge = np.array([2.0**L for L in sums])
    V = np.vander(edge[:3], 3)
    for j in range(2):
        coef = np.linalg.solve(V, np.array([sums[L][j] for L in (3, 4, 5)]))
        for L in (6, 10):
            want = np.polyval(coef, 2.0**L)
            assert abs(sums[L][j] - want) <= 1e-12 * want, (L, j)


@pytest.mark.parametrize("dtype", [hg.F64, hg.F32, hg.F16])
@pytest.mark.parametrize("nvec", [2, 8, 64])
@pytest.mark.parametrize("name,levels", [("octa", (1, 2, 3, 4)), ("shell", (1, 2))])
def test_p2_restriction_of_interleaved_vectors(ctx, name, levels, nvec, dtype):
    """each vector as alone, whether its face points fill a wavefront or share it with
    other vectors"""
    st = _storage(ctx, name) if name == "octa" else hg.PrimitiveStorage.shell(ctx, 2, 2, 0.55, 1.0)
    for L in levels:
        f, g = hg.P2Function("f", st, L - 1, L, dtype, nvec=nvec), hg.P2Function("g", st, L - 1, L, dtype)
        rng = np.random.default_rng(nvec + L)
        # values that every type holds exactly
        fine = rng.uniform(-1, 1, (st.p2_ndofs(L), nvec)).astype(np.float16).astype(np.float64)
        print(f"P2 restriction {name} {L}->{L - 1} nvec {nvec} dtype {dtype}", flush=True)
        f.upload(L, fine)
        f.upload(L - 1, np.zeros((st.p2_ndofs(L - 1), nvec)))
        hg.restrict(f, L, hg.ALL)
        got = f.download(L - 1)
        for k in {0, 1, nvec // 2, nvec - 1}:
            g.upload(L, fine[:, k])
            g.upload(L - 1, np.zeros(st.p2_ndofs(L - 1)))
            hg.restrict(g, L, hg.ALL)
            assert np.array_equal(got[:, k], g.download(L - 1)), (L, k)  # the same sums in the same order
        f.destroy()
        g.destroy()


@pytest.mark.parametrize("cells", [1, 3])
@pytest.mark.parametrize("L", [2, 3, 4])
def test_stokes_blocks_over_odd_tile_counts(ctx, cells, L):
    X, c = octahedron()
    c = np.ascontiguousarray(c[:cells])
    used = np.unique(c)
    lut = np.zeros(len(X), dtype=c.dtype)
    lut[used] = np.arange(len(used))
    X, c = np.ascontiguousarray(X[used]), lut[c]
    _apply_parity(hg.PrimitiveStorage.from_cells(ctx, X, c), po.Mesh.from_arrays(X, c), L, (0.3, 0.5))


# (mesh, level): launches of 24 tiles (one result box a tile), 480 (result boxes a wavefront),
# 720 and 1200 (the last layer apart for the viscous masks only), 960 (three tiles in four
# in the last layer) and 1920 of one micro-cell; level 2 has last-layer tiles only
@pytest.mark.parametrize("mesh,L", [("cube", 3), ("cube", 2), ((2, 3), 3), ((3, 2), 3), ((3, 2), 2), ("cube32", 4),
                                    ((2, 2), 4), ((5, 3), 0)])
def test_stokes_masks_agree_over_the_forms(ctx, mesh, L):
    """the blocks one by one, in pairs and all together, whose launches take different
    forms, and the velocity block on FP32 and FP16 functions"""
    st = (hg.PrimitiveStorage.shell(ctx, *mesh, 0.55, 1.0) if isinstance(mesh, tuple) else
          hg.PrimitiveStorage.cuboid(ctx, n=(3, 2, 1) if mesh == "cube32" else (1, 1, 1)))
    # (a viscosity whose results stay in the FP16 range, also at the cube's corner r = 0)
    A = hg.P2P1StokesOperator(st, L, L, 0.3, 0.5)
    src, dst = (hg.P2P1TaylorHoodFunction("f", st, L, L) for _ in range(2))
    for k, f in enumerate([*src.uvw, src.p]):
        f.interpolate_random(7 + k, -1.0, 1.0, L)

    def apply(mask):
        for f in (*dst.uvw, dst.p):
            f.interpolate(0.0, L)
        print(f"Stokes forms {mesh} L{L} mask {mask}", flush=True)
        A.apply(src, dst, L, hg.ALL, hg.REPLACE, mask)
        return dst.download(L)

    u1, u2, p4 = apply(1)[0], apply(2)[0], apply(4)[1]
    scale, pscale = np.abs(u1).max(), np.abs(p4).max()
    # every result: sums over the micro-cells around a DoF (at most some hundred terms) in
    # another order, of terms within a small factor of the largest result
    tol = 1024 * EPS[hg.F64]
    for mask in (3, 5, 6, 7):
        u, p = apply(mask)
        ref = (u1 if mask & 1 else 0.0) + (u2 if mask & 2 else 0.0)
        assert np.abs(u - ref).max() <= tol * (scale if mask & 1 else np.abs(u2).max()), mask
        if mask & 4:
            assert np.abs(p - p4).max() <= tol * pscale, mask
    for dtype in (hg.F32, hg.F16):
        low, out = ([hg.P2Function("f", st, L, L, dtype) for _ in range(3)] for _ in range(2))
        for a, f in zip(src.uvw, low):
            f.copy_from(a, L)
            a.copy_from(f, L)  # rounded to the storage type
        ref = apply(1)[0]
        hs, hd = (np.array([*(f.h for f in fs), 0], dtype=np.int64) for fs in (low, out))
        print(f"Stokes forms {mesh} L{L} dtype {dtype}", flush=True)
        ctx.check(lib().hg_stokes_apply(ctx.h, A.h, hs.ctypes.data_as(C.c_void_p), hd.ctypes.data_as(C.c_void_p), L, hg.ALL,
                                        1, hg.REPLACE), "Stokes apply")
        got = np.concatenate([f.download(L) for f in out])
        # FP32 arithmetic throughout; FP16 results are rounded once a tile that adds to them
        assert np.abs(got - ref).max() <= (1024 * EPS[hg.F32] if dtype == hg.F32 else 32 * EPS[hg.F16]) * np.abs(ref).max()
        for f in (*low, *out):
            f.destroy()
    A.destroy()


@pytest.mark.parametrize("dtype", [hg.F64, hg.F32])
def test_stokes_kernel_time_of_a_first_apply_is_the_kernels(ctx, dtype):
    """the first apply on a storage builds its tile lists ahead of the timed kernels"""
    L, first, later = 4, [], []
    ctx.event_timing(True)
    try:
        for k in range(6):
            st = hg.PrimitiveStorage.cuboid(ctx, n=(3, 2, 1))
            A = hg.P2P1StokesOperator(st, L, L, 0.3, 0.5)
            fs = [hg.P2Function("f", st, L, L, dtype) for _ in range(6)]
            hs, hd = (np.array([*(f.h for f in x), 0], dtype=np.int64) for x in (fs[:3], fs[3:]))
            for f in fs[:3]:
                f.interpolate_random(k, -1.0, 1.0, L)
            for j in range(4):
                print(f"Stokes kernel time, dtype {dtype}, storage {k}, apply {j}", flush=True)
                ctx.check(lib().hg_stokes_apply(ctx.h, A.h, hs.ctypes.data_as(C.c_void_p), hd.ctypes.data_as(C.c_void_p), L,
                                                hg.GMG_FLAG, 1, hg.REPLACE), "Stokes apply")
                ctx.synchronize()
                (later if j else first).append(ctx.last_ms())
            for f in fs:
                f.destroy()
            A.destroy()
    finally:
        ctx.event_timing(False)
    # (the first storage's launch loads the kernel's code)
    assert min(first[1:]) < 2 * np.median(later), (first, np.median(later))


def test_stokes_masks_can_be_captured_after_one_of_them(ctx):
    """720 tiles, where the viscous masks and B^T read different tile lists: a capture,
    which cannot allocate, finds the lists of every mask after an apply of one"""
    L = 4
    for eager, captured in ((1, 2), (2, 7)):
        st = hg.PrimitiveStorage.cuboid(ctx, n=(3, 2, 1))
        A = hg.P2P1StokesOperator(st, L, L, 0.3, 0.5)
        src, dst = (hg.P2P1TaylorHoodFunction("f", st, L, L) for _ in range(2))
        for k, f in enumerate([*src.uvw, src.p]):
            f.interpolate_random(7 + k, -1.0, 1.0, L)
        print(f"Stokes mask {captured} captured after mask {eager}", flush=True)
        A.apply(src, dst, L, hg.ALL, hg.REPLACE, eager)
        graph = C.c_int64()
        ctx.check(lib().hg_graph_begin_capture(ctx.h), "begin capture")
        try:
            A.apply(src, dst, L, hg.ALL, hg.REPLACE, captured)
        finally:
            ctx.check(lib().hg_graph_end_capture(ctx.h, C.byref(graph)), "end capture")
        A.apply(src, dst, L, hg.ALL, hg.REPLACE, captured)
        ref = dst.download(L)[0]
        for _ in range(3):
            dst.interpolate(0.0, L)
            ctx.check(lib().hg_graph_launch(ctx.h, graph), "graph launch")
            assert relmax(dst.download(L)[0], ref) <= 64 * EPS[hg.F64]  # atomics, in any order
        ctx.check(lib().hg_graph_destroy(ctx.h, graph), "graph destroy")
        src.destroy()
        dst.destroy()
        A.destroy()


@pytest.mark.parametrize("L", [1, 2, 3, 4, 5])
def test_a_face_of_three_cells(ctx, L):
    """applies, sweeps and restriction, whose sums over a face's cells take the general kernel"""
    X, c = three_on_a_face()
    st, om = hg.PrimitiveStorage.from_cells(ctx, X, c), po.Mesh.from_arrays(X, c)
    rng = np.random.default_rng(L)
    n, n2, fl = om.ndofs(L), om.ndofs(L + 1), om.flags(L)
    assert n == st.ndofs(L)
    A, op = hg.P1ConstantLaplaceOperator(st, L, L), po.P1Op(om, L)
    colour, _ = A.sor_colours(L)
    csr, x0, b = op.csr(), rng.uniform(-1, 1, n), rng.uniform(-1, 1, n)
    for nvec in (1, 4):
        x, y = (hg.P1Function("f", st, L, L, nvec=nvec) for _ in range(2))

        def put(f, v):
            f.upload(L, v if nvec == 1 else np.repeat(v[:, None], nvec, axis=1))

        def get(f):
            return f.download(L).reshape(n, nvec)

        print(f"three cells on a face: P1 L{L} nvec {nvec}", flush=True)
        put(x, x0)
        A.apply(x, y, L, hg.ALL)
        ref = np.zeros(n)
        op.apply(x0, ref, hg.ALL)
        assert relmax(get(y), ref[:, None]) < 1e-12
        for backward in (False, True):
            put(x, x0)
            put(y, b)
            (A.smooth_sor_backwards if backward else A.smooth_sor)(x, y, 1.2, L, hg.ALL)
            ref = po.sor_multicolour(csr, colour, (fl & hg.ALL) != 0, x0.copy(), b, 1.2, backward)
            assert relmax(get(x), ref[:, None]) < 1e-12, backward
        x.destroy()
        y.destroy()
    k = problems.shell_coefficient(3)
    A2 = hg.P2DivKGradOperator(st, L, L, *k)
    f = hg.P2Function("f", st, L - 1, L)
    g = hg.P2Function("g", st, L, L)
    v = rng.uniform(-1, 1, n2)
    f.upload(L, v)
    print(f"three cells on a face: P2 L{L}", flush=True)
    A2.apply(f, g, L, hg.ALL)
    ref = np.zeros(n2)
    po.P2Op(om, L, po.KCoeff(*k)).apply(v, ref, hg.ALL, False)
    assert relmax(g.download(L), ref) < 1e-12
    ref = np.zeros(n)
    f.upload(L - 1, ref)
    hg.restrict(f, L, hg.ALL)
    om.p2_restrict(L, v, ref, hg.ALL)
    assert relmax(f.download(L - 1), ref) < 1e-12
    f.destroy()
    g.destroy()
    A2.destroy()
