"""The fused step, and the kernels around it, at the sizes where their tables and tiles can go wrong.

Comparisons are value for value unless a test says otherwise: the fused step does the arithmetic of the
eager calls in FP64, in the same order."""
import ctypes

import numpy as np
import pytest

import _oracle
from _oracle import NC, ND
from sequences import OracleBackend

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    import panslbm2_amd as pa

    c = pa.Context(0)
    yield c
    c.close()


def _fields(b, N, d3, rng, adjoint):
    u = lambda lo, hi: rng.uniform(lo, hi, N)
    b.put("rho", u(0.95, 1.05))
    b.put("alpha", u(0.0, 0.5))
    b.put("dif", u(0.02, 0.2))
    for n in ("ux", "uy", "uz", "vx", "vy", "vz", "qx", "qy", "qz"):
        b.put(n, u(-0.05, 0.05))
    b.put("tem", u(0.5, 1.5))
    if adjoint:
        for n in ("ip", "iux", "iuy", "iuz", "imx", "imy", "imz", "item", "iqx", "iqy", "iqz"):
            b.put(n, u(-0.1, 0.1))
    return (lambda n: n if d3 else None)


def _collide(b, p, q, z, adjoint):
    if adjoint:
        b.aad_collide_fc(p, "rho", "ux", "uy", z("uz"), "ip", "iux", "iuy", z("iuz"), "imx", "imy", z("imz"), "alpha",
                         0.05, q, "tem", "item", "iqx", "iqy", z("iqz"), "dif")
    else:
        b.ad_collide_fc(p, "rho", "ux", "uy", z("uz"), "alpha", 0.05, q, "tem", "qx", "qy", z("qz"), "dif")


def _result(b, p, q, z, adjoint):
    out = {"f": b.pops(p), "g": b.pops(q)}
    for n in ("ip", "iux", "imx", "item", "iqx") if adjoint else ("rho", "ux", "uy", z("uz"), "tem", "qx"):
        if n:
            out[n] = b.get(n)
    return out


def _operators(b, p, q, z, N, rng, adjoint, values):
    """Ten calls, so that nodes on two or three faces run up to 30 operators; `values`: "random" draws masks
    and values per node, "uniform" gives every node of the box the same, "patch" makes one node differ."""
    def field(lo, hi):
        if values == "random":
            return rng.uniform(lo, hi, N)
        v = np.full(N, rng.uniform(lo, hi))
        if values == "patch":
            v[N // 3] = rng.uniform(lo, hi)
        return v

    def mask(top=1):
        if values == "random":
            return rng.integers(0, top + 1, N).astype(np.int32)
        m = np.full(N, int(rng.integers(0, top + 1)), np.int32)
        if values == "patch":
            m[N // 2] = top
        return m

    v = ("vx", "vy", z("vz"))
    if adjoint:
        b.bc(p, mask(2), adjoint=True)
        b.ans_iset_u(p, mask(), field(0, 0.1), field(0, 0.1), field(0, 0.1), eps=0.3)
        b.ans_iset_rho(p, mask())
        b.ans_iset_u(p, mask(), field(0, 0.1), field(0, 0.1), field(0, 0.1), eps=0.7)
        b.aad_iset_t(q, mask(), *v)
        b.aad_iset_q(q, mask(), *v, eps=0.2)
        b.aad_iset_q(q, mask(), *v, eps=0.4)
        b.aad_iset_q(q, mask(), *v, eps=0.6)
        b.bc(q, mask(2), adjoint=True)
        if ND[p.kind] == 2:  # no 3D form
            b.aad_iset_rho(p, q, mask(2), "rho", *v, "tem", eps=0.5)
    else:
        b.bc(p, mask(2))
        b.ns_set_u(p, mask(), field(0, 0.1), field(0, 0.1), field(0, 0.1))
        b.ns_set_rho(p, mask(), field(0.9, 1.1), field(0, 0.1), field(0, 0.1))
        b.ns_set_u(p, mask(), field(0, 0.1), field(0, 0.1), field(0, 0.1))
        b.ad_set_t(q, mask(), field(0.5, 1.5), *v)
        b.ad_set_q(q, mask(), field(0, 0.1), *v, "dif")
        b.ad_set_q(q, mask(), field(0, 0.1), *v, 0.07)
        b.ad_set_q(q, mask(), field(0, 0.1), *v, 0.11)
        b.ad_set_t(q, mask(), field(0.5, 1.5), *v)
        b.bc(q, mask(2))


def _run(b, kinds, dims, seed, adjoint, steps, ops):
    rng = np.random.default_rng(seed)
    N = dims[0] * dims[1] * dims[2]
    p, q = (b.lattice(k, *dims) for k in kinds)
    z = _fields(b, N, ND[kinds[0]] == 3, rng, adjoint)
    for h, k in ((p, kinds[0]), (q, kinds[1])):
        b.set_pops(h, rng.uniform(0.02, 0.2, (NC[k], N)))
    state = rng.bit_generator.state
    for _ in range(steps):
        rng.bit_generator.state = state  # the same recording in each step
        for h in (p, q):
            (b.istream if adjoint else b.stream)(h)
        ops(p, q, z, N, rng)
        _collide(b, p, q, z, adjoint)
    return _result(b, p, q, z, adjoint)


def _same(got, want):
    for k, w in want.items():
        np.testing.assert_array_equal(np.asarray(got[k]), np.asarray(w), err_msg=k)


PAIRS = {"q9q9": ("D2Q9", "D2Q9"), "q9q5": ("D2Q9", "D2Q5"), "q15q15": ("D3Q15", "D3Q15"), "q15q7": ("D3Q15", "D3Q7"),
         "q27q7": ("D3Q27", "D3Q7")}
DIMS2 = [(2, 2, 1), (3, 2, 1), (5, 4, 1), (131, 9, 1)]
DIMS3 = [(2, 3, 2), (4, 3, 3), (65, 5, 7)]


@pytest.mark.parametrize("values", ["uniform", "patch", "random"])
@pytest.mark.parametrize("adjoint", [False, True], ids=["fwd", "adj"])
@pytest.mark.parametrize("pair", sorted(PAIRS))
def test_operator_lists_match_oracle(ctx, pair, adjoint, values):
    """Lists longer than the eight operators of a node's header, several values of one kind at a node,
    places of the box with one list and with many, grids of two nodes up to several workgroups."""
    from gpu_backend import FusedGpuBackend

    kinds = tuple(getattr(_oracle, n) for n in PAIRS[pair])
    for dims in DIMS2 if ND[kinds[0]] == 2 else DIMS3:
        print("operator lists", pair, dims, "adjoint" if adjoint else "forward", values, flush=True)

        def run(b):
            return _run(b, kinds, dims, sum(dims), adjoint, 2,
                        lambda p, q, z, N, rng: _operators(b, p, q, z, N, rng, adjoint, values))

        fb = FusedGpuBackend(ctx)
        got = run(fb)
        assert fb.fused_calls == 2
        _same(got, run(OracleBackend()))


@pytest.mark.parametrize("own", [True, False], ids=["reads-saved", "reads-other"])
@pytest.mark.parametrize("which", ["f", "g", "fg"])
@pytest.mark.parametrize("pair", sorted(PAIRS))
def test_smoothing_matches_oracle(ctx, pair, which, own):
    """One or both lattices smoothed.  Where the operators read arrays that the collide writes
    ("reads-saved") the smoothed nodes are done after the pass, otherwise inside it."""
    from gpu_backend import FusedGpuBackend

    kinds = tuple(getattr(_oracle, n) for n in PAIRS[pair])
    for dims in [(3, 3, 1), (5, 4, 1), (70, 3, 1)] if ND[kinds[0]] == 2 else [(3, 3, 3), (4, 3, 5), (19, 5, 35)]:
        print("smoothing", pair, dims, which, "saved" if own else "other", flush=True)

        def run(b):
            def ops(p, q, z, N, rng):
                b.bc(p, np.ones(N, np.int32))
                b.ns_set_u(p, rng.integers(0, 2, N).astype(np.int32), *(rng.uniform(0, 0.1, (3, N))))
                u = ("ux", "uy", z("uz")) if own else ("vx", "vy", z("vz"))
                b.ad_set_t(q, rng.integers(0, 2, N).astype(np.int32), rng.uniform(0.5, 1.5, N), *u)
                for h, name in ((p, "f"), (q, "g")):
                    if name in which:
                        b.smooth(h)

            return _run(b, kinds, dims, 5, False, 2, ops)

        fb = FusedGpuBackend(ctx)
        got = run(fb)
        assert fb.fused_calls == 2
        _same(got, run(OracleBackend()))


def test_grid_beyond_the_cache_matches_eager(ctx):
    """A 3D step of 329 MB of populations, read and written past the caches (non-temporal), odd sides."""
    from gpu_backend import FusedGpuBackend, GpuBackend

    kinds, dims = (_oracle.D3Q15, _oracle.D3Q7), (121, 101, 77)

    def run(b):
        def ops(p, q, z, N, rng):
            b.bc(p, np.ones(N, np.int32))
            b.ad_set_t(q, np.ones(N, np.int32), np.full(N, 1.2), "vx", "vy", "vz")

        return _run(b, kinds, dims, 8, False, 2, ops)

    print("beyond the cache", dims, flush=True)
    _same(run(FusedGpuBackend(ctx)), run(GpuBackend(ctx)))


@pytest.mark.parametrize("dims", [(97, 89, 67), (101, 97, 73), (129, 101, 79)], ids=["plain", "loads", "loads-stores"])
def test_grids_on_each_side_of_the_non_temporal_lines_match_eager(ctx, dims):
    """204 MB of populations (plain accesses), 252 MB (loads non-temporal) and 362 MB (stores too)."""
    from gpu_backend import FusedGpuBackend, GpuBackend

    kinds = (_oracle.D3Q15, _oracle.D3Q7)

    def run(b):
        def ops(p, q, z, N, rng):
            b.bc(p, np.ones(N, np.int32))
            b.ad_set_t(q, np.ones(N, np.int32), np.full(N, 1.2), "vx", "vy", "vz")

        return _run(b, kinds, dims, 8, False, 2, ops)

    print("non-temporal lines", dims, flush=True)
    _same(run(FusedGpuBackend(ctx)), run(GpuBackend(ctx)))


@pytest.mark.parametrize("count", [0, 1, 1023, 1024, 1025, 5000])
def test_gather_sum_is_the_serial_sum(ctx, count):
    """The sum in the order of the list, one addition after the other, over chunks in LDS."""
    import panslbm2_amd as pa

    print("gather sum", count, flush=True)
    rng = np.random.default_rng(count)
    v = rng.standard_normal(7001)
    idx = rng.integers(0, v.size, count).astype(np.int32)
    want = 0.0
    for x in v[idx]:
        want += float(x)
    out = ctypes.c_double(-1.0)
    a = ctx.array(v.shape, data=v)
    pa.check(ctx.lib.lbm_gather_sum(ctx.h, a.ptr, pa.hptr(idx) if count else None, count, ctypes.byref(out)))
    assert out.value == want


@pytest.mark.parametrize("have_prev", [0, 1])
@pytest.mark.parametrize("dims,box,plate", [((2, 2, 2), (2, 2, 2), 0), ((9, 7, 5), (6, 7, 4), 2), ((33, 8, 3), (20, 3, 3), 1)])
def test_duct_coefficients_match_numpy(ctx, dims, box, plate, have_prev):
    """The formulas in numpy's order of operations, value for value."""
    import panslbm2_amd as pa

    print("duct coefficients", dims, box, plate, have_prev, flush=True)
    lx, ly, lz = dims
    N = lx * ly * lz
    n = np.arange(N)
    i, j, k = n % lx, n // lx % ly, n // (lx * ly)
    rng = np.random.default_rng(N)
    s, prev = rng.uniform(0, 1, N), rng.uniform(0, 1, N)
    am, qf, qg, dfl, dso = 1e4, 1e-2, 1e-3, 0.007, 0.11
    dev = {m: ctx.array((N,), data=a) for m, a in (("gamma", s), ("prev", prev))}
    for m in ("dgamma", "alpha", "dads", "diff", "dkds"):
        dev[m] = ctx.array((N,), fill=-7.0)
    d = ctypes.c_double
    pa.check(ctx.lib.lbm_duct_coefficients(
        ctx.h, lx, ly, lz, *box, plate, d(am), d(qf), d(qg), d(dfl), d(dso), dev["gamma"].ptr, dev["prev"].ptr,
        have_prev, *(dev[m].ptr for m in ("dgamma", "alpha", "dads", "diff", "dkds"))))
    s[~((i < box[0]) & (j < box[1]) & (k < box[2]))] = 1.0
    s[k < plate] = 0.0
    want = {"gamma": s, "prev": s, "dgamma": s - prev if have_prev else np.zeros(N),
            "alpha": am / (ly - 1.0) * qf * (1.0 - s) / (s + qf),
            "dads": -am / (ly - 1.0) * qf * (1.0 + qf) / (s + qf) ** 2,
            "diff": dso + (dfl - dso) * s * (1.0 + qg) / (s + qg), "dkds": (dfl - dso) * qg * (1.0 + qg) / (s + qg) ** 2}
    _same({m: dev[m].download() for m in want}, want)


def _route(b):
    """(symbols, most operators at a node, smoothing) of the backend's last fused collide."""
    import panslbm2_amd as pa

    v = [ctypes.c_int(-9) for _ in range(3)]
    pa.check(b.L.lbm_program_fused_route(b._pending, *(ctypes.byref(x) for x in v)))
    return tuple(x.value for x in v)


def test_route_before_a_fused_collide_is_an_error(ctx):
    import panslbm2_amd as pa

    p = pa.Lattice(ctx, pa.D2Q9, 5, 4, 1)
    prog, v = ctypes.c_void_p(), ctypes.c_int()
    pa.check(ctx.lib.lbm_record_begin(ctx.h))
    pa.check(ctx.lib.lbm_stream(p.h))
    pa.check(ctx.lib.lbm_record_end(ctx.h, ctypes.byref(prog)))
    r = [ctypes.byref(v)] * 3
    assert ctx.lib.lbm_program_fused_route(prog, *r) < 0
    assert ctx.lib.lbm_program_fused_route(None, *r) < 0
    ctx.lib.lbm_program_destroy(prog)


@pytest.mark.parametrize("smooth,own", [("", False), ("fg", False), ("fg", True)], ids=["plain", "in-pass", "after-pass"])
@pytest.mark.parametrize("pair", ["q9q5", "q15q7"])
def test_route_of_a_program_in_one_order(ctx, pair, smooth, own):
    """Two calls on every face: a symbol per call and face, and one per smoothed lattice; a corner of the
    grid has both calls on each of its faces.  Smoothed nodes inside the pass, or after it where an
    operator reads what the collide writes."""
    from gpu_backend import FusedGpuBackend

    kinds = tuple(getattr(_oracle, n) for n in PAIRS[pair])
    nd = ND[kinds[0]]
    dims = (9, 7, 1) if nd == 2 else (6, 5, 4)
    print("route", pair, smooth, own, flush=True)

    def run(b):
        def ops(p, q, z, N, rng):
            b.bc(p, np.ones(N, np.int32))
            u = ("ux", "uy", z("uz")) if own else ("vx", "vy", z("vz"))
            b.ad_set_t(q, np.ones(N, np.int32), np.full(N, 1.2), *u)
            for h, name in ((p, "f"), (q, "g")):
                if name in smooth:
                    b.smooth(h)

        return _run(b, kinds, dims, 5, False, 2, ops)

    fb = FusedGpuBackend(ctx)
    got = run(fb)
    assert _route(fb) == (4 * nd + len(smooth), 2 * nd + len(smooth), 0 if not smooth else (2 if own else 1))
    _same(got, run(OracleBackend()))


@pytest.mark.parametrize("calls", [11, 18], ids=["11", "18"])
@pytest.mark.parametrize("pair", ["q9q5", "q15q7"])
def test_route_of_a_program_position_by_position(ctx, pair, calls):
    """Programs around the limit of 64 symbols, one per call, face and type that some node of the face has:
    `calls` bounce-back calls with types drawn per node, both of them in every other call.  Beyond it the operators are taken
    position by position, here with lists of up to 54, most of them past the eight in a list's header."""
    from gpu_backend import FusedGpuBackend

    kinds = tuple(getattr(_oracle, n) for n in PAIRS[pair])
    nd = ND[kinds[0]]
    dims = (131, 9, 1) if nd == 2 else (65, 5, 7)
    print("route", pair, calls, flush=True)

    n = np.arange(dims[0] * dims[1] * dims[2])
    at = (n % dims[0], n // dims[0] % dims[1], n // (dims[0] * dims[1]))
    faces = [at[f // 2] == (f % 2) * (dims[f // 2] - 1) for f in range(2 * nd)]
    symbols = set()

    def run(b):
        def ops(p, q, z, N, rng):
            for c in range(calls):
                t = rng.integers(0, 3, N) if c % 2 else rng.integers(0, 2, N)
                t[:] = np.where(np.arange(N) == 0, 1, t)  # the longest list is the first corner's
                symbols.update((c, f, x) for f, on in enumerate(faces) for x in set(t[on]) if x)
                b.bc(q if c % 3 else p, t.astype(np.int32))

        return _run(b, kinds, dims, 5, False, 2, ops)

    fb = FusedGpuBackend(ctx)
    got = run(fb)
    assert (len(symbols) > 64) == ((calls, nd) != (11, 2))
    assert _route(fb) == (len(symbols) if len(symbols) <= 64 else 0, calls * nd, 0)
    _same(got, run(OracleBackend()))


@pytest.mark.parametrize("dims", [(200, 400, 1), (65, 49, 33)], ids=["2d", "3d"])
def test_mixed_operator_lists_cost_little_more_than_uniform_ones(ctx, dims):
    """A step waits for the wavefront with the most operators.  With masks drawn per node a wavefront of
    64 wall nodes has up to 64 different lists, of six calls (24 or 36 symbols) together; with the same
    two calls everywhere it has 2 or 3 of 4 to 6 symbols.  A wavefront runs each symbol once, so the
    ratio of the step times is below that of the symbols, 24 / 4 = 6, and of the operators' share in a
    step, of which about half is not operators: 3."""
    import time

    import panslbm2_amd as pa
    from panslbm2_amd import D, check, hptr

    L, (lx, ly, lz) = ctx.lib, dims
    N, d3 = lx * ly * lz, lz > 1
    kinds = (pa.D3Q15, pa.D3Q7) if d3 else (pa.D2Q9, pa.D2Q5)
    rng = np.random.default_rng(3)

    def arr(v):
        return ctx.array((N,), data=np.full(N, v))

    one, zero, alpha, diff = arr(1.0), arr(0.0), arr(0.1), arr(0.1)
    out = [arr(0.0) for _ in range(8)]
    uz = zero.ptr if d3 else None

    def face(a, dt=np.float64):
        return pa.to_face(kinds[0], lx, ly, lz, np.broadcast_to(a, (N,)), dt)

    def step_us(masks):
        p, q = (pa.Lattice(ctx, k, lx, ly, lz) for k in kinds)
        m = [face(a, np.int32) for a in masks]
        u, r, z = face(0.01), face(1.0), face(0.0)
        check(L.lbm_record_begin(ctx.h))
        for h in (p, q):
            check(L.lbm_stream(h.h))
        check(L.lbm_bc(p.h, hptr(m[0])))
        check(L.lbm_ns_set_u(p.h, hptr(m[1]), hptr(u), hptr(z), hptr(z)))
        check(L.lbm_ns_set_rho(p.h, hptr(m[2]), hptr(r), hptr(z), hptr(z)))
        check(L.lbm_ad_set_t(q.h, hptr(m[3]), hptr(u), zero.ptr, zero.ptr, uz))
        check(L.lbm_ad_set_q(q.h, hptr(m[4]), hptr(z), zero.ptr, zero.ptr, uz, diff.ptr, D(0)))
        check(L.lbm_bc(q.h, hptr(m[5])))
        prog, g = ctypes.c_void_p(), ctypes.c_void_p()
        check(L.lbm_record_end(ctx.h, ctypes.byref(prog)))
        check(L.lbm_ns_initial_condition(p.h, one.ptr, zero.ptr, zero.ptr, uz))
        check(L.lbm_ad_initial_condition(q.h, zero.ptr, zero.ptr, zero.ptr, uz))

        def step():
            check(L.lbm_ad_macro_brinkman_collide_force_convection_p(
                prog, p.h, *(x.ptr for x in out[:3]), out[3].ptr, alpha.ptr, D(0.1), q.h,
                *(x.ptr for x in out[4:7]), out[7].ptr, diff.ptr, 0, None, None))

        step()
        step()
        check(L.lbm_graph_begin(ctx.h))
        for _ in range(100):
            step()
        check(L.lbm_graph_end(ctx.h, ctypes.byref(g)))
        best = np.inf
        for _ in range(6):
            ctx.sync()
            t0 = time.perf_counter()
            check(L.lbm_graph_launch(g))
            ctx.sync()
            best = min(best, time.perf_counter() - t0)
        L.lbm_graph_destroy(g)
        L.lbm_program_destroy(prog)
        return 1e4 * best

    uniform = step_us([np.ones(N, np.int32)] + [np.zeros(N, np.int32)] * 2 + [np.ones(N, np.int32)] +
                      [np.zeros(N, np.int32)] * 2)
    mixed = step_us([rng.integers(0, top + 1, N).astype(np.int32) for top in (2, 1, 1, 1, 1, 2)])
    print("mixed lists", dims, "%.1f us, uniform %.1f us" % (mixed, uniform), flush=True)
    assert mixed <= 3.0 * uniform


def test_eager_call_does_not_pay_for_the_fused_kernels_tables(ctx):
    """An eager boundary call uploads its operators and 4 bytes per boundary slot; recording the same call
    also builds what a fused collide reads, some 100 bytes per slot.  So the eager call, its kernel and
    its wait included, takes less than three quarters of the recording's time (best of 15 each)."""
    import time

    import panslbm2_amd as pa
    from panslbm2_amd import check, hptr

    L, (lx, ly, lz) = ctx.lib, (96, 96, 48)
    N = lx * ly * lz
    p = pa.Lattice(ctx, pa.D3Q15, lx, ly, lz)
    one, zero = ctx.array((N,), fill=1.0), ctx.array((N,), fill=0.0)
    check(L.lbm_ns_initial_condition(p.h, one.ptr, zero.ptr, zero.ptr, zero.ptr))

    def face(a, dt=np.float64):
        return pa.to_face(pa.D3Q15, lx, ly, lz, a, dt)

    inlet, u, z = face(np.arange(N) % lx == 0, np.int32), face(np.full(N, 0.03)), face(np.zeros(N))

    def eager():
        check(L.lbm_ns_set_u(p.h, hptr(inlet), hptr(u), hptr(z), hptr(z)))

    def record():
        prog = ctypes.c_void_p()
        check(L.lbm_record_begin(ctx.h))
        eager()
        check(L.lbm_record_end(ctx.h, ctypes.byref(prog)))
        L.lbm_program_destroy(prog)

    def best(call):
        b = np.inf
        for _ in range(15):
            ctx.sync()
            t0 = time.perf_counter()
            call()
            ctx.sync()
            b = min(b, time.perf_counter() - t0)
        return 1e6 * b

    e, r = best(eager), best(record)
    print("eager call %.0f us, recorded %.0f us" % (e, r), flush=True)
    assert e < 0.75 * r
