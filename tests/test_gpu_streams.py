"""Untuned S=1/2 plans above the cached sizes (tile size, threads and non-temporal streams by
vector size) against the state-major kernel on the same vectors."""
import numpy as np
import pytest

from pned_amd import gpu, lattice, model

pytestmark = pytest.mark.gpu


# 2^22 elements: first size with 2^12-state tiles; 256 MiB (16 columns): v0 non-temporal, v1
# cached; 1 GiB and 512 MiB: both non-temporal where the runs are whole lines (complex64 with
# one column reads 64-byte runs)
@pytest.mark.parametrize("spec,cols,dtype", [("1x11", 1, gpu.C128), ("2x5", 16, gpu.C128), ("1x13", 1, gpu.C128),
                                             ("1x13", 1, gpu.C64), ("2x5", 64, gpu.C64)])
def test_untuned_plan_matches_state_major(spec, cols, dtype):
    cl = lattice.get_cluster(spec)
    ctx = gpu.Context(model.build_operator(cl, 20, 126.0, field=0.1))
    x, a, b = (ctx.vector(cols, dtype) for _ in range(3))
    ctx.set_initial_vec(x, 5)
    ctx.set_initial_vec(a, 6)
    b.copy_from(a)
    pa = np.atleast_1d(ctx.p_mltply_v3(x, a, 0.03))
    ctx.s12_kernel(0)
    pb = np.atleast_1d(ctx.p_mltply_v3(x, b, 0.03))
    # about 80 terms a state, each kernel rounding once a term in the storage precision
    tol = 1e-13 if dtype == gpu.C128 else 2e-6
    nb = np.sqrt(np.atleast_1d(ctx.calc_vec_inprdct(b, b)).real)
    ctx.axpby(np.full(cols, -1.0 + 0j), b, np.full(cols, 1.0 + 0j), a)
    nd = np.sqrt(np.atleast_1d(ctx.calc_vec_inprdct(a, a)).real)
    assert np.all(nd <= tol * nb), (nd, nb)
    assert np.all(np.abs(pa - pb) <= tol * nb)   # |<x|Hx>| <= |Hx| for the unit x


# hv_s12_split (short vectors, untuned) against hv_s12_tm on 256 threads: the same values and sums bit
# for bit.  One tile and several, more and fewer columns than workgroups per tile, 256 and 1024 threads
@pytest.mark.parametrize("spec,cols,dtype", [("2x2", 1, gpu.C128), ("2x2", 64, gpu.C64), ("2x3", 1, gpu.C64),
                                             ("2x3", 16, gpu.C64), ("2x3", 32, gpu.C128), ("2x4", 1, gpu.C128),
                                             ("2x4", 2, gpu.C64), (18, 1, gpu.C128)])
def test_split_matches_tiles(spec, cols, dtype):
    cl = lattice.get_cluster(spec)
    got = []
    for threads in (0, 256):
        ctx = gpu.Context(model.build_operator(cl, 20, 126.0, field=0.1))
        if threads:
            ctx.tune(0, 0, threads)
        x, y = ctx.vector(cols, dtype), ctx.vector(cols, dtype)
        ctx.set_initial_vec(x, 5)
        ctx.set_initial_vec(y, 6)
        out = [np.atleast_1d(ctx.p_mltply_v3(x, y, 0.03)), y.download()]
        if cols == 1 and dtype == gpu.C128:
            _, a, b, _ = ctx.lnc1(x, y, fixed_steps=9, nvec=1)
            out += [a, b, x.download(), y.download()]
        got.append(out)
    for p, q in zip(*got):
        assert np.array_equal(p, q)


# hv_spin_split against the per-state gather kernel: one tile, several, parts of one and of q
# slots, complex coefficients (field), tiles of few states, and tiles too many for it (hv_spin_pass;
# 4 states on 12 sites with a non-temporal v1)
@pytest.mark.parametrize("spec,q,tile", [("2x2", 3, 0), ("2x2", 3, 6), ("2x3", 3, 0), ("2x3", 3, 7), ("2x3", 3, 4),
                                         ("2x2", 4, 0), ("2x2", 4, 4), ("2x3", 4, 0), ("2x2", 5, 0), ("2x2", 5, 3)])
@pytest.mark.parametrize("field", [0.0, 0.2])
def test_spin_split_matches_gather(spec, q, tile, field):
    ctx = gpu.Context(model.build_operator(lattice.get_cluster(spec), 20, 108.0, q=q, field=field))
    if tile:
        ctx.tune(tile_bits=tile)
    x, a, b = (ctx.vector() for _ in range(3))
    ctx.set_initial_vec(x, 5)
    ctx.set_initial_vec(a, 6)
    b.copy_from(a)
    pa = ctx.p_mltply_v3(x, a, 0.03)
    ctx.spin_kernel(False)
    pb = ctx.p_mltply_v3(x, b, 0.03)
    a, b = a.download(), b.download()
    # at most 18 bonds of 9 elements a state, one rounding each: 162 * 1.1e-16, twice
    assert np.linalg.norm(a - b) <= 1e-13 * np.linalg.norm(b)
    assert abs(pa - pb) <= 1e-13 * np.linalg.norm(b)


# one operator per column: the untuned plan (512 threads on 2^11-state tiles, and on 2^12-state tiles above
# 2^21 elements) against 256 threads on the same plan rules
@pytest.mark.parametrize("spec,cols", [("2x4", 8), (18, 2), ("2x5", 4)])
def test_batch_threads(spec, cols):
    cl = lattice.get_cluster(spec)
    ops = [model.build_operator(cl, 20, 126.0 + 23.0 * c, field=0.1 + 0.01 * c) for c in range(cols)]
    got = []
    for threads in (0, 256):
        ctx = gpu.Context(ops[0], batch_ops=ops)
        if threads:
            ctx.tune(0, 0, threads)
        x, y = ctx.vector(cols), ctx.vector(cols)
        ctx.set_initial_vec(x, 5)
        a, b = ctx.lanczos_batch_steps(x, y, np.ones(cols, dtype=np.int32), np.zeros(cols), np.zeros(cols), 5)
        got.append((a, b, x.download(), y.download()))
    # the sums over 2^16 and more products differ in order: sqrt of their number times 1.1e-16, and five
    # steps that each divide by a beta of order one
    for p, q in zip(*got):
        assert np.linalg.norm(p - q) <= 1e-12 * np.linalg.norm(q)
