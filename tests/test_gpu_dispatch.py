"""H.v at sizes where the choice of tile, threads or kernel changes, against the oracle."""
import numpy as np
import pytest

import oracle
from pned_amd import gpu, lattice, model

pytestmark = pytest.mark.gpu


def _offdiagonal(cl, phi, field):
    c = model.set_lattice(20, phi)
    c.I11, c.I12, c.I11p, c.I12p, c.I11pp, c.I12pp = 0.21, 0.13, 0.21, 0.13, 0.21, 0.13
    H = model.bond_matrices(c, 2, "s12", field=field)
    mask, parity = model.local_mask(H, 2, "s12")
    return model.Operator(cl.n, 2, cl.ipair, cl.ibond_type, H, mask, parity, "s12", 0.0)


def _columns(ctx, ops, dtype, tol):
    """One H.v of a batch context (one operator per column), every column against the oracle."""
    cols = len(ops)
    x, y = ctx.vector(cols, dtype), ctx.vector(cols, dtype)
    ctx.set_initial_vec(x, 5)
    ctx.set_initial_vec(y, 6)
    X, Y = x.download().astype(complex), y.download().astype(complex)
    pr = ctx.p_mltply_v3(x, y, 0.03)
    got = y.download()
    for c in {0, 1, cols - 1}:
        xc, want = np.ascontiguousarray(X[:, c]), Y[:, c].copy()
        ref = oracle.hv(oracle.OracleOp(ops[c]), xc, want, eperbd=0.03)
        assert np.linalg.norm(got[:, c] - want) <= tol * np.linalg.norm(want), c
        assert abs(pr[c] - ref) <= tol * np.linalg.norm(xc) * np.linalg.norm(want - Y[:, c]), c


# 18 sites: 2^13-state tiles would save a pass, but leave the columns' coefficients no room in LDS.
# At most 9 terms a bond and 3 a site, one rounding each: 300 * 1.1e-16 (complex64 6e-8 with 3 roundings a term)
@pytest.mark.parametrize("cols,dtype,tol", [(16, gpu.C128, 1e-13), (64, gpu.C128, 1e-13), (64, gpu.C64, 2e-5)])
def test_batch_coefficients_beside_the_tile(cols, dtype, tol):
    cl = lattice.get_cluster("3x3")
    ops = [_offdiagonal(cl, 20.0 + 3.0 * c, 0.1 + 0.01 * c) for c in range(cols)]
    _columns(gpu.Context(ops[0], batch_ops=ops), ops, dtype, tol)


# sectors: 26 sites with few states on 1024 threads, 28 sites with more states than the grid's threads
@pytest.mark.parametrize("spec,k", [("1x13", 3), ("2x7", 6)])
def test_sector_grids(spec, k):
    op = model.build_operator(lattice.get_cluster(spec), 20, 180.0)
    ctx = gpu.Context(op)
    ctx.sz_sector(k)
    x, y = ctx.vector(), ctx.vector()
    ctx.set_initial_vec(x, 5)
    ctx.set_initial_vec(y, 6)
    xh, yh = x.download(), y.download()
    pr = ctx.p_mltply_v3(x, y, 0.05)
    want = yh.copy()
    ref = oracle.hv_sector(oracle.OracleOp(op), k, xh, want, eperbd=0.05)
    # at most 42 partners a state, each rounded once
    assert np.linalg.norm(y.download() - want) <= 1e-14 * np.linalg.norm(want)
    assert abs(pr - ref) <= 1e-13 * np.linalg.norm(xh) * np.linalg.norm(want - yh)


# more columns than hv_s12_split can sum (8 sites, 2^17 elements): <x|Hx> of every column
def test_512_columns():
    op = model.build_operator(lattice.get_cluster("2x2"), 20, 126.0, field=0.1)
    ctx = gpu.Context(op)
    rng = np.random.default_rng(3)
    xh, yh = (rng.standard_normal((256, 512)) + 1j * rng.standard_normal((256, 512)) for _ in range(2))
    x, y = ctx.vector(512), ctx.vector(512)
    x.upload(xh)
    y.upload(yh)
    pr = ctx.p_mltply_v3(x, y, 0.03)
    got = y.download()
    for c in (0, 1, 255, 256, 300, 511):
        want = yh[:, c].copy()
        ref = oracle.hv(oracle.OracleOp(op), np.ascontiguousarray(xh[:, c]), want, eperbd=0.03)
        assert np.linalg.norm(got[:, c] - want) <= 1e-13 * np.linalg.norm(want), c
        assert abs(pr[c] - ref) <= 1e-13 * np.linalg.norm(xh[:, c]) * np.linalg.norm(want - yh[:, c]), c


# complex couplings, which the real instances leave out: tables in LDS under 256 and 1024 threads, in memory
@pytest.mark.parametrize("spec,k", [("2x4", 8), ("1x11", 4), ("1x15", 2)])
def test_sector_complex_coefficients(spec, k):
    op = model.build_operator(lattice.get_cluster(spec), 20, 0.0)
    op.xlocal = op.xlocal * (1.0 + 0.3j)
    ctx = gpu.Context(op)
    ctx.sz_sector(k)
    x, y = ctx.vector(), ctx.vector()
    ctx.set_initial_vec(x, 5)
    ctx.set_initial_vec(y, 6)
    xh, yh = x.download(), y.download()
    pr = ctx.p_mltply_v3(x, y, 0.05)
    want = yh.copy()
    ref = oracle.hv_sector(oracle.OracleOp(op), k, xh, want, eperbd=0.05)
    # at most 45 partners a state, four products each
    assert np.linalg.norm(y.download() - want) <= 3e-14 * np.linalg.norm(want)
    assert abs(pr - ref) <= 1e-13 * np.linalg.norm(xh) * np.linalg.norm(want - yh)
    assert abs(pr.imag) > 1e-3 * abs(pr)


# COCG on the tiled kernel (shift, p^T y and scalars on the device) against the per-state gather kernel and
# the host's scalars: the same iterates after a few steps, also where the run ends without convergence
@pytest.mark.parametrize("spec,q", [("2x2", 3), ("2x2", 4), ("2x2", 5)])
def test_cocg_paths(spec, q):
    op = model.build_operator(lattice.get_cluster(spec), 20, 108.0, q=q)
    got = []
    for tiled in (True, False):
        ctx = gpu.Context(op)
        ctx.spin_kernel(tiled)
        b, x, r, p, y = (ctx.vector() for _ in range(5))
        ctx.set_initial_vec(b, 9)
        with pytest.raises(gpu.PnedError) as e:
            ctx.cocg(-5.0, 1.0, b, x, r, p, y, max_it=4, tol=1e-11)
        assert e.value.code == gpu.E_NOCONV
        got.append([v.download() for v in (x, r, p)])
        it, resid = ctx.cocg(-5.0, 1.0, b, x, r, p, y, tol=1e-11)
        assert resid < 1e-11
        # (H - e0 + i eta) x = b
        xh, bh = x.download(), b.download()
        ctx.hv_fresh(x, y, -5.0 / op.ibond)
        assert np.linalg.norm(y.download() + 1j * xh - bh) <= 1e-10 * np.linalg.norm(bh)
        got[-1].append(xh)
    # four steps grow a rounding difference of 1e-15 by the condition of the shifted operator, below 100 each
    for a, c in zip(*got):
        assert np.linalg.norm(a - c) <= 1e-10 * np.linalg.norm(c)


# every two-site term on all pairs of 8 sites, 64 operators: passes beyond the LDS on the state-major kernel,
# the others term-major, and all of them state-major.  448 products a state, one rounding each: 5e-14 at
# most (complex64 3e-5)
@pytest.mark.parametrize("dtype,tol", [(gpu.C128, 1e-13), (gpu.C64, 3e-5)])
def test_coefficients_beyond_the_lds(dtype, tol):
    ops = []
    for c in range(64):
        rng = np.random.default_rng(c)
        pairs = np.array([(a + 1, b + 1) for a in range(8) for b in range(a + 1, 8)], dtype=np.int32)
        H = rng.standard_normal((9, 4, 4)) + 1j * rng.standard_normal((9, 4, 4))
        H = H + np.conj(np.transpose(H, (0, 2, 1)))
        ops.append(model.Operator(8, 2, pairs.reshape(-1), (np.arange(28) % 9 + 1).astype(np.int32), H,
                                  np.zeros(H.shape, dtype=bool), 1, "s12", 0.0))
    ctx = gpu.Context(ops[0], batch_ops=ops)
    for kernel in (1, 0, 1):
        ctx.s12_kernel(kernel)
        _columns(ctx, ops, dtype, tol)
