"""Sector H.v by table place and block size, and sector Lanczos steps from captured graphs."""
import numpy as np
import pytest

import oracle
from pned_amd import gpu, lattice, model

pytestmark = pytest.mark.gpu


# 705432 states (1024 threads, a ragged last block), 28 sites (98 KB of tables in LDS), 30 sites
# (tables in global memory)
@pytest.mark.parametrize("spec,k", [("1x11", 11), ("2x7", 4), ("1x15", 3)])
def test_sector_hv_tables(spec, k):
    cl = lattice.get_cluster(spec)
    op = model.build_operator(cl, 20, 180.0)
    ctx = gpu.Context(op)
    ctx.sz_sector(k)
    rng = np.random.default_rng(3)
    x, y = (rng.standard_normal(ctx.dim) + 1j * rng.standard_normal(ctx.dim) for _ in range(2))
    v1, v0 = ctx.vector(), ctx.vector()
    v1.upload(x)
    v0.upload(y)
    pr = ctx.p_mltply_v3(v1, v0, 0.05)
    want = y.copy()
    pr_ref = oracle.hv_sector(oracle.OracleOp(op), k, x, want, eperbd=0.05)
    # at most 45 partners a state, each rounded once
    assert np.linalg.norm(v0.download() - want) <= 1e-14 * np.linalg.norm(want)
    assert abs(pr - pr_ref) <= 1e-13 * np.linalg.norm(x) * np.linalg.norm(want - y)


def test_sector_lanczos_graphs_match_launches():
    cl = lattice.get_cluster("2x4")
    got = []
    for graphs in (True, False):
        ctx = gpu.Context(model.build_operator(cl, 20, 0.0))
        ctx.sz_sector(8)
        ctx.graphs(graphs)
        v1, v0 = ctx.vector(), ctx.vector()
        ctx.set_initial_vec(v1, 7)
        _, a, b, _ = ctx.lnc1(v1, v0, fixed_steps=23, nvec=1)
        got.append((a, b, v1.download(), v0.download()))
    for p, q in zip(*got):
        assert np.array_equal(p, q)
