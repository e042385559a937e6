"""Which kernels the host code launches, and in which shape, by size (no GPU: see record.py)."""
import os
import shutil
import subprocess

import numpy as np
import pytest

from pned_amd import gpu, lattice, model
from tests.record import record  # noqa: F401  (fixture)

LDS = 160 * 1024


def test_batch_contexts_have_a_kernel(record):
    """One operator per column, complex128 and complex64: every size and operator count gets a kernel
    whose tile and staged coefficients fit the LDS, on wider tiles only while they do."""
    got = record("""
out = []
for l1, l2 in [(1, 4), (2, 3), (1, 7), (2, 4), (1, 9), (2, 5), (1, 11)]:
    for cols in (2, 8, 16, 32, 64):
        for field in (0.0, 0.1):
            ops = [offdiagonal(l1, l2, 20.0 + c, field) for c in range(cols)]
            for dtype in (gpu.C128, gpu.C64):
                if 2 * l1 * l2 + cols.bit_length() - 1 > 26:
                    continue
                ctx = gpu.Context(ops[0], batch_ops=ops)
                x, y = ctx.vector(cols, dtype), ctx.vector(cols, dtype)
                try:
                    k = launches(lambda: ctx.hv_fresh(x, y))
                except gpu.PnedError as e:
                    k = str(e)
                out.append([2 * l1 * l2, cols, field, dtype, k])
print(json.dumps(out))
""")
    assert len(got) == 2 * 2 * 33
    failed = [g[:4] + [g[4]] for g in got if isinstance(g[4], str)]
    assert not failed, failed
    for *case, k in got:
        assert k[-1][0] == "reduce_partials"
        for name, targs, grid, block, lds, limit in k[:-1]:
            assert name in ("hv_s12_tm", "hv_s12_pass") and targs[0] == block, (case, name)
            assert lds <= limit <= LDS, (case, name, lds, limit)


@pytest.mark.parametrize("cost,keeps", [(0.5, True), (5.0, False)])
def test_autotune_times_the_untuned_plan(record, cost, keeps):
    """The untuned plan of a short vector is the only one on hv_s12_split: autotuning keeps it (zeros)
    where it is the fastest and sets an explicit plan where it is not."""
    tune, names = record(f"""
rec.record_cost(b"hv_s12_split", ctypes.c_float({cost}))
ctx = gpu.Context(model.build_operator(T(2, 3), 20, 126.0, field=0.1))
x, y = ctx.vector(), ctx.vector()
r = ctx.autotune(x, y, 2)
print(json.dumps([[r["tile_bits"], r["low_bits"], r["threads"]], [k[0] for k in launches(lambda: ctx.hv_fresh(x, y))]]))
""")
    assert (tune == [0, 0, 0]) == keeps
    assert ("hv_s12_split" in names) == keeps and ("hv_s12_tm" in names) != keeps


def test_launches_set_their_lds_limit(record):
    """Every launch runs under a limit of its function that covers its own LDS, also when passes and
    contexts of different LDS sizes share an instance."""
    got = record("""
out = []
ctxs = []
for q, l1, l2, f in [(3, 2, 3, 0.0), (3, 2, 2, 0.0), (3, 1, 5, 0.2), (3, 2, 3, 0.2), (4, 2, 2, 0.0), (4, 1, 5, 0.1), (5, 2, 2, 0.1)]:
    ctx = gpu.Context(model.build_operator(T(l1, l2), 20, 108.0, q=q, field=f))
    ctxs.append((ctx, ctx.vector(), ctx.vector()))
for _ in range(2):
    for ctx, x, y in ctxs:
        out += launches(lambda: ctx.hv_fresh(x, y))
print(json.dumps(out))
""")
    assert len({(k[0], k[4]) for k in got if k[0] == "hv_spin_split"}) > 6
    short = [k for k in got if k[4] > k[5]]
    assert not short, short


@pytest.fixture(scope="module")
def nt_streams(tmp_path_factory):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(gpu.LIB_PATH) or not os.path.exists(hipcc):
        pytest.skip("needs libpned_gpu.so and hipcc")
    d = tmp_path_factory.mktemp("nt")
    libdir = os.path.dirname(gpu.LIB_PATH)
    subprocess.run([hipcc, "-O1", "-std=c++17", os.path.join(os.path.dirname(__file__), "native", "nt_streams.cpp"), "-o",
                    str(d / "nt"), "-L" + libdir, "-lpned_gpu", "-Wl,-rpath," + libdir], check=True, capture_output=True)

    def run(op, colbits, tile_bits, dtype):
        with open(d / "op.bin", "wb") as f:
            np.array([op.n, op.ibond, colbits, tile_bits, dtype], dtype=np.int32).tofile(f)
            np.asarray(op.ipair, dtype=np.int32).tofile(f)
            np.asarray(op.ibond_type, dtype=np.int32).tofile(f)
            np.ascontiguousarray(op.fortran_xlocal()).view(np.float64).tofile(f)
            np.asarray(op.fortran_llocal(), dtype=np.int32).tofile(f)
        return [int(x) for x in subprocess.run([str(d / "nt"), str(d / "op.bin")], check=True, capture_output=True).stdout.split()]

    return run


# vectors within the 256 MB cache, one of two beyond it, both beyond it; in complex64 a plan whose first pass
# alone reads whole lines (24 sites, a field), and one with whole lines throughout
@pytest.mark.parametrize("l1,l2,field,colbits,tile_bits,dtype,want", [
    (2, 5, 0.1, 2, 12, 0, 0), (3, 4, 0.1, 0, 12, 0, 2), (3, 4, 0.1, 1, 13, 0, 3), (3, 4, 0.1, 2, 14, 1, 0),
    (3, 4, 0.1, 1, 13, 1, 0), (3, 4, 0.1, 4, 13, 1, 3), (1, 13, 0.1, 0, 13, 1, 3), (2, 7, 0.0, 0, 13, 1, 0)])
def test_streams_need_whole_lines_in_every_pass(nt_streams, l1, l2, field, colbits, tile_bits, dtype, want):
    op = model.build_operator(lattice.torus(l1, l2), 20, 126.0, field=field)
    run, nt = nt_streams(op, colbits, tile_bits, dtype)
    assert nt == want
    assert nt == 0 or (16, 8)[dtype] << run >= 128


def test_batch_threads_by_blocks_per_cu(record):
    """2^12-state tiles of a batch context: 512 threads while two blocks fit a CU, else 1024."""
    got = record("""
out = []
for l1, l2, cols in [(2, 5, 8), (1, 11, 8), (2, 5, 64), (1, 9, 64)]:
    ops = [model.build_operator(T(l1, l2), 20, 126.0 + c, field=0.1) for c in range(cols)]
    ctx = gpu.Context(ops[0], batch_ops=ops)
    x, y = ctx.vector(cols), ctx.vector(cols)
    out.append(launches(lambda: ctx.hv_fresh(x, y))[:-1])
print(json.dumps(out))
""")
    tiles = {name for k in got for name, *_ in k}
    assert tiles == {"hv_s12_tm"}
    threads = set()
    for k in got:
        if k[0][1][0] * k[0][1][1] == 1 << 12:
            two = all(2 * lds <= LDS for *_, lds, limit in k)
            assert all(block == (512 if two else 1024) for _, _, _, block, _, _ in k), k
            threads.add(k[0][3])
    assert threads == {512, 1024}


def test_sector_blocks_are_resident(record):
    """Sector H.v: tables of 12 KB and more in LDS are staged by 1024 threads, on no more blocks than the
    CUs hold at once."""
    got = record("""
out = []
for l1, l2, k in [(2, 4, 8), (2, 5, 10), (1, 11, 2), (1, 11, 11), (3, 4, 3), (3, 4, 7), (1, 13, 3), (1, 13, 7), (2, 7, 6)]:
    ctx = gpu.Context(model.build_operator(T(l1, l2), 20, 0.0))
    ctx.sz_sector(k)
    x, y = ctx.vector(), ctx.vector()
    out.append([2 * l1 * l2, launches(lambda: ctx.hv_fresh(x, y))[0]])
print(json.dumps(out))
""")
    for n, (name, targs, grid, block, lds, limit) in got:
        assert name == "hv_sector_kernel" and targs == [1, n <= 28, block] and lds <= limit
        assert block == (1024 if 20 < n <= 28 else 256)
        if block == 1024:   # 16 KB of block sums beside the tables
            assert grid <= 256 * min(2, LDS // (lds + 16384)), (n, grid, lds)


def test_split_kernel_by_columns(record):
    """Short vectors: several workgroups per tile up to 2^18 elements in one complex128 column, 2^16 in 2 to
    16, 2^17 in more and in complex64."""
    got = record("""
out = []
for l1, l2, cols, dtype in [(3, 3, 1, 0), (2, 5, 1, 0), (2, 4, 1, 0), (1, 7, 4, 0), (1, 7, 8, 0), (2, 4, 2, 0), (2, 3, 16, 0), (2, 3, 32, 0), (1, 5, 128, 0),
                            (1, 7, 8, 1), (2, 4, 2, 1), (2, 4, 4, 1), (3, 3, 1, 1)]:
    ctx = gpu.Context(model.build_operator(T(l1, l2), 20, 126.0, field=0.1))
    x, y = ctx.vector(cols, dtype), ctx.vector(cols, dtype)
    out.append([2 * l1 * l2, cols, dtype, launches(lambda: ctx.hv_fresh(x, y))[0][0]])
print(json.dumps(out))
""")
    for n, cols, dtype, name in got:
        limit = 17 if dtype == 1 or cols > 16 else 16 if cols > 1 else 18
        assert (name == "hv_s12_split") == (n + cols.bit_length() - 1 <= limit), (n, cols, dtype, name)


@pytest.mark.parametrize("l1,l2,field,split", [(3, 3, 0.0, False), (3, 3, 0.1, True), (1, 9, 0.0, False), (2, 4, 0.0, True)])
def test_split_kernel_by_terms(record, l1, l2, field, split):
    """2^18 elements in one column take the split kernel where the passes have many terms."""
    names = record(f"""
ctx = gpu.Context(model.build_operator(T({l1}, {l2}), 20, 126.0, field={field}))
x, y = ctx.vector(), ctx.vector()
print(json.dumps([k[0] for k in launches(lambda: ctx.hv_fresh(x, y))]))
""")
    assert (names[0] == "hv_s12_split") == split


@pytest.mark.parametrize("cols,split", [(256, True), (512, False)])
def test_split_kernel_columns_fit_its_sums(record, cols, split):
    """hv_s12_split sums as 256 threads would: more columns than that stay with hv_s12_tm, whose block
    then has a thread for each."""
    k = record(f"""
ctx = gpu.Context(model.build_operator(T(2, 2), 20, 126.0, field=0.1))
x, y = ctx.vector({cols}), ctx.vector({cols})
print(json.dumps(launches(lambda: ctx.hv_fresh(x, y))))
""")
    assert (k[0][0] == "hv_s12_split") == split
    assert split or k[0][3] >= cols


@pytest.mark.parametrize("dtype", [0, 1])
def test_coefficients_beyond_the_lds(record, dtype):
    """64 operators with every two-site term: some passes leave their coefficients no room, so the
    state-major kernel runs there; the address tables are rebuilt whenever a pass's threads change with the kernel."""
    first, second, third, bytes1, bytes2 = record(f"""
ops = [general(8, c) for c in range(64)]
ctx = gpu.Context(ops[0], batch_ops=ops)
x, y = ctx.vector(64, {dtype}), ctx.vector(64, {dtype})
a = launches(lambda: ctx.hv_fresh(x, y))
ctx.s12_kernel(0)
n0 = rec.record_uploaded()
b = launches(lambda: ctx.hv_fresh(x, y))
n1 = rec.record_uploaded()
ctx.s12_kernel(1)
c = launches(lambda: ctx.hv_fresh(x, y))
print(json.dumps([a, b, c, n1 - n0, rec.record_uploaded() - n1]))
""")
    assert first == third
    assert {(k[0], k[3]) for k in first[:-1]} == {("hv_s12_pass", 256), ("hv_s12_tm", 512 if dtype else 1024)}
    assert {(k[0], k[3]) for k in second[:-1]} == {("hv_s12_pass", 512)}
    assert bytes1 > 0 and bytes2 > 0
