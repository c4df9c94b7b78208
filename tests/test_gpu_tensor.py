"""MTTKRP and TTM on the GPU vs the CPU oracle, through the C ABI.

Structure (output rows / fibers) must be bit-exact; values within
|x - y| <= 1e-12 * max(|y|, sum|terms|).
"""
import time

import numpy as np
import pytest

import oracle
from sparsews_amd import formats, gen, taco
from sparsews_amd.device import Context, DeviceArray, DeviceCSF, mttkrp, set_ttm_method, ttm

pytestmark = pytest.mark.gpu
TOL = 1e-12


def dense(X):
    D = np.zeros(X.dims)
    D[X.idx[:, 0], X.idx[:, 1], X.idx[:, 2]] = X.vals
    return D


def run_mttkrp(ctx, X, Bf, Cf):
    R = Bf.shape[1]
    csf = formats.csf3_from_coo(X, (1, 2, 0))
    rows, M = mttkrp(ctx, DeviceCSF.upload(ctx, csf), X.dims[0], X.dims[1], X.dims[2], R,
                     DeviceArray.from_host(ctx, np.ascontiguousarray(Bf.ravel())),
                     DeviceArray.from_host(ctx, np.ascontiguousarray(Cf.ravel())))
    return rows.to_host(), M.to_host().reshape(X.dims[0], R)


def run_ttm(ctx, X, U, method=0):
    R = U.shape[1]
    csf = formats.csf3_from_coo(X, (0, 2, 1))
    set_ttm_method(ctx, method)
    try:
        fi, fj, Y = ttm(ctx, DeviceCSF.upload(ctx, csf), X.dims[0], X.dims[1], X.dims[2], R,
                        DeviceArray.from_host(ctx, np.ascontiguousarray(U.ravel())))
        return fi.to_host(), fj.to_host(), Y.to_host().reshape(-1, R)
    finally:
        set_ttm_method(ctx, 0)


@pytest.mark.parametrize("R", [32, 8, 48])
def test_mttkrp_small(ctx, R):
    print(f"case: mttkrp small R={R}", flush=True)
    X = gen.zipf_coo3((400, 300, 200), 20000, (1.5, 1.5, 1.5), 11, 5, 0.0, 1.0)
    rng = np.random.default_rng(R)
    Bf, Cf = rng.random((300, R)), rng.random((200, R))
    rows, M = run_mttkrp(ctx, X, Bf, Cf)
    csf = formats.csf3_from_coo(X, (1, 2, 0))
    oi, orr, ov = oracle.mttkrp_hash(csf, formats.dense_as_dcsr(Bf), formats.dense_as_dcsr(Cf), 400, R, 1 << 16)
    np.testing.assert_array_equal(np.repeat(rows, R), oi)
    absM = np.einsum("ijk,jr,kr->ir", np.abs(dense(X)), np.abs(Bf), np.abs(Cf))
    assert oracle.max_value_error(M[rows].ravel(), ov, absM[rows].ravel()) <= TOL
    # rows without a nonzero stay exactly zero
    empty = np.setdiff1d(np.arange(400), rows)
    assert np.all(M[empty] == 0)


def check_mttkrp(ctx, dims, idx, Bf, Cf, seed):
    """MTTKRP of the coordinates idx (distinct) against extended-precision
    sums."""
    rng = np.random.default_rng(seed)
    idx = np.asarray(idx, dtype=np.int32)
    idx = idx[np.lexsort((idx[:, 2], idx[:, 1], idx[:, 0]))]
    X = gen.COO3(dims, idx, rng.uniform(-1.0, 1.0, len(idx)))
    rows, M = run_mttkrp(ctx, X, Bf, Cf)
    np.testing.assert_array_equal(rows, np.unique(idx[:, 0]))
    exact = np.zeros((dims[0], Bf.shape[1]), dtype=np.longdouble)
    absum = np.zeros((dims[0], Bf.shape[1]))
    for at in range(0, len(idx), 1 << 18):
        i, j, k = idx[at:at + (1 << 18)].T
        t = (X.vals[at:at + (1 << 18), None] * Bf[j]) * Cf[k]
        u, start = np.unique(i, return_index=True)
        exact[u] += np.add.reduceat(t.astype(np.longdouble), start, axis=0)
        absum[u] += np.add.reduceat(np.abs(t), start, axis=0)
    assert oracle.max_value_error(M.ravel(), exact.astype(np.float64).ravel(), absum.ravel()) <= TOL


# ranks at the edges of a group's lanes and slices; rows of one nonzero, rows
# that end on a segment or a tile, one row over many tiles
@pytest.mark.parametrize("R", [1, 16, 17, 32, 33, 64])
@pytest.mark.parametrize("shape", ["one", "singles", "segments", "hot"])
def test_mttkrp_segment_edges(ctx, R, shape):
    print(f"case: mttkrp segments {shape} R={R}", flush=True)
    dims = (3000, 200, 150)
    if shape == "one":
        idx = [(5, 7, 9)]
    elif shape == "singles":  # every nonzero its own row
        idx = [(i, i % 200, i % 150) for i in range(2049)]
    elif shape == "segments":  # rows of 31, 32, 33, 255, 256, 257, 511, 513 nonzeros
        idx = [(3 * q, e % 200, e // 200) for q, c in enumerate((31, 32, 33, 255, 256, 257, 511, 513, 1, 1))
               for e in range(c)]
    else:  # one row of every (j, k), rows of one nonzero on both sides
        dims = (3000, 2000, 600) if R == 32 else dims
        j, k = np.meshgrid(np.arange(dims[1]), np.arange(dims[2]), indexing="ij")
        idx = np.stack([np.full(j.size, 1500), j.ravel(), k.ravel()], axis=1)
        idx = np.concatenate([idx, [(i, i % 200, i % 150) for i in range(1400, 1600) if i != 1500]])
    rng = np.random.default_rng(R)
    check_mttkrp(ctx, dims, idx, rng.uniform(-1, 1, (dims[1], R)), rng.uniform(-1, 1, (dims[2], R)), 5)


def test_mttkrp_factor_over_4_gib(ctx):
    """A factor of more than 2^32 bytes (64-bit addresses)."""
    print("case: mttkrp wide factor", flush=True)
    dims, R = (40, 30, 8_400_000), 64
    rng = np.random.default_rng(6)
    k = np.concatenate([rng.integers(0, dims[2], 300), [0, dims[2] - 1]])
    Cf = np.zeros((dims[2], R))
    Cf[k] = rng.uniform(-1, 1, (len(k), R))
    idx = np.unique(np.stack([rng.integers(0, 40, len(k)), rng.integers(0, 30, len(k)), k], axis=1), axis=0)
    check_mttkrp(ctx, dims, idx, rng.uniform(-1, 1, (dims[1], R)), Cf, 7)


# leaf modes of fewer bits than the sort's first digit (it then reaches into
# the root's bits), of as many and of more; one to three passes; nonzero counts
# at the edges of its tiles of 4,096; fibers longer than a tile
@pytest.mark.parametrize("dims,nnz", [
    ((70_000, 1, 9), 5000), ((70_000, 2, 9), 4097), ((3000, 5, 700), 8192), ((300, 513, 40), 4095), ((2, 2, 50), 150),
    ((5, 20_000, 3), 60_000), ((1, 1, 1), 1), ((40, 262_145, 3), 4096),
])
def test_tensor_sort_sources(ctx, dims, nnz):
    print(f"case: sort from the CSF dims={dims} nnz={nnz}", flush=True)
    rng = np.random.default_rng(nnz)
    I, J, K = dims
    at = np.unique(rng.choice(I * J * K, nnz, replace=False)) if I * J * K < 1 << 22 else \
        np.unique(rng.integers(0, I * J * K, 2 * nnz))
    at = np.sort(rng.permutation(at)[:nnz])
    X = gen.COO3(dims, np.stack([at // (J * K), at // K % J, at % K], axis=1).astype(np.int32),
                 rng.uniform(-1, 1, len(at)))
    U = rng.uniform(-1, 1, (K, 7))
    fi, fj, Y = run_ttm(ctx, X, U, method=1)
    fib, start = np.unique(at // K, return_index=True)  # (i, j) and its first nonzero
    np.testing.assert_array_equal(fi, fib // J)
    np.testing.assert_array_equal(fj, fib % J)
    t = X.vals[:, None] * U[X.idx[:, 2]]
    assert oracle.max_value_error(Y.ravel(), np.add.reduceat(t, start, axis=0).ravel(),
                                  np.add.reduceat(np.abs(t), start, axis=0).ravel()) <= TOL
    check_mttkrp(ctx, dims, X.idx, rng.uniform(-1, 1, (J, 7)), U, 9)


def test_mttkrp_taco_entry():
    print("case: mttkrp taco entry", flush=True)
    X = gen.zipf_coo3((120, 90, 70), 3000, (1.5, 1.5, 1.5), 12, 5, 0.0, 1.0)
    R = 16
    rng = np.random.default_rng(12)
    Bf, Cf = rng.random((90, R)), rng.random((70, R))
    csf = formats.csf3_from_coo(X, (1, 2, 0))
    At = taco.init_taco_tensor_COO([120, R])
    Bt = taco.csf_to_taco_tensor(csf)
    Ct = taco.CC_to_taco_tensor(formats.dense_as_dcsr(Bf), 90, R)
    Dt = taco.CC_to_taco_tensor(formats.dense_as_dcsr(Cf), 70, R)
    taco.mttkrp_compute(At, Bt, Ct, Dt, 1 << 10)
    gi, gr, gv = taco.taco_coo(At)
    oi, orr, ov = oracle.mttkrp_hash(csf, formats.dense_as_dcsr(Bf), formats.dense_as_dcsr(Cf), 120, R, 1 << 10)
    np.testing.assert_array_equal(gi, oi)
    np.testing.assert_array_equal(gr, orr)
    absM = np.einsum("ijk,jr,kr->ir", np.abs(dense(X)), np.abs(Bf), np.abs(Cf))
    assert oracle.max_value_error(gv, ov, absM[oi, orr]) <= TOL


@pytest.mark.parametrize("R", [16, 5, 40])
def test_ttm_small(ctx, R):
    print(f"case: ttm small R={R}", flush=True)
    X = gen.zipf_coo3((500, 400, 60), 20000, (1.5, 1.5, None), 13, 5, -1.0, 1.0)
    U = np.random.default_rng(R).uniform(-1, 1, (60, R))
    fi, fj, Y = run_ttm(ctx, X, U)
    csf = formats.csf3_from_coo(X, (0, 2, 1))
    ok, oj, ol, ov = oracle.ttm_hash_il(csf, formats.dense_as_dcsr(U), 500, 400, R)
    np.testing.assert_array_equal(np.repeat(fi, R), ok)
    np.testing.assert_array_equal(np.repeat(fj, R), oj)
    absY = np.einsum("ijk,kr->ijr", np.abs(dense(X)), np.abs(U))
    assert oracle.max_value_error(Y.ravel(), ov, absY[fi, fj].ravel()) <= TOL


TTM_ROOT_CASES = [
    # (dims, nnz, exponents, seed): Zipf roots -- a few heavy roots of many
    # 2,048-nonzero tiles and light ones; uniform roots -- light roots only;
    # Zipf roots over many roots -- both kinds, heavy ones of one tile
    ((60, 5000, 300), 200_000, (1.2, 1.5, None), 23),
    ((5000, 3000, 50), 100_000, (None, None, None), 24),
    ((20_000, 4000, 200), 300_000, (1.1, 1.3, None), 25),
]


@pytest.mark.parametrize("R", [16, 5, 32, 40, 64])
@pytest.mark.parametrize("case", range(len(TTM_ROOT_CASES)))
def test_ttm_roots_and_windows(ctx, R, case):
    """The roots-and-windows path (light roots sorted in registers, heavy
    roots bucketed by column window and added in dense LDS windows of
    1024 / R' columns): every fiber summed from 0.0 over k in increasing
    order, so structure and values equal the sequential hash_il oracle bit
    for bit; the sorting path gives the same structure and values within
    the tolerance (it splits fibers of more than 128 nonzeros into partial
    sums)."""
    dims, nnz, exps, seed = TTM_ROOT_CASES[case]
    print(f"case: ttm roots and windows R={R} dims={dims} nnz={nnz}", flush=True)
    X = gen.zipf_coo3(dims, nnz, exps, seed, 5, -1.0, 1.0)
    U = np.random.default_rng(50 + R).uniform(-1, 1, (dims[2], R))
    fi, fj, Y = run_ttm(ctx, X, U, method=2)
    csf = formats.csf3_from_coo(X, (0, 2, 1))
    ok, oj, ol, ov = oracle.ttm_hash_il(csf, formats.dense_as_dcsr(U), dims[0], dims[1], R)
    np.testing.assert_array_equal(np.repeat(fi, R), ok)
    np.testing.assert_array_equal(np.repeat(fj, R), oj)
    np.testing.assert_array_equal(Y.ravel(), ov)
    si, sj, SY = run_ttm(ctx, X, U, method=1)
    np.testing.assert_array_equal(si, fi)
    np.testing.assert_array_equal(sj, fj)
    scale = np.abs(Y).max() + 1.0
    assert np.max(np.abs(SY - Y)) <= 1e-12 * scale * 16


def test_ttm_roots_declines_wide_output_mode(ctx):
    """More column windows than the per-root counters hold (J = 300,000 at
    R = 16): method 2 refuses with SPWS_ERR_UNSUPPORTED, the automatic method
    takes the sorting path."""
    print("case: ttm roots path declines wide J", flush=True)
    from sparsews_amd._lib import SpwsError
    X = gen.zipf_coo3((40, 300_000, 30), 5000, (None, None, None), 26, 5, -1.0, 1.0)
    U = np.random.default_rng(7).uniform(-1, 1, (30, 16))
    with pytest.raises(SpwsError):
        run_ttm(ctx, X, U, method=2)
    fi, fj, Y = run_ttm(ctx, X, U)
    csf = formats.csf3_from_coo(X, (0, 2, 1))
    ok, oj, ol, ov = oracle.ttm_hash_il(csf, formats.dense_as_dcsr(U), 40, 300_000, 16)
    np.testing.assert_array_equal(np.repeat(fi, 16), ok)
    np.testing.assert_array_equal(np.repeat(fj, 16), oj)


# fibers at the edges of a segment (32 to 128 nonzeros) and of a group's reach
# beyond it (128), alone, after short ones and over many segments; ranks at the
# edges of a group's lanes and slices
@pytest.mark.parametrize("R", [1, 16, 17, 33, 64, 65, 256])
@pytest.mark.parametrize("lengths", [
    (1,), (128,), (129,), (1200,),
    tuple([1] * 515),
    (31, 33, 32, 127, 129, 128, 1, 161, 160, 159, 257, 1, 1, 255, 383, 1000, 3, 1200, 1200, 2),
    (7, 1200, 64, 64, 64, 96, 32, 1199, 1, 17, 500, 300),
])
def test_ttm_segment_edges(ctx, R, lengths):
    """Fibers of at most 128 nonzeros bit for bit the sum in increasing k;
    longer ones within the tolerance and the same again on a second call."""
    print(f"case: ttm segments R={R} lengths={lengths[:8]}", flush=True)
    K, J = 1200, 90
    rng = np.random.default_rng(R)
    idx = [(q // J, q % J, k) for q, c in enumerate(lengths) for k in sorted(rng.permutation(K)[:c])]
    idx = np.asarray(idx, dtype=np.int32)
    X = gen.COO3((len(lengths) // J + 1, J, K), idx, rng.uniform(-1, 1, len(idx)))
    U = rng.uniform(-1, 1, (K, R))
    fi, fj, Y = run_ttm(ctx, X, U, method=1)
    q = np.arange(len(lengths))
    np.testing.assert_array_equal(fi, q // J)
    np.testing.assert_array_equal(fj, q % J)
    at = 0
    for f, c in enumerate(lengths):
        t = X.vals[at:at + c, None] * U[idx[at:at + c, 2]]
        at += c
        seq = np.add.accumulate(np.concatenate([np.zeros((1, R)), t]), axis=0)[-1]
        if c <= 128:
            np.testing.assert_array_equal(Y[f], seq)
        assert oracle.max_value_error(Y[f], seq, np.abs(t).sum(axis=0)) <= TOL
    np.testing.assert_array_equal(run_ttm(ctx, X, U, method=1)[2], Y)


def test_ttm_segments_of_64(ctx):
    """A nonzero count whose segments hold 64: every fiber of 300."""
    print("case: ttm segments of 64", flush=True)
    dims, R = (20, 400, 300), 16
    i, j, k = np.meshgrid(*(np.arange(d) for d in dims), indexing="ij")
    idx = np.stack([i.ravel(), j.ravel(), k.ravel()], axis=1).astype(np.int32)
    rng = np.random.default_rng(3)
    X = gen.COO3(dims, idx, rng.uniform(-1, 1, len(idx)))
    U = rng.uniform(-1, 1, (dims[2], R))
    fi, fj, Y = run_ttm(ctx, X, U, method=1)
    np.testing.assert_array_equal(fi, np.repeat(np.arange(20), 400))
    np.testing.assert_array_equal(fj, np.tile(np.arange(400), 20))
    V = X.vals.reshape(-1, 300)
    exact = (V.astype(np.longdouble) @ U.astype(np.longdouble)).astype(np.float64)
    assert oracle.max_value_error(Y.ravel(), exact.ravel(), (np.abs(V) @ np.abs(U)).ravel()) <= TOL


def test_ttm_time_of_a_long_fiber(ctx):
    """One fiber of 300,000 nonzeros by sorting: its parts are added one after
    another, but not one slice of 16 ranks after another (four slices then
    take 3.2 times as long as one)."""
    print("case: ttm time of a long fiber", flush=True)
    K = 300_000
    X = gen.COO3((1, 1, K), np.stack([np.zeros(K), np.zeros(K), np.arange(K)], axis=1).astype(np.int32),
                 np.random.default_rng(9).uniform(-1, 1, K))
    dX = DeviceCSF.upload(ctx, formats.csf3_from_coo(X, (0, 2, 1)))
    times = []
    try:
        set_ttm_method(ctx, 1)
        for R in (16, 64):
            U = np.random.default_rng(R).uniform(-1, 1, (K, R))
            dU = DeviceArray.from_host(ctx, U.ravel())
            took = []
            for _ in range(6):
                ctx.sync()
                t = time.perf_counter()
                Y = ttm(ctx, dX, 1, 1, K, R, dU)[2]
                ctx.sync()
                took.append(time.perf_counter() - t)
            times.append(min(took[1:]))
            assert oracle.max_value_error(Y.to_host(), X.vals @ U, np.abs(X.vals) @ np.abs(U)) <= TOL
    finally:
        set_ttm_method(ctx, 0)
    print(f"R = 16 {times[0] * 1e6:.0f} us, R = 64 {times[1] * 1e6:.0f} us", flush=True)
    assert times[1] <= 2 * times[0]


@pytest.mark.parametrize("method", [0, 1])
@pytest.mark.parametrize("R", [16, 40])
def test_ttm_long_fibers(ctx, R, method):
    """Fibers of 139-200 nonzeros, by roots and windows (the automatic choice
    here) and by sorting: there most are longer than the group that starts
    them follows (segments of 32 and 128 nonzeros beyond), so segments inside
    them leave partial sums; ranks in three 16-lane slices for R = 40."""
    print(f"case: ttm long fibers R={R} method {method}", flush=True)
    X = gen.zipf_coo3((20, 30, 400), 100000, (None, None, None), 21, 5, -1.0, 1.0)
    U = np.random.default_rng(30 + R).uniform(-1, 1, (400, R))
    fi, fj, Y = run_ttm(ctx, X, U, method)
    csf = formats.csf3_from_coo(X, (0, 2, 1))
    ok, oj, ol, ov = oracle.ttm_hash_il(csf, formats.dense_as_dcsr(U), 20, 30, R)
    np.testing.assert_array_equal(np.repeat(fi, R), ok)
    np.testing.assert_array_equal(np.repeat(fj, R), oj)
    absY = np.einsum("ijk,kr->ijr", np.abs(dense(X)), np.abs(U))
    assert oracle.max_value_error(Y.ravel(), ov, absY[fi, fj].ravel()) <= TOL


@pytest.mark.parametrize("method", [0, 1])
def test_ttm_many_short_fibers(ctx, method):
    """~400k short fibers, by roots and windows (all of them light roots) and
    by sorting: there each 16-lane group writes about thirty fibers of its
    segment of 32 nonzeros."""
    print(f"case: ttm many short fibers method {method}", flush=True)
    X = gen.zipf_coo3((3000, 3000, 50), 400000, (None, None, None), 22, 5, -1.0, 1.0)
    R = 16
    U = np.random.default_rng(40).uniform(-1, 1, (50, R))
    fi, fj, Y = run_ttm(ctx, X, U, method)
    csf = formats.csf3_from_coo(X, (0, 2, 1))
    ok, oj, ol, ov = oracle.ttm_hash_il(csf, formats.dense_as_dcsr(U), 3000, 3000, R)
    np.testing.assert_array_equal(np.repeat(fi, R), ok)
    np.testing.assert_array_equal(np.repeat(fj, R), oj)
    # |X| |U| per fiber from the sorted coordinates (no dense 3000 x 3000 x 50 copy)
    order = np.lexsort((X.idx[:, 2], X.idx[:, 1], X.idx[:, 0]))
    xi, xj, xk = (X.idx[order, m].astype(np.int64) for m in range(3))
    fid = np.searchsorted(fi.astype(np.int64) * 3000 + fj, xi * 3000 + xj)
    absY = np.zeros((len(fi), R))
    np.add.at(absY, fid, np.abs(X.vals[order])[:, None] * np.abs(U[xk]))
    assert oracle.max_value_error(Y.ravel(), ov, absY.ravel()) <= TOL


def test_ttm_wide_coordinates(ctx):
    """Dimensions whose packed (i, j, k) coordinates need more than 64 bits
    (2^24 x 2^24 x 2^17): the fibers are grouped through the hash table
    instead of one sort on (i, j, k).  Fibers and their sums are checked
    against a numpy grouping of the nonzeros, summed in increasing k."""
    print("case: ttm 65-bit coordinates", flush=True)
    dims = (1 << 24, 1 << 24, 1 << 17)
    X = gen.zipf_coo3(dims, 3000, (1.5, 1.5, None), 16, 5, -1.0, 1.0)
    R = 4
    U = np.random.default_rng(16).uniform(-1, 1, (dims[2], R))
    fi, fj, Y = run_ttm(ctx, X, U)
    i, j, k, v = X.idx[:, 0], X.idx[:, 1], X.idx[:, 2], X.vals
    order = np.lexsort((k, j, i))
    i, j, k, v = i[order], j[order], k[order], v[order]
    head = np.ones(len(i), dtype=bool)
    head[1:] = (i[1:] != i[:-1]) | (j[1:] != j[:-1])
    np.testing.assert_array_equal(fi, i[head])
    np.testing.assert_array_equal(fj, j[head])
    fib = np.cumsum(head) - 1
    ref = np.zeros((head.sum(), R))
    ab = np.zeros((head.sum(), R))
    for p in range(len(i)):  # in increasing k within each fiber
        ref[fib[p]] += v[p] * U[k[p]]
        ab[fib[p]] += np.abs(v[p] * U[k[p]])
    assert oracle.max_value_error(Y.ravel(), ref.ravel(), ab.ravel()) <= TOL


def test_ttm_frostt_file(ctx, tmp_path):
    """A FROSTT .tns file read with its values, then TTM on the device."""
    print("case: ttm on a FROSTT file", flush=True)
    from sparsews_amd import io as spio
    X0 = gen.zipf_coo3((300, 200, 40), 8000, (1.5, 1.5, None), 17, 5, -1.0, 1.0)
    path = tmp_path / "x.tns"
    spio.write_tns(path, X0)
    X = spio.read_tns(path, dims=X0.dims)
    R = 8
    U = np.random.default_rng(17).uniform(-1, 1, (40, R))
    fi, fj, Y = run_ttm(ctx, X, U)
    csf = formats.csf3_from_coo(X, (0, 2, 1))
    ok, oj, ol, ov = oracle.ttm_hash_il(csf, formats.dense_as_dcsr(U), 300, 200, R)
    np.testing.assert_array_equal(np.repeat(fi, R), ok)
    np.testing.assert_array_equal(np.repeat(fj, R), oj)
    absY = np.einsum("ijk,kr->ijr", np.abs(dense(X)), np.abs(U))
    assert oracle.max_value_error(Y.ravel(), ov, absY[fi, fj].ravel()) <= TOL


def test_ttm_taco_entry():
    print("case: ttm taco entry", flush=True)
    X = gen.zipf_coo3((80, 70, 30), 2500, (1.5, 1.5, None), 14, 5, -1.0, 1.0)
    R = 16
    U = np.random.default_rng(14).uniform(-1, 1, (30, R))
    csf = formats.csf3_from_coo(X, (0, 2, 1))
    At = taco.init_taco_tensor_COO([80, 70, R])
    taco.ttm_compute(At, taco.csf_to_taco_tensor(csf), taco.CC_to_taco_tensor(formats.dense_as_dcsr(U), 30, R), 1)
    gk, gj, gl, gv = taco.taco_coo(At)
    ok, oj, ol, ov = oracle.ttm_hash_il(csf, formats.dense_as_dcsr(U), 80, 70, R)
    np.testing.assert_array_equal(gk, ok)
    np.testing.assert_array_equal(gj, oj)
    np.testing.assert_array_equal(gl, ol)
    absY = np.einsum("ijk,kr->ijr", np.abs(dense(X)), np.abs(U))
    assert oracle.max_value_error(gv, ov, absY[ok, oj, ol]) <= TOL


@pytest.mark.parametrize("col_density", [1.0, 0.5])
def test_mttkrp_taco_hypersparse_factors(col_density):
    """DCSR factors with missing rows (and, at density 0.5, rows storing only
    some columns) through the taco entry point: the co-iteration of
    hash_free.h:277-300 on the device (factor row masks); entries, their
    order and values against the oracle."""
    print(f"case: mttkrp hypersparse factors density {col_density}", flush=True)
    X = gen.zipf_coo3((120, 90, 70), 3000, (1.5, 1.5, 1.5), 16, 5, 0.0, 1.0)
    R = 16
    rng = np.random.default_rng(16)
    Bf, Cf = rng.random((90, R)), rng.random((70, R))
    Bd = formats.partial_dcsr(Bf, rng.random(90) < 0.6, col_density, 161)
    Cd = formats.partial_dcsr(Cf, rng.random(70) < 0.7, col_density, 162)
    csf = formats.csf3_from_coo(X, (1, 2, 0))
    At = taco.init_taco_tensor_COO([120, R])
    taco.mttkrp_compute(At, taco.csf_to_taco_tensor(csf), taco.CC_to_taco_tensor(Bd, 90, R),
                        taco.CC_to_taco_tensor(Cd, 70, R), 1 << 10)
    gi, gr, gv = taco.taco_coo(At)
    oi, orr, ov = oracle.mttkrp_hash(csf, Bd, Cd, 120, R, 1 << 10)
    assert len(oi) < 120 * R
    np.testing.assert_array_equal(gi, oi)
    np.testing.assert_array_equal(gr, orr)
    Bz, _ = formats.dcsr_dense_and_mask(Bd)
    Cz, _ = formats.dcsr_dense_and_mask(Cd)
    absM = np.einsum("ijk,jr,kr->ir", np.abs(dense(X)), np.abs(Bz), np.abs(Cz))
    assert oracle.max_value_error(gv, ov, absM[oi, orr]) <= TOL


@pytest.mark.parametrize("col_density", [1.0, 0.5])
def test_ttm_taco_hypersparse_factor(col_density):
    """A DCSR U with missing rows (and partial rows at density 0.5) through
    the taco entry point: hash_il's co-iteration of the contracted level with
    U's rows on the device; fibers, entries and values against the oracle."""
    print(f"case: ttm hypersparse factor density {col_density}", flush=True)
    X = gen.zipf_coo3((80, 70, 30), 2500, (1.5, 1.5, None), 17, 5, -1.0, 1.0)
    R = 16
    rng = np.random.default_rng(17)
    U = rng.uniform(-1, 1, (30, R))
    Ud = formats.partial_dcsr(U, rng.random(30) < 0.5, col_density, 171)
    csf = formats.csf3_from_coo(X, (0, 2, 1))
    At = taco.init_taco_tensor_COO([80, 70, R])
    taco.ttm_compute(At, taco.csf_to_taco_tensor(csf), taco.CC_to_taco_tensor(Ud, 30, R), 1)
    gk, gj, gl, gv = taco.taco_coo(At)
    ok, oj, ol, ov = oracle.ttm_hash_il(csf, Ud, 80, 70, R)
    np.testing.assert_array_equal(gk, ok)
    np.testing.assert_array_equal(gj, oj)
    np.testing.assert_array_equal(gl, ol)
    Uz, _ = formats.dcsr_dense_and_mask(Ud)
    absY = np.einsum("ijk,kr->ijr", np.abs(dense(X)), np.abs(Uz))
    assert oracle.max_value_error(gv, ov, absY[ok, oj, ol]) <= TOL


@pytest.mark.parametrize("R", [16, 40])
def test_ttm_masked_long_fibers(R):
    """Stored columns of fibers over several segments: each is stored by one
    of its parts only (U row k stores column k mod R, half the rows none)."""
    print(f"case: ttm masked long fibers R={R}", flush=True)
    X = gen.zipf_coo3((5, 6, 900), 20_000, (None, None, None), 18, 5, -1.0, 1.0)
    k = np.arange(0, 900, 2)
    Ud = formats.DCSR(900, R, k.astype(np.int32), np.arange(len(k) + 1, dtype=np.int32), (k % R).astype(np.int32),
                      np.random.default_rng(18).uniform(-1, 1, len(k)))
    At = taco.init_taco_tensor_COO([5, 6, R])
    taco.ttm_compute(At, taco.csf_to_taco_tensor(formats.csf3_from_coo(X, (0, 2, 1))),
                     taco.CC_to_taco_tensor(Ud, 900, R), 1)
    gk, gj, gl, gv = taco.taco_coo(At)
    ok, oj, ol, ov = oracle.ttm_hash_il(formats.csf3_from_coo(X, (0, 2, 1)), Ud, 5, 6, R)
    for got, want in ((gk, ok), (gj, oj), (gl, ol)):
        np.testing.assert_array_equal(got, want)
    absY = np.einsum("ijk,kr->ijr", np.abs(dense(X)), np.abs(formats.dcsr_dense_and_mask(Ud)[0]))
    assert oracle.max_value_error(gv, ov, absY[ok, oj, ol]) <= TOL


def test_tensor_edge_cases(ctx):
    print("case: tensor edge cases", flush=True)
    X = gen.zipf_coo3((10, 9, 8), 1, (None, None, None), 15, 5, 0.5, 1.0)
    Bf, Cf = np.ones((9, 4)), np.ones((8, 4))
    rows, M = run_mttkrp(ctx, X, Bf, Cf)
    np.testing.assert_array_equal(rows, [X.idx[0, 0]])
    np.testing.assert_array_equal(M[X.idx[0, 0]], np.full(4, X.vals[0]))
    fi, fj, Y = run_ttm(ctx, X, np.ones((8, 3)))
    np.testing.assert_array_equal(fi, [X.idx[0, 0]])
    np.testing.assert_array_equal(fj, [X.idx[0, 1]])


def sample_rows_reference(X, Bf, Cf, rows):
    """M(rows, :) from the nonzeros of the sampled rows, and sum|terms|."""
    sel = np.isin(X.idx[:, 0], rows)
    xi, xj, xk, xv = X.idx[sel, 0], X.idx[sel, 1], X.idx[sel, 2], X.vals[sel]
    where = np.searchsorted(rows, xi)
    R = Bf.shape[1]
    ref = np.zeros((len(rows), R))
    ab = np.zeros((len(rows), R))
    t = (xv[:, None] * Bf[xj]) * Cf[xk]
    np.add.at(ref, where, t)
    np.add.at(ab, where, np.abs(t))
    return ref, ab


def test_mttkrp_full_workload(ctx):
    """50,000 x 40,000 x 30,000, 20M nonzeros, R = 32: present rows exact and
    256 sampled rows against a float reference."""
    print("case: mttkrp full workload (generating)", flush=True)
    X, Bf, Cf = gen.mttkrp_tensor()
    print("case: mttkrp full workload (running)", flush=True)
    rows, M = run_mttkrp(ctx, X, Bf, Cf)
    np.testing.assert_array_equal(rows, np.unique(X.idx[:, 0]))
    samp = np.sort(np.random.default_rng(5).choice(rows, 256, replace=False))
    ref, ab = sample_rows_reference(X, Bf, Cf, samp)
    assert oracle.max_value_error(M[samp].ravel(), ref.ravel(), ab.ravel()) <= TOL


def test_ttm_full_workload(ctx):
    """100,000 x 80,000 x 2,000, 10M nonzeros, R = 16: fiber list exact and
    sampled fibers against a float reference."""
    print("case: ttm full workload (generating)", flush=True)
    X, U = gen.ttm_tensor()
    print("case: ttm full workload (running)", flush=True)
    fi, fj, Y = run_ttm(ctx, X, U)
    key = X.idx[:, 0].astype(np.int64) * X.dims[1] + X.idx[:, 1]
    fib = np.unique(key)
    np.testing.assert_array_equal(fi.astype(np.int64) * X.dims[1] + fj, fib)
    samp = np.sort(np.random.default_rng(6).choice(len(fib), 512, replace=False))
    sel = np.isin(key, fib[samp])
    where = np.searchsorted(fib[samp], key[sel])
    t = X.vals[sel, None] * U[X.idx[sel, 2]]
    ref = np.zeros((len(samp), U.shape[1]))
    ab = np.zeros_like(ref)
    np.add.at(ref, where, t)
    np.add.at(ab, where, np.abs(t))
    assert oracle.max_value_error(Y[samp].ravel(), ref.ravel(), ab.ravel()) <= TOL
