"""Size-edge tests of the paths chosen by sizes, ranks and layouts.

Each test takes its sizes where the path it names can go wrong (edges of
chunks, runs and tables, remainders, the smallest and largest of a range) and
compares with a plain restatement or the float64 oracle.  Tolerances:
counts, orders and index arrays exact; float32 sums within 1e-5 relative
(Frobenius) of float64, 2^-24 per rounding over the at most a few hundred
roundings of a row's partial sums, with room for their growth."""
import numpy as np
import pytest

from test_gpu_builder import random_tensor

pytestmark = pytest.mark.gpu


# ---- which tree order a mode gets: the working set of its gathers ----------------

def footprint(ind, rows, frac=0.9):
    """Rows that hold `frac` of the nonzeros, most used first."""
    c = np.sort(np.bincount(ind, minlength=rows))[::-1].astype(np.int64)
    before = np.concatenate([[0], np.cumsum(c)[:-1]])
    return int((before < frac * len(ind)).sum())


@pytest.mark.parametrize("dims,skew,nnz", [
    ([40, 30, 20], [None, None, None], 1),            # one nonzero
    ([300, 200, 100], [1.2, None, None], 20_000),
    ([30_000, 9000, 500], [None, 1.2, None], 60_000),  # more rows than the counting table holds
    ([20_000, 30_000, 400], [1.2, 1.1, None], 150_000),
    ([9000, 8192, 8193], [None, None, None], 100_000),
    # the concentrated mode above the leaf; pairs counted exactly up to 2^16
    # nonzeros, by a sample of the pairs past it
    ([30_000, 3000, 2000], [1.5, None, None], 65_500),
    ([30_000, 3000, 2000], [1.5, None, None], 66_000),
    ([30_000, 5000, 4000], [1.4, None, None], 700_001),
    ([3000, 2000, 1000], [1.4, None, None], 700_001),
])
def test_mode_tree_orders_follow_the_footprints(cuda, dims, skew, nnz):
    import mmcsf
    rng = np.random.default_rng(nnz)
    inds, vals = random_tensor(rng, dims, nnz, skew)
    f = mmcsf.Format(mmcsf.Tensor.from_numpy(dims, inds, vals), 12, fbr_threshold=128)
    info = f.info()
    hot = [footprint(inds[m], dims[m]) for m in range(3)]
    n = len(vals)
    for m in (0, 1):
        a, b = sorted((x for x in range(3) if x != m), key=lambda x: dims[x])
        # the default order ends in b; the swapped one in a
        pairs = {x: len(np.unique(inds[m].astype(np.int64) * dims[x] + inds[x])) for x in (a, b)}
        sampled = n > 1 << 16  # counts within 3 %: either order is right nearer to a line
        if 2 * hot[a] < hot[b] or 2 * hot[b] < hot[a]:
            dense, spread = (a, b) if hot[a] < hot[b] else (b, a)
            x, y = pairs[spread] / n, pairs[dense] / n
            if sampled and min(abs(x / 0.9 - 1), abs(y / 0.65 - 1)) < 0.03:
                continue
            want = [m, dense, spread] if x >= 0.9 and y <= 0.65 else [m, spread, dense]
        else:
            if sampled and abs(pairs[a] / pairs[b] - 1) < 0.03:
                continue
            want = [m, b, a] if pairs[b] < pairs[a] else [m, a, b]
        assert info["modeTreeOrder"][m] == want, (m, hot)


# ---- builder: sorted keys unpacked, values carried, start bits by windows ---------

def rel(a, b):
    b = np.asarray(b, dtype=np.float64)
    n = np.linalg.norm(b)
    return float(np.linalg.norm(np.asarray(a, np.float64) - b) / (n if n > 0 else 1.0))


def fibers_tensor(rng, fibers, per_fiber, leaf_dim):
    """`fibers` leaf fibers of `per_fiber` nonzeros each, in random order."""
    f = np.repeat(np.arange(fibers, dtype=np.int64), per_fiber)
    leaf = np.concatenate([np.sort(rng.choice(leaf_dim, per_fiber, replace=False)) for _ in range(fibers)])
    p = rng.permutation(len(f))
    inds = [(f // 50)[p], (f % 50)[p], leaf[p].astype(np.int64)]
    dims = [int(inds[0].max()) + 1, 50, leaf_dim]
    return dims, inds, (rng.random(len(f)) + 0.25).astype(np.float32)


@pytest.mark.parametrize("fibers,per_fiber", [(1, 1), (2047, 1), (2048, 3), (2049, 2), (2048, 32), (2049, 33), (4100, 40)])
def test_fiber_start_bits(cuda, fibers, per_fiber):
    """A block of the start-bit kernel marks 2048 fibers in a window of 65536
    nonzeros: one fiber below, at and above the block, at and past the window."""
    import torch
    import mmcsf
    import oracle as O
    from test_gpu_builder import check_format
    rng = np.random.default_rng(fibers)
    dims, inds, vals = fibers_tensor(rng, fibers, per_fiber, 64)
    t = mmcsf.Tensor.from_numpy(dims, inds, vals)
    U = [rng.random((d, 8)).astype(np.float32) for d in dims]
    Ud = [torch.from_numpy(u).to(cuda) for u in U]
    for fmt_type in (8, 10):
        fmt, _ = check_format(mmcsf, t, fmt_type, dims, inds, vals, 0, 1 << 30)
        assert rel(mmcsf.mttkrp(fmt, 0, Ud).cpu().numpy(), O.mttkrp_coo_f64(inds, vals, 0, U)) < 1e-5


@pytest.mark.parametrize("dims", [[1 << 21, 1 << 21, 1 << 21], [(1 << 21) + 1, 1 << 21, (1 << 22) - 1],
                                  [1 << 16, 1 << 16, 1 << 16, 1 << 16], [1 << 20, (1 << 18) + 5, 1 << 19, 1 << 17]])
@pytest.mark.parametrize("fmt_type", [3, 8, 10, 12])
def test_sort_key_widths(cuda, dims, fmt_type):
    """Coordinates of 63, 64 and more than 64 bits in all: one sort whose keys
    are unpacked, and two of which the second holds only the upper levels."""
    import mmcsf
    from test_gpu_builder import check_format
    rng = np.random.default_rng(len(dims) + fmt_type)
    inds, vals = random_tensor(rng, dims, 3000, [1.3] + [None] * (len(dims) - 1))
    for a, d in zip(inds, dims):
        a[rng.integers(0, len(a), 20)] = d - 1  # the largest coordinate
    key = np.stack(inds)
    _, first = np.unique(key, axis=1, return_index=True)
    first = np.sort(first)
    inds, vals = [a[first] for a in inds], vals[first]
    t = mmcsf.Tensor.from_numpy(dims, inds, vals)
    for mode in ([2] if fmt_type == 12 else range(len(dims))):
        check_format(mmcsf, t, fmt_type, dims, inds, vals, mode, 128)


# ---- MTTKRP at ranks that no vector width divides ---------------------------------

def offset_copy(t, off):
    """A contiguous device copy of t that starts `off` floats into its storage."""
    import torch
    s = torch.empty(t.numel() + off, dtype=t.dtype, device=t.device)
    v = s[off:].view(t.shape)
    v.copy_(t)
    return v


@pytest.mark.parametrize("R", [1, 3, 4, 5, 6, 7, 8, 9, 10, 15, 17, 25, 31, 33, 50, 63, 65, 127, 129, 253, 255])
@pytest.mark.parametrize("dims,skew,nnz", [([211, 90, 57], [1.2, None, 1.1], 9000),
                                           ([60, 37, 25, 14], [1.1, None, 1.2, None], 7001)])
def test_mttkrp_ragged_ranks(cuda, dims, skew, nnz, R):
    """Each side of the row groups' widths (4, 8, 16, 32, 64, 128, 256 columns);
    factors and output at 4-byte boundaries where the rank allows them."""
    import torch
    import mmcsf
    import oracle as O
    rng = np.random.default_rng(R)
    inds, vals = random_tensor(rng, dims, nnz, skew)
    t = mmcsf.Tensor.from_numpy(dims, inds, vals)
    U = [rng.random((d, R)).astype(np.float32) for d in dims]
    off = 1 if R % 4 else 0
    Ud = [offset_copy(torch.from_numpy(u).to(cuda), off) for u in U]
    ref = [O.mttkrp_coo_f64(inds, vals, m, U) for m in range(len(dims))]
    f = mmcsf.Format(t, 12, fbr_threshold=16)
    for m in range(len(dims)):
        out = offset_copy(torch.full((dims[m], R), 7.0, device=cuda), off)
        mmcsf.mttkrp(f, m, Ud, out=out)
        assert rel(out.cpu().numpy(), ref[m]) < 1e-5, f"mode {m}"
    for fmt_type in (8, 10):
        g = mmcsf.Format(t, fmt_type, mode=1, fbr_threshold=16)
        assert rel(mmcsf.mttkrp(g, 1, Ud).cpu().numpy(), ref[1]) < 1e-5, f"type {fmt_type}"


# ---- COO type as a walk -------------------------------------------------------------

@pytest.mark.parametrize("nnz", [1, 63, 64, 65, 4097, 40_000])
@pytest.mark.parametrize("rows", [1, 50, 100_000])  # one slice, slices over many chunks, a slice per nonzero
@pytest.mark.parametrize("N", [3, 4])
def test_coo_walk(cuda, N, rows, nnz):
    import torch
    import mmcsf
    import oracle as O
    rng = np.random.default_rng(nnz + rows)
    dims = [rows, 300, 170, 90][:N]
    inds, vals = random_tensor(rng, dims, nnz, [1.3 if rows > 50 else None] + [None] * (N - 1))
    f = mmcsf.Format(mmcsf.Tensor.from_numpy(dims, inds, vals), 3, mode=0)
    for R in (3, 4, 10, 16, 32, 64, 136):
        U = [rng.random((d, R)).astype(np.float32) for d in dims]
        Ud = [torch.from_numpy(u).to(cuda) for u in U]
        ref = O.mttkrp_coo_f64(inds, vals, 0, U)
        out = torch.full((rows, R), 5.0, device=cuda)
        assert rel(mmcsf.mttkrp(f, 0, Ud, out=out).cpu().numpy(), ref) < 1e-5, R
        if R % 4 == 0:
            # bfloat16 rows at 16 and (accepted, per-group kernel) 8 byte boundaries
            Ub = [u.to(torch.bfloat16) for u in Ud]
            Ur = [u.float().cpu().numpy() for u in Ub]
            ref = O.mttkrp_coo_f64(inds, vals, 0, Ur)
            for off in (0, 4):
                got = mmcsf.mttkrp(f, 0, [offset_copy(u, off) for u in Ub])
                assert rel(got.cpu().numpy(), ref) < 1e-5, (R, off)


# ---- modes below the root of a tree that serves every mode ------------------------

ONE_TREE = [(9, {}), (13, {}), (14, {}), (9, {"mode_trees": False}), (13, {"mode_trees": False}),
            (14, {"mode_trees": False}), (12, {"mode_trees": False}), (12, {"mixed": True})]


@pytest.mark.parametrize("dims,skew,nnz", [
    ([40, 30, 20], [None, None, None], 1),
    ([40, 30, 20], [None, None, None], 64),
    ([300, 20, 9], [1.2, None, 1.1], 65),
    ([500, 400, 60], [1.2, 1.2, None], 20_000),
    ([3000, 1, 700], [None, None, 1.3], 4097),  # one row takes everything
    ([30, 25, 20, 15], [None, None, None, None], 129),
    ([60, 37, 25, 14], [1.1, None, 1.2, None], 12_000),
])
@pytest.mark.parametrize("fmt_type,kw", ONE_TREE)
def test_one_tree_every_mode(cuda, dims, skew, nnz, fmt_type, kw):
    import torch
    import mmcsf
    import oracle as O
    if kw.get("mixed") and (nnz < 1000 or 1 in dims):
        pytest.skip("the mixed-mode partition refuses tensors of one slice")
    rng = np.random.default_rng(nnz + fmt_type)
    inds, vals = random_tensor(rng, dims, nnz, skew)
    f = mmcsf.Format(mmcsf.Tensor.from_numpy(dims, inds, vals), fmt_type, mode=0, fbr_threshold=16, **kw)
    for R in (1, 3, 4, 10, 16, 32, 64, 136):
        U = [rng.random((d, R)).astype(np.float32) for d in dims]
        Ud = [torch.from_numpy(u).to(cuda) for u in U]
        outs, _ = mmcsf.mttkrp_allmode(f, Ud)
        for m in range(len(dims)):
            assert rel(outs[m].cpu().numpy(), O.mttkrp_coo_f64(inds, vals, m, U)) < 1e-5, (R, m)
        if R % 8 == 0:
            # bfloat16 rows at 16 byte boundaries, and, for modes below the root, at
            # 8 (per-group kernels)
            Ub = [u.to(torch.bfloat16) for u in Ud]
            Ur = [u.float().cpu().numpy() for u in Ub]
            root = f.info()["modeOrder"][0]
            for off in (0, 4):
                for m in range(len(dims)):
                    if off and (m == root or kw.get("mixed")):
                        continue
                    got = mmcsf.mttkrp(f, m, [offset_copy(u, off) for u in Ub])
                    assert rel(got.cpu().numpy(), O.mttkrp_coo_f64(inds, vals, m, Ur)) < 1e-5, (R, m, off)


@pytest.mark.parametrize("name,dims,fmt_type,kw", [("one_tree_3d", [17, 11, 9], 14, {"mode_trees": False}),
                                                   ("single_tree_4d", [9, 7, 6, 5], 12, {"mode_trees": False}),
                                                   ("mixed_3d", [17, 11, 9], 12, {"mixed": True})])
def test_version_1_caches_load(cuda, golden_dir, tmp_path, name, dims, fmt_type, kw):
    """Files of the cache's first version hold ranked-row tables where a format
    now derives level maps; they load and equal a fresh build."""
    import torch
    import mmcsf
    import oracle as O
    rng = np.random.default_rng(11)
    inds, vals = random_tensor(rng, dims, 150, [1.4] + [None] * (len(dims) - 1))
    f = mmcsf.Format.load(f"{golden_dir}/{name}_v1.fmt")
    fresh = mmcsf.Format(mmcsf.Tensor.from_numpy(dims, inds, vals), fmt_type, mode=1, fbr_threshold=4, **kw)
    assert f.info() == fresh.info()
    f.save(tmp_path / "a.fmt")
    fresh.save(tmp_path / "b.fmt")
    assert (tmp_path / "a.fmt").read_bytes() == (tmp_path / "b.fmt").read_bytes()
    U = [rng.random((d, 12)).astype(np.float32) for d in dims]
    Ud = [torch.from_numpy(u).to(cuda) for u in U]
    for m in range(len(dims)):
        assert rel(mmcsf.mttkrp(f, m, Ud).cpu().numpy(), O.mttkrp_coo_f64(inds, vals, m, U)) < 1e-5


# ---- TTM without a cleared output ---------------------------------------------------

@pytest.mark.parametrize("fibers,per_fiber", [(1, 1), (1, 64), (63, 1), (64, 1), (65, 2), (3, 4000), (5000, 1),
                                              (200_000, 1), (1000, 63), (1000, 64), (777, 65), (90, 3000)])
def test_ttm_writes_every_row(cuda, fibers, per_fiber):
    """Fibers shorter and longer than chunks, runs and blocks; the output holds
    other numbers before the call."""
    import torch
    import mmcsf
    rng = np.random.default_rng(fibers + per_fiber)
    n = fibers * per_fiber
    f = np.repeat(np.arange(fibers, dtype=np.int64), per_fiber)
    leaf = np.tile(np.arange(per_fiber, dtype=np.int64), fibers)
    dims = [(fibers - 1) // 50 + 1, 50, max(4000, per_fiber)]
    vals = (rng.random(n) + 0.25).astype(np.float32)
    t = mmcsf.Tensor.from_numpy(dims, [f // 50, f % 50, leaf], vals)
    fm = mmcsf.Format(t, 8, mode=0)
    assert fm.info()["modeOrder"] == [0, 1, 2]
    for R in (4, 32, 72):
        U = rng.random((dims[2], R)).astype(np.float32)
        Y = torch.full((fibers, R), 3.0, device=cuda)
        mmcsf.ttm(fm, torch.from_numpy(U).to(cuda), out=Y)
        want = np.einsum("fl,lr->fr", vals.astype(np.float64).reshape(fibers, per_fiber), U[:per_fiber].astype(np.float64))
        assert rel(Y.cpu().numpy(), want) < 1e-5, R


def test_ttm_large_output(cuda):
    """More than 256 MB of rows, which are written around the caches."""
    import torch
    import mmcsf
    fibers, R = 1_050_001, 64
    f = np.arange(fibers, dtype=np.int64)
    inds = [np.concatenate([f // 1000, f[:500] // 1000]), np.concatenate([f % 1000, f[:500] % 1000]),
            np.concatenate([f % 37, 40 + f[:500] % 9])]
    rng = np.random.default_rng(5)
    vals = (rng.random(fibers + 500) + 0.25).astype(np.float32)
    dims = [fibers // 1000 + 1, 1000, 2000]
    fm = mmcsf.Format(mmcsf.Tensor.from_numpy(dims, inds, vals), 8, mode=0)
    assert fm.info()["nLevel"][1] == fibers and fibers * R * 4 > 256 << 20
    U = rng.random((dims[2], R)).astype(np.float32)
    Y = torch.full((fibers, R), 3.0, device=cuda)
    mmcsf.ttm(fm, torch.from_numpy(U).to(cuda), out=Y)
    want = vals[:fibers, None].astype(np.float64) * U[inds[2][:fibers]]
    want[:500] += vals[fibers:, None].astype(np.float64) * U[inds[2][fibers:]]
    assert rel(Y.cpu().numpy(), want) < 1e-5


# ---- all modes in one launch -------------------------------------------------------

@pytest.mark.parametrize("dims,skew,nnz", [
    ([4, 3, 2], [None] * 3, 1),
    ([300, 200, 100], [None] * 3, 64),
    ([300, 1, 100], [None] * 3, 4000),
    ([5000, 70, 900], [1.2, None, 1.1], 16_384 * 8),   # a chunk per wave and more
    ([900, 800, 700], [None] * 3, 1_000_000),
    ([90, 80, 70, 60], [None] * 4, 333),
    ([900, 80, 70, 600], [1.1, None, None, 1.2], 300_000),
])
def test_allmode_in_one_launch(cuda, dims, skew, nnz):
    """All modes side by side equal each mode by itself, which goes through a
    launch of its own, and float64; outputs hold other numbers before."""
    import torch
    import mmcsf
    import oracle as O
    rng = np.random.default_rng(nnz)
    inds, vals = random_tensor(rng, dims, nnz, skew)
    f = mmcsf.Format(mmcsf.Tensor.from_numpy(dims, inds, vals), 12, fbr_threshold=128)
    for R, dt in ((4, "f32"), (10, "f32"), (32, "f32"), (32, "bf16"), (64, "bf16"), (132, "f32")):
        Ud = [torch.from_numpy(rng.random((d, R)).astype(np.float32)).to(cuda) for d in dims]
        if dt == "bf16":
            Ud = [u.to(torch.bfloat16) for u in Ud]
        outs = [torch.full((d, R), 9.0, device=cuda) for d in dims]
        mmcsf.mttkrp_allmode(f, Ud, outs=outs)
        for m in range(len(dims)):
            one = mmcsf.mttkrp(f, m, Ud)
            assert rel(outs[m].cpu().numpy(), one.cpu().numpy()) < 1e-6, (R, dt, m)
            if nnz <= 200_000 and R in (10, 32):
                ref = O.mttkrp_coo_f64(inds, vals, m, [u.float().cpu().numpy() for u in Ud])
                assert rel(outs[m].cpu().numpy(), ref) < 1e-5, (R, dt, m)


# ---- MTTKRP in passes over columns ---------------------------------------------------

@pytest.mark.parametrize("R,dt", [(64, "f32"), (65, "f32"), (66, "f32"), (67, "f32"), (68, "f32"), (72, "bf16"),
                                  (76, "bf16"), (96, "f32"), (127, "f32"), (128, "f32"), (128, "bf16"), (129, "f32"),
                                  (136, "bf16"), (140, "bf16"), (200, "bf16"), (255, "f32"), (256, "f32"),
                                  (256, "bf16")])
@pytest.mark.parametrize("dims,skew", [([800, 300, 90], [1.2, None, 1.1]),
                                       ([90, 30_000, 200, 60_000], [1.2, None, None, 1.2])])
def test_mttkrp_column_passes(cuda, dims, skew, R, dt):
    """Widths around the passes' 64 columns; the 4-D tensor's tables are past
    24 MB from R = 68 on, where R = 96, 128 and 256 go 32 columns at a time;
    bfloat16 rows go in one pass.  Trees, COO and level maps; one launch per mode and all
    modes in one."""
    import torch
    import mmcsf
    import oracle as O
    rng = np.random.default_rng(R)
    inds, vals = random_tensor(rng, dims, 9001, skew)
    t = mmcsf.Tensor.from_numpy(dims, inds, vals)
    Ud = [torch.from_numpy(rng.random((d, R)).astype(np.float32)).to(cuda) for d in dims]
    if dt == "bf16":
        Ud = [u.to(torch.bfloat16) for u in Ud]
    U = [u.float().cpu().numpy() for u in Ud]
    ref = [O.mttkrp_coo_f64(inds, vals, m, U) for m in range(len(dims))]
    for fmt_type, kw in ((12, {}), (14, {"mode_trees": False}), (12, {"mixed": True})):
        f = mmcsf.Format(t, fmt_type, fbr_threshold=64, **kw)
        outs, _ = mmcsf.mttkrp_allmode(f, Ud)
        for m in range(len(dims)):
            assert rel(outs[m].cpu().numpy(), ref[m]) < 1e-5, (fmt_type, m)
            assert rel(mmcsf.mttkrp(f, m, Ud).cpu().numpy(), ref[m]) < 1e-5, (fmt_type, m)
    for fmt_type in (3, 8, 10):
        f = mmcsf.Format(t, fmt_type, mode=1)
        assert rel(mmcsf.mttkrp(f, 1, Ud).cpu().numpy(), ref[1]) < 1e-5, fmt_type


# ---- CP-ALS row solve and Gram on float64 matrix instructions -----------------------

@pytest.mark.parametrize("dims", [[513, 512, 17], [511, 64, 65], [1025, 33, 15], [131_073, 40, 30]])
@pytest.mark.parametrize("R", [4, 12, 16, 20, 28, 32])
def test_cpd_row_solve_edges(cuda, dims, R):
    """Rows at the edges of 16-row tiles, 64-row waves, 512-row spans and of a
    second round of spans; one and two column tiles, full and partial.  Bounds of
    test_gpu_cpd.py: fits within 1e-4 of the float64 ALS, the model on the
    observed entries within 1e-3."""
    import torch
    import mmcsf
    from oracle import dense as D
    from test_gpu_cpd import planted_tensor
    rng = np.random.default_rng(R + dims[0])
    inds, vals = planted_tensor(rng, dims, 40_000, R)
    U0 = [(rng.random((d, R)) * 6 - 3).astype(np.float32) for d in dims]
    fmt = mmcsf.Format(mmcsf.Tensor.from_numpy(dims, inds, vals), 12, fbr_threshold=128)
    iters = 4
    Ud = [torch.from_numpy(u.copy()).to(cuda) for u in U0]
    lam, st = mmcsf.cpd_als(fmt, Ud, iters=iters, tol=0.0)
    fits, U64, lam64 = D.cpd_als(inds, vals, dims, [u.astype(np.float64) for u in U0], iters, tol=0.0)
    np.testing.assert_allclose(st["fit_history"], fits, atol=1e-4, rtol=0)
    mg = D.cp_model_values(inds, [u.cpu().double().numpy() * (lam if m == 0 else 1.0) for m, u in enumerate(Ud)])
    m64 = D.cp_model_values(inds, [u * (lam64 if m == 0 else 1.0) for m, u in enumerate(U64)])
    assert np.linalg.norm(mg - m64) / np.linalg.norm(m64) < 1e-3
    # the allocation-free call takes the same path
    Un = [torch.from_numpy(u.copy()).to(cuda) for u in U0]
    lamn, stn = mmcsf.cpd_als(fmt, Un, iters=iters, tol=0.0, no_alloc=True)
    np.testing.assert_allclose(stn["fit_history"], fits, atol=1e-4, rtol=0)
