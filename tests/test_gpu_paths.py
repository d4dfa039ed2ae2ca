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
])
def test_mode_tree_orders_follow_the_footprints(cuda, dims, skew, nnz):
    import mmcsf
    rng = np.random.default_rng(nnz)
    inds, vals = random_tensor(rng, dims, nnz, skew)
    f = mmcsf.Format(mmcsf.Tensor.from_numpy(dims, inds, vals), 12, fbr_threshold=128)
    info = f.info()
    hot = [footprint(inds[m], dims[m]) for m in range(3)]
    for m in (0, 1):
        a, b = sorted((x for x in range(3) if x != m), key=lambda x: dims[x])
        # the default order ends in b; the swapped one in a
        if 2 * hot[a] < hot[b]:
            want = [m, b, a]
        elif 2 * hot[b] < hot[a]:
            want = [m, a, b]
        else:
            # the order with fewer level-1 entries, counted with the -f 128 split
            na, nb = ([-(-c // 128) for c in np.unique(inds[m].astype(np.int64) * dims[x] + inds[x],
                                                       return_counts=True)[1]] for x in (a, b))
            na, nb = sum(na), sum(nb)
            want = [m, b, a] if nb < na else [m, a, b]
        assert info["modeTreeOrder"][m] == want, (m, hot)
