"""Blocks with a NaN among their entries beside regular ones: the pivot search takes no NaN while a number is
left, so the elimination ends at the first column whose remaining rows are all NaN (or zero); info names that
column, the block is zeroed and the other members are untouched.  An infinite pivot is an ordinary one with
reciprocal zero: its row and column of the inverse are zero and the rest is the inverse without them."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 31, 32, 33, 63, 64, 65, 96, 97, 128, 160, 255, 257, 384, 385]


@pytest.fixture(scope="module")
def qt():
    from quantum_transport_amd import rgf

    rgf.init(0)
    return rgf


def _info(A):
    """First column (1-based) without a pivot in unblocked Gauss-Jordan by components: the largest |re| + |im|
    among the rows not yet taken, a NaN never; 0 if every column has one."""
    n = len(A)
    re, im = A.real.copy(), A.imag.copy()
    left = np.ones(n, bool)
    with np.errstate(all="ignore"):
        for j in range(n):
            key = np.where(left, np.abs(re[:, j]) + np.abs(im[:, j]), -1.0)
            if not np.fmax.reduce(key) > 0.0:
                return j + 1
            p = int(np.nanargmax(key))
            left[p] = False
            x, y = re[p, j], im[p, j]
            if abs(x) >= abs(y):
                r = y / x
                d = x + y * r
                dx, dy = 1.0 / d, -r / d
            else:
                r = x / y
                d = y + x * r
                dx, dy = r / d, -1.0 / d
            gx, gy = re[:, j] * dx - im[:, j] * dy, re[:, j] * dy + im[:, j] * dx
            ur, ui = re[p].copy(), im[p].copy()
            re -= np.outer(gx, ur) - np.outer(gy, ui)
            im -= np.outer(gx, ui) + np.outer(gy, ur)
            re[:, j], im[:, j] = -gx, -gy
            re[p], im[p], re[p, j], im[p, j] = ur, ui, 1.0, 0.0
    return 0


def _blocks(n):
    rng = np.random.default_rng(n)
    blk = lambda: rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n)) + 4.0 * np.sqrt(n) * np.eye(n)
    bad = {}
    for name, r, c in (("first", 0, 0), ("last", n - 1, n - 1), ("inside", n // 2, n // 3), ("corner", n - 1, 0)):
        bad[name] = blk()
        bad[name][r, c] = np.nan
    for name, at in (("row", np.s_[n // 2]), ("column", np.s_[:, n // 2]), ("lanes 16-31", np.s_[16:32]),
                     ("all", np.s_[:])):
        bad[name] = blk()
        bad[name][at] = np.nan
    bad["imaginary part"] = blk()
    bad["imaginary part"][n // 3, n // 2] = complex(1.0, np.nan)
    if n <= 16:
        del bad["lanes 16-31"]
    if n > 1:
        bad["tiny pivots"] = blk() * 1e-312  # their reciprocals overflow
    return blk, bad


@pytest.mark.parametrize("n", SIZES)
def test_blocks_with_nan(qt, n):
    blk, bad = _blocks(n)
    A = []
    for B in bad.values():
        A += [blk(), B]
    A = np.stack(A + [blk()])
    regular = A.copy()
    regular[1::2] = [blk() for _ in bad]
    print("n", n, "blocks with NaN", len(bad), flush=True)
    X, info = qt.invert_batched(A)
    ref, ref_info = qt.invert_batched(regular)
    assert not ref_info.any()
    assert np.array_equal(X[0::2], ref[0::2]) and not info[0::2].any()
    for i, (name, B) in enumerate(bad.items()):
        want = _info(B)
        assert want > 0 and info[2 * i + 1] == want, name
        assert not X[2 * i + 1].any(), name


@pytest.mark.parametrize("n", SIZES)
def test_infinite_pivot(qt, n):
    rng = np.random.default_rng(n)
    blk = lambda: (rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))
                   + (8.0 + 4.0 * np.sqrt(n)) * np.eye(n))  # every column's pivot is its diagonal entry
    where = [(r, v) for r in sorted({0, n // 2, n - 1})
             for v in (complex(np.inf, 1.0), complex(-1.0, -np.inf), complex(-np.inf, 0.0))]
    A = np.stack([blk() for _ in where] + [blk()])
    for b, (r, v) in enumerate(where):
        A[b, r, r] = v
    print("n", n, "blocks with an infinite pivot", len(where), flush=True)
    X, info = qt.invert_batched(A)
    assert not info.any()
    assert np.array_equal(X[-1], qt.invert_batched(A[-1:])[0][0])
    for b, (r, v) in enumerate(where):
        assert not X[b, r].any() and not X[b, :, r].any(), (r, v)
        rest = np.delete(np.arange(n), r)
        a, x = A[b][np.ix_(rest, rest)], X[b][np.ix_(rest, rest)]
        bound = 8 * n * np.finfo(float).eps * np.linalg.norm(a) * np.linalg.norm(x)
        assert n == 1 or np.abs(a @ x - np.eye(n - 1)).max() <= bound, (r, v)
