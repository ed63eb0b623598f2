"""The arithmetic of the RSi16 int8 MFMA contractions with two signed byte limbs (parity and syndromes,
rsi16_contract_kernel) and of the root search (rsi16_repair_lane_kernel, rsi16_roots_wave_kernel), restated
in numpy and checked on the CPU: the limbs and the residue they miss, the scale of each output row, the sums'
bounds in int32, contract_value over its whole range, and the values against the oracle."""
import numpy as np
import pytest

from oracle import oracle as O
from rsi16_words import P, Words, inv

MISSED = 32640


def fold16(x):
    return (x & 0xFFFF) - (x >> 16)


def limbs(g):
    """Signed byte limbs of canonical residues other than MISSED."""
    assert (g != MISSED).all()
    v = np.where(g > 32639, g - P, g)
    lo = ((v + 128) & 255) - 128
    return lo, (v - lo) >> 8


def contract_value(p0, p1, sinv):
    t = p0 + 256 * fold16(p1)
    assert (np.abs(t) < 2 ** 31).all()
    f = fold16(fold16(t))
    assert (np.abs(f * sinv) < 2 ** 31).all()
    r = fold16(fold16(f * sinv))
    return r + np.where(r < 0, P, 0)


def scales(mat):
    """Per column the first power of 3 that keeps its entries off MISSED and whose inverse has a sign bit free."""
    third, out = inv(3), []
    for col in mat.T:
        s, si = 1, 1
        while (col == MISSED * si % P).any() or si in (32768, P - 32768):
            s, si = s * 3 % P, si * third % P
        out.append((s, si - P if si > 32768 else si))
    return np.array(out, np.int64).T


def contract(mat, sym):
    """sym [N, rows] u16 symbols, mat [rows, E] -> canonical sum_m sym mat mod P, as the kernel computes it."""
    s, si = scales(mat)
    g = mat * s % P
    g0, g1 = limbs(g)
    assert all((np.abs(x + 0.5) <= 127.5).all() for x in (g0, g1))
    y0, y1 = (sym & 255) - 128, (sym >> 8) - 128
    K = (g * (128 * 257) + g1).sum(0) % P
    p0 = y0 @ g0 + ~y1 @ g1 + K
    p1 = y1 @ g0 + y0 @ g1
    assert np.abs(p0).max() < 2 ** 30 and np.abs(p1).max() < 2 ** 30
    return contract_value(p0, p1, si)


def test_limbs_reach_every_residue_but_one():
    g = np.delete(np.arange(P), MISSED)
    lo, hi = limbs(g)
    assert lo.min() == -128 and lo.max() == 127 and hi.min() == -128 and hi.max() == 127
    assert ((256 * hi + lo - g) % P == 0).all()
    pairs = (256 * np.arange(-128, 128)[:, None] + np.arange(-128, 128)).ravel() % P
    assert not (pairs == MISSED).any() and np.unique(pairs).size == P - 1


def test_contract_value_over_its_range():
    rng = np.random.default_rng(1)
    edge = np.array([-2 ** 30 + 1, -65537, -65536, -1, 0, 1, 65535, 65536, 65537, 2 ** 30 - 1])
    v = np.r_[edge, rng.integers(-2 ** 30 + 1, 2 ** 30, 3000)]
    s = np.r_[1, -1, 32767, -32767, rng.integers(-32767, 32768, 60)]
    p0, p1 = np.meshgrid(v, v[::37])
    for si in s:
        assert (contract_value(p0, p1, si) == (p0 + 256 * p1) * si % P).all()


@pytest.mark.parametrize("n,ecc", [(24, 8), (256, 8), (208, 16), (256, 32), (512, 64), (640, 128)])
def test_parity_and_syndromes(n, ecc):
    o = O.RSi16(n, ecc)
    w, rng, k = Words(o), np.random.default_rng(n + ecc), n - ecc
    V = np.ones((n, ecc), np.int64)                     # row m: X_m^j
    for j in range(1, ecc):
        V[:, j] = V[:, j - 1] * w.X % P
    msgs = np.concatenate([rng.integers(0, 65536, (40, k)), np.zeros((1, k), np.int64), np.full((1, k), 65535),
                           np.arange(k)[None] % 2 * 65535, np.full((1, k), 32768), np.full((1, k), 255)])
    par = rng.integers(0, 65536, (len(msgs), ecc))
    syn = contract(V, np.concatenate([msgs, par], 1))
    for s, m, e in zip(syn, msgs, par):
        assert np.array_equal(s, o.synds(m.astype(np.uint16), e.astype(np.uint16)))
    G = np.array([-(w.Vi @ row % P) % P for row in V[:k]])   # the parity that cancels the unit message at m
    assert np.array_equal(contract(G, msgs) & 0xFFFF, o.encode(msgs.astype(np.uint16), vector_lanes=False))


def test_scaled_rows():
    """Columns that hold the missed residue, and ones whose next scales meet it or a forbidden inverse again."""
    rng = np.random.default_rng(5)
    third = inv(3)
    mat = rng.integers(0, P, (192, 16))
    for j in range(8):
        for t in range(j + 1):
            mat[t, j] = MISSED * pow(third, t, P) % P
    sym = rng.integers(0, 65536, (30, 192))
    sym[0], sym[1] = 65535, 0
    assert (scales(mat)[0] != 1).sum() >= 8
    want = np.array([[sum(int(a) * int(b) for a, b in zip(r, c)) % P for c in mat.T] for r in sym])
    assert np.array_equal(contract(mat, sym), want)


@pytest.mark.parametrize("n,ecc", [(16, 8), (1024, 16), (256, 32), (128, 64), (1024, 128), (512, 256)])
def test_root_search(n, ecc):
    w, T = Words(O.RSi16(n, ecc)), ecc // 2
    rng = np.random.default_rng(3 * n + ecc)
    third = inv(3)
    xi = np.array([inv(x) for x in w.X], np.int64)
    M = np.ones((T, n), np.int64) * (xi * third % P)
    for i in range(1, T):
        M[i] = M[i - 1] * M[0] % P
    g0, g1 = limbs(M)                                   # never the missed residue
    pow3 = np.array([pow(3, i, P) for i in range(1, T + 1)], np.int64)
    for roots in (0, 1, T // 2, T):
        loc = [int(rng.integers(1, P))]
        for p in rng.choice(n, roots, replace=False):
            loc = [(a - int(w.X[p]) * b) % P for a, b in zip(loc + [0], [0] + loc)]
        a = np.array(loc + [0] * (T + 1 - len(loc)), np.int64)
        while a[0] == 65536 or (a[1:] * pow3 % P == MISSED).any():
            a = a * 3 % P                               # another multiple has the same roots
        v0, v1 = limbs(a[1:] * pow3 % P)
        p0 = v0 @ g0 + ~v1 @ g1 + g1.sum(0) + a[0]
        p1 = v1 @ g0 + v0 @ g1
        assert np.abs(p1).max() <= 2 ** 22 and np.abs(p0 + 256 * p1).max() < 2 ** 31
        f = fold16(fold16(p0 + 256 * p1))
        at = np.zeros(n, np.int64)
        for c in a[::-1]:
            at = (at * xi + c) % P
        assert np.array_equal(f % P, at) and np.array_equal(f == 0, at == 0) and (f == 0).sum() == roots
