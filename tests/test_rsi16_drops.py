"""The RSi16 key-equation solvers' rules for words whose remainders drop by more than one degree, restated
in plain Python against the oracle: which words the regular steps may finish (LaneSolve, ecc_len 8 to 32,
and WaveSolve, 64 to 256: the remainder is shorter than ecc / 2), and how many evaluator coefficients the
root search of ecc_len 64 to 256 has to read (the remainder may be longer than the steps taken).
The continuation after an irregular step (WaveSolve::irregular) is restated too. The GPU tests compare the
kernels themselves."""
import numpy as np
import pytest

from oracle import oracle as O
from rsi16_words import P, Words, inv
from test_sugiyama_forms import div_ok


def length(r):
    nz = np.nonzero(r)[0]
    return int(nz[-1]) + 1 if nz.size else 0


def shift(v):
    return np.r_[0, v[:-1]]


def regular(S):
    """Steps done, then (r2, r1, a2, a1) after them."""
    E = len(S)
    T = E // 2
    S = np.asarray(S, np.int64)
    zero, one = np.zeros(E, np.int64), np.r_[1, np.zeros(E - 1, np.int64)]
    if S[E - 1] == 0:
        return 0, None
    a11 = -inv(S[E - 1]) % P
    a10 = int(S[E - 2]) * a11 * a11 % P
    r2, a2, r1, a1 = S, one, (a10 * S + a11 * shift(S)) % P, zero.copy()
    a1[:2] = a10, a11
    s = 1
    while s < T and r1[E - 1 - s]:
        g = E - s
        a0 = inv(r1[g - 1])
        w = a0 * int(r1[g - 2]) % P
        q1 = a0 * int(r2[g]) % P
        q0 = a0 * (int(r2[g - 1]) - w * int(r2[g])) % P
        r2, r1 = r1, (r2 - q0 * r1 - q1 * shift(r1)) % P
        a2, a1 = a1, (a2 - q0 * a1 - q1 * shift(a1)) % P
        s += 1
    return s, (r2, r1, a2, a1)


def irregular(s, E, r2, r1, a2, a1):
    """WaveSolve::irregular: the solved locator and evaluator, or None (left to the general code)."""
    T = E // 2
    r2_len, r1_len, a2_deg, a1_deg = E + 1 - s, length(r1), s - 1, s
    for _ in range(s + 1, T + 1):
        if r1_len < T:
            return (a1, r1) if div_ok(E, r2_len, r1_len) else None
        g = r1_len
        if r2_len >= g:
            q = r2_len - g
            if q not in (1, 2):
                return None
            at = lambda v, i: int(v[i]) if i < E else 0
            a0, v1, f0, f1 = inv(r1[g - 1]), int(r1[g - 2]), at(r2, g), int(r2[g - 1])
            if q == 1:
                n = [a0 * (f1 - a0 * v1 * f0) % P, a0 * f0 % P, 0]
            else:
                v2, up, f2 = int(r1[g - 3]), at(r2, g + 1), int(r2[g - 2])
                c1 = -a0 * a0 * v1 % P
                b0 = -a0 * (c1 * v1 + a0 * v2) % P
                n = [(b0 * f0 + c1 * f1 + a0 * f2) % P, (b0 * up + c1 * f0 + a0 * f1) % P, (c1 * up + a0 * f0) % P]
            a2_deg = max(a2_deg, a1_deg + q)
            if a2_deg > T:
                return None
            x, xa = r1, a1
            for u in n:
                r2, a2, x, xa = (r2 - u * x) % P, (a2 - u * xa) % P, shift(x), shift(xa)
        r2, r1, a2, a1, a2_deg, a1_deg = r1, r2, a1, a2, a1_deg, a2_deg
        r2_len, r1_len = r1_len, length(r1)
    return a1, r1


def lane_solve(S):
    """LaneSolve: None where the codeword is left to the general kernel."""
    E, T = len(S), len(S) // 2
    s, st = regular(S)
    if s == 0:
        return None
    r1, a1 = st[1], st[3]
    if s < T:
        high, low = r1[T - 1:E - 1 - s].any(), r1[:T].any()
        if high or not low:
            return None
    return None if a1[0] == 0 else (s, a1, r1, T)


def wave_solve(S):
    """WaveSolve: (steps, locator, evaluator, evaluator coefficients read) or None."""
    E, T = len(S), len(S) // 2
    s, st = regular(S)
    if s == 0:
        return None
    n = length(st[1]) if s < T else 0
    if s < T and n == 0:
        return None
    if n >= T:  # finished by the general code's root search, over every coefficient
        r = irregular(s, E, *st)
        return None if r is None or r[0][0] == 0 else (s, *r, E)
    return None if st[3][0] == 0 else (s, st[3], st[1], -(-max(s, n) // 8) * 8)


def evaluate(c, x):
    v = np.zeros_like(x)
    for a in c[::-1]:
        v = (v * x + int(a)) % P
    return v


def corrected(w, cw, a, r):
    """The word after Forney's corrections at the locator's roots, and its status."""
    xi = np.array([inv(x) for x in w.X], np.int64)
    out, at = cw.copy(), np.nonzero(evaluate(a, xi) == 0)[0]
    num, den = evaluate(r, xi[at]), evaluate([i * int(v) % P for i, v in enumerate(a)][1:], xi[at])
    for p, u, d in zip(at, num, den):
        q = int(u) * inv(d) % P if d else int(u) * inv(a[0]) % P
        out[p] = (int(cw[p]) + q * int(w.X[p])) % P & 0xffff
    return out, 2 if at.size else 4


@pytest.mark.parametrize("n,ecc", [(16, 8), (64, 8), (64, 16), (96, 32), (256, 32), (128, 64), (256, 128), (512, 256)])
def test_solvers_against_oracle(n, ecc):
    w, rng = Words(O.RSi16(n, ecc)), np.random.default_rng(5 * n + ecc)
    k, T, solved = n - ecc, ecc // 2, 0
    for s, d, cw in w.drops(rng):
        m, e = cw[:k].copy(), cw[k:].copy()
        S = w.o.synds(m, e)
        st = w.o.repair(m, e)
        got = lane_solve(S) if ecc <= 32 else wave_solve(S)
        if d + 1 < T:
            assert got is not None, (s, d)      # within the regular steps
        if got is None:
            continue
        solved += 1
        L, loc, ev = w.o.sugiyama(S)
        _, a, r, read = got
        f = inv(a[0])
        assert np.array_equal(a * f % P, loc) and np.array_equal(r * f % P, ev), (s, d)
        assert not r[read:].any(), (s, d)
        want = corrected(w, cw, a, r[:read])
        assert st == want[1] and np.array_equal(np.r_[m, e], want[0]), (s, d)
    assert solved > 5
