"""The three-term quotient of the RSi16 Sugiyama solver in coefficient form (pr_sugiyama's q_len == 3
step), restated in plain Python, against NTT::poly_div_ntt (ntt.hpp:363-564) through its transforms,
over every divisor length that step meets, on random and sparse polynomials, also ones with
coefficients at and above their lengths (which the cyclic products read)."""
import random

import pytest

from test_sugiyama_forms import Code, P, add, inttr, inv, mul, nttr, poly_div, sub


def three_term(E, f, f_len, g, g_len, f0):
    mask = E - 1
    a0 = inv(g[g_len - 1])
    v = [g[(g_len - 1 - j) & mask] for j in range(-2, 3)]
    c1 = sub(0, mul(mul(a0, a0), v[3]))
    hh = [sub(2 if j == 1 else 0, add(mul(a0, v[j + 1]), mul(c1, v[j]))) for j in range(4)]
    ai = [0, 0, 0]
    for j in range(3):
        ai[2 - j] = add(mul(a0, hh[j + 1]), mul(c1, hh[j]))
    right_n = min(3, E - g_len)
    q = []
    for i in range(3):
        at = g_len + i if i < right_n else i - right_n
        s = 0
        for u in range(3):
            k = (at - u) & mask
            s = add(s, mul(ai[u], sub(f[k], f0) if k == 0 else f[k]))
        q.append(s)
    return q


@pytest.mark.parametrize("E", [8, 16, 32])
def test_three_term_quotient(E):
    C, rng = Code(E), random.Random(7 + E)
    for g_len in range(E // 2, E - 1):
        for kind in range(6):
            f_len = g_len + 2
            pick = (lambda: rng.randrange(P)) if kind % 2 == 0 else (lambda: rng.choice([0, 0, 1, P - 1, 65535]))
            f = [pick() if i < f_len or kind >= 4 else 0 for i in range(E)]
            g = [pick() if i < g_len or kind >= 4 else 0 for i in range(E)]
            f[f_len - 1] = f[f_len - 1] or 1
            g[g_len - 1] = g[g_len - 1] or 5
            Q, q_len = poly_div(C, nttr(C, f), f_len, nttr(C, g), g_len, f[0], g[g_len - 1])
            assert q_len == 3
            want = inttr(C, Q)
            assert three_term(E, f, f_len, g, g_len, f[0]) == want[:3] and not any(want[3:])
