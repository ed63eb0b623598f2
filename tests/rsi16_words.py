"""RSi16 words with chosen syndromes. S = Omega / Lambda mod x^ecc for a locator Lambda of s positions
and an evaluator Omega of degree d: the remainder sequence of x^ecc and S drops from degree ecc - s to d
after s regular steps. Random damage meets a drop of more than one degree about once in 65,537 words."""
import numpy as np

P = 65537


def inv(a):
    return pow(int(a), P - 2, P)


def _inverse(M):
    """Inverse of a square matrix mod P (Gauss-Jordan)."""
    E = M.shape[0]
    A = np.concatenate([M % P, np.eye(E, dtype=np.int64)], 1)
    for c in range(E):
        piv = c + int(np.nonzero(A[c:, c])[0][0])
        if piv != c:
            A[[c, piv]] = A[[piv, c]]
        A[c] = A[c] * inv(A[c, c]) % P
        f = A[:, c].copy()
        f[c] = 0
        A = (A - f[:, None] * A[c]) % P
    return A[:, E:]


class Words:
    """Words of one RSi16(n, ecc); `oracle` is its oracle codec."""

    def __init__(self, oracle):
        self.o = oracle
        self.n, self.E = oracle.block_len, oracle.ecc_len
        self.k = self.n - self.E
        roots, bits = oracle.table("roots_ntt").astype(np.int64), oracle.ntt_len.bit_length() - 1
        rbo = [int(format(m, f"0{bits}b")[::-1], 2) for m in range(self.n)]
        self.X = roots[rbo]                           # locator of position m
        V = np.ones((self.E, self.E), np.int64)       # syndromes of the parity symbols
        for j in range(1, self.E):
            V[j] = V[j - 1] * self.X[self.k:] % P
        self.Vi = _inverse(V)

    def with_syndromes(self, S, rng):
        """A word of random message symbols whose syndromes are S."""
        S = np.asarray(S, np.int64)
        zero = np.zeros(self.E, np.uint16)
        while True:
            msg = rng.integers(0, 65536, self.k).astype(np.uint16)
            rhs = (S - self.o.synds(msg, zero)) % P
            par = np.zeros(self.E, np.int64)
            for b in range(0, self.E, 64):            # sums of 64 products stay below 2^63
                par = (par + self.Vi[:, b:b + 64] @ rhs[b:b + 64]) % P
            if (par != 65536).all():
                cw = np.r_[msg, par.astype(np.uint16)]
                assert np.array_equal(self.o.synds(cw[:self.k].copy(), cw[self.k:].copy()), S)
                return cw

    def syndromes(self, positions, omega):
        """Omega / prod (1 - X_p x) mod x^ecc."""
        lam = [1]
        for p in positions:
            x = int(self.X[p])
            lam = [(a - x * b) % P for a, b in zip(lam + [0], [0] + lam)]
        S = []
        for j in range(self.E):
            v = int(omega[j]) if j < len(omega) else 0
            S.append((v - sum(lam[i] * S[j - i] for i in range(1, min(j, len(lam) - 1) + 1))) % P)
        return S

    def drop(self, s, d, rng, dense=True):
        """Syndromes with s locator positions and an evaluator of degree d."""
        pos = rng.choice(self.n, s, replace=False)
        omega = rng.integers(1, P, d + 1)
        if not dense:
            omega[1:d] = 0
        return self.syndromes(pos, omega)

    def drops(self, rng, extra=()):
        """(s, d, word) over the steps s and degrees d where a solver's rules can part: within the radius
        (d < s), coefficients in one more block of eight than the steps, remainders just below, at and above
        ecc / 2, and no drop at all."""
        T, E = self.E // 2, self.E
        for s in sorted({1, 2, 3, T // 4, T // 2, T - 2, T - 1} | set(extra)):
            if not 1 <= s < T:
                continue
            r8 = -(-s // 8) * 8
            for d in sorted({s - 1, s, r8 - 1, r8, T // 2, T - 3, T - 2, T - 1, T, T + 1, E - 2 - s, E - 1 - s}):
                if s - 1 <= d <= E - 1 - s:
                    yield s, d, self.with_syndromes(self.drop(s, d, rng, dense=(s + d) % 2 == 0), rng)
