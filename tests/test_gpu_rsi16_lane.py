"""The one-codeword-per-lane RSi16 repair (ecc_len 8, 16, 32) and the automatic choice (one codeword
per wave for small launches) against the general register kernel (syndromes in the repair kernel)
and, on a sample, the oracle: every error count from none to beyond
the radius, partial waves, the smallest and largest block lengths, 0 / 65535 / constant symbols,
parity-only damage, and patterns whose remainders drop by more than one degree (left to the general
kernel)."""
import numpy as np
import pytest

from libffrs_amd import workloads as W

pytestmark = pytest.mark.gpu

SHAPES = [(16, 8, 700), (24, 8, 64), (1024, 8, 65), (32, 16, 1000), (208, 16, 129), (64, 32, 1), (96, 32, 63), (256, 32, 2017),
          (256, 32, 20000), (4096, 32, 500), (16384, 16, 100)]


def _structured(n, ecc, k):
    rows = []
    for step in (1, 2, max(2, n // ecc), ecc, n // 2):
        for start in (0, 1, k - 1, k):
            cw = np.zeros(n, np.int64)
            cw[start::step] += 1 + start % 3
            rows.append(cw)
    for a in (1, 2, ecc // 2, ecc // 2 + 1, ecc):
        cw = np.zeros(n, np.int64)
        cw[k:k + a] = 7
        rows.append(cw)
        cw = np.zeros(n, np.int64)
        cw[:a] = 65535
        rows.append(cw)
    rows.append(np.full(n, 65535))
    rows.append(np.arange(n) % 65536)
    return np.array(rows, np.uint16)


@pytest.mark.parametrize("n,ecc,count", SHAPES)
def test_lane_repair_matches_general(n, ecc, count):
    from libffrs_amd import capi
    from oracle import oracle as O
    k = n - ecc
    print(f"lane repair ({n},{ecc}) x {count}", flush=True)
    ctx = capi.Context(0)
    codec = capi.RSi16Codec(ctx, n, ecc)
    msgs, errs, s = W.rsi16_plain(count, n, ecc, min(n, ecc // 2 + 3), seed=17 + n + count)
    d_m, d_p = ctx.alloc(msgs.nbytes), ctx.alloc(count * ecc * 2)
    d_m.upload(msgs)
    codec.encode_device(d_m, count, d_p)
    par = np.empty((count, ecc), np.uint16)
    d_p.download(par)
    cws = np.concatenate([msgs, par], 1)
    W.rsi16_corrupt(cws, errs, s)
    cws = np.concatenate([cws, _structured(n, ecc, k)])
    total = cws.shape[0]
    for b in (d_m, d_p):
        b.free()
    d_m, d_p, d_s = ctx.alloc(total * k * 2), ctx.alloc(total * ecc * 2), ctx.alloc(total)
    outs = []
    for mode in (1, 2, 0):
        codec.set_repair_syndromes(mode)
        d_m.upload(np.ascontiguousarray(cws[:, :k]))
        d_p.upload(np.ascontiguousarray(cws[:, k:]))
        codec.repair_device(d_m, d_p, total, d_s)
        m, e, st = np.empty((total, k), np.uint16), np.empty((total, ecc), np.uint16), np.empty(total, np.uint8)
        d_m.download(m)
        d_p.download(e)
        d_s.download(st)
        outs.append((m, e, st))
    for b in (d_m, d_p, d_s):
        b.free()
    codec.close()
    ctx.close()
    m0, e0, s0 = outs[0]
    for m1, e1, s1 in outs[1:]:
        bad = np.nonzero((s0 != s1) | (m0 != m1).any(1) | (e0 != e1).any(1))[0]
        assert bad.size == 0, (bad[:8], s0[bad[:8]], s1[bad[:8]])
    rows = np.unique(np.r_[0:min(count, 40), count:count + 20])
    m, e = np.ascontiguousarray(cws[rows, :k]), np.ascontiguousarray(cws[rows, k:])
    st = O.RSi16(n, ecc).repair_batch(m, e)
    bad = np.nonzero((st != s1[rows]) | (m != m1[rows]).any(1) | (e != e1[rows]).any(1))[0]
    assert bad.size == 0, (rows[bad], st[bad], s1[rows[bad]], cws[rows[bad]][:4])
