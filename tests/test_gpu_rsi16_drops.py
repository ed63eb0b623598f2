"""RSi16 repair of words whose remainders drop by more than one degree (built from their syndromes), one,
17 and many to a launch, in every mode, against the oracle: the regular steps must not finish a word whose
remainder is exactly ecc / 2 long, and Forney's numerator has all coefficients of an evaluator that is longer
than the number of steps."""
import numpy as np
import pytest

from oracle import oracle as O
from rsi16_words import Words

pytestmark = pytest.mark.gpu


def _check(n, ecc, counts, extra=()):
    from libffrs_amd import capi
    k = n - ecc
    print(f"drops ({n},{ecc})", flush=True)
    o = O.RSi16(n, ecc)
    base = np.array([w for _, _, w in Words(o).drops(np.random.default_rng(3 * n + ecc), extra)])
    wm, we = np.ascontiguousarray(base[:, :k]), np.ascontiguousarray(base[:, k:])
    wst = o.repair_batch(wm, we)
    # the general kernels give 4 or 255 where the reference's lengths run past ecc symbols and it raises
    keep = wst != 255
    base, wm, we, wst = base[keep], wm[keep], we[keep], wst[keep]
    ctx = capi.Context(0)
    codec = capi.RSi16Codec(ctx, n, ecc)
    top = max(counts)
    d_m, d_p, d_s = ctx.alloc(top * k * 2), ctx.alloc(top * ecc * 2), ctx.alloc(top)
    for count in counts:
        for first in range(0, len(base), count):
            idx = (first + np.arange(count)) % len(base)
            for mode in (0, 1, 2):
                codec.set_repair_syndromes(mode)
                d_m.upload(np.ascontiguousarray(base[idx, :k]))
                d_p.upload(np.ascontiguousarray(base[idx, k:]))
                codec.repair_device(d_m, d_p, count, d_s)
                m, e, st = np.empty((count, k), np.uint16), np.empty((count, ecc), np.uint16), np.empty(count, np.uint8)
                d_m.download(m)
                d_p.download(e)
                d_s.download(st)
                bad = np.nonzero((st != wst[idx]) | (m != wm[idx]).any(1) | (e != we[idx]).any(1))[0]
                assert bad.size == 0, (count, mode, idx[bad[:8]], st[bad[:8]], wst[idx[bad[:8]]])
    for b in (d_m, d_p, d_s):
        b.free()
    codec.close()
    ctx.close()


@pytest.mark.parametrize("n,ecc,counts", [(128, 64, (1, 17, 3000)), (384, 128, (1, 17, 20000)), (512, 256, (1, 17, 1100))])
def test_evaluator_longer_than_the_steps(n, ecc, counts):
    _check(n, ecc, counts)


@pytest.mark.parametrize("n,ecc,counts", [(16, 8, (1, 70000)), (1024, 8, (17, 2000)), (64, 16, (1, 30000)),
                                          (96, 32, (17, 20000)), (256, 32, (1, 17000))])
def test_remainder_of_half_the_parity(n, ecc, counts):
    _check(n, ecc, counts, extra=range(1, ecc // 2))


def test_remainder_of_half_the_parity_found_word():
    """A word beyond the radius of RSi16(1024,8) whose remainder is 4 long after three steps: the oracle finds
    no location."""
    from libffrs_amd import capi
    n, ecc, count = 1024, 8, 2048
    k = n - ecc
    cw = np.zeros(n, np.uint16)
    cw[:8] = (7139, 55613, 11942, 57933, 12862, 37347, 12777, 45739)
    m, e = cw[:k].copy(), cw[k:].copy()
    assert O.RSi16(n, ecc).repair(m, e) == 4 and np.array_equal(np.r_[m, e], cw)
    ctx = capi.Context(0)
    codec = capi.RSi16Codec(ctx, n, ecc)
    d_m, d_p, d_s = ctx.alloc(count * k * 2), ctx.alloc(count * ecc * 2), ctx.alloc(count)
    for mode in (0, 1, 2):
        codec.set_repair_syndromes(mode)
        d_m.upload(np.tile(cw[:k], (count, 1)))
        d_p.upload(np.tile(cw[k:], (count, 1)))
        codec.repair_device(d_m, d_p, count, d_s)
        m, e, st = np.empty((count, k), np.uint16), np.empty((count, ecc), np.uint16), np.empty(count, np.uint8)
        d_m.download(m)
        d_p.download(e)
        d_s.download(st)
        assert (st == 4).all() and (m == cw[:k]).all() and (e == cw[k:]).all(), mode
    for b in (d_m, d_p, d_s):
        b.free()
    codec.close()
    ctx.close()


def test_plan_with_irregular_words():
    """The plan kernels, which leave irregular steps to the transforms, on the same words."""
    from libffrs_amd import capi
    codes = [(16, 8), (64, 16), (256, 32), (128, 64), (256, 128), (512, 256)]
    ws, wants, sts, shape = [], [], [], []
    for n, ecc in codes:
        o = O.RSi16(n, ecc)
        base = np.array([w for _, _, w in Words(o).drops(np.random.default_rng(7 * n + ecc))])
        wm, we = np.ascontiguousarray(base[:, :n - ecc]), np.ascontiguousarray(base[:, n - ecc:])
        st = o.repair_batch(wm, we)
        for i in np.nonzero(st != 255)[0]:
            ws.append(base[i])
            wants.append(np.r_[wm[i], we[i]])
            sts.append(st[i])
            shape.append((n, ecc))
    print(f"plan of {len(ws)} irregular words", flush=True)
    n, ecc = np.array(shape).T
    k = n - ecc
    mo, eo = np.r_[0, np.cumsum(k)], np.r_[0, np.cumsum(ecc)]
    ctx = capi.Context(0)
    plan = capi.RSi16Plan(ctx, n, ecc, mo[:-1], eo[:-1])
    d_m, d_e, d_s = ctx.alloc(2 * int(mo[-1])), ctx.alloc(2 * int(eo[-1])), ctx.alloc(len(ws))
    d_m.upload(np.concatenate([w[:a] for w, a in zip(ws, k)]))
    d_e.upload(np.concatenate([w[a:] for w, a in zip(ws, k)]))
    plan.repair(d_m, d_e, d_s)
    m, e, st = np.empty(int(mo[-1]), np.uint16), np.empty(int(eo[-1]), np.uint16), np.empty(len(ws), np.uint8)
    for b, a in zip((d_m, d_e, d_s), (m, e, st)):
        b.download(a)
        b.free()
    plan.close()
    ctx.close()
    bad = [i for i, w in enumerate(wants) if st[i] != sts[i] or
           not np.array_equal(np.r_[m[mo[i]:mo[i + 1]], e[eo[i]:eo[i + 1]]], w)]
    assert not bad, [(shape[i], st[i], sts[i]) for i in bad[:8]]
