"""The one-codeword-per-lane RSi16 repair by what its waves hold: clean codewords alone, irregular ones alone or
beside clean and damaged ones (the wave takes them one at a time after its own), and a last wave that is not
full; against the oracle. And the automatic choice at the counts where it changes, against the general kernel."""
import numpy as np
import pytest

from libffrs_amd import workloads as W
from oracle import oracle as O
from rsi16_words import Words

pytestmark = pytest.mark.gpu


def _repair(codec, ctx, m, e, mode):
    k, ecc, count = m.shape[1], e.shape[1], len(m)
    d = [ctx.alloc(count * k * 2), ctx.alloc(count * ecc * 2), ctx.alloc(count)]
    d[0].upload(m)
    d[1].upload(e)
    codec.set_repair_syndromes(mode)
    codec.repair_device(*d[:2], count, d[2])
    out = [np.empty_like(m), np.empty_like(e), np.empty(count, np.uint8)]
    for b, a in zip(d, out):
        b.download(a)
        b.free()
    return out


@pytest.mark.parametrize("n,ecc", [(16, 8), (1024, 8), (48, 16), (256, 32)])
def test_waves(n, ecc):
    from libffrs_amd import capi
    k = n - ecc
    print(f"waves ({n},{ecc})", flush=True)
    rng, o = np.random.default_rng(n + ecc), O.RSi16(n, ecc)
    msgs, errs, s = W.rsi16_plain(64, n, ecc, ecc // 2, seed=n)
    clean = np.concatenate([msgs, o.encode(msgs)], 1)
    damaged = clean.copy()
    W.rsi16_corrupt(damaged, errs, s)
    odd = np.array([w for s, d, w in Words(o).drops(rng) if ecc // 2 <= d + 1 < ecc - s])
    st = o.repair_batch(np.ascontiguousarray(odd[:, :k]), np.ascontiguousarray(odd[:, k:]))
    odd = odd[st != 255]
    pick = lambda a, q: a[np.arange(q) % len(a)]
    waves = [clean, np.concatenate([pick(odd, 1), clean[1:]]), pick(odd, 64),
             np.concatenate([pick(odd, 20), pick(damaged, 24), pick(clean, 20)]), damaged,
             np.concatenate([pick(clean, 63), damaged[-1:]]), pick(odd, 5)]
    cws = np.concatenate(waves)
    m, e = np.ascontiguousarray(cws[:, :k]), np.ascontiguousarray(cws[:, k:])
    ctx = capi.Context(0)
    codec = capi.RSi16Codec(ctx, n, ecc)
    got = _repair(codec, ctx, m, e, 2)
    codec.close()
    ctx.close()
    st = o.repair_batch(m, e)
    for a, b in zip(got, (m, e, st)):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("n,ecc,counts", [(1024, 16, (6144, 6145)), (128, 16, (8192, 8193)), (256, 32, (11263, 11264)),
                                          (512, 32, (18431, 18432)), (2048, 32, (8447, 8448))])
def test_lines(n, ecc, counts):
    from libffrs_amd import capi
    k, sub = n - ecc, 500
    ctx = capi.Context(0)
    codec = capi.RSi16Codec(ctx, n, ecc)
    msgs, errs, s = W.rsi16_plain(sub, n, ecc, ecc // 2 + 1, seed=n + ecc)
    cws = np.concatenate([msgs, O.RSi16(n, ecc).encode(msgs)], 1)
    W.rsi16_corrupt(cws, errs, s)
    m, e = np.ascontiguousarray(cws[:, :k]), np.ascontiguousarray(cws[:, k:])
    want = _repair(codec, ctx, m, e, 1)
    for count in counts:
        print(f"lines ({n},{ecc}) x {count}", flush=True)
        rows = np.arange(count) % sub
        for a, b in zip(_repair(codec, ctx, m[rows], e[rows], 0), want):
            assert np.array_equal(a, b[rows])
    codec.close()
    ctx.close()
