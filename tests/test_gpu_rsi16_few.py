"""The one-launch RSi16 repair of a few codewords (ecc_len 64 to 256): clean and damaged words, words whose
remainders drop by more than one degree or that the general code solves, on aligned and unaligned buffers, against
the oracle; and the automatic choice at the counts where it ends, against the general kernel."""
import numpy as np
import pytest

from libffrs_amd import workloads as W
from oracle import oracle as O
from rsi16_words import Words

pytestmark = pytest.mark.gpu


class View:
    def __init__(self, buf, offset):
        self.ptr = buf.ptr + offset


def _repair(codec, ctx, m, e, mode, offset=0):
    k, ecc, count = m.shape[1], e.shape[1], len(m)
    from libffrs_amd import capi
    d = [ctx.alloc(m.nbytes + 64), ctx.alloc(e.nbytes + 64), ctx.alloc(count)]
    v = [View(d[0], offset), View(d[1], offset), View(d[2], 0)]
    out = [np.empty_like(m), np.empty_like(e), np.empty(count, np.uint8)]
    for x, a in zip(v, (m, e)):
        capi.check(capi.lib().ffrs_memcpy_h2d(ctx.h, x.ptr, a.ctypes.data, a.nbytes), "h2d")
    codec.set_repair_syndromes(mode)
    codec.repair_device(*v[:2], count, v[2])
    for x, a in zip(v, out):
        capi.check(capi.lib().ffrs_memcpy_d2h(ctx.h, a.ctypes.data, x.ptr, a.nbytes), "d2h")
    for b in d:
        b.free()
    return out


@pytest.fixture
def ctx():
    from libffrs_amd import capi
    c = capi.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("n,ecc", [(128, 64), (192, 64), (2048, 64), (256, 128), (896, 128), (8192, 128), (512, 256),
                                   (768, 256), (4096, 256)])
def test_few(ctx, n, ecc):
    from libffrs_amd import capi
    k, o, rng = n - ecc, O.RSi16(n, ecc), np.random.default_rng(n + ecc)
    w = Words(o)
    print(f"few ({n},{ecc})", flush=True)
    msgs, errs, s = W.rsi16_plain(40, n, ecc, ecc // 2 + 2, seed=n + 1)
    cws = np.concatenate([msgs, o.encode(msgs)], 1)
    clean = cws[:4].copy()
    W.rsi16_corrupt(cws, errs, s)
    odd = [x for i, (_, _, x) in enumerate(w.drops(rng)) if n < 1000 or i % 5 == 0]
    for a in (1, ecc // 2, ecc):              # the last syndromes zero, and all but a few
        S = rng.integers(0, 65537, ecc)
        S[ecc - a:] = 0
        odd.append(w.with_syndromes(S, rng))
        odd.append(w.with_syndromes(np.where(np.arange(ecc) < a, 0, rng.integers(1, 65537, ecc)), rng))
    cws = np.concatenate([clean, cws, odd])
    m, e = np.ascontiguousarray(cws[:, :k]), np.ascontiguousarray(cws[:, k:])
    st = o.repair_batch(m, e)
    keep = np.nonzero(st != 255)[0]           # where the reference raises: as the general kernel, below
    codec = capi.RSi16Codec(ctx, n, ecc)
    general = _repair(codec, ctx, np.ascontiguousarray(cws[:, :k]), np.ascontiguousarray(cws[:, k:]), 1)
    for size, offset in ((1, 0), (16, 0), (16, 2), (len(cws), 2 if n > 2048 else 0)):
        for b in range(0, len(cws), size):
            got = _repair(codec, ctx, np.ascontiguousarray(cws[b:b + size, :k]), np.ascontiguousarray(cws[b:b + size, k:]),
                          0, offset)
            for g, x, y in zip(got, (m, e, st), general):
                at = keep[(keep >= b) & (keep < b + size)]
                assert np.array_equal(g[at - b], x[at]) and np.array_equal(g, y[b:b + size]), (size, b)
    codec.close()


@pytest.mark.parametrize("n,ecc,counts", [(128, 64, (8192, 8193)), (1024, 64, (1024, 1025)), (1024, 128, (2048, 2049)),
                                          (4096, 128, (16, 17)), (512, 256, (1024, 1025)), (8192, 256, (256, 257))])
def test_lines(ctx, n, ecc, counts):
    from libffrs_amd import capi
    k, sub = n - ecc, 200
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
