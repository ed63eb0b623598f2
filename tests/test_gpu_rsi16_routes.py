"""The automatic choice of the RSi16 repair at the counts where it changes between one codeword per
wave, the general kernel with and without given syndromes, and one codeword per lane, against the
general kernel with its own syndromes (every error count up to beyond the radius) and, on a sample,
the oracle."""
import numpy as np
import pytest

from libffrs_amd import workloads as W

pytestmark = pytest.mark.gpu

SHAPES = [(16, 2, 1025), (64, 8, 1025), (64, 8, 16385), (128, 8, 8193), (64, 16, 513), (256, 16, 2049), (512, 16, 4097),
          (512, 16, 20479), (2048, 16, 8193), (256, 32, 1025), (512, 32, 2049), (512, 32, 16383), (512, 32, 16384),
          (2048, 32, 4097), (896, 128, 16), (896, 128, 17)]


@pytest.mark.parametrize("n,ecc,count", SHAPES)
def test_automatic_repair_matches_general(n, ecc, count):
    from libffrs_amd import capi
    from oracle import oracle as O
    k = n - ecc
    print(f"automatic repair ({n},{ecc}) x {count}", flush=True)
    ctx = capi.Context(0)
    codec = capi.RSi16Codec(ctx, n, ecc)
    sub = min(count, 512)
    msgs, errs, s = W.rsi16_plain(sub, n, ecc, min(n, ecc // 2 + 2), seed=23 + n + count)
    d_m, d_p, d_s = ctx.alloc(count * k * 2), ctx.alloc(count * ecc * 2), ctx.alloc(count)
    d_m.upload(msgs)
    codec.encode_device(d_m, sub, d_p)
    par = np.empty((sub, ecc), np.uint16)
    d_p.download(par)
    cws = np.concatenate([msgs, par], 1)
    W.rsi16_corrupt(cws, errs, s)
    cws = np.tile(cws, (-(-count // sub), 1))[:count]
    outs = []
    for mode in (1, 0):
        codec.set_repair_syndromes(mode)
        d_m.upload(np.ascontiguousarray(cws[:, :k]))
        d_p.upload(np.ascontiguousarray(cws[:, k:]))
        codec.repair_device(d_m, d_p, count, d_s)
        m, e, st = np.empty((count, k), np.uint16), np.empty((count, ecc), np.uint16), np.empty(count, np.uint8)
        d_m.download(m)
        d_p.download(e)
        d_s.download(st)
        outs.append((m, e, st))
    for b in (d_m, d_p, d_s):
        b.free()
    codec.close()
    ctx.close()
    for x, y in zip(*outs):
        assert np.array_equal(x, y)
    rows = np.unique(np.r_[0:min(20, count), max(0, count - 20):count])
    m, e = np.ascontiguousarray(cws[rows, :k]), np.ascontiguousarray(cws[rows, k:])
    st = O.RSi16(n, ecc).repair_batch(m, e)
    got_m, got_e, got_s = outs[1]
    assert np.array_equal(st, got_s[rows]) and np.array_equal(m, got_m[rows]) and np.array_equal(e, got_e[rows])
