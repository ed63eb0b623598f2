"""RSi16 repair for ecc_len 64 to 256 where codewords with irregular remainder sequences, repaired from
a list beside the root search, stand at the end of a launch of many workgroups: they are finished before
the workgroups that cover them start, and must not be searched again. Against the general kernel."""
import numpy as np
import pytest

from libffrs_amd import workloads as W

pytestmark = pytest.mark.gpu


def _irregular(n, k):
    rows = []
    for step in (1, 2, 4, n // 8):
        for start in (0, 1, k - 1):
            cw = np.zeros(n, np.uint16)
            cw[start::step] = 1 + start % 3
            rows.append(cw)
    for a in (1, 2, 7, 30, 31):
        cw = np.zeros(n, np.uint16)
        cw[k:k + a] = 7
        rows.append(cw)
    return np.array(rows, np.uint16)


@pytest.mark.parametrize("n,ecc,count", [(128, 64, 60000), (256, 128, 20000), (512, 256, 10000), (512, 256, 700)])
def test_listed_codewords_at_the_end(n, ecc, count):
    from libffrs_amd import capi
    k = n - ecc
    print(f"listed codewords ({n},{ecc}) x {count}", flush=True)
    ctx = capi.Context(0)
    codec = capi.RSi16Codec(ctx, n, ecc)
    sub = 512
    msgs, errs, s = W.rsi16_plain(sub, n, ecc, ecc // 2, seed=29 + n)
    d_m, d_p, d_s = ctx.alloc(count * k * 2), ctx.alloc(count * ecc * 2), ctx.alloc(count)
    d_m.upload(msgs)
    codec.encode_device(d_m, sub, d_p)
    par = np.empty((sub, ecc), np.uint16)
    d_p.download(par)
    cws = np.concatenate([msgs, par], 1)
    W.rsi16_corrupt(cws, errs, s)
    cws = np.tile(cws, (-(-count // sub), 1))[:count]
    odd = _irregular(n, k)
    cws[-200:] = np.tile(odd, (-(-200 // len(odd)), 1))[:200]
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
