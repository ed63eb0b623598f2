"""RS256 repair of small launches (one codeword per wave) and of every ecc_len <= 32 in the pipeline
(Berlekamp-Massey unrolled for the next of 2, 4, 8, 16, 24, 32), against the one-codeword-per-lane
kernel and, on a sample, the oracle: message lengths around the wave's runs of eight positions, error
counts from none to beyond the radius, and counts on both sides of the line between the two."""
import numpy as np
import pytest

from libffrs_amd import workloads as W

pytestmark = pytest.mark.gpu

CASES = [(e, k, 257) for e in (1, 2, 3, 4, 5, 7, 8, 9, 12, 15, 16, 17, 21, 23, 24, 25, 31, 32)
         for k in (1, 8, 61, 255 - e)] + [(32, 223, 12288), (32, 223, 12289), (21, 130, 12289), (3, 9, 12289)]


@pytest.mark.parametrize("ecc,k,count", CASES)
def test_small_and_pipeline_repairs_agree(ecc, k, count):
    from libffrs_amd import capi
    from oracle import oracle as O
    n = k + ecc
    s = W.Stream(31 * ecc + k + count)
    msgs = s.bytes(count * k).reshape(count, k)
    counts = np.minimum(s.ints(0, ecc // 2 + 3, count), n)
    print(f"rs256 small ({n},{k}) x {count}", flush=True)
    ctx = capi.Context(0)
    codec = capi.RS256Codec(ctx, ecc)
    d_m, d_p, d_s = ctx.alloc(msgs.nbytes), ctx.alloc(count * ecc), ctx.alloc(count)
    try:
        d_m.upload(msgs)
        codec.encode_device(k, d_m, count, d_p)
        par = np.empty((count, ecc), np.uint8)
        d_p.download(par)
        cws = np.concatenate([msgs, par], 1)
        W.rs256_corrupt(cws, counts, s)
        outs = []
        for mode in (2, 1, 0):
            codec.set_repair_mode(mode)
            d_m.upload(np.ascontiguousarray(cws[:, :k]))
            d_p.upload(np.ascontiguousarray(cws[:, k:]))
            codec.repair_device(k, d_m, d_p, count, d_s)
            m, e, st = np.empty((count, k), np.uint8), np.empty((count, ecc), np.uint8), np.empty(count, np.uint8)
            d_m.download(m)
            d_p.download(e)
            d_s.download(st)
            outs.append((m, e, st))
        for o in outs[1:]:
            for a, b in zip(outs[0], o):
                assert (a == b).all()
        rows = np.r_[0:40, count - 8:count]
        m, e = np.ascontiguousarray(cws[rows, :k]), np.ascontiguousarray(cws[rows, k:])
        st = O.RS256(ecc).decode_batch(m, e)
        assert (st == outs[2][2][rows]).all() and (m == outs[2][0][rows]).all() and (e == outs[2][1][rows]).all()
    finally:
        for b in (d_m, d_p, d_s):
            b.free()
        codec.close()
        ctx.close()
