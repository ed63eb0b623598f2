"""The int8 MFMA contractions of RSi16 (encode and syndromes) at the edges of their tiles: 16 and 64
codewords per workgroup, partial and single groups, every output-tile split (ecc_len 16 to 256),
messages that are no whole number of 64-symbol chunks, and both launch shapes (from 64 codewords per
CU on). The parity must equal the butterfly kernels' and, on a sample, the oracle's; a repair with
contracted syndromes must equal the one that computes them in the repair kernel."""
import numpy as np
import pytest

from libffrs_amd import workloads as W

pytestmark = pytest.mark.gpu

SHAPES = [(48, 16), (96, 32), (192, 64), (384, 128), (512, 256), (4096, 256)]


def _counts(n):
    big = [64 * 256 + 1] if n <= 512 else []  # 64 codewords per workgroup on 256 CUs, and one more
    return [1, 15, 17, 64, 65] + big


@pytest.mark.parametrize("n,ecc", SHAPES)
def test_contraction_tiles(n, ecc):
    from libffrs_amd import capi
    from oracle import oracle as O
    k = n - ecc
    ctx = capi.Context(0)
    codec = capi.RSi16Codec(ctx, n, ecc)
    try:
        for count in _counts(n):
            print(f"contraction ({n},{ecc}) x {count}", flush=True)
            msgs, errs, s = W.rsi16_plain(count, n, ecc, ecc // 2, seed=5 + n + count)
            msgs[count // 2] = 65535
            msgs[count - 1, ::2] = 0
            d_m, d_p, d_s = ctx.alloc(msgs.nbytes), ctx.alloc(count * ecc * 2), ctx.alloc(count)
            d_m.upload(msgs)
            par = []
            for kernel in (1, 2):
                codec.set_encode_kernel(kernel)
                codec.encode_device(d_m, count, d_p, False)
                o = np.empty((count, ecc), np.uint16)
                d_p.download(o)
                par.append(o)
            assert (par[0] == par[1]).all()
            rows = np.unique([0, count // 2, count - 1])
            assert (O.RSi16(n, ecc).encode(np.ascontiguousarray(msgs[rows]), vector_lanes=False) == par[1][rows]).all()
            cws = np.concatenate([msgs, par[1]], 1)
            W.rsi16_corrupt(cws, errs, s)
            outs = []
            for mode in (1, 2):
                codec.set_repair_syndromes(mode)
                d_m.upload(np.ascontiguousarray(cws[:, :k]))
                d_p.upload(np.ascontiguousarray(cws[:, k:]))
                codec.repair_device(d_m, d_p, count, d_s)
                m, e, st = np.empty((count, k), np.uint16), np.empty((count, ecc), np.uint16), np.empty(count, np.uint8)
                d_m.download(m)
                d_p.download(e)
                d_s.download(st)
                outs.append((m, e, st))
            for a, b in zip(*outs):
                assert (a == b).all()
            for b in (d_m, d_p, d_s):
                b.free()
    finally:
        codec.close()
        ctx.close()
