"""CIRC16's row kernels (inner ecc_len 2, 4, 8, one wave per row) and the known-position repair as a
matrix per interleave block, at the edges of their tiles: rows shorter and longer than a wave and no
multiple of it, column counts around 64, one to ecc_len error rows (message and parity rows), several
interleave blocks with different rows, and outer codes above the matrix's limit. The inner parity
must equal RSi16's; every pattern of up to ecc_len lost rows is within the code, so the repair must
restore the message and the ecc."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# inner block, inner ecc, outer block, outer ecc, interleave
SHAPES = [(6, 2, 16, 8, 1), (10, 2, 24, 8, 3), (132, 4, 32, 16, 2), (136, 8, 48, 16, 1), (264, 8, 64, 32, 2),
          (516, 4, 512, 256, 1), (20, 4, 1024, 512, 1)]


@pytest.mark.parametrize("shape", SHAPES, ids=["x".join(map(str, s)) for s in SHAPES])
def test_lost_rows_are_restored(shape):
    import libffrs_amd as L
    ib, ie, ob, oe, I = shape
    ik, ok = ib - ie, ob - oe
    rs = L.CIRC16(ib, ie, ob, oe, I)
    rng = np.random.default_rng(sum(shape))
    msg = rng.integers(0, 65536, rs.message_len).astype(np.uint16)
    ecc = np.frombuffer(bytes(rs.encode(msg.tobytes())), np.uint16)
    inner = L.RSi16(ib, ie)
    rso = oe * ik * I
    want = np.frombuffer(bytes(inner.encode(msg.tobytes())), np.uint16)
    assert (ecc[rso:rso + want.size] == want).all()
    for lost in sorted({1, 2, 7, 8, 9, oe - 1, oe}):
        if lost > oe:
            continue
        print(f"circ16 {shape} lost rows {lost}", flush=True)
        bm, be = msg.reshape(ok, I, ik).copy(), ecc.copy()
        outer = be[:rso].reshape(oe, I, ik)
        for kk in range(I):
            for row in rng.choice(ob, lost if kk == 0 else max(1, lost // 2), replace=False):
                at = bm[row, kk] if row < ok else outer[row - ok, kk]
                at[:] = (at.astype(np.int64) + rng.integers(1, 65536, ik)) % 65536
        bm, be = bytearray(bm.tobytes()), bytearray(be.tobytes())
        assert rs.repair(bm, be) is False
        got_m, got_e = np.frombuffer(bm, np.uint16), np.frombuffer(be, np.uint16)
        assert (got_m == msg).all() and (got_e == ecc).all()
