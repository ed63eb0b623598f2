"""The choice between CIRC16's two known-position repairs (a matrix per interleave block, or column by column
where the rows are short and the outer code long), the matrices' turns where they do not fit their memory
together, and blocks with different numbers of lost rows, none among them: the message and the ecc must be
restored. And what the repair of a clean block and of one with a lost row leaves reserved on the device."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# inner block, inner ecc, outer block, outer ecc, interleave, most lost rows of a block
SHAPES = [(10, 2, 1024, 64, 2048, 16),   # column by column
          (10, 2, 512, 256, 2048, 72),   # matrices, in two turns
          (68, 4, 512, 256, 64, 9),      # matrices of 16 words a row
          (68, 4, 4096, 64, 1, 64),      # column by column, one block
          (2052, 4, 512, 256, 4, 255),   # matrices
          (20, 4, 64, 32, 1024, 9),      # 32,768 short inner rows: lane groups, not a wave a row
          (16, 8, 64, 32, 2048, 9)]


def _case(L, shape, rng):
    ib, ie, ob, oe, I, _ = shape
    rs = L.CIRC16(ib, ie, ob, oe, I)
    msg = rng.integers(0, 65536, rs.message_len).astype(np.uint16)
    return rs, msg, np.frombuffer(bytes(rs.encode(msg.tobytes())), np.uint16)


@pytest.mark.parametrize("shape", SHAPES, ids=["x".join(map(str, s)) for s in SHAPES])
def test_lost_rows_are_restored(shape):
    import libffrs_amd as L
    ib, ie, ob, oe, I, most = shape
    ik, ok = ib - ie, ob - oe
    rng = np.random.default_rng(sum(shape))
    rs, msg, ecc = _case(L, shape, rng)
    bm, be = msg.reshape(ok, I, ik).copy(), ecc.copy()
    outer = be[:oe * ik * I].reshape(oe, I, ik)
    for kk in range(I):
        for row in rng.choice(ob, most if kk % 7 == 0 else int(rng.integers(0, most + 1)), replace=False):
            at = bm[row, kk] if row < ok else outer[row - ok, kk]
            at[:] = (at.astype(np.int64) + rng.integers(1, 65536, ik)) % 65536
    print(f"circ16 known rows {shape}", flush=True)
    bm, be = bytearray(bm.tobytes()), bytearray(be.tobytes())
    assert rs.repair(bm, be) is False
    got_m, got_e = np.frombuffer(bm, np.uint16), np.frombuffer(be, np.uint16)
    assert (got_m == msg).all() and (got_e == ecc).all()


def test_memory_reserved():
    import libffrs_amd as L
    from libffrs_amd import capi
    shape = (10, 2, 512, 256, 8191, 1)
    rng = np.random.default_rng(3)
    rs, msg, ecc = _case(L, shape, rng)
    ctx = capi.Context(0)
    free = ctx.info()[2]
    print("circ16 reserved memory", flush=True)
    assert rs.repair(bytearray(msg.tobytes()), bytearray(ecc.tobytes())) is False
    bm = msg.reshape(256, 8191, 8).copy()
    bm[9, 77] ^= rng.integers(1, 65536, 8).astype(np.uint16)
    m = bytearray(bm.tobytes())
    assert rs.repair(m, bytearray(ecc.tobytes())) is False
    assert bytes(m) == msg.tobytes()
    # what a block takes: u16 message and ecc, u32 outer parity, inner parity and syndromes, row flags
    rows = 512 * 8191
    block = 2 * msg.size + 2 * ecc.size + 4 * 256 * 8 * 8191 + 2 * 4 * 2 * rows + rows
    used = free - ctx.info()[2]
    ctx.close()
    assert used < block + (600 << 20)
