"""The device workspace of the RSi16 repair: two threads on one codec, capture with and without a call before
it, replays after the workspace has been outgrown, and batches larger than one workspace takes. Against the
general kernel, which uses none."""
import threading

import numpy as np
import pytest

from libffrs_amd import workloads as W

pytestmark = pytest.mark.gpu


class Batch:
    """Damaged codewords in device buffers, and what the general kernel makes of them."""

    def __init__(self, ctx, codec, count, seed, distinct=512):
        n, ecc, k = codec.block_len, codec.ecc_len, codec.message_len
        sub = min(count, distinct)
        msgs, errs, s = W.rsi16_plain(sub, n, ecc, ecc // 2, seed=seed)
        self.codec, self.count = codec, count
        self.d = [ctx.alloc(count * k * 2), ctx.alloc(count * ecc * 2), ctx.alloc(count)]
        self.d[0].upload(msgs)
        codec.encode_device(self.d[0], sub, self.d[1])
        par = np.empty((sub, ecc), np.uint16)
        self.d[1].download(par)
        cws = np.concatenate([msgs, par], 1)
        W.rsi16_corrupt(cws, errs, s)
        self.rows = np.arange(count) % sub
        self.src = [np.ascontiguousarray(cws[:, :k]), np.ascontiguousarray(cws[:, k:])]
        codec.set_repair_syndromes(1)
        self.upload(sub)
        codec.repair_device(*self.d[:2], sub, self.d[2])
        self.want = self.results(sub)
        codec.set_repair_syndromes(0)
        self.upload()

    def upload(self, count=None):
        for d, a in zip(self.d, self.src):
            d.upload(a[self.rows[:count]])

    def repair(self):
        self.codec.repair_device(*self.d[:2], self.count, self.d[2])

    def results(self, count):
        out = [np.empty((count, a.shape[1]), np.uint16) for a in self.src] + [np.empty(count, np.uint8)]
        for d, a in zip(self.d, out):
            d.download(a)
        return out

    def check(self):
        for a, b in zip(self.results(self.count), self.want):
            assert (a == b[self.rows]).all()

    def free(self):
        for d in self.d:
            d.free()


@pytest.fixture
def ctx():
    from libffrs_amd import capi
    c = capi.Context(0)
    yield c
    c.close()


def _codec(ctx, n, ecc):
    from libffrs_amd import capi
    print(f"workspace ({n},{ecc})", flush=True)
    return capi.RSi16Codec(ctx, n, ecc)


@pytest.mark.parametrize("n,ecc,counts", [(64, 8, (30000, 45000)), (256, 32, (20000, 17000)), (128, 64, (9000, 10000)),
                                          (256, 128, (8300, 9000)), (512, 256, (1100, 2000))])
def test_two_threads_on_one_codec(ctx, n, ecc, counts):
    codec = _codec(ctx, n, ecc)
    batches = [Batch(ctx, codec, c, 7 + c) for c in counts]
    errors = []

    def work(b):
        try:
            for _ in range(40):
                b.repair()
        except Exception as e:
            errors.append(e)

    for _ in range(3):
        for b in batches:
            b.upload()
        threads = [threading.Thread(target=work, args=(b,)) for b in batches]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert not errors
        ctx.sync()
        for b in batches:  # the calls after the first found repaired words
            m, e, st = b.results(b.count)
            assert (m == b.want[0][b.rows]).all() and (e == b.want[1][b.rows]).all()
            b.repair()
            assert (st == b.results(b.count)[2]).all()
    for b in batches:
        b.free()
    codec.close()


@pytest.mark.parametrize("n,ecc,small,large", [(64, 8, 30000, 100000), (256, 32, 20000, 50000), (128, 64, 9000, 30000),
                                               (256, 128, 8300, 20000), (512, 256, 1100, 4000)])
def test_capture_and_growth(ctx, n, ecc, small, large):
    codec = _codec(ctx, n, ecc)
    first, later = Batch(ctx, codec, small, 11), Batch(ctx, codec, large, 13)
    graphs = []
    for warm in (False, True):
        if warm:
            first.repair()
        ctx.capture_begin()
        first.repair()
        graphs.append(ctx.capture_end())
    for _ in range(3):
        for g in graphs:
            first.upload()
            g.launch()
            first.check()
        later.upload()
        later.repair()  # outgrows the workspace the second graph was captured with
        later.check()
    for g in graphs:
        g.close()
    first.free()
    later.free()
    codec.close()


def test_batch_larger_than_the_workspace(ctx):
    codec = _codec(ctx, 512, 256)
    b = Batch(ctx, codec, 261120 + 1000, 17)
    b.repair()
    b.check()
    b.free()
    codec.close()
