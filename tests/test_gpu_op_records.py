"""The one-kernel ops' step records and selection scratch: each op runs under
its own record whatever ran before it, and selections from several threads on
one device do not mix."""
import threading

import numpy as np
import pytest

import _oracle as orc
import frizzle_amd as fz
from helpers import assert_same_bits, q4_blocks

pytestmark = pytest.mark.gpu


def test_ops_between_records(device):
    # A product of 5 rows between two of 40, each with its own row count.
    rng = np.random.default_rng(3)
    rows, cols = 96, 1152
    w = q4_blocks(rng, rows, cols)
    codes, scales = (device.array(a) for a in fz.block_split(2, w))
    x = rng.normal(0, 1, (40, cols)).astype(np.float32)
    dx = device.array(x)
    for tokens in (40, 5, 40):
        dy = device.array(np.full((40, rows), 7.0, np.float32))
        fz._lib.check(fz.load().frz_op_gemv(device.handle, codes.ptr, scales.ptr, rows, cols,
                                            dx.ptr, cols, dy.ptr, rows, tokens, 0))
        got = dy.numpy()
        for t in (0, tokens - 1):
            assert_same_bits(got[t], orc.gemv_format(2, w, rows, cols, x[t]), f"token {t}")
        assert (got[tokens:] == 7.0).all()


def _topk(device, dl, count, dc):
    fz._lib.check(fz.load().frz_op_topk(device.handle, dl.ptr, count, dc.ptr))


# The device's own scratch serves up to 1,048,576 logits.
@pytest.mark.parametrize("count", [64, 1 << 20, (1 << 20) + 1])
def test_topk_at_the_scratch_limit(device, count):
    logits = np.random.default_rng(count).permutation(count).astype(np.float32)
    dl, dc = device.array(logits), device.empty((64, 2), np.uint32)
    _topk(device, dl, count, dc)
    want = np.argsort(-logits)[:64]
    assert (dc.numpy()[:, 1] == want).all()


def test_topk_from_threads(device):
    count, threads, calls = 262144, 4, 20
    rng = np.random.default_rng(8)
    sets = [rng.permutation(count).astype(np.float32) for _ in range(threads)]
    bufs = [(device.array(s), device.empty((64, 2), np.uint32)) for s in sets]
    bad = []

    def work(i):
        want = np.argsort(-sets[i])[:64]
        for _ in range(calls):
            _topk(device, bufs[i][0], count, bufs[i][1])
            if not (bufs[i][1].numpy()[:, 1] == want).all():
                bad.append(i)

    ts = [threading.Thread(target=work, args=(i,)) for i in range(threads)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad
