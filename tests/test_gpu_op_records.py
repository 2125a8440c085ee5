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


def _together(jobs):
    """Runs each job in a thread of its own; raises the first failure."""
    bad = []

    def run(job):
        try:
            job()
        except BaseException as e:  # noqa: BLE001
            bad.append(e)

    threads = [threading.Thread(target=run, args=(j,)) for j in jobs]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    if bad:
        raise bad[0]


def test_products_from_threads_keep_their_own_records(device):
    # Each thread's product has its own row count; every buffer has room for
    # the largest, so a record that another op replaced would show as rows
    # unwritten or overwritten, nothing worse.
    rng = np.random.default_rng(11)
    rows, cols, most = 96, 1152, 40
    w = q4_blocks(rng, rows, cols)
    codes, scales = (device.array(a) for a in fz.block_split(2, w))
    counts = (3, 40, 17, 29)
    xs = [rng.normal(0, 1, (most, cols)).astype(np.float32) for _ in counts]
    want = [np.stack([orc.gemv_format(2, w, rows, cols, x[t]) for t in range(n)])
            for x, n in zip(xs, counts)]
    bufs = [(device.array(x), device.empty((most, rows), np.float32)) for x in xs]
    unwritten = np.full((most, rows), 7.0, np.float32)

    def job(i):
        dx, dy = bufs[i]
        for _ in range(40):
            dy.upload(unwritten)
            fz._lib.check(fz.load().frz_op_gemv(device.handle, codes.ptr, scales.ptr, rows, cols,
                                                dx.ptr, cols, dy.ptr, rows, counts[i], 0))
            got = dy.numpy()
            assert_same_bits(got[:counts[i]], want[i], f"{counts[i]} rows")
            assert (got[counts[i]:] == 7.0).all(), f"rows past {counts[i]}"

    _together([lambda i=i: job(i) for i in range(len(counts))])


def test_attention_from_threads_keeps_its_own_states(device):
    # The entry point that allocates nothing: one workspace for every call.
    slots, d = 4096, 256
    cases = []
    for i, (position, window) in enumerate([(4000, 4096), (700, 512), (63, 512)]):
        rng = np.random.default_rng(20 + i)
        qkv = rng.normal(0, 2, 6 * d).astype(np.float32)
        gains = (1 + 0.1 * rng.normal(0, 1, (2, d))).astype(np.float32)
        k, v = ((rng.integers(-96, 97, slots * d) / 32.0).astype(np.float16).view(np.uint16)
                for _ in range(2))
        dev = [device.array(a) for a in (qkv, fz.rope_turns(1e6, d), gains[0], gains[1], k, v)]
        cases.append((dev, device.empty((4 * d,), np.float32), window, position))

    def call(name, case):
        dev, out, window, position = case
        fz._lib.check(getattr(fz.load(), name)(device.handle, *(a.ptr for a in dev), out.ptr,
                                               slots, window, 1e-6, 0.0625, position))
        return out.numpy()

    want = [call("frz_op_rope_attention", c) for c in cases]

    def job(i):
        for _ in range(40):
            assert_same_bits(call("frz_op_rope_attention_noalloc", cases[i]), want[i],
                             f"position {cases[i][3]}")

    _together([lambda i=i: job(i) for i in range(len(cases))])
