"""The products of steps of 2 to 512 rows through the C ABI, bit for bit the
oracle's, at the edges of their token tiles and of the rules that choose a
kernel for a step's rows."""
import numpy as np
import pytest

import _oracle as orc
import frizzle_amd as fz
from helpers import assert_same_bits, format_blocks, q4_blocks

pytestmark = pytest.mark.gpu


def _dev(device, fmt, blocks):
    codes, scales = fz.block_split(fmt, blocks)
    return device.array(codes), device.array(scales)


def _check_rows(got, want_row, tokens):
    """Every token's row when they are few; else both edges of each 16-token
    tile and a stride through the rest."""
    rows = set(range(tokens)) if tokens <= 40 else (
        {t for t in range(tokens) if t % 16 in (0, 15)} | set(range(0, tokens, 7)) | {tokens - 1})
    for t in sorted(rows):
        assert_same_bits(got[t], want_row(t), f"token {t}")


@pytest.mark.parametrize("fmt,rows,cols,tokens", [
    (2, 1536, 1152, 17), (2, 1152, 1024, 31), (2, 1152, 6912, 33), (2, 100, 1152, 64),
    (2, 1152, 6912, 256), (2, 1152, 6912, 257), (2, 1536, 1152, 255), (2, 8192, 1152, 17),
    (2, 8191, 1152, 17), (3, 1152, 6912, 49), (8, 1152, 6912, 130), (3, 40, 1152, 300),
    (2, 1152, 6912, 497), (2, 1536, 1152, 512), (2, 1152, 1024, 401), (8, 36, 6912, 512),
    (3, 36, 6912, 511), (2, 40, 992, 77), (2, 40, 16416, 17),
    (2, 1536, 1152, 113), (2, 1500, 1152, 300), (2, 1137, 1024, 176), (2, 600, 2048, 512),
    (2, 600, 2080, 512),
    (2, 1152, 1056, 19),
    # Where a wave a tile is sooner: 32 x 32 tiles, and 16 x 16 ones.
    (2, 4096, 1152, 512), (3, 1600, 2080, 500), (8, 1024, 4096, 512)])
def test_row_products_bit_exact(device, fmt, rows, cols, tokens):
    rng = np.random.default_rng(rows + cols + tokens)
    w = format_blocks(rng, fmt, rows, cols)
    x = rng.normal(0, 1, (tokens, cols)).astype(np.float32)
    codes, scales = _dev(device, fmt, w)
    dx, dy = device.array(x), device.empty((tokens, rows), np.float32)
    fz._lib.check(fz.load().frz_op_gemv_format(device.handle, fmt, codes.ptr, scales.ptr, rows,
                                               cols, dx.ptr, cols, dy.ptr, rows, tokens, 0))
    _check_rows(dy.numpy(), lambda t: orc.gemv_format(fmt, w, rows, cols, x[t]), tokens)


# A pass a wave, the wide tiles (of 32 neurons or of 16; K of fewer groups than
# ranges goes there at any rows) and, over long ranges of one length, a wave a
# tile: each form where product_rules.h takes it.
@pytest.mark.parametrize("rows,tokens,cols", [
    (6912, 17, 1152), (1000, 48, 1152), (96, 256, 1152), (96, 257, 1152), (100, 512, 1152),
    (95, 208, 1152), (1000, 209, 1152), (6900, 510, 1152), (6900, 385, 1056), (33, 300, 1056),
    (50, 2, 32), (40, 9, 96), (70, 161, 992), (70, 225, 1024),
    (6900, 380, 1152), (5000, 33, 96), (8200, 33, 1024), (3000, 511, 4096)])
def test_gated_rows_bit_exact(device, rows, tokens, cols):
    rng = np.random.default_rng(rows + tokens)
    layers, layer, position = 2, 1, 30
    g, u = q4_blocks(rng, rows, cols), q4_blocks(rng, rows, cols)
    x = rng.normal(0, 1, (tokens, cols)).astype(np.float32)
    # Pins that start and end inside the step, at the first and last neurons.
    edits = [fz.Edit(layer, n, fz.EditKind.SET, 0.5 * n + 1, 3, 3 + tokens // 2)
             for n in (0, 15, 16, rows - 1)]
    table = fz.edit_table(edits, layers, origin=position)
    (gc, gs), (uc, us) = _dev(device, 2, g), _dev(device, 2, u)
    dx, dt = device.array(x), device.array(table)
    da = device.empty((tokens, rows), np.float32)
    fz._lib.check(fz.load().frz_op_gated(device.handle, gc.ptr, gs.ptr, uc.ptr, us.ptr, rows,
                                         cols, dx.ptr, da.ptr, tokens, position, dt.ptr, layer))

    def want(t):
        row = orc.gated(g, u, rows, cols, x[t])
        orc.lib().orc_edit_row(table.ctypes.data, layer, position + t, rows, row.ctypes.data)
        return row

    _check_rows(da.numpy(), want, tokens)


# Past 16 tokens a product's steps are held in a table: K past what it holds
# is refused, before anything is launched, at every row count.
@pytest.mark.parametrize("rows,cols,tokens,ok", [
    (1536, 16384, 512, True), (1536, 16416, 512, False), (32, 32768, 17, True),
    (32, 32800, 17, False), (32, 32800, 16, True)])
def test_row_products_of_long_k(device, rows, cols, tokens, ok):
    rng = np.random.default_rng(cols)
    w = q4_blocks(rng, rows, cols)
    codes, scales = _dev(device, 2, w)
    x = rng.normal(0, 1, (tokens, cols)).astype(np.float32)
    dx, dy = device.array(x), device.array(np.full((tokens, rows), 7.0, np.float32))

    def call():
        fz._lib.check(fz.load().frz_op_gemv(device.handle, codes.ptr, scales.ptr, rows, cols,
                                            dx.ptr, cols, dy.ptr, rows, tokens, 0))
    if ok:
        call()
        for t in (0, tokens - 1):
            assert_same_bits(dy.numpy()[t], orc.gemv_format(2, w, rows, cols, x[t]), f"token {t}")
    else:
        with pytest.raises(fz.FrzError):
            call()
        assert (dy.numpy() == 7.0).all()


def test_gated_rows_of_long_k(device):
    rows, cols = 32, 16416
    rng = np.random.default_rng(2)
    (gc, gs), (uc, us) = (_dev(device, 2, q4_blocks(rng, rows, cols)) for _ in range(2))
    dx = device.array(rng.normal(0, 1, (17, cols)).astype(np.float32))
    da = device.array(np.full((17, rows), 7.0, np.float32))
    for tokens, ok in ((16, True), (17, False)):
        rc = fz.load().frz_op_gated(device.handle, gc.ptr, gs.ptr, uc.ptr, us.ptr, rows, cols,
                                    dx.ptr, da.ptr, tokens, 0, None, 0)
        assert (rc == 0) == ok, tokens
