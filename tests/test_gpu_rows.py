"""softmax and layernorm on the GPU against the pinned fp64 references.

Tolerance: max abs <= 1e-4 (e2e_softmax_test.cpp:308, e2e_layernorm_test.cpp:
320). Shapes: the reference's {(4096,1024), (16384,4096), (1,8192)}, the
BASELINE inputs (N(0, 4^2) rows; gamma U[0.5,1.5], beta U[-0.1,0.1]), odd
widths that take the scalar path, the stability and constant-row special
cases, and the reference's negative controls (uniform softmax; eps = 0).
"""
import numpy as np
import pytest

import kernelh as kh
import oracle as O
from khtest import down, empty, say, up

pytestmark = pytest.mark.gpu

SHAPES = [(4096, 1024), (16384, 4096), (1, 8192), (3, 1000), (5, 7), (64, 256), (2, 65536), (33, 2048)]


def _softmax(x, rows, cols):
    dx, dy = up(x), empty(rows * cols)
    say(f"softmax {rows}x{cols}")
    kh.softmax(dx, dy, rows, cols)
    return down(dy, rows * cols).reshape(rows, cols)


@pytest.mark.parametrize("rows,cols", SHAPES)
def test_softmax_vs_fp64_reference(dev, rows, cols):
    x, _ = O.lcg_fill(rows * cols, 0x27AB13)
    got = _softmax(x, rows, cols)
    ref = O.ref_softmax(x, rows, cols)
    assert np.all(np.isfinite(got))
    err = np.max(np.abs(got - ref))
    print(f"softmax {rows}x{cols} max-abs={err:.3e}")
    assert err <= 1e-4


def test_softmax_bench_inputs(dev):
    rows, cols = 4096, 1024
    x = O.normal(rows * cols, 0x50F7, 0.0, 4.0)
    got = _softmax(x, rows, cols)
    assert np.max(np.abs(got - O.ref_softmax(x, rows, cols))) <= 1e-4
    assert np.max(np.abs(got.astype(np.float64).sum(axis=1) - 1.0)) <= 1e-5


def test_softmax_stability_case(dev):
    rows = cols = 1024
    pat = np.array([1000.0, -1000.0, 0.0, 0.5, -0.5], np.float32)
    x = np.tile(np.resize(pat, cols), rows)
    got = _softmax(x, rows, cols)
    assert np.all(np.isfinite(got))
    assert np.max(np.abs(got - O.ref_softmax(x, rows, cols))) <= 1e-4


def test_softmax_negative_control_uniform(dev):
    rows = cols = 256
    x, _ = O.lcg_fill(rows * cols, 0x51AC0D3)
    got = _softmax(x, rows, cols)
    assert np.any(np.abs(got - 1.0 / cols) > 1e-4)


def test_softmax_reference_geometry(dev):
    rows, cols = 300, 1024
    x, _ = O.lcg_fill(rows * cols, 0x27AB13)
    dx, dy = up(x), empty(rows * cols)
    f = kh.template_function("softmax")
    args = kh.LaunchArgs().add_memref(dx, [rows, cols]).add_memref(dy, [rows, cols])
    assert args.param_count() == 14
    say("softmax reference geometry rows x 256")
    kh.kernel_launch(f, (rows, 1, 1), (256, 1, 1), args)
    assert np.max(np.abs(down(dy, rows * cols).reshape(rows, cols) - O.ref_softmax(x, rows, cols))) <= 1e-4


@pytest.mark.parametrize("symbol", ["softmax", "softmax_wave", "softmax_wide", "layernorm", "layernorm_wave",
                                    "layernorm_wide", "layernorm_wide_many", "layernorm_wide_parts"])
@pytest.mark.parametrize("cols", [64, 256, 512, 1000, 1024, 2048, 4096, 5000])
def test_every_row_symbol_at_every_width(dev, symbol, cols):
    # Each symbol of a template computes the same result at every width (the
    # launcher picks one by width; raw callers may launch either).
    rows = 37
    x, seed = O.lcg_fill(rows * cols, 0x27AB13)
    g, seed = O.lcg_fill(cols, seed)
    b, seed = O.lcg_fill(cols, seed)
    m = kh.GpuModule(kh.code_object(symbol.split("_")[0]))
    f = m.get_function(symbol)
    dx, dy = up(x), empty(rows * cols)
    args = kh.LaunchArgs().add_memref(dx, [rows, cols])
    if symbol.startswith("layernorm"):
        dg, db = up(g), up(b)
        args.add_memref(dg, [cols]).add_memref(db, [cols])
        ref = O.ref_layernorm(x, g, b, rows, cols)
    else:
        ref = O.ref_softmax(x, rows, cols)
    args.add_memref(dy, [rows, cols])
    say(f"{symbol} rows={rows} cols={cols}")
    kh.kernel_launch(f, (5, 1, 1), (256, 1, 1), args)
    got = down(dy, rows * cols).reshape(rows, cols)
    assert np.max(np.abs(got - ref)) <= 1e-4



@pytest.mark.parametrize("block", [64, 128, 192])
@pytest.mark.parametrize("cols", [128, 1024])
def test_layernorm_narrow_block_sizes(dev, block, cols):
    # The narrow symbol copies gamma and beta into LDS with the block's
    # threads before its rows: any multiple of 64 threads per block, with
    # grid-strided rows, gives the same result.
    rows = 45
    x, seed = O.lcg_fill(rows * cols, 0x51ED27)
    g, seed = O.lcg_fill(cols, seed)
    b, seed = O.lcg_fill(cols, seed)
    f = kh.GpuModule(kh.code_object("layernorm")).get_function("layernorm")
    dx, dg, db, dy = up(x), up(g), up(b), empty(rows * cols)
    args = kh.LaunchArgs().add_memref(dx, [rows, cols]).add_memref(dg, [cols]).add_memref(db, [cols])
    args.add_memref(dy, [rows, cols])
    say(f"layernorm block={block} rows={rows} cols={cols}")
    kh.kernel_launch(f, (4, 1, 1), (block, 1, 1), args)
    got = down(dy, rows * cols).reshape(rows, cols)
    assert np.max(np.abs(got - O.ref_layernorm(x, g, b, rows, cols))) <= 1e-4

def _layernorm(x, g, b, rows, cols):
    dx, dg, db, dy = up(x), up(g), up(b), empty(rows * cols)
    say(f"layernorm {rows}x{cols}")
    kh.layernorm(dx, dg, db, dy, rows, cols)
    return down(dy, rows * cols).reshape(rows, cols)


@pytest.mark.parametrize("rows,cols", SHAPES)
def test_layernorm_vs_fp64_reference(dev, rows, cols):
    x, seed = O.lcg_fill(rows * cols, 0x2E2E8A)
    g, seed = O.lcg_fill(cols, seed)
    b, seed = O.lcg_fill(cols, seed)
    got = _layernorm(x, g, b, rows, cols)
    err = np.max(np.abs(got - O.ref_layernorm(x, g, b, rows, cols)))
    print(f"layernorm {rows}x{cols} max-abs={err:.3e}")
    assert err <= 1e-4


def test_layernorm_bench_inputs(dev):
    rows, cols = 4096, 1024
    x = O.normal(rows * cols, 0x1A7E, 0.0, 4.0)
    g = O.uniform(cols, 0x1A7F, 0.5, 1.5)
    b = O.uniform(cols, 0x1A80, -0.1, 0.1)
    got = _layernorm(x, g, b, rows, cols)
    assert np.max(np.abs(got - O.ref_layernorm(x, g, b, rows, cols))) <= 1e-4


def test_layernorm_constant_rows_and_eps0_control(dev):
    rows, cols = 64, 1024
    x = np.full(rows * cols, 3.0, np.float32)
    g, seed = O.lcg_fill(cols, 0xC0578A)
    b, seed = O.lcg_fill(cols, seed)
    got = _layernorm(x, g, b, rows, cols)
    assert np.all(np.isfinite(got))
    assert np.max(np.abs(got - O.ref_layernorm(x, g, b, rows, cols))) <= 1e-4
    # Negative control (e2e_layernorm_test.cpp:336-425): the eps = 0 reference
    # is NaN everywhere, the kernel's eps = 1e-5 output is finite beta.
    ref0 = O.ref_layernorm(x, g, b, rows, cols, eps=0.0)
    assert np.all(np.isnan(ref0)) and not np.any(np.abs(got - ref0) <= 1e-4)


@pytest.mark.parametrize("template", ["softmax", "layernorm"])
@pytest.mark.parametrize("cols", [100, 40, 200])
def test_rows_blocks_of_partial_waves(dev, template, cols):
    # The reference's rows x min(cols, 256) geometry (kernelh_backend.cpp:
    # 256-257) with cols < 256 not a multiple of 64: blocks of `cols`
    # threads. The verified launch refuses them, as the reference's launch
    # verifier does; a raw launch (plain hipModuleLaunchKernel) is still
    # correct: the kernels give each thread whole rows when the block is not
    # whole wavefronts.
    rows = 70
    x, seed = O.lcg_fill(rows * cols, 0x51ED27)
    g, seed = O.lcg_fill(cols, seed)
    b, seed = O.lcg_fill(cols, seed)
    dx, dy = up(x), empty(rows * cols)
    args = kh.LaunchArgs().add_memref(dx, [rows, cols])
    if template == "layernorm":
        dg, db = up(g), up(b)
        args.add_memref(dg, [cols]).add_memref(db, [cols])
        ref = O.ref_layernorm(x, g, b, rows, cols)
    else:
        ref = O.ref_softmax(x, rows, cols)
    args.add_memref(dy, [rows, cols])
    say(f"{template} partial-wave blocks rows={rows} cols={cols} block={min(cols, 256)}")
    f = kh.template_function(template)
    with pytest.raises(kh.KhrtError, match="multiple of the wavefront size"):
        kh.kernel_launch(f, (rows, 1, 1), (min(cols, 256), 1, 1), args)
    kh.launch_raw(f, (rows, 1, 1), (min(cols, 256), 1, 1), args)
    kh.synchronize()
    got = down(dy, rows * cols).reshape(rows, cols)
    assert np.max(np.abs(got - ref)) <= 1e-4


# Edges of softmax's row paths: 16 lanes (one, two, four float4 each), a wave,
# a workgroup of 4, 8 and 16 float4 per thread, two sweeps; one column either
# side of each and widths that leave 1-3 floats in the last float4.
SOFTMAX_EDGES = [1, 3, 63, 64, 65, 127, 129, 254, 256, 257, 511, 513, 1023, 1025, 2047, 2048, 2049, 4095, 4096, 4097,
                 12288, 12289, 16383, 16385, 24576, 24577, 32767, 32768, 32769, 65535, 65536, 65537]


@pytest.mark.parametrize("cols", SOFTMAX_EDGES)
def test_softmax_path_edges(dev, cols):
    # Rows at odd addresses, a guard after the output, and 5 rows so that a
    # wave's last group of four is partial. Each output is e/s with exponents
    # of magnitude up to ~30 (error 2^-24 * 30 each before it cancels), two
    # roundings of e and 1/s and a sum of positive terms: 1e-6 of the largest.
    rows, guard = 5, 64
    x = O.normal(rows * cols, 0x50F7 + cols, 0.0, 4.0)
    ref = O.ref_softmax(x, rows, cols)
    dx, dy = up(np.concatenate([np.full(1, np.nan, np.float32), x])), empty(rows * cols + guard, -7.0)
    say(f"softmax rows={rows} cols={cols}")
    kh.softmax(dx.ptr + 4, dy, rows, cols)
    out = down(dy, rows * cols + guard)
    assert np.all(out[rows * cols:] == -7.0)
    assert np.max(np.abs(out[:rows * cols].reshape(rows, cols) - ref)) <= 1e-6 * np.max(ref)


@pytest.mark.parametrize("rows,cols,symbol", [
    (1664, 2049, "softmax_block"), (1000, 4095, "softmax_block"), (2560, 2051, "softmax_block"), (970, 4096, "softmax_block"),
    (257, 24577, "softmax_block"), (300, 32001, "softmax_block"), (7170, 514, "softmax_wave"), (8191, 1023, "softmax_wave"),
])
def test_softmax_path_of_many_rows(dev, rows, cols, symbol):
    # Launches whose symbol depends on the number of rows too: odd addresses, a
    # guard, and the tolerance as above.
    guard = 64
    x = O.normal(rows * cols, 0x50F8 + cols, 0.0, 4.0)
    ref = O.ref_softmax(x, rows, cols)
    dx, dy = up(np.concatenate([np.full(1, np.nan, np.float32), x])), empty(rows * cols + guard, -7.0)
    say(f"softmax rows={rows} cols={cols}")
    assert kh.launch_symbol("softmax", f"rows={rows},cols={cols}") == symbol
    kh.softmax(dx.ptr + 4, dy, rows, cols)
    out = down(dy, rows * cols + guard)
    assert np.all(out[rows * cols:] == -7.0)
    assert np.max(np.abs(out[:rows * cols].reshape(rows, cols) - ref)) <= 1e-6 * np.max(ref)


@pytest.mark.parametrize("cols", [40, 200, 300, 700, 1500, 3001, 5000, 20001, 40001, 70001])
def test_softmax_extreme_rows(dev, cols):
    # Rows of the type's lowest value, of one large value, half masked with
    # either, and with an infinity or NaN: uniform, the softmax of the rest,
    # or NaN, as in 64 bits.
    low = np.finfo(np.float32).min
    x = O.normal(8 * cols, 0xE27, 0.0, 1.0).reshape(8, cols)
    x[0], x[1], x[2] = low, 1e9, -np.inf
    x[3, :cols // 2], x[4, : cols // 2] = -np.inf, low
    x[5, 0], x[6, cols - 1], x[7] = np.inf, np.nan, -3e38
    with np.errstate(invalid="ignore"):
        e = np.exp(x.astype(np.float64) - np.max(x.astype(np.float64), axis=1, keepdims=True))
        ref = e / e.sum(axis=1, keepdims=True)
    got = _softmax(x.ravel(), 8, cols)
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    assert np.nanmax(np.abs(got - ref)) <= 1e-6


@pytest.mark.parametrize("symbol,block", [("softmax", 40), ("softmax_wave", 40), ("softmax_wave", 128)])
@pytest.mark.parametrize("cols", [40, 100, 250, 700])
def test_softmax_extreme_rows_raw_launches(dev, symbol, block, cols):
    # The same rows in blocks that are not whole waves, a thread per row, and in
    # the wave symbol at widths the launcher does not give it.
    low = np.finfo(np.float32).min
    x = O.normal(7 * cols, 0xE28, 0.0, 1.0).reshape(7, cols)
    x[0], x[1], x[2], x[3, : cols // 2], x[4, 0], x[5, : cols // 2] = low, 3e38, -np.inf, low, np.inf, -np.inf
    with np.errstate(invalid="ignore"):
        e = np.exp(x.astype(np.float64) - np.max(x.astype(np.float64), axis=1, keepdims=True))
        ref = e / e.sum(axis=1, keepdims=True)
    dx, dy = up(x.ravel()), empty(7 * cols)
    args = kh.LaunchArgs().add_memref(dx, [7, cols]).add_memref(dy, [7, cols])
    f = kh.GpuModule(kh.code_object("softmax")).get_function(symbol)
    say(f"{symbol} extreme rows, cols={cols}, block={block}")
    kh.launch_raw(f, (3, 1, 1), (block, 1, 1), args)
    got = down(dy, 7 * cols).reshape(7, cols)
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    assert np.nanmax(np.abs(got - ref)) <= 1e-6


@pytest.mark.parametrize("symbol", ["softmax", "softmax_wave", "softmax_wide", "softmax_block"])
@pytest.mark.parametrize("cols", [30, 250, 1500, 4096, 9000])
@pytest.mark.parametrize("block", [64, 256])
def test_softmax_padded_rows_any_symbol(dev, symbol, cols, block):
    # Rows further apart than their width (x and y each by its own stride):
    # pads are NaN in x and keep their value in y.
    rows, xs, ys = 11, cols + 5, cols + 3
    x = O.normal(rows * cols, 0x77, 0.0, 4.0)
    xp = np.full((rows, xs), np.nan, np.float32)
    xp[:, :cols] = x.reshape(rows, cols)
    dx, dy = up(xp.ravel()), empty(rows * ys, -7.0)
    args = kh.LaunchArgs().add_memref(dx, [rows, cols]).add_memref(dy, [rows, cols])
    args.slots[5], args.slots[7 + 5] = xs, ys
    f = kh.GpuModule(kh.code_object("softmax")).get_function(symbol)
    say(f"{symbol} rows={rows} cols={cols} strides={xs},{ys} block={block}")
    kh.kernel_launch(f, (2, 1, 1), (block, 1, 1), args)
    out = down(dy, rows * ys).reshape(rows, ys)
    assert np.all(out[:, cols:] == -7.0)
    assert np.max(np.abs(out[:, :cols] - O.ref_softmax(x, rows, cols))) <= 1e-6


@pytest.mark.parametrize("cols", SOFTMAX_EDGES)
def test_layernorm_path_edges(dev, cols):
    # The same edges, every operand at an odd address. Rows of N(3, 4^2): the
    # mean carries 2^-24 * 12 (the sum's rounding) and the deviations, scaled
    # to |d| <= ~5 by up to 1/4 (sqrt(1/eps) for the single column, whose
    # deviation is an exact 0), 2^-24 of themselves: 1e-5 covers both.
    rows, guard = 5, 64
    x = O.normal(rows * cols, 0x1A7E + cols, 3.0, 4.0)
    if cols > 1:  # no row whose few values happen to lie close together
        x[::cols], x[1::cols] = 9.0, -3.0
    g = O.uniform(cols, 0x1A7F, 0.5, 1.5)
    b = O.uniform(cols, 0x1A80, -0.1, 0.1)
    ref = O.ref_layernorm(x, g, b, rows, cols)
    nan = np.full(1, np.nan, np.float32)
    dx, dg, db = (up(np.concatenate([nan, t, nan])) for t in (x, g, b))
    dy = empty(rows * cols + guard, -7.0)
    say(f"layernorm rows={rows} cols={cols}")
    kh.layernorm(dx.ptr + 4, dg.ptr + 4, db.ptr + 4, dy, rows, cols)
    out = down(dy, rows * cols + guard)
    assert np.all(out[rows * cols:] == -7.0)
    assert np.max(np.abs(out[:rows * cols].reshape(rows, cols) - ref)) <= 1e-5


@pytest.mark.parametrize("rows,cols,symbol", [(12289, 2689, "layernorm_wide_parts"), (12290, 4095, "layernorm_wide_parts"),
                                              (300, 24579, "layernorm_block"), (8200, 131, "layernorm"),
                                              (6001, 254, "layernorm_wave"), (511, 1026, "layernorm_wide"),
                                              (895, 2047, "layernorm_wide"), (1025, 1027, "layernorm_wide_many")])
def test_layernorm_path_of_many_rows(dev, rows, cols, symbol):
    # Launches whose symbol depends on the number of rows too: every operand at an
    # odd address, a guard, and the tolerance as above.
    guard = 64
    x = O.normal(rows * cols, 0x1A81 + cols, 3.0, 4.0)
    g, b = O.uniform(cols, 0x1A7F, 0.5, 1.5), O.uniform(cols, 0x1A80, -0.1, 0.1)
    ref = O.ref_layernorm(x, g, b, rows, cols)
    nan = np.full(1, np.nan, np.float32)
    dx, dg, db = (up(np.concatenate([nan, t, nan])) for t in (x, g, b))
    dy = empty(rows * cols + guard, -7.0)
    say(f"layernorm rows={rows} cols={cols}")
    assert kh.launch_symbol("layernorm", f"rows={rows},cols={cols}") == symbol
    kh.layernorm(dx.ptr + 4, dg.ptr + 4, db.ptr + 4, dy, rows, cols)
    out = down(dy, rows * cols + guard)
    assert np.all(out[rows * cols:] == -7.0)
    assert np.max(np.abs(out[:rows * cols].reshape(rows, cols) - ref)) <= 1e-5


@pytest.mark.parametrize("cols", [40, 100, 200, 300, 700, 1500, 3001, 5000, 20001, 40001, 70001])
def test_layernorm_infinities_and_nan(dev, cols):
    # A row with an infinity or NaN has no finite mean: all NaN, as in 64 bits,
    # and the rows beside it (four to a wave, one or a workgroup) are untouched.
    rows = 9
    x = O.normal(rows * cols, 0x1A82, 3.0, 4.0).reshape(rows, cols)
    x[1, 0], x[3, cols - 1], x[4, cols // 2], x[6, 5:9] = np.inf, np.nan, -np.inf, [np.inf, -np.inf, np.inf, np.nan]
    g, b = O.uniform(cols, 0x1A7F, 0.5, 1.5), O.uniform(cols, 0x1A80, -0.1, 0.1)
    dx, dg, db, dy = up(x.ravel()), up(g), up(b), empty(rows * cols)
    say(f"layernorm infinities and NaN, cols={cols}")
    kh.layernorm(dx, dg, db, dy, rows, cols)
    got = down(dy, rows * cols).reshape(rows, cols)
    bad = [1, 3, 4, 6]
    ok = [r for r in range(rows) if r not in bad]
    assert np.all(np.isnan(got[bad]))
    assert np.max(np.abs(got[ok] - O.ref_layernorm(x[ok].ravel(), g, b, len(ok), cols))) <= 1e-5


@pytest.mark.parametrize("symbol", ["layernorm", "layernorm_wave", "layernorm_wide", "layernorm_wide_many",
                                    "layernorm_wide_parts", "layernorm_block"])
@pytest.mark.parametrize("cols", [30, 250, 1500, 4096, 9000])
@pytest.mark.parametrize("block", [64, 256])
def test_layernorm_padded_rows_any_symbol(dev, symbol, cols, block):
    rows, xs, ys = 11, cols + 5, cols + 3
    x = O.normal(rows * cols, 0x77, 0.0, 4.0)
    g, b = O.uniform(cols, 0x78, 0.5, 1.5), O.uniform(cols, 0x79, -0.1, 0.1)
    xp = np.full((rows, xs), np.nan, np.float32)
    xp[:, :cols] = x.reshape(rows, cols)
    dx, dg, db, dy = up(xp.ravel()), up(g), up(b), empty(rows * ys, -7.0)
    args = kh.LaunchArgs().add_memref(dx, [rows, cols]).add_memref(dg, [cols]).add_memref(db, [cols])
    args.add_memref(dy, [rows, cols])
    args.slots[5], args.slots[17 + 5] = xs, ys
    f = kh.GpuModule(kh.code_object("layernorm")).get_function(symbol)
    say(f"{symbol} rows={rows} cols={cols} strides={xs},{ys} block={block}")
    kh.kernel_launch(f, (2, 1, 1), (block, 1, 1), args)
    out = down(dy, rows * ys).reshape(rows, ys)
    assert np.all(out[:, cols:] == -7.0)
    assert np.max(np.abs(out[:, :cols] - O.ref_layernorm(x, g, b, rows, cols))) <= 1e-5


@pytest.mark.parametrize("template", ["softmax", "layernorm"])
@pytest.mark.parametrize("cols", [5000, 12289, 24577, 32768, 65535, 65536])
def test_row_is_read_whole_before_it_is_written(dev, template, cols):
    # Up to 65536 columns a workgroup holds the row in registers, so an output
    # that overlaps the input further on is the one beside it; a second sweep
    # over the row would read what the first chunk's outputs replaced.
    shift = 16384 if cols > 16384 else 1024
    x = O.normal(cols, 0x0E1A, 0.0, 4.0)
    g, b = O.uniform(cols, 0x1A7F, 0.5, 1.5), O.uniform(cols, 0x1A80, -0.1, 0.1)
    buf = up(np.concatenate([x, np.zeros(shift, np.float32)]))
    say(f"{template} rows=1 cols={cols}, y {shift} floats into x")
    if template == "softmax":
        ref = _softmax(x, 1, cols)
        kh.softmax(buf.ptr, buf.ptr + 4 * shift, 1, cols)
    else:
        ref = _layernorm(x, g, b, 1, cols)
        dg, db = up(g), up(b)
        kh.layernorm(buf.ptr, dg, db, buf.ptr + 4 * shift, 1, cols)
    assert np.array_equal(down(buf, shift + cols)[shift:], ref.ravel())


@pytest.mark.parametrize("template", ["softmax", "layernorm"])
@pytest.mark.parametrize("rows,cols", [(203, 132), (203, 160), (17000, 196), (17000, 255), (9300, 224), (4097, 252)])
@pytest.mark.parametrize("odd", [0, 1, 8])
def test_rows_that_share_cache_lines(dev, template, rows, cols, odd):
    # Outputs whose rows' starts and ends are parts of cache lines, and whole
    # ones, from starts of several alignments, with guards on both sides.
    guard = 64
    x = O.normal(rows * cols, 0x5AC + cols, 0.0, 4.0)
    g, b = O.uniform(cols, 0x1A7F, 0.5, 1.5), O.uniform(cols, 0x1A80, -0.1, 0.1)
    dx, dy = up(x), empty(guard + rows * cols + guard, -7.0)
    say(f"{template} rows={rows} cols={cols} y {odd} floats past a line")
    if template == "softmax":
        kh.softmax(dx, dy.ptr + 4 * odd, rows, cols)
        ref = O.ref_softmax(x, rows, cols)
    else:
        dg, db = up(g), up(b)
        kh.layernorm(dx, dg, db, dy.ptr + 4 * odd, rows, cols)
        ref = O.ref_layernorm(x, g, b, rows, cols)
    out = down(dy, guard + rows * cols + guard)
    assert np.all(out[:odd] == -7.0) and np.all(out[odd + rows * cols:] == -7.0)
    assert np.max(np.abs(out[odd:odd + rows * cols].reshape(rows, cols) - ref)) <= 1e-5
