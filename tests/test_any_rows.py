"""Softmax rows of any length and element alignment on the vector tiers (softmax_short, softmax_rows_any and the
co-resident tier's instantiation for such rows): the sizes where a row's last vector, a wave's share or a chunk begins
to be used, base pointers off a 16-byte boundary, -inf elements and rows, against the oracle within the bounds of the
softmax tests (fp32 1e-5 relative, and 2^-147 below the normal range; bf16 1 ulp). The emulated cases run the kernels'
source on the CPU between guard pages, so an access outside a row's tensor ends them; a stopped clock makes a wait end
by its pairs only."""

import ctypes
import os

import pytest
import torch

from _emu import build, run
from _util import assert_rel, assert_ulp, bits16


@pytest.fixture(scope="module")
def emu_softmax(tmp_path_factory):
    return build(tmp_path_factory.mktemp("emu_any_rows"), "softmax.hip", "emu_softmax.cpp")


# cols around one vector, one wave's vectors, and the steps of the waves and of the vectors per lane
EDGES = {0: [4, 5, 255, 257, 1023, 1025, 2047, 4097, 8191], 1: [8, 9, 511, 513, 2049, 3001, 4095, 8193]}


@pytest.mark.parametrize("dtype,cols", [(d, c) for d in EDGES for c in EDGES[d]])
def test_emulated_row_edges(emu_softmax, dtype, cols):
    # offset 1: the buffers begin one element past a 16-byte boundary (and rows of a whole number of vectors are
    # unaligned)
    run(emu_softmax, [9, cols, dtype, 1, cols, 0, 0, 1, "special"])


# rows of one vector to 64 of them (fp32 4 to 256 columns, bf16 8 to 512) in softmax_short, numbers of rows that leave a
# wave's sets empty or take several steps
SHORT = [(1, 4, 0), (3, 5, 0), (17, 63, 0), (16, 64, 0), (9, 65, 0), (33, 127, 0), (8200, 130, 0), (1, 8, 1),
         (70, 9, 1), (15, 127, 1), (40, 129, 1), (8, 256, 1), (8193, 257, 1)]


@pytest.mark.parametrize("pattern", ["randn", "special"])
@pytest.mark.parametrize("rows,cols,dtype", SHORT)
def test_emulated_short_rows(emu_softmax, rows, cols, dtype, pattern):
    run(emu_softmax, [rows, cols, dtype, 0, cols, 0, 0, cols % 4, pattern], env=dict(os.environ, EMU_SHORT="1"))


# where rows begin to share waves (256 CUs): workgroups of one wave of 16 or 8 rows, or of four waves of a row each
@pytest.mark.parametrize("rows,cols,dtype,offset,workgroups", [(64, 64, 0, 0, 16), (4095, 64, 0, 0, 512),
                                                               (4096, 64, 0, 0, 256),
                                                               (64, 128, 1, 1, 16), (4096, 200, 1, 0, 512),
                                                               (4096, 200, 0, 0, 512), (8192, 200, 0, 0, 256)])
def test_emulated_few_short_rows(emu_softmax, rows, cols, dtype, offset, workgroups):
    out = run(emu_softmax, [rows, cols, dtype, 0, rows, 0, 0, offset])
    assert int(out.split("workgroups ")[1].split(",")[0]) == workgroups, out


@pytest.mark.parametrize("dtype,waves,nv", [(0, 1, 8), (0, 2, 4), (0, 16, 1), (1, 1, 8), (1, 8, 2)])
@pytest.mark.parametrize("env", [{}, {"EMU_WAVE_AHEAD": "1"}], ids=["lanes", "waves_ahead"])
def test_emulated_row_shapes(emu_softmax, dtype, waves, nv, env):
    run(emu_softmax, [21, 1999, dtype, 1, 5, waves, nv, 3, "randn"], env=dict(os.environ, **env))


# rows, cols, dtype, row groups: chunks of 16384 elements and of a quarter of them (few rows), a last chunk of one
# vector
COOP = [(2, 65539, 0, 0), (1, 4 * 4096 + 1, 0, 0), (3, 40001, 1, 0), (5, 16384 * 2 + 5, 0, 2), (5, 16384 * 3 - 1, 1, 3)]


@pytest.mark.parametrize("rows,cols,dtype,groups", COOP)
@pytest.mark.parametrize("pattern", ["randn", "special"])
def test_emulated_coresident(emu_softmax, rows, cols, dtype, groups, pattern):
    run(emu_softmax, [rows, cols, dtype, 4, 3, 0, groups, 1, pattern, 3], env=dict(os.environ, EMU_CLOCK_STOPPED="1"),
        concurrent=True, weak=True, timeout=300)


@pytest.mark.parametrize("rows,cols,dtype,groups", COOP)
def test_emulated_coresident_fallback(emu_softmax, rows, cols, dtype, groups):
    run(emu_softmax, [rows, cols, dtype, 4, 3, 0, groups, 1, "special", 2, 1])


# rows whose middle half is masked, NaN among the masked elements or elsewhere: whole chunks of -inf and NaN. tier 0 is
# the automatic choice (rows of the row tier's lengths that an eager launch hands to the co-resident tier), 4 the
# co-resident tier; rows, cols, dtype, tier, row groups
NAN_ROWS = [(2, 30000, 0, 0, 0), (2, 49999, 0, 0, 0), (2, 49152, 1, 0, 0), (2, 60001, 1, 0, 0), (5, 70000, 0, 4, 0),
            (5, 70001, 0, 4, 0), (5, 49152, 1, 4, 0), (5, 49153, 1, 4, 0), (5, 70000, 0, 4, 2), (5, 70001, 0, 4, 2),
            (5, 70000, 1, 4, 2), (5, 70001, 1, 4, 2)]


@pytest.mark.parametrize("rows,cols,dtype,tier,groups", NAN_ROWS)
@pytest.mark.parametrize("ticks", [0, 1], ids=["pairs", "fallback"])
def test_emulated_coresident_nan(emu_softmax, rows, cols, dtype, tier, groups, ticks):
    env = dict(os.environ) if ticks else dict(os.environ, EMU_CLOCK_STOPPED="1")
    run(emu_softmax, [rows, cols, dtype, tier, 3, 0, groups, 0, "nan", 1, ticks], env=env, concurrent=not ticks,
        timeout=300)


# bf16 rows by expf and a division (the scalar kernel) or in the row tier before the vector tiers took them: 32-bit
# arithmetic is off by a few 2^-24 before the one rounding to bf16, whose boundaries lie 1 / 185 of the value's inverse
# apart on the mean: 3.2e-7 on the mean rounds 6e-5 of the elements otherwise (exp_narrow's error 1.3e-4 and more)
BITS = [(2000, 200, 1), (9000, 500, 1), (400, 1000, 1), (300, 1001, 0), (600, 301, 0), (60, 40000, 0), (12, 40001, 0)]


@pytest.mark.parametrize("rows,cols,offset", BITS)
def test_emulated_bf16_rounding(emu_softmax, rows, cols, offset):
    env = dict(os.environ, EMU_CLOCK_STOPPED="1")
    out = run(emu_softmax, [rows, cols, 1, 0, 1, 0, 0, offset], env=env, concurrent=cols > 32768)
    assert int(out.split("other bits ")[1].split()[0]) <= 6e-5 * rows * cols, out


@pytest.mark.parametrize("cols,dtype,groups", [(4 * 4096 + 1, 1, 0), (4 * 4096 + 7, 1, 0), (2 * 16384 + 3, 1, 1),
                                               (4097, 0, 0), (16384 + 3, 0, 1)])
def test_emulated_last_chunk_writes_its_own(emu_softmax, cols, dtype, groups):
    # a last chunk of less than a vector, whose workgroup loads the row's last whole vector: the elements of the chunk
    # before are its workgroup's to write, whose rounding may be another; two rows, so that one group loops
    own = cols % 4096 if groups == 0 else cols % 16384
    chunks = cols // (4096 if groups == 0 else 16384) + 1
    env = dict(os.environ, EMU_ONLY=str(chunks - 1))
    rows = 2 if groups else 1
    out = run(emu_softmax, [rows, cols, dtype, 4, 3, 0, groups, 0, "randn", 1, 1], env=env, expect_ok=False)
    written = [int(i) for i in out.split("written")[0].split()]
    assert written == [r * cols + i for r in range(rows) for i in range(cols - own, cols)]


@pytest.mark.parametrize("cols", [3, 5, 300])
def test_emulated_exponential(emu_softmax, cols):
    # rows of 0, d and -inf with d down to -104: exp(d) / (1 + exp(d)) by the exponential (about an ulp), the sum and
    # the quotient (half an ulp each), against the fp64 value rounded once (half an ulp): 2.5 ulps; by expf in the
    # scalar kernel (3 columns) as well
    out = run(emu_softmax, [6000, cols, 0, 0, 1, 0, 0, 0, "pair"])
    assert float(out.split("worst ")[1].split()[0]) <= 2.5, out


# rows, cols, dtype, kernel nodes of a captured launch: rows that an eager launch takes from the row tier stay there
# (one node), longer ones have the co-resident tier's tag node before theirs
CAPTURED = [(8, 30000, 0, 1), (8, 30001, 0, 1), (8, 60000, 1, 1), (8, 60001, 1, 1), (2, 33000, 0, 2), (2, 65537, 1, 2)]


@pytest.mark.parametrize("rows,cols,dtype,nodes", CAPTURED)
def test_emulated_captured_launches(emu_softmax, rows, cols, dtype, nodes):
    env = dict(os.environ, EMU_CLOCK_STOPPED="1", EMU_GRAPH="1")
    out = run(emu_softmax, [rows, cols, dtype, 0, 1, 0, 0, 0, "randn", 2], env=env, concurrent=True)
    assert int(out.split("graph nodes ")[1].split(",")[0]) == nodes, out


SAME = [(5, 50000, 0, 0), (5, 50001, 0, 0), (6, 70000, 0, 2), (6, 70001, 0, 2), (60, 20000, 0, 0), (6, 50000, 1, 2),
        (6, 50001, 1, 2), (4, 70000, 1, 0), (4, 70001, 1, 0)]


@pytest.mark.parametrize("rows,cols,dtype,groups", SAME)
@pytest.mark.parametrize("pattern", ["randn", "special"])
def test_emulated_coresident_same_bits(emu_softmax, rows, cols, dtype, groups, pattern):
    # by the pairs, and with the wait timed out (one workgroup after another: all but a row's last take pairs from x)
    args = [rows, cols, dtype, 4, 3, 0, groups, 0, pattern, 1]
    pairs = run(emu_softmax, args, env=dict(os.environ, EMU_CLOCK_STOPPED="1"), concurrent=True)
    alone = run(emu_softmax, [*args, 1])
    assert pairs.split("outputs ")[1][:16] == alone.split("outputs ")[1][:16]


# one row per workgroup: the workgroups of the chunk length chosen (256 CUs), where half of it would put more on a CU
# (bf16) and where it would not; fp32 a quarter
GRIDS = [(48, 33000, 1, 48 * 5), (24, 33000, 1, 24 * 9), (8, 70000, 1, 8 * 18), (20, 70000, 1, 20 * 9),
         (96, 33000, 1, 96 * 5), (50, 20000, 0, 50 * 5), (110, 20000, 0, 110 * 5),
         (14, 70000, 0, 14 * 18), (16, 70000, 0, 16 * 9)]


@pytest.mark.parametrize("rows,cols,dtype,workgroups", GRIDS)
def test_emulated_chunk_lengths(emu_softmax, rows, cols, dtype, workgroups):
    out = run(emu_softmax, [rows, cols, dtype, 0, 1, 0, 0, 0, "randn", 1, 1])
    assert int(out.split("workgroups ")[1].split(",")[0]) == workgroups, out


@pytest.mark.parametrize("rows,cols,offset", [(200, 5003, 0), (200, 8193, 0), (200, 10000, 1), (100, 16383, 0)])
def test_emulated_fp32_row_sums(emu_softmax, rows, cols, offset):
    # a row's outputs add up to 1 but for the error of its own sum (a common factor of the row): six additions at nearly
    # the whole sum, each off by 2.5e-8 on the mean square, are 6e-8; the scalar kernel's sums 6.8e-8 to 9.1e-8 here
    out = run(emu_softmax, [rows, cols, 0, 0, 1, 0, 0, offset])
    assert float(out.split("row sums off by ")[1].split()[0]) <= 6.6e-8, out


@pytest.mark.parametrize("rows,cols,dtype,waves", [(5, 4096, 0, 16), (5, 20000, 0, 4), (5, 8192, 1, 16),
                                                   (5, 2048, 1, 4)])
def test_emulated_stream_nan(emu_softmax, rows, cols, dtype, waves):
    # with a vector or two per lane, some lanes hold masked elements only
    run(emu_softmax, [rows, cols, dtype, 2, 3, waves, 0, 0, "nan"])


def _check(pkg, oracle, dev, rows, cols, dtype, offset=0, special=False):
    print(f"[softmax any] {rows}x{cols} {dtype} offset {offset}", flush=True)
    g = torch.Generator().manual_seed(rows * 131 + cols)
    x = torch.randn(rows, cols, generator=g) * 3
    if special:
        x[0, ::3] = float("-inf")
        x[-1] = float("-inf")
    x = x.to(dtype)
    n = rows * cols
    # at an offset into a buffer whose other elements must stay as they were: into another buffer, and in place
    buf = torch.full((n + 32,), 7.0, dtype=dtype)
    buf[offset:offset + n] = x.view(-1)
    lib = pkg.candidate("softmax")._lib
    for inplace in (False, True):
        src = buf.to(dev)
        dst = src if inplace else torch.full_like(src, 7.0)
        at = offset * src.element_size()
        err = lib.launch(src.data_ptr() + at, dst.data_ptr() + at, rows, cols, 0 if dtype == torch.float32 else 1, 256,
                         1024, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
        assert err == 0
        out = dst.cpu()
        assert (out[:offset] == 7).all() and (out[offset + n:] == 7).all()
        y = out[offset:offset + n].view(rows, cols)
        what = f"{rows}x{cols} in place {inplace}"
        if dtype == torch.float32:
            assert_rel(y.numpy(), oracle.softmax(x.numpy(), "fp32"), 1e-5, what, 2.0 ** -147)
        else:
            assert_ulp(bits16(y), oracle.softmax(bits16(x), "bf16"), 1, what)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
@pytest.mark.parametrize("rows,cols", [(3, 8), (70, 9), (40000, 8), (5000, 63), (70001, 64), (16385, 131), (9000, 255),
                                       (8191, 256), (8192, 257), (9001, 511), (20000, 512), (513, 255), (700, 513),
                                       (5, 2049), (300, 3001), (9, 8191), (600, 16383), (3, 16384), (40, 20001),
                                       (2, 32767),
                                       (300, 20000), (5, 65535), (3, 70001), (2, 262143), (70, 262143), (1, 1048576),
                                       (2, 1048577), (3, 16385), (9, 36869), (300, 49153)])
def test_gpu_rows(pkg, oracle, dev, dtype, rows, cols):
    _check(pkg, oracle, dev, rows, cols, dtype, offset=1, special=True)


@pytest.mark.gpu
@pytest.mark.parametrize("short", [1, 2], ids=["short", "row"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
@pytest.mark.parametrize("rows,cols,offset", [(3, 8, 0), (70, 9, 0), (1000, 64, 0), (333, 131, 0), (9000, 255, 1),
                                              (777, 256, 0), (5, 200, 3), (40000, 8, 0), (8193, 100, 0)])
def test_gpu_short_rows_either_way(pkg, oracle, dev, dtype, rows, cols, offset, short):
    lib = pkg.candidate("softmax")._lib
    lib.softmax_tune(9, short)
    try:
        _check(pkg, oracle, dev, rows, cols, dtype, offset=offset, special=True)
    finally:
        lib.softmax_tune(9, 0)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
@pytest.mark.parametrize("offset", [0, 1, 2, 3, 5, 7, 8])
def test_gpu_offsets(pkg, oracle, dev, dtype, offset):
    for rows, cols in ((7, 1024), (7, 1027), (3, 40000)):
        _check(pkg, oracle, dev, rows, cols, dtype, offset=offset)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
@pytest.mark.parametrize("rows,cols", [(5, 3001), (5, 4096), (5, 30000), (5, 49152), (5, 49999), (40, 70000),
                                       (5, 70001), (300, 70000), (300, 70001), (5, 1200000)])
@pytest.mark.parametrize("ticks", [0, 1])
def test_gpu_nan_among_masked(pkg, oracle, dev, dtype, rows, cols, ticks):
    # as test_emulated_coresident_nan: the row's middle half masked, in the row tiers and in the co-resident tier
    print(f"[softmax nan] {rows}x{cols} {dtype} ticks {ticks}", flush=True)
    x = torch.randn(rows, cols, generator=torch.Generator().manual_seed(cols)) * 3
    x[:, cols // 4:cols - cols // 4] = float("-inf")
    x[1::5, cols // 4:cols - cols // 4] = float("nan")
    x[0::5, cols // 2] = float("nan")
    x[2::5, cols - 1] = float("nan")
    x[3::5, 0] = float("inf")
    x = x.to(dtype)
    lib = pkg.candidate("softmax")._lib
    try:
        lib.softmax_tune(7, ticks)
        y = pkg.softmax(x.to(dev)).cpu()
    finally:
        lib.softmax_tune(7, 0)
    if dtype == torch.float32:
        assert_rel(y.numpy(), oracle.softmax(x.numpy(), "fp32"), 1e-5, "nan", 2.0 ** -147)
    else:
        assert_ulp(bits16(y), oracle.softmax(bits16(x), "bf16"), 1, "nan")


def _fp64(rows, cols, dtype, offset, seed, dev):
    """x at an offset into its buffer, and its softmax in fp64."""
    g = torch.Generator(device=dev).manual_seed(seed)
    buf = torch.empty(rows * cols + offset, device=dev, dtype=dtype)
    x = buf[offset:].view(rows, cols)
    x.copy_(torch.randn(rows, cols, device=dev, generator=g) * (3 if dtype == torch.bfloat16 else 1))
    return x, torch.softmax(x.double(), -1)


def _softmax_at(pkg, x, offset):
    y = torch.empty(x.numel() + offset, device=x.device, dtype=x.dtype)[offset:].view_as(x)
    dtype = 0 if x.dtype == torch.float32 else 1
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    assert pkg.candidate("softmax")._lib.launch(x.data_ptr(), y.data_ptr(), *x.shape, dtype, 256, 1024, stream) == 0
    return y


@pytest.mark.gpu
@pytest.mark.parametrize("rows,cols,offset", [(4096, 200, 1), (20000, 500, 1), (2000, 3001, 0), (512, 10000, 1),
                                              (600, 40000, 0), (600, 40000, 1), (300, 60000, 0), (256, 128256, 1)])
def test_gpu_bf16_rounding(pkg, dev, rows, cols, offset):
    # the elements rounded otherwise than the fp64 softmax's, as test_emulated_bf16_rounding; longer rows hold more
    # small elements, whose x - max is itself rounded (6.6e-5 of 600 x 40000 by expf and a division)
    print(f"[softmax bits] {rows}x{cols} offset {offset}", flush=True)
    x, e = _fp64(rows, cols, torch.bfloat16, offset, cols, dev)
    y = _softmax_at(pkg, x, offset)
    bits, unit = e.view(torch.int64), 1 << 45  # the lowest bit of bf16's seven in fp64's fraction
    once = ((bits + unit // 2 - 1 + ((bits >> 45) & 1)) & ~(unit - 1)).view(torch.float64)
    share = ((y.double() != once) & (e > 1e-37)).double().mean().item()
    assert share <= 9.5e-5, share


@pytest.mark.gpu
@pytest.mark.parametrize("rows,cols,offset", [(16, 50000, 0), (16, 128256, 0), (64, 128256, 0), (4, 262144, 0),
                                              (16, 262144, 1)])
def test_gpu_fp32_error_of_few_long_rows(pkg, dev, rows, cols, offset):
    # chunks of a half and a quarter of the longest: no further from the fp64 softmax than the longest ones (mean
    # relative error 1.34e-7 to 1.55e-7 over these shapes; 1.0e-7 to 1.1e-7 with one exponential of x - max)
    x, e = _fp64(rows, cols, torch.float32, offset, cols, dev)
    error = ((_softmax_at(pkg, x, offset).double() - e).abs() / e).mean().item()
    assert error <= 1.3e-7, error


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
@pytest.mark.parametrize("rows,cols,offset", [(16, 20000, 0), (5, 50000, 0), (5, 50000, 1), (24, 128256, 0),
                                              (1, 262143, 0), (300, 49152, 0), (300, 50000, 1), (300, 262144, 0)])
def test_gpu_timed_out_rows_have_the_same_bits(pkg, dev, dtype, rows, cols, offset):
    print(f"[softmax timed out] {rows}x{cols} {dtype} offset {offset}", flush=True)
    x, _ = _fp64(rows, cols, dtype, offset, cols, dev)
    lib = pkg.candidate("softmax")._lib
    by_pairs = _softmax_at(pkg, x, offset)
    try:
        lib.softmax_tune(7, 1)
        for _ in range(3):
            assert torch.equal(_softmax_at(pkg, x, offset), by_pairs)
    finally:
        lib.softmax_tune(7, 0)


@pytest.mark.gpu
def test_gpu_rows_on_two_streams(pkg, oracle, dev):
    # long rows on two streams at once, over and over: each launch has pair slots of its own
    g = torch.Generator().manual_seed(5)
    xs = [torch.randn(24, 30000, generator=g) for _ in range(2)]
    refs = [oracle.softmax(x.numpy(), "fp32") for x in xs]
    streams = [torch.cuda.Stream() for _ in range(2)]
    ds = [x.to(dev) for x in xs]
    torch.cuda.synchronize()
    ys = [[], []]
    for _ in range(20):
        for i in range(2):
            with torch.cuda.stream(streams[i]):
                ys[i].append(pkg.softmax(ds[i]))
    torch.cuda.synchronize()
    for i in range(2):
        for y in ys[i]:
            assert_rel(y.cpu().numpy(), refs[i], 1e-5, f"stream {i}", 2.0 ** -147)


@pytest.mark.gpu
def test_gpu_captured_rows_take_the_row_tier(pkg, oracle, dev):
    # a captured launch of rows that an eager launch hands to the co-resident tier, whose rounding is another: replays
    # on new values give the row tier's bits
    x = torch.empty(8, 30000, device=dev)
    lib = pkg.candidate("softmax")._lib
    pkg.softmax(x)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = pkg.softmax(x)
    for seed in range(3):
        h = torch.randn(8, 30000, generator=torch.Generator().manual_seed(seed)) * 3
        x.copy_(h)
        pkg.softmax(x + 1)
        graph.replay()
        torch.cuda.synchronize()
        assert_rel(y.cpu().numpy(), oracle.softmax(h.numpy(), "fp32"), 1e-5, f"replay {seed}", 2.0 ** -147)
        assert not torch.equal(y, pkg.softmax(x))
        try:
            lib.softmax_tune(5, 1)
            assert torch.equal(y, pkg.softmax(x))
        finally:
            lib.softmax_tune(5, 0)


@pytest.mark.gpu
@pytest.mark.parametrize("cols", [3, 5, 300])
def test_gpu_exponential(pkg, dev, cols):
    # as test_emulated_exponential, with the hardware's exp2 (an ulp) inside the exponential: 3 ulps
    print(f"[softmax exponential] {cols}", flush=True)
    d = torch.linspace(-103.9, 0, 60000, device=dev)
    x = torch.full((60000, cols), float("-inf"), device=dev)
    x[:, 0] = 0
    x[:, 1] = d
    y = pkg.softmax(x)[:, 1].double()
    exact = d.double().exp() / (1 + d.double().exp())
    ulp = torch.exp2((exact.log2().floor() - 23).clamp(min=-149))
    worst = ((y - exact).abs() / ulp).max().item()
    assert worst <= 3, worst


@pytest.mark.gpu
@pytest.mark.parametrize("rows,cols,dtype", [(600, 40000, torch.bfloat16), (1024, 50001, torch.bfloat16),
                                             (500, 20000, torch.float32), (64, 262144, torch.float32)])
def test_gpu_two_launches_that_fill_the_gpu(pkg, dev, rows, cols, dtype):
    # on two streams at once, over and over: each has the bits that it has alone
    print(f"[softmax two] {rows}x{cols} {dtype}", flush=True)
    xs = [(torch.randn(rows, cols, device=dev, generator=torch.Generator(device=dev).manual_seed(i)) * 3).to(dtype)
          for i in range(2)]
    alone = [pkg.softmax(x) for x in xs]
    streams = [torch.cuda.Stream() for _ in range(2)]
    torch.cuda.synchronize()
    for _ in range(4):
        ys = [[], []]
        for _ in range(5):
            for i in range(2):
                with torch.cuda.stream(streams[i]):
                    ys[i].append(pkg.softmax(xs[i]))
        torch.cuda.synchronize()
        assert all(torch.equal(y, alone[i]) for i in range(2) for y in ys[i])


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
def test_gpu_captured_unaligned_long_rows(pkg, oracle, dev, dtype):
    # unaligned rows beyond the row tier, recorded into a graph: fresh tags at every replay, eager launches in between
    x = torch.empty(3, 70001, device=dev, dtype=dtype)
    pkg.softmax(x)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = pkg.softmax(x)
    for seed in range(4):
        h = (torch.randn(3, 70001, generator=torch.Generator().manual_seed(seed)) * 3).to(dtype)
        x.copy_(h)
        if seed % 2:
            pkg.softmax(x + 1)
        graph.replay()
        torch.cuda.synchronize()
        if dtype == torch.float32:
            assert_rel(y.cpu().numpy(), oracle.softmax(h.numpy(), "fp32"), 1e-5, f"replay {seed}", 2.0 ** -147)
        else:
            assert_ulp(bits16(y), oracle.softmax(bits16(h), "bf16"), 1, f"replay {seed}")
