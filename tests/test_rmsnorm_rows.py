"""RMSNorm of short rows (rmsnorm_short: sixteen lanes per row, sixteen rows per wave and step): rows of one vector, of
just under, exactly and just over one and two vectors per lane, and numbers of rows that leave sets, waves and blocks
partly empty or take several steps; and of rows of any length and element alignment (the row kernel's kAny form), where
a row's last vector, a wave's share or the next shape begins, with the fused residual in place, whose last vector overlaps
another lane's. Bit for bit against the oracle, as every RMSNorm path. The emulated cases run the kernels' source on the
CPU between guard pages."""

import os

import pytest
import torch

from _emu import build, run
from _util import bits16, same_bits16


@pytest.fixture(scope="module")
def emu_rmsnorm(tmp_path_factory):
    return build(tmp_path_factory.mktemp("emu_short_rmsnorm"), "rmsnorm.hip", "emu_rmsnorm.cpp")


# rows, cols, dtype (1 bf16, 2 fp16), mode (0 plain, 1 weighted), seed
CASES = [(1, 8, 1, 1), (3, 64, 2, 0), (4, 120, 1, 1), (15, 128, 1, 1), (16, 128, 2, 1), (17, 136, 1, 1),
         (65, 192, 2, 0), (100, 248, 1, 1), (33, 256, 1, 1)]


@pytest.mark.parametrize("rows,cols,dtype,mode", CASES)
def test_emulated_short_rows(emu_rmsnorm, rows, cols, dtype, mode):
    run(emu_rmsnorm, [rows, cols, dtype, mode, rows + cols, 0, 0, 0, 0], env=dict(os.environ, EMU_SHORT="1"))


# where rows begin to share waves (256 CUs): one-wave workgroups of sixteen rows, or four-wave ones of a row a wave
@pytest.mark.parametrize("rows,cols,workgroups", [(64, 128, 16), (3071, 128, 768), (3072, 128, 192), (64, 256, 16),
                                                  (7168, 256, 448)])
def test_emulated_few_short_rows(emu_rmsnorm, rows, cols, workgroups):
    out = run(emu_rmsnorm, [rows, cols, 1, 1, rows, 0, 0, 0, 0])
    assert int(out.split("workgroups ")[1].split()[0]) == workgroups, out


# rows, cols, mode (0 plain, 1 weighted, 2 add, 3 add in place), waves, nv, offset (elements off a 16-byte boundary)
ANY = [(5, 9, 1, 0, 0, 0), (9, 511, 0, 0, 0, 0), (9, 513, 3, 0, 0, 0), (6, 2049, 3, 0, 0, 0), (5, 4097, 3, 0, 0, 0),
       (7, 1030, 3, 2, 2, 0), (7, 4096, 1, 0, 0, 3), (5, 128, 1, 0, 0, 1), (3, 1025, 2, 4, 1, 0), (9, 3001, 3, 8, 1, 0)]


@pytest.mark.parametrize("env", [{}, {"EMU_WAVE_AHEAD": "1"}], ids=["lanes", "waves_ahead"])
@pytest.mark.parametrize("rows,cols,mode,waves,nv,offset", ANY)
def test_emulated_any_rows(emu_rmsnorm, rows, cols, mode, waves, nv, offset, env):
    run(emu_rmsnorm, [rows, cols, 1, mode, rows + cols, waves, nv, 1, offset], env=dict(os.environ, **env))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("rows,cols", [(3, 9), (700, 100), (513, 511), (600, 513), (2000, 1129), (1100, 2049),
                                       (300, 5121), (520, 4095), (40, 16385), (20, 65533), (2, 65537)])
def test_gpu_any_rows(pkg, oracle, dev, dtype, rows, cols):
    print(f"[rmsnorm any] {rows}x{cols} {dtype}", flush=True)
    g = torch.Generator().manual_seed(rows + cols)
    x, r = (torch.randn(rows, cols, generator=g).to(dtype) for _ in range(2))
    x[:, ::7] = -0.0
    w = (torch.rand(cols, generator=g) + 0.5).to(dtype)
    fp16 = dtype == torch.float16
    name = "fp16" if fp16 else "bf16"
    y = pkg.rmsnorm(x.to(dev), w.to(dev))
    assert same_bits16(bits16(y), oracle.rmsnorm(bits16(x), bits16(w), dtype=name), fp16)
    ry, rh = oracle.rmsnorm_add(bits16(x), bits16(r), bits16(w), dtype=name)
    y, h = pkg.rmsnorm_add(x.to(dev), r.to(dev), w.to(dev))
    assert same_bits16(bits16(h), rh, fp16) and same_bits16(bits16(y), ry, fp16)
    # everything in place, one element past a 16-byte boundary: residual_out = residual, y = x
    def off(t):
        buf = torch.zeros(t.numel() + 16, dtype=dtype, device=dev)
        buf[1:1 + t.numel()] = t.view(-1).to(dev)
        return buf
    xd, rd, wd = off(x), off(r), off(w)
    lib, at = pkg.candidate("rmsnorm")._lib, lambda t: t.data_ptr() + 2
    assert lib.rmsnorm_add_launch(at(xd), at(rd), at(wd), at(xd), at(rd), rows, cols, 2 if fp16 else 1, 1e-6, 256,
                                  torch.cuda.current_stream().cuda_stream) == 0
    n = rows * cols
    assert same_bits16(bits16(rd[1:1 + n].view(rows, cols)), rh, fp16)
    assert same_bits16(bits16(xd[1:1 + n].view(rows, cols)), ry, fp16)
    assert (xd[0] == 0) and (xd[1 + n:] == 0).all() and (rd[0] == 0) and (rd[1 + n:] == 0).all()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("cols", [7, 64, 256, 1000, 1001, 4096, 5120, 16384, 70000])
def test_gpu_negative_zeros(pkg, oracle, dev, dtype, cols):
    # -0 stays -0 through both products in every form of the kernel: short, part and full rows, any rows, scalar rows
    print(f"[rmsnorm -0] 9x{cols} {dtype}", flush=True)
    g = torch.Generator().manual_seed(cols)
    x = torch.randn(9, cols, generator=g).to(dtype)
    x[:, ::3] = -0.0
    x[4] = -0.0
    r = torch.randn(9, cols, generator=g).to(dtype)
    r[:, ::2] = -0.0
    w = (torch.rand(cols, generator=g) - 0.5).to(dtype)
    fp16 = dtype == torch.float16
    name = "fp16" if fp16 else "bf16"
    for weight in (w, None):
        y = pkg.rmsnorm(x.to(dev), None if weight is None else weight.to(dev))
        ref = oracle.rmsnorm(bits16(x), None if weight is None else bits16(weight), dtype=name)
        assert same_bits16(bits16(y), ref, fp16)
    ry, rh = oracle.rmsnorm_add(bits16(x), bits16(r), bits16(w), dtype=name)
    y, h = pkg.rmsnorm_add(x.to(dev), r.to(dev), w.to(dev))
    assert same_bits16(bits16(h), rh, fp16) and same_bits16(bits16(y), ry, fp16)


@pytest.mark.gpu
@pytest.mark.parametrize("short", [0, 1], ids=["auto", "short"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("rows,cols", [(1, 8), (5, 64), (16, 80), (17, 96), (4095, 128), (16384, 128), (16401, 136),
                                       (40000, 192), (163841, 128), (70000, 256), (300, 264), (70001, 512)])
def test_gpu_short_rows(pkg, oracle, dev, dtype, rows, cols, short):
    print(f"[rmsnorm short] {rows}x{cols} {dtype} {short}", flush=True)
    lib = pkg.candidate("rmsnorm")._lib
    lib.rmsnorm_tune(5, short)
    try:
        _short_rows(pkg, lib, oracle, dev, dtype, rows, cols)
    finally:
        lib.rmsnorm_tune(5, 0)


def _short_rows(pkg, lib, oracle, dev, dtype, rows, cols):
    g = torch.Generator().manual_seed(rows + cols)
    x = (torch.randn(rows, cols, generator=g) * torch.rand(rows, 1, generator=g) * 3).to(dtype)
    x[rows // 2, cols // 2] = float("nan")
    x[0] = 0
    w = (torch.rand(cols, generator=g) + 0.5).to(dtype)
    fp16 = dtype == torch.float16
    name = "fp16" if fp16 else "bf16"
    for weight in (w, None):
        y = pkg.rmsnorm(x.to(dev), None if weight is None else weight.to(dev), 1e-5)
        ref = oracle.rmsnorm(bits16(x), None if weight is None else bits16(weight), eps=1e-5, dtype=name)
        assert same_bits16(bits16(y), ref, fp16)
    d = x.to(dev)  # in place through the C entry point
    assert lib.launch(d.data_ptr(), d.data_ptr(), rows, cols, 2 if fp16 else 1, 1e-5, 256,
                      torch.cuda.current_stream().cuda_stream) == 0
    assert same_bits16(bits16(d), ref, fp16)
