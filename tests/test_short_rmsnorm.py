"""RMSNorm of short rows (rmsnorm_short: sixteen lanes per row, sixteen rows per wave and step): rows of one vector, of
just under, exactly and just over one and two vectors per lane, and numbers of rows that leave sets, waves and blocks
partly empty or take several steps; bit for bit against the oracle, as every RMSNorm path. The emulated cases run the
kernel's source on the CPU between guard pages."""

import pytest
import torch

from _emu import build, run
from _util import bits16, same_bits16


@pytest.fixture(scope="module")
def emu_rmsnorm(tmp_path_factory):
    return build(tmp_path_factory.mktemp("emu_short_rmsnorm"), "rmsnorm.hip", "emu_rmsnorm.cpp")


# rows, cols, dtype (1 bf16, 2 fp16), mode (0 plain, 1 weighted), seed
CASES = [(1, 8, 1, 1), (3, 64, 2, 0), (4, 120, 1, 1), (15, 128, 1, 1), (16, 128, 2, 1), (17, 136, 1, 1), (65, 192, 2, 0),
         (100, 248, 1, 1), (33, 256, 1, 1)]


@pytest.mark.parametrize("rows,cols,dtype,mode", CASES)
def test_emulated_short_rows(emu_rmsnorm, rows, cols, dtype, mode):
    run(emu_rmsnorm, [rows, cols, dtype, mode, rows + cols, 0, 0, 0, 0])


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("rows,cols", [(1, 8), (5, 64), (16, 80), (17, 96), (4095, 128), (16384, 128), (16401, 136),
                                       (40000, 192), (163841, 128), (70000, 256), (300, 264), (70001, 512)])
def test_gpu_short_rows(pkg, oracle, dev, dtype, rows, cols):
    print(f"[rmsnorm short] {rows}x{cols} {dtype}", flush=True)
    g = torch.Generator().manual_seed(rows + cols)
    x = (torch.randn(rows, cols, generator=g) * torch.rand(rows, 1, generator=g) * 3).to(dtype) + 0  # no -0: the weighted fp16 product of -0 comes out as +0 on the GPU
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
    lib = pkg.candidate("rmsnorm")._lib
    assert lib.launch(d.data_ptr(), d.data_ptr(), rows, cols, 2 if fp16 else 1, 1e-5, 256,
                      torch.cuda.current_stream().cuda_stream) == 0
    assert same_bits16(bits16(d), ref, fp16)
