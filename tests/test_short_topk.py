"""Top-k of short rows (topk_short): every lane layout at its smallest and largest row, k from 1 to a whole row, ties,
negative rows and the all-ones NaN, rows that do not fill a wave or a workgroup; bit for bit against the oracle. The
emulated cases run the kernel's source on the CPU between guard pages."""

import os

import numpy as np
import pytest
import torch

from _emu import build, run
from _util import bits16


@pytest.fixture(scope="module")
def emu_topk(tmp_path_factory):
    return build(tmp_path_factory.mktemp("emu_short_topk"), "topk.hip", "emu_topk.cpp")


# rows, cols, dtype, ks, pattern: cols at the edges of the layouts (64, 128, 256, 512, 1024), odd ones between
CASES = [(1, 1, 0, "1", "randn"), (7, 3, 1, "1,3", "ints"), (5, 61, 0, "7,61", "randn"), (17, 64, 0, "8,64", "negative"),
         (18, 65, 0, "2,33", "allones"), (33, 128, 1, "8,64", "ints"), (19, 129, 0, "16,64", "randn"),
         (9, 256, 1, "1,64", "allones"), (6, 257, 1, "16,33", "negative"), (3, 512, 0, "32", "descending"),
         (5, 513, 1, "13,32", "ints"), (4, 1023, 0, "1,16", "ascending"), (3, 1024, 1, "32", "outlier")]


@pytest.mark.parametrize("rows,cols,dtype,ks,pattern", CASES)
def test_emulated_short_rows(emu_topk, rows, cols, dtype, ks, pattern):
    run(emu_topk, [rows, cols, dtype, ks, 0, 2048, 1, cols, -1, pattern])


@pytest.mark.parametrize("rows,cols,dtype,ks,pattern", CASES[3:6])
def test_emulated_short_rows_shuffled_and_low_guard(emu_topk, rows, cols, dtype, ks, pattern):
    run(emu_topk, [rows, cols, dtype, ks, 0, 2048, 1, 5, 99, pattern], env=dict(os.environ, EMU_ALIGN_START="1"))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
@pytest.mark.parametrize("rows,cols", [(1, 16), (50, 63), (4097, 64), (1000, 65), (16384, 128), (300, 129), (77, 256),
                                       (2048, 257), (65535, 40), (63, 512), (9, 513), (2050, 1024), (31, 1023)])
def test_gpu_short_rows(pkg, oracle, dev, dtype, rows, cols):
    g = torch.Generator().manual_seed(rows + cols)
    for k in sorted({1, min(8, cols), min(16, cols), min(33, cols), min(64, cols)}):
        x = torch.randn(rows, cols, generator=g) * 2
        if k % 2 == 0:
            x = x.round()  # ties
        x = x.to(dtype)
        x[0] = float("-inf")
        x[-1, ::2] = float("nan")
        print(f"[topk short] {rows}x{cols} {dtype} k={k}", flush=True)
        v, i = pkg.topk(x.to(dev), k)
        raw = x.numpy() if dtype == torch.float32 else bits16(x)
        rv, ri = oracle.topk(raw, k, "fp32" if dtype == torch.float32 else "bf16")
        got = v.cpu().numpy().view(np.uint32) if dtype == torch.float32 else bits16(v)
        ref = rv.view(np.uint32) if dtype == torch.float32 else rv
        assert np.array_equal(i.cpu().numpy(), ri) and np.array_equal(got, ref)
