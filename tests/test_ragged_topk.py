"""Top-k of rows at any element alignment (16-byte loads at the rows' own alignment, the last vector of a tile shifted
into place): every remainder of a row by the vector width, tiles and chunks ending anywhere, rows shorter than a
vector, for each kernel (k = 1, up to 64, up to 1024); bit for bit against the oracle. The emulated cases run the
kernels' source on the CPU between guard pages, so a load outside the row's tensor ends them."""

import os

import numpy as np
import pytest
import torch

from _emu import build, run
from _util import bits16


@pytest.fixture(scope="module")
def emu_topk(tmp_path_factory):
    return build(tmp_path_factory.mktemp("emu_ragged_topk"), "topk.hip", "emu_topk.cpp")


# rows, cols, dtype, ks, chunk (0: plan's), pattern
CASES = [(2, 20001, 0, "1,50,300", 4096, "randn"), (2, 20003, 1, "1,50,300", 4096, "randn"),
         (2, 16385, 1, "1,13,100", 16385, "ints"), (1, 32767, 1, "1,50,1024", 0, "randn"),
         (2, 2053, 1, "1,64,65", 2052, "negative"), (2, 30001, 0, "50,300", 4100, "ascending"),
         (2, 49999, 1, "1,50", 0, "allones"), (1, 5, 1, "1,2,5", 0, "randn"), (1, 3, 0, "1,3", 0, "randn")]


@pytest.mark.parametrize("rows,cols,dtype,ks,chunk,pattern", CASES)
def test_emulated_ragged_rows(emu_topk, rows, cols, dtype, ks, chunk, pattern):
    run(emu_topk, [rows, cols, dtype, ks, chunk, 2048, 1, cols, -1, pattern])


@pytest.mark.parametrize("dtype", [0, 1])
def test_emulated_ragged_rows_low_guard(emu_topk, dtype):
    run(emu_topk, [2, 18003, dtype, "1,50,100", 6004, 2048, 1, 3, 9, "randn"], env=dict(os.environ, EMU_ALIGN_START="1"),
        concurrent=True, weak=True)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
@pytest.mark.parametrize("rows,cols", [(3, 16001), (2, 16002), (5, 16003), (1, 20004), (2, 20005), (3, 20006), (2, 20007),
                                       (4, 16385), (3, 32767), (64, 49999), (1, 128257), (20, 65537), (300, 30011),
                                       (2, 1500), (7, 1025)])
def test_gpu_ragged_rows(pkg, oracle, dev, dtype, rows, cols):
    g = torch.Generator().manual_seed(rows + cols)
    x = torch.randn(rows, cols, generator=g) * 2
    x[:, -1] = 9.0  # the last element is among the largest: the shifted vector's values and indices are seen
    x[:, -3:-1] = 9.0
    x[0, 0] = 9.0
    x = x.to(dtype)
    raw = x.numpy() if dtype == torch.float32 else bits16(x)
    name = "fp32" if dtype == torch.float32 else "bf16"
    for k in (1, 2, 50, 64, 65, 300, 1024):
        print(f"[topk ragged] {rows}x{cols} {name} k={k}", flush=True)
        k = min(k, cols)
        v, i = pkg.topk(x.to(dev), k)
        rv, ri = oracle.topk(raw, k, name)
        got, ref = (v.cpu().numpy().view(np.uint32), rv.view(np.uint32)) if name == "fp32" else (bits16(v), rv)
        assert np.array_equal(i.cpu().numpy(), ri) and np.array_equal(got, ref)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
def test_gpu_rows_off_a_vector_boundary(pkg, oracle, dev, dtype):
    # rows of whole vectors in a tensor that begins 1 to 7 elements past a 16-byte boundary
    g = torch.Generator().manual_seed(8)
    x = (torch.randn(3, 24000, generator=g) * 2).to(dtype)
    name = "fp32" if dtype == torch.float32 else "bf16"
    rv, ri = oracle.topk(x.numpy() if name == "fp32" else bits16(x), 50, name)
    for offset in range(1, 8):
        buf = torch.zeros(x.numel() + 8, dtype=dtype, device=dev)
        at = buf[offset:offset + x.numel()].view(3, 24000)
        at.copy_(x)
        v, i = pkg.topk(at, 50)
        assert np.array_equal(i.cpu().numpy(), ri)
        assert np.array_equal(v.cpu().numpy() if name == "fp32" else bits16(v), rv)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
@pytest.mark.parametrize("rows,cols", [(64, 50000), (39, 17920), (16, 132352), (143, 33536), (300, 17152), (2, 41984),
                                       (4, 17152), (90, 37070), (300, 49160)])
def test_gpu_rows_whose_last_chunk_would_be_short(pkg, oracle, dev, dtype, rows, cols):
    # full chunks of 16384 (or 8192) columns would leave a short one at the end; the launch makes the chunks equal
    g = torch.Generator().manual_seed(rows + cols)
    x = (torch.randn(rows, cols, generator=g) * 2).to(dtype)
    x[:, -1] = 11.0
    raw = x.numpy() if dtype == torch.float32 else bits16(x)
    name = "fp32" if dtype == torch.float32 else "bf16"
    for k in (1, 8, 64, 100, 1024):
        print(f"[topk chunks] {rows}x{cols} {name} k={k}", flush=True)
        v, i = pkg.topk(x.to(dev), k)
        rv, ri = oracle.topk(raw, k, name)
        got, ref = (v.cpu().numpy().view(np.uint32), rv.view(np.uint32)) if name == "fp32" else (bits16(v), rv)
        assert np.array_equal(i.cpu().numpy(), ri) and np.array_equal(got, ref)
