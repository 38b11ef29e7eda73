"""Atomic split-K on wave tiles of 32, 64 and 128 columns, whose adds leave as
64 consecutive dwords (two rows of 32, one of 64, half a row of 128), or from
a few workgroups of one 64-column wave as four dwords a lane, at the row and
column edges: the result against f64, the padding columns unwritten.

Bound per element: f32 products and sums in any order are off by at most
(K + splits + 1) eps times the sum of the magnitudes added."""
import numpy as np
import pytest
import torch

import mini_triton_nvgpu_v1_amd as tb
import oracle

pytestmark = pytest.mark.gpu

# (block, wave grid): wave tiles of 32, 64 (16-row passes, then 32) and 128 columns
TILES = [((64, 64, 64), (2, 2)), ((128, 64, 32), (4, 1)), ((128, 128, 64), (2, 2)),
         ((256, 128, 64), (4, 1)),
         # one wave: of 64 columns, 8 workgroups or fewer (with 3 splits one or two
         # tiles) add four columns a lane and more whole lines; of 128 whole lines
         ((64, 64, 32), (1, 1)), ((64, 128, 64), (1, 1))]


@pytest.mark.parametrize("block,grid", TILES)
@pytest.mark.parametrize("M,N", [(1, 8), (33, 136), (40, 72), (128, 128), (257, 72)])
def test_atomic_edges(block, grid, M, N, device):
    K, split, pad = 5 * block[2] + 8, 3, 8
    print(f"atomic {M}x{N}x{K} block {block} grid {grid}", flush=True)
    tiles = -(-M // block[0]) * -(-N // block[1])
    desc = tb.GemmDesc.from_config(
        m=M, n=N, k=K, lda=K, ldb=N, ldc=N + pad, c_dtype=tb.DTYPE_F32,
        acc_init=tb.ACC_INIT_LOAD_C, block_m=block[0], block_n=block[1], block_k=block[2],
        num_waves=grid[0] * grid[1], wave_grid_m=grid[0], wave_grid_n=grid[1], stages=2,
        mapping=tb.MAP_SPLIT_K, group_m=1, split_k=split, reduction=tb.RED_ATOMIC,
        num_programs=tiles * split, xcd_remap=0)
    A, B = oracle.config_inputs(M, N, K, 0x5EED0800 + M + N, oracle.UNIFORM)
    C0 = np.random.default_rng(M).standard_normal((M, N + pad)).astype(np.float32)
    dC = torch.from_numpy(C0.copy()).to(device)
    desc.launch(torch.from_numpy(A).to(device), torch.from_numpy(B).to(device), dC)
    got = dC.cpu().numpy()
    a, b = A.astype(np.float64), B.astype(np.float64)
    ref = C0[:, :N] + a @ b
    bound = (K + split + 1) * 2.0 ** -24 * (np.abs(C0[:, :N]) + np.abs(a) @ np.abs(b))
    assert (np.abs(got[:, :N] - ref) <= bound).all()
    assert np.array_equal(got[:, N:], C0[:, N:])
