"""The shrink over the whole reduction per workgroup (GPU) at the edges of its
tiles and pieces: rows 1 and 17 of 16-row tiles, K around the eight waves'
128-byte pieces, every block count, unaligned rows, rank-0 and clamped ranks."""

import pytest
import torch

from multi_lora_amd.kernels.lora_ops import Workspace, apply_segments, shrink
from multi_lora_amd.synthetic import make_meta
from oracle.lora_ref import apply_f64
from tests.gpu_helpers import assert_tol_f64
from tests.test_gpu_segments import case

pytestmark = pytest.mark.gpu

LENS, SLOTS, RANKS = [17, 1, 64, 0, 33, 150], [0, 1, 2, 0, 3, 1], [16, 5, 0, 12]


def run(dev, in_dim, n_slices, r_max, dtype, pad=0, ranks=RANKS, lens=LENS, slots=SLOTS):
    outs = [96] * n_slices
    x, a, b, base, cols, meta_cpu, scal = case(dev, lens, slots, ranks, in_dim, outs, r_max, dtype, in_dim + r_max)
    meta = make_meta(lens, slots, ranks, scal, dev, dtype)
    rows = torch.full((x.shape[0], in_dim + pad), float("nan"), dtype=dtype, device=dev)
    rows[:, :in_dim] = x.to(dev)
    xd, ad, bd = rows[:, :in_dim], [t.to(dev) for t in a], [t.to(dev) for t in b]
    got = base.to(dev)
    apply_segments(xd, ad, bd, meta, got, cols, workspace=Workspace())
    assert_tol_f64(got.cpu(), apply_f64(x, a, b, meta_cpu, base, cols), f"{in_dim} {n_slices}x{r_max} {dtype}")
    mid = torch.full((x.shape[0], n_slices * r_max + 3), 7.0, dtype=dtype, device=dev)
    shrink(xd, ad, meta, mid, workspace=Workspace())
    want = torch.zeros(x.shape[0], n_slices, r_max, dtype=torch.float64)
    r0 = 0
    for n, s in zip(lens, slots):
        r = min(ranks[s], r_max)
        for i in range(n_slices):
            want[r0:r0 + n, i, :r] = x[r0:r0 + n].double() @ a[i][s, :r].double().T
        r0 += n
    assert_tol_f64(mid[:, :n_slices * r_max].cpu(), want.reshape(x.shape[0], -1))
    assert bool((mid[:, n_slices * r_max:] == 7).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("in_dim", [8, 64, 72, 504, 512, 520, 1000, 1096])
def test_k_edges(dev, in_dim, dtype):
    run(dev, in_dim, 1, 16, dtype)


@pytest.mark.parametrize("n_slices,r_max,ranks", [(1, 8, [8, 3, 0, 8]), (2, 16, RANKS), (3, 16, RANKS), (2, 32, [32, 17, 0, 9]),
                                                  (3, 32, [32, 17, 0, 30]), (4, 32, [20, 32, 0, 1]), (1, 128, [128, 70, 0, 100]),
                                                  (3, 64, [64, 20, 0, 48])])
def test_block_counts(dev, n_slices, r_max, ranks):
    run(dev, 328, n_slices, r_max, torch.float16, ranks=ranks)
    run(dev, 328, n_slices, r_max, torch.float32, ranks=ranks)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("in_dim,pad", [(1, 0), (63, 0), (65, 1), (511, 0), (1001, 0), (1024, 4), (1024, 1)])
def test_unaligned_rows(dev, in_dim, pad, dtype):
    run(dev, in_dim, 2, 12, dtype, pad=pad)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("in_dim", [4101, 2111])
@pytest.mark.parametrize("n_slices,r_max,ranks", [(1, 16, [16, 5, 0, 12]), (2, 16, [16, 5, 0, 12]),
                                                  (2, 32, [32, 17, 0, 9]), (4, 32, [32, 20, 0, 30])])
def test_unaligned_long_k(dev, in_dim, n_slices, r_max, ranks, dtype):
    # Long enough for every wave to load pieces again, by block count.
    run(dev, in_dim, n_slices, r_max, dtype, ranks=ranks)


@pytest.mark.parametrize("in_dim,r_max", [(4100, 16), (2052, 48)])
def test_fp32_long_k(dev, in_dim, r_max):
    run(dev, in_dim, 1, r_max, torch.float32, ranks=[r_max, 5, 0, 12])


def test_many_one_row_segments_in_fp32(dev):
    run(dev, 520, 2, 16, torch.float32, ranks=[16, 8, 0, 3], lens=[1] * 150, slots=[i % 4 for i in range(150)])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("in_dim,r_max,pad,lens", [(4101, 8, 0, [17]), (14001, 64, 0, [20, 1]), (14336, 16, 4, [300])])
def test_unaligned_rows_of_few_tiles_are_split(dev, in_dim, r_max, pad, lens, dtype):
    # The last shape plans 128-row tiles when its rows are aligned.
    run(dev, in_dim, 1, r_max, dtype, pad=pad, ranks=[r_max, 5], lens=lens, slots=list(range(len(lens))))


def test_unaligned_decode_rows_get_the_workspace_they_need(dev):
    run(dev, 4096, 1, 20, torch.bfloat16, pad=4, ranks=[20, 9, 0, 17], lens=[1] * 200, slots=[i % 4 for i in range(200)])
