"""Paged and contiguous calls of 2 .. 9 query tokens per sequence against the
oracle: row groups whose keys are split over the waves of a workgroup (two or
four wave sets, dvattention_amd/csrc/dv_chunk.hip) and the first size past it.
Lengths end inside the first stage, the first step of a split and a later one,
so some wave sets see no key; ragged batches also leave pieces of a few keys to
merge.  Packed batches mix short row groups with long ones.  Tolerances:
test_gpu_parity.close."""
import numpy as np
import pytest
import torch

from oracle import dvattn_oracle as O
from test_gpu_parity import close, dv, rand_paged, rand_varlen, run_paged, run_varlen  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("S", [2, 3, 4, 5, 8, 9])
@pytest.mark.parametrize("W,Hkv,bs,lens", [(2, 1, 16, [1]), (3, 2, 16, [33, 5]), (1, 4, 24, [128, 97]),
                                           (5, 8, 16, [1500]), (2, 2, 32, [700, 0, 261])])
def test_paged_few_tokens(dv, gpu, dtype, S, W, Hkv, bs, lens):  # noqa: F811
    F = len(lens)
    rng = np.random.default_rng(17 * S + sum(lens))
    loc = rng.integers(-1, max(lens), size=(F, W, 1)) - S + 1 + np.arange(S)  # causal, some rows see no key
    d = rand_paged(F, W, S, Hkv, bs, lens, 64, dtype, seed=S + bs, loc=loc, k_scale=2.0)
    close(run_paged(dv, d, 0.1, gpu), O.paged_sdpa(0.1, **d), dtype, f"S={S}")


@pytest.mark.parametrize("S", [2, 4, 7])
def test_contiguous_few_tokens(dv, gpu, S):  # noqa: F811
    F, W, Hkv, Ls = 2, 3, 2, [300, 45]
    g = torch.Generator().manual_seed(S)
    q = torch.randn(F, W, 16 * Hkv, S, 128, generator=g).to(torch.bfloat16)
    ks = [torch.randn(W, Hkv, L, 128, generator=g).to(torch.bfloat16) for L in Ls]
    vs = [torch.randn(W, Hkv, L, 128, generator=g).to(torch.bfloat16) for L in Ls]
    loc = torch.from_numpy(np.random.default_rng(S).integers(-1, 310, size=(F, W, S)).astype(np.int32))
    fl = torch.tensor(Ls, dtype=torch.int32)
    out = dv.dvattn_sdpa(q.to(gpu), loc.to(gpu), [k.to(gpu) for k in ks], [v.to(gpu) for v in vs], 0.1, fl.to(gpu))
    close(out, O.contig_sdpa(0.1, loc, q, fl, ks, vs), torch.bfloat16, f"S={S}")


# tokens per sequence: groups of 4 or fewer split their keys, longer ones in the same
# launch do not; pages that are and are not a power of two, pieces cut inside groups
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("bs", [16, 24])
@pytest.mark.parametrize("counts,lens", [
    ([1, 1, 40, 1, 3], [700]), ([4, 5, 16, 17, 20, 21, 0, 1], [90, 40]), ([2, 2], [50]), ([16, 32], [300]),
    ([4] * 4, [600]), ([1, 1, 1, 29], [500]), ([1, 3], [9000]), ([3, 36], [5000]), ([1] * 6 + [30], [2000, 33, 0])])
def test_varlen_mixed_groups(dv, gpu, dtype, bs, counts, lens):  # noqa: F811
    W, T = len(counts), sum(counts)
    d = rand_varlen(len(lens), W, T, np.concatenate([[0], np.cumsum(counts)]), 2, bs, lens, 64, dtype, seed=T)
    close(run_varlen(dv, d, 0.1, gpu), O.varlen_paged_sdpa(0.1, **d), dtype, f"{counts}")


# keys per view around the number from which a short group's keys are split (96), one
# view and three, beside a long group
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("lens", [[95], [96], [97], [100, 100, 87], [100, 100, 88], [250, 38, 1]])
def test_varlen_split_from_96_keys(dv, gpu, dtype, lens):  # noqa: F811
    counts = [1, 4, 20, 2]
    W, T, F = len(counts), sum(counts), len(lens)
    d = rand_varlen(F, W, T, np.concatenate([[0], np.cumsum(counts)]), 2, 16, lens, 64, dtype, seed=sum(lens))
    d["locations"] = torch.from_numpy(np.repeat(np.array(lens, np.int32)[:, None] - 1, T, axis=1))
    close(run_varlen(dv, d, 0.1, gpu), O.varlen_paged_sdpa(0.1, **d), dtype, f"{lens}")


# views of one, two and more steps of a split (its loads end with the last step), and
# contiguous views below and above the length from which 5 - 8 tokens are split
@pytest.mark.parametrize("S", [3, 7])
@pytest.mark.parametrize("lens", [[47], [48, 48], [129, 63, 65], [128, 128, 128, 256], [600, 385, 17]])
def test_split_steps(dv, gpu, S, lens):  # noqa: F811
    F, W, Hkv, dtype = len(lens), 2, 2, torch.bfloat16
    loc = np.array(lens)[:, None, None] - S + np.arange(S) + np.zeros((F, W, 1), int)
    d = rand_paged(F, W, S, Hkv, 16, lens, 64, dtype, seed=S + sum(lens), loc=loc)
    close(run_paged(dv, d, 0.1, gpu), O.paged_sdpa(0.1, **d), dtype, f"paged S={S} {lens}")
    g = torch.Generator().manual_seed(S)
    q = torch.randn(F, W, 16 * Hkv, S, 128, generator=g).to(dtype)
    ks = [torch.randn(W, Hkv, L, 128, generator=g).to(dtype) for L in lens]
    vs = [torch.randn(W, Hkv, L, 128, generator=g).to(dtype) for L in lens]
    fl, lc = torch.tensor(lens, dtype=torch.int32), torch.from_numpy(loc.astype(np.int32))
    out = dv.dvattn_sdpa(q.to(gpu), lc.to(gpu), [k.to(gpu) for k in ks], [v.to(gpu) for v in vs], 0.1, fl.to(gpu))
    close(out, O.contig_sdpa(0.1, lc, q, fl, ks, vs), dtype, f"contiguous S={S} {lens}")


def test_varlen_mixed_unsorted_table(dv, gpu):  # noqa: F811
    # a table that is not non-decreasing, and tokens past its last entry
    d = rand_varlen(2, 4, 45, np.array([0, 3, 2, 30, 29]), 1, 16, [60, 200], 32, torch.bfloat16, seed=5)
    close(run_varlen(dv, d, 0.1, gpu), O.varlen_paged_sdpa(0.1, **d), torch.bfloat16, "unsorted")


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("S", [2, 4, 8, 9])
def test_nan_beside_an_empty_wave_set(dv, gpu, dtype, S):  # noqa: F811
    # the first wave set's keys have no page, another set's keys are NaN: one piece
    # gives NaN with and without the split (S = 9)
    d = rand_paged(1, 1, S, 1, 32, [64], 64, dtype, seed=S, loc=np.full((1, 1, S), 63))
    bt, kc = d["block_tables"].clone(), d["k_cache"].clone()
    kc[bt[0, 1]] = float("nan")
    bt[0, 0] = 10 ** 6
    assert run_paged(dv, dict(d, block_tables=bt, k_cache=kc), 0.1, gpu).isnan().all()
