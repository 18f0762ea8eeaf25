"""Paged decode of one token against the oracle at the lengths and page sizes
where a stage of 32 keys takes one load path or the other
(dvattention_amd/csrc/dv_stream.h, issue_stage): pages of 8, 16, 24, 32 and 64
keys, ranges that start and end inside a stage, views that start off a multiple
of 32 logical positions, and rows short enough that a cut leaves a piece without
keys.  Tolerances: test_gpu_parity.close."""
import numpy as np
import pytest
import torch

from oracle import dvattn_oracle as O
from test_gpu_parity import close, dv, rand_paged, run_paged  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("bs", [8, 16, 24, 32, 64])
@pytest.mark.parametrize("W,Hkv,lens", [(1, 1, [1]), (1, 4, [31]), (2, 2, [32]), (1, 8, [3001]), (3, 4, [65]),
                                        (2, 4, [37, 100, 5]), (66, 4, [130]), (2, 1, [9000])])
def test_paged_stage_paths(dv, gpu, dtype, bs, W, Hkv, lens):  # noqa: F811
    F = len(lens)
    rng = np.random.default_rng(bs + sum(lens))
    loc = np.array(lens)[:, None, None] - 1 - rng.integers(0, min(lens), size=(F, W, 1))
    d = rand_paged(F, W, 1, Hkv, bs, lens, 64, dtype, seed=bs, loc=loc, k_scale=1.5)
    close(run_paged(dv, d, 0.1, gpu), O.paged_sdpa(0.1, **d), dtype, f"bs={bs} {lens}")


@pytest.mark.parametrize("bs", [16, 32])
def test_invalid_page_in_a_full_stage(dv, gpu, bs):  # noqa: F811
    # a page outside the pool in the middle of a row: its keys are masked, the
    # stage's other keys are not
    d = rand_paged(1, 1, 1, 1, bs, [320], 64, torch.bfloat16, seed=3, loc=np.array([[[319]]]))
    bt = d["block_tables"].clone()
    bt[0, 3] = 10 ** 6
    out = run_paged(dv, dict(d, block_tables=bt), 0.1, gpu).cpu()
    pos = np.array([i for i in range(320) if i // bs != 3])
    pages = d["block_tables"][0].numpy()[pos // bs]
    rq = O.rope_q(d["queries"], d["cosines"], d["sines"])[0, 0, :, 0].float()
    k = d["k_cache"][pages, pos % bs, 0].float()
    v = d["v_cache"][pages, pos % bs, 0].float()
    close(out[0, :, 0], torch.softmax(0.1 * (rq @ k.T), -1) @ v, torch.bfloat16, f"bs={bs}")


# rows of more than 64 views, whose table is walked 64 at a time: one view more than a
# block, two blocks, views without keys (some of them unseen by their query), page
# positions past the first block
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("F,bs", [(64, 16), (65, 16), (129, 24), (140, 32)])
def test_paged_many_views(dv, gpu, dtype, F, bs):  # noqa: F811
    rng = np.random.default_rng(F)
    lens = rng.integers(0, 90, size=F)
    lens[[0, 63, -1]] = [70, 33, 41]
    loc = rng.integers(-1, 90, size=(F, 3, 1))
    d = rand_paged(F, 3, 1, 4, bs, list(lens), 32, dtype, seed=bs, loc=loc)
    close(run_paged(dv, d, 0.1, gpu), O.paged_sdpa(0.1, **d), dtype, f"F={F}")
    loc[64:] = -1  # no view of the later blocks is seen
    d = rand_paged(F, 3, 1, 4, bs, list(lens), 32, dtype, seed=bs, loc=loc)
    close(run_paged(dv, d, 0.1, gpu), O.paged_sdpa(0.1, **d), dtype, f"F={F}, first block only")


# short rows, which get a workgroup each where all have one length: lengths up to and
# past the limits of that (96, 128 and 256 keys), more and fewer than 64 rows, one row
# of another length among them
@pytest.mark.parametrize("W,Hkv", [(3, 2), (20, 8), (70, 4)])
@pytest.mark.parametrize("lens", [[1], [60], [96], [97], [130], [256], [257], [40, 60], [100, 29]])
@pytest.mark.parametrize("odd", [None, 0, 1])
def test_paged_short_rows(dv, gpu, W, Hkv, lens, odd):  # noqa: F811
    loc = np.array(lens)[:, None, None] - 1 + np.zeros((len(lens), W, 1), int)
    if odd is not None:
        loc[-1, odd] -= 1
    d = rand_paged(len(lens), W, 1, Hkv, 16, lens, 64, torch.bfloat16, seed=W, loc=loc)
    close(run_paged(dv, d, 0.1, gpu), O.paged_sdpa(0.1, **d), torch.bfloat16, f"W={W} {lens} {odd}")
