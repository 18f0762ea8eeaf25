"""Paged calls with a negative entry in fragment_lengths (device data no host check
sees): the view itself has no keys, the next view starts at a negative logical
position, and its keys there are invisible while the others are not.  The expected
result attends to the keys at positions >= 0 only.  Tolerances:
test_gpu_parity.close."""
import numpy as np
import pytest
import torch

from oracle import dvattn_oracle as O
from test_gpu_parity import close, dv, rand_paged, run_paged  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("bs", [16, 24, 64])
@pytest.mark.parametrize("S", [1, 4, 17])
@pytest.mark.parametrize("neg,n", [(32, 200), (64, 96), (100, 3000), (70, 64), (4096, 5000)])
def test_view_at_a_negative_position(dv, gpu, dtype, bs, neg, n, S):  # noqa: F811
    W, Hkv = 2, 2
    loc = np.stack([np.full((W, S), -1), n - S + np.arange(S)[None].repeat(W, 0)])
    d = rand_paged(2, W, S, Hkv, bs, [0, n], 64, dtype, seed=neg + bs, loc=loc)
    out = run_paged(dv, dict(d, fragment_lengths=torch.tensor([-neg, n], dtype=torch.int32)), 0.1, gpu)
    # the keys at positions 0 .. n - neg - 1 are keys neg .. n - 1 of the view
    seen = max(0, n - neg)
    want = O.paged_sdpa(0.1, **dict(d, locations=torch.from_numpy(np.maximum(loc - neg, -1).astype(np.int32)),
                                    fragment_lengths=torch.tensor([0, seen], dtype=torch.int32)))
    close(out, want, dtype, f"bs={bs} -{neg} {n} S={S}")
