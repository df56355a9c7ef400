"""The MLA reduce alone against the oracle's merge, at the edges of its forms:
8 and 9 groups (value dims over four waves or one; 6 groups of few pieces: one), piece counts around the 8
and 16 in flight and the 64 a wave looks up at a time, pieces with lse -inf
whose rows hold NaN, and a group whose pieces are all such.

Bar: the weights are ratios of float32 exponentials (relative 2^-18 at the
tested lse range of +-8), the sums round once per piece, the output once to
bfloat16: |out - ref| <= 2^-8 |ref| + (2^-18 + n 2^-23) * wabs, wabs the
weighted mean of |x|; lse within 2e-5 + 1e-5 |lse|.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from flydsl_amd.mla_decode import mla_reduce_v1
from oracle.mla import mla_reduce_ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("groups", [1, 8, 9])
def test_reduce_piece_counts(groups):
    counts = [(1, 8, 9, 16, 17, 64, 65, 130, 7)[(g + (groups == 1) * 6) % 9] for g in range(groups)]
    n = sum(counts)
    rng = np.random.default_rng(groups)
    so = rng.standard_normal((n, 1, 128, 512)).astype(np.float32)
    sl = rng.uniform(-8, 8, (n, 1, 128, 1)).astype(np.float32)
    perm = rng.permutation(n).astype(np.int32)
    indptr = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    skipped = [perm[indptr[g + 1] - 1] for g in range(groups) if counts[g] > 1]  # last pieces: no visible key
    if groups == 9:
        skipped += list(perm[indptr[8]:indptr[9]])  # and every piece of a group
    so_ref = so.copy()
    so_ref[skipped] = 0.0
    so[skipped] = np.nan
    sl[skipped] = -np.inf
    fmap = np.array([[g, g + 1] for g in range(groups)], np.int32)
    dev = lambda x: torch.from_numpy(x).cuda()  # noqa: E731
    out = torch.full((groups, 128, 512), float("nan"), dtype=torch.bfloat16, device="cuda")
    lse = torch.full((groups, 128), float("nan"), dtype=torch.float32, device="cuda")
    mla_reduce_v1(dev(so), dev(sl), dev(indptr), dev(fmap), dev(perm), 1, out, lse)
    got, got_lse = out.float().cpu().numpy(), lse.cpu().numpy()
    live = 8 if groups == 9 else groups
    want = mla_reduce_ref(so_ref[:, 0].astype(np.float64), sl[:, 0, :, 0].astype(np.float64), indptr, fmap, perm, live)
    wabs = mla_reduce_ref(np.abs(so_ref[:, 0]).astype(np.float64), sl[:, 0, :, 0].astype(np.float64), indptr, fmap,
                          perm, live)
    for g in range(live):
        tol = 2.0 ** -8 * np.abs(want[g][0]) + (2.0 ** -18 + counts[g] * 2.0 ** -23) * wabs[g][0] + 1e-30
        assert np.all(np.abs(got[g] - want[g][0]) <= tol), g
        assert np.all(np.abs(got_lse[g] - want[g][1]) <= 2e-5 + 1e-5 * np.abs(want[g][1])), g
    if groups == 9:
        assert np.all(got[8] == 0) and np.all(np.isneginf(got_lse[8]))


@pytest.mark.parametrize("groups", [2, 6, 9])
def test_reduce_shows_nan_and_infinity(groups):
    """Every piece with an lse other than -inf takes part: a (row, head) whose
    lse are NaN, alone or beside -inf, and one whose weightless piece (its lse
    140 below the other's: exp(-140) is 0 in float32) holds NaN or an infinity come out
    as NaN; the other heads as without them."""
    pieces = 3
    rng = np.random.default_rng(groups)
    so = rng.standard_normal((groups * pieces, 1, 128, 512)).astype(np.float32)
    sl = rng.uniform(-8, 8, (groups * pieces, 1, 128, 1)).astype(np.float32)
    sl[:, 0, 1:5] = 0.0
    sl[:3, 0, 1] = np.nan  # every piece
    sl[:3, 0, 2] = [[np.nan], [-np.inf], [-np.inf]]
    sl[1, 0, 3:5] = -140.0
    so[1, 0, 3, 7], so[1, 0, 4, 8] = np.nan, np.inf
    dev = lambda x: torch.from_numpy(x).cuda()  # noqa: E731
    args = [dev(np.arange(0, groups * pieces + 1, pieces, dtype=np.int32)),
            dev(np.array([[g, g + 1] for g in range(groups)], np.int32)),
            dev(np.arange(groups * pieces, dtype=np.int32))]
    out = torch.zeros((groups, 128, 512), dtype=torch.bfloat16, device="cuda")
    mla_reduce_v1(dev(so), dev(sl), *args, 1, out)
    bad = torch.isnan(out).cpu()
    want = torch.zeros_like(bad)
    want[0, 1:3] = True
    want[0, 3, 7] = want[0, 4, 8] = True
    assert torch.equal(bad, want)
