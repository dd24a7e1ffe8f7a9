"""Decode launches of more groups than are resident at once, on an MI355X: the
launch takes what fits and deals it to the sequences by their pages.  Batches
at the deal's edges (a lane's run of 1 to 4 sequences; past 256 the
proportional deal), ragged, equal, empty and one-token lengths, group counts
that divide evenly and not, paired and single heads, fp16 and INT8 with the
last page's residual, and split counts the workspace allows far more of than
are launched, all against the oracle."""

from __future__ import annotations

import numpy as np
import pytest

import oracle
from tests.cases import assert_close, int8_case, paged_case

torch = pytest.importorskip("torch")

pytestmark = [
    pytest.mark.gpu,
    pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU"),
]


def _lens(kind, b):
    rng = np.random.default_rng(b)
    if kind == "equal":
        return [333] * b
    lens = rng.integers(1, 700, b)
    lens[rng.integers(0, b, max(1, b // 8))] = 0
    lens[0] = 1
    lens[b // 2] = 1500
    return lens.tolist()


def _gpu(xs):
    return [torch.from_numpy(np.ascontiguousarray(x)).cuda() for x in xs]


@pytest.mark.parametrize("kind", ["ragged", "equal"])
@pytest.mark.parametrize("b,h,splits", [(1, 2, 700), (1, 3, 600), (5, 4, 26), (48, 8, 2),
                                        (48, 8, 7), (63, 1, 40), (64, 2, 5), (65, 2, 4),
                                        (70, 8, 2), (129, 2, 3), (256, 2, 2), (257, 2, 2)])
def test_fp16(kind, b, h, splits):
    from latentserve_amd.kernels.hip import paged_decode_hip as pdh
    lens = _lens(kind, b)
    case = paged_case(lens, h_kv=h, n_rep=4, seed=b + h)
    q, k, v, t, l = _gpu(case)
    want = oracle.paged_decode(*case)
    for max_len in (max(lens), 0, 100):           # the host's split exact, absent, too short
        for _ in range(2):                        # (the counters are left at zero)
            got = pdh.paged_decode_hip(q, k, v, t, l, max_len, num_splits=splits)
        assert_close(got.float().cpu().numpy(), want, 2e-3, 1e-2, f"{kind} {b} {h} {splits}")


@pytest.mark.parametrize("asym", [False, True])
@pytest.mark.parametrize("b,h,splits", [(5, 4, 26), (48, 2, 9), (40, 1, 20)])
def test_int8(asym, b, h, splits):
    from latentserve_amd.kernels.hip import paged_decode_hip as pdh
    lens = [max(1, x) for x in _lens("ragged", b)]
    case, extra = int8_case(lens, asym=asym, h_kv=h, n_rep=6, seed=b)
    want = oracle.paged_decode(*case, **extra)
    dev = {n: _gpu([x])[0] for n, x in extra.items()}
    got = pdh.paged_decode_hip(*_gpu(case), max(lens), num_splits=splits, **dev)
    assert_close(got.float().cpu().numpy(), want, 2e-3, 1e-2, f"{asym} {b} {h} {splits}")


def test_chosen_splits_are_resident_or_dealt():
    """More than 4 splits a sequence: never more groups than are resident."""
    from latentserve_amd.kernels.hip import paged_decode_hip as pdh
    for int8 in (False, True):
        for h in range(1, 17):
            for b in range(1, 300):
                s = pdh.choose_splits(b, h, 4096, torch.device("cuda", 0), int8=int8)
                groups, fit = (b * h // 2, 256) if h % 2 == 0 else (b * h, 512)
                assert s <= 4 or groups * s <= fit, (b, h, s)
                s = pdh.choose_splits(b, h, 4096, torch.device("cuda", 0), int8=int8, dealt=False)
                assert s == 1 or groups * s <= fit, (b, h, s)


@pytest.mark.parametrize("over", [0, 1, 2, 3, 40])
@pytest.mark.parametrize("b,h,splits", [(2, 2, 5), (3, 3, 5), (60, 8, 2)])
def test_host_partition_over_the_even_one(b, h, splits, over):
    """A host length whose shares are that many pages over even ones (the host's
    partition up to two, even shares past it), equal lengths, full and ragged
    last pages, undealt and dealt groups."""
    from latentserve_amd.kernels.hip import paged_decode_hip as pdh
    for tokens in (50 * 16, 50 * 16 - 3, 47 * 16 + 1):
        max_len = (10 + over) * 16 * splits if splits == 5 else (25 + over) * 16 * splits
        case = paged_case([tokens] * b, h_kv=h, n_rep=4, seed=b + over, width=max_len // 16 if b < 9 else None)
        got = pdh.paged_decode_hip(*_gpu(case), max_len, num_splits=splits)
        assert_close(got.float().cpu().numpy(), oracle.paged_decode(*case), 2e-3, 1e-2,
                     f"{b} {h} {splits} {tokens} {max_len}")
        case, extra = int8_case([tokens] * b, asym=False, h_kv=h, n_rep=4, seed=b + over)
        dev = {n: _gpu([x])[0] for n, x in extra.items()}
        got = pdh.paged_decode_hip(*_gpu(case), max_len, num_splits=splits, **dev)
        assert_close(got.float().cpu().numpy(), oracle.paged_decode(*case, **extra), 2e-3, 1e-2,
                     f"int8 {b} {h} {splits} {tokens} {max_len}")
