"""GPU tests of the filtered draw's two-launch form (k_first, k_finer, k_finish) where its selection can go wrong:
ties at a threshold, one score for the whole row, more candidates than a list holds in the first bins or in
the finer ones, masked rows, the first top-k past the form's limit, and rows that leave a workgroup's slice
empty.  Tokens equal the sampling oracle's (a knife edge of the oracle aside, as in test_gpu_sampling)."""

import numpy as np
import pytest
import torch

from test_gpu_sampling import _compare, _gpu_sample

pytestmark = pytest.mark.gpu

V = 151936


def _row(kind, n, rng):
    if kind == "normal":
        return rng.normal(0, 2, n)
    if kind == "shifted":  # far from 0: coarse key bins, cut into the finer ones
        return rng.normal(40, 2, n)
    if kind == "equal":  # one score: no list
        return np.full(n, 1.25)
    if kind == "two":  # two scores a hair apart, thousands of each: one finer bin each
        return np.where(rng.random(n) < 0.5, 1.0, 1.0009765625)
    if kind == "dense":  # distinct scores within one bin, thousands in each of its finer ones
        return 3.0 + rng.random(n) * 0.01
    if kind == "near":  # a few hundred scores, tens of thousands in each finer bin: no list holds them
        return 3.0 + rng.random(n) * 1e-4
    if kind == "flat":
        return rng.normal(0, 0.01, n)
    if kind == "masked":  # a handful of live scores
        x = np.full(n, -np.inf)
        x[rng.choice(n, 5, replace=False)] = rng.normal(0, 1, 5)
        return x
    if kind == "lowest":
        x = np.full(n, np.finfo(np.float32).min)
        x[rng.choice(n, 5, replace=False)] = rng.normal(0, 1, 5)
        return x
    return np.round(rng.normal(0, 2, n) * 8) / 8  # "ties": hundreds of scores at every value


@pytest.mark.parametrize("k,p", [(0, 0.9), (50, 1.0), (50, 0.9), (4096, 0.95), (4097, 0.95), (1, 0.5), (0, 0.001)])
@pytest.mark.parametrize("kind", ["normal", "shifted", "equal", "two", "dense", "near", "flat", "masked", "lowest", "ties"])
def test_filtered_draw_forms(kind, k, p):
    rng = np.random.default_rng(len(kind) * 100 + k)
    rows = np.stack([_row(kind, V, rng) for _ in range(2)]).astype(np.float32)
    _compare(rows, 0.8, k, p, 77, [3, 1 << 33])


@pytest.mark.parametrize("n", [1, 2, 63, 64, 1000, 2049])
def test_filtered_draw_small_vocabularies(n):
    rng = np.random.default_rng(n)
    rows = rng.normal(0, 2, (5, n)).astype(np.float32)
    for k, p in ((0, 0.8), (max(1, n // 2), 1.0), (max(1, n // 2), 0.7)):
        _compare(rows, 1.1, k, p, 5, list(range(5)))


@pytest.mark.parametrize("rows", [128, 129, 256, 257])
def test_row_groups(rows):
    """Rows at the edges of a launch sequence's rows (128 of the two-launch form, 256 of the others): every
    form draws what it draws for each row alone, and leaves the work clear."""
    rng = np.random.default_rng(rows)
    x = rng.normal(0, 2, (rows, 700)).astype(np.float32)
    ctr = list(range(rows))
    for T, k, p in ((0.0, 0, 1.0), (0.9, 0, 1.0), (0.9, 30, 1.0), (0.9, 0, 0.8), (0.9, 30, 0.8), (0.9, 5000, 1.0)):
        got = _compare(x, T, k, p, 11, ctr)
        some = [0, 127, 128 % rows, rows - 1]
        assert [got[r] for r in some] == [_gpu_sample(x[r:r + 1], T, k, p, 11, [ctr[r]])[0] for r in some]


def test_work_is_clear_after_every_form():
    """A call of each form after each other form on one stream gives what it gives alone."""
    rng = np.random.default_rng(9)
    rows = rng.normal(0, 2, (3, 5000)).astype(np.float32)
    rows[1] = 0.5
    forms = [(0, 1.0), (0, 0.9), (40, 1.0), (40, 0.9), (4500, 0.9), (4500, 1.0)]
    alone = {}
    for k, p in forms:
        with torch.cuda.stream(torch.cuda.Stream()):
            alone[k, p] = _gpu_sample(rows, 0.9, k, p, 3, [1, 2, 3])
    for a in forms:
        for b in forms:
            assert _gpu_sample(rows, 0.9, *a, 3, [1, 2, 3]) == alone[a]
            assert _gpu_sample(rows, 0.9, *b, 3, [1, 2, 3]) == alone[b]
