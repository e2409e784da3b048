"""Greedy sampling on the device (pkv_greedy_tokens) against NumPy's argmax, which is the
reference's greedy_token (sampling.py:28-30): bit-exact token ids, including ties (lowest id),
NaN (first NaN wins), -inf rows, signed zeros, odd vocabulary sizes and strided rows. The
whole config-1 run sampled on the device is in test_gpu_replay.py."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from paged_kv_serving_amd import ops

pytestmark = pytest.mark.gpu


def _argmax_rows(logits: np.ndarray) -> np.ndarray:
    return np.asarray([int(np.argmax(row)) for row in logits], dtype=np.int32)


@pytest.mark.parametrize("vocab", [1, 3, 4, 255, 256, 1000, 32_000, 128_256])
def test_random_rows_match_numpy(device, vocab) -> None:
    rng = np.random.default_rng(vocab)
    logits = rng.standard_normal((37, vocab)).astype(np.float32)
    got = ops.greedy_tokens(torch.from_numpy(logits).to(device)).cpu().numpy()
    assert np.array_equal(got, _argmax_rows(logits))


def test_ties_nan_infinities_and_signed_zeros(device) -> None:
    vocab = 1031  # not a multiple of 4: exercises the tail of the vector path
    rows = np.zeros((10, vocab), dtype=np.float32)
    rows[0, [5, 700, 1030]] = 2.0  # tie -> lowest id
    rows[1, :] = -np.inf  # all -inf -> 0
    rows[2, [9, 400]] = np.nan  # first NaN wins over everything
    rows[2, 3] = np.inf
    rows[3, 1030] = np.nan  # a NaN in the tail
    rows[3, 2] = 1e30
    rows[4, :] = -0.0
    rows[4, 600] = 0.0  # -0.0 and +0.0 tie -> 0
    rows[5, 1029] = np.inf
    rows[5, 1030] = np.inf  # tie of infinities in the tail
    rows[6, :] = np.float32(-3.0)
    rows[6, 1027] = np.float32(-2.9999998)  # one ulp above
    rows[7, 256 * 3 + 1] = 1.0  # one element, in another thread's stretch
    rows[8, :] = np.arange(vocab, dtype=np.float32)[::-1]  # maximum at 0
    rows[9, :] = np.arange(vocab, dtype=np.float32)  # maximum at the last id
    with np.errstate(invalid="ignore"):
        want = _argmax_rows(rows)
    got = ops.greedy_tokens(torch.from_numpy(rows).to(device)).cpu().numpy()
    assert np.array_equal(got, want), (got, want)


def test_strided_and_misaligned_rows(device) -> None:
    rng = np.random.default_rng(1)
    big = torch.from_numpy(rng.standard_normal((16, 300)).astype(np.float32)).to(device)
    view = big[:, 1:258]  # stride 300, base one float past 16-byte alignment
    got = ops.greedy_tokens(view).cpu().numpy()
    assert np.array_equal(got, _argmax_rows(big[:, 1:258].cpu().numpy()))
    aligned = big[::2, :256]  # stride 600, aligned: the vector path
    assert np.array_equal(ops.greedy_tokens(aligned).cpu().numpy(), _argmax_rows(aligned.cpu().numpy()))


@pytest.mark.parametrize("vocab", [1, 2, 3, 5, 4095, 4096, 4099, 16_387, 50_257])
def test_every_alignment_and_edge_of_a_row(device, vocab) -> None:
    """Rows start at each of the four offsets from a 16-byte boundary, with the maximum at the
    row's ends and around its aligned body's ends (the first three and last four ids), at ids a
    workgroup's stride of 4,096 apart (ties go to the lowest) and with a NaN behind each."""
    picks = sorted({i % vocab for i in (0, 1, 2, 3, -1, -2, -3, -4, 4095, 4096, 4100, vocab // 2)})
    for offset in range(4):
        rows = np.full((2 * len(picks), vocab), -1.0, dtype=np.float32)
        for r, i in enumerate(picks):
            rows[r, i:: 4096] = 7.0
            rows[len(picks) + r, 0] = np.inf
            rows[len(picks) + r, i:: 4096] = np.nan
        held = torch.zeros((rows.shape[0], vocab + 4), device=device)
        flat = held.view(-1)[offset : offset + rows.size].view(rows.shape)  # rows vocab apart
        flat.copy_(torch.from_numpy(rows))
        got = ops.greedy_tokens(flat).cpu().numpy()
        assert np.array_equal(got, _argmax_rows(rows)), (offset, got)


@pytest.mark.parametrize(
    ("vocab", "count"), [(v, 8) for v in (1, 5, 510, 513, 4094, 4097, 32_767, 32_771)] + [(32_771, 130)]
)
def test_every_workgroup_size(device, vocab, count) -> None:
    """Both sides of the vocabularies and row counts at which the workgroup's size changes: random
    rows, rows of -inf alone or but for one element, ties, a NaN, and +inf before a NaN."""
    rng = np.random.default_rng(vocab)
    rows = rng.standard_normal((count, vocab)).astype(np.float32)
    at = rng.integers(0, vocab, 8)
    rows[1] = -np.inf
    rows[2] = -np.inf
    rows[2, at[2]] = -np.finfo(np.float32).max
    rows[3] = 0.0
    rows[3, ::2] = -0.0
    rows[4, at[4]] = np.nan
    rows[5, 0], rows[5, at[5]] = np.inf, np.nan
    rows[6, -1] = np.inf
    rows[7] = np.nan
    for offset in (0, 1):
        held = torch.zeros(rows.size + 4, device=device)[offset : offset + rows.size].view(rows.shape)
        held.copy_(torch.from_numpy(rows))
        got = ops.greedy_tokens(held).cpu().numpy()
        assert np.array_equal(got, _argmax_rows(rows)), (offset, got[:8])
