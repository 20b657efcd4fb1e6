"""The sampler's bins at their edges, against the oracle's draws: rows whose
candidates crowd one bin (equal logits, a narrow spread), rows spread past the
bins' range (low temperatures, infinitely unlikely tokens), vocabularies around
a chunk's and a bin search's sizes, cuts that keep one, all or almost all
candidates, and the largest draw there is."""
import numpy as np
import pytest

import oracle as O
from huggingfaceeacp_amd import gemma_q8 as G
from test_gpu_sampling import DeviceSampler, agree

pytestmark = pytest.mark.gpu
S = G.SamplingOptions


def cuts(vocab):
    # 0.47: with p = 1/2 of an even number of equal masses the running mass
    # reaches p exactly, and the rounding of the sums (here about n 2^-53, in
    # the oracle's sequential loop too) decides whether one more is kept
    return [S(1.0, seed=1), S(0.7, top_k=1, seed=2), S(1.0, top_k=vocab - 1, seed=3),
            S(1.0, top_k=min(40, vocab), top_p=0.9, seed=4), S(1.1, top_p=0.47, seed=5),
            S(1.0, top_p=0.999, seed=6), S(1.0, top_k=vocab, seed=7)]


@pytest.mark.parametrize("vocab", [2, 511, 513, 1024, 8191, 8192, 8193, 16385])
def test_vocabulary_edges(torch_cuda, vocab):
    row = np.random.default_rng(vocab).normal(0, 2, vocab).astype(np.float32)
    for options in cuts(vocab):
        agree(torch_cuda, row, options, draws=12)


@pytest.mark.parametrize("spread", [0.0, 1e-4, 0.05])
def test_crowded_bins(torch_cuda, spread):
    vocab = 60000
    row = np.random.default_rng(9).normal(0, 1, vocab).astype(np.float32) * np.float32(spread)
    for options in cuts(vocab) + [S(1.0, top_k=30000, seed=8)]:
        agree(torch_cuda, row, options, draws=6)


@pytest.mark.parametrize("temperature", [0.001, 0.02, 0.2])
def test_low_temperatures(torch_cuda, temperature):
    vocab = 40000
    row = np.random.default_rng(10).normal(0, 3, vocab).astype(np.float32)
    row[::3] = -np.inf
    for options in (S(temperature, top_k=40, seed=11), S(temperature, top_p=0.95, seed=12),
                    S(temperature, top_k=30000, top_p=0.99999, seed=13), S(temperature, seed=14)):
        agree(torch_cuda, row, options, draws=6)


def test_a_row_without_a_number_keeps_its_last_candidate(torch_cuda):
    """No running mass is a number: the draw falls to the last kept candidate
    of the ranking, or with no cut to the last unmasked token
    (Sampler.cpp:196-213)."""
    import torch
    vocab = 3000
    row = np.linspace(-3, 3, vocab).astype(np.float32)
    for value, k_th in ((np.inf, 10), (np.nan, 10)):
        bad = row.copy()
        bad[5] = value  # ranks first
        dev = torch.from_numpy(bad).cuda()
        n = G.sample_workspace_bytes(vocab)
        ws = torch.empty(n, dtype=torch.uint8, device="cuda")
        token = torch.zeros(1, dtype=torch.int32, device="cuda")

        def sample(options):
            G.sample_row(dev.data_ptr(), None, vocab, options, 0.25, token.data_ptr(), ws.data_ptr(), n)
            return int(token.item())

        # the tokens from the top down follow the planted one
        assert sample(S(1.0, top_k=k_th)) == vocab - (k_th - 1)
        assert sample(S(1.0, top_p=0.5)) == 0
        assert sample(S(1.0)) == vocab - 1


def drawn(torch, row, options, uniform):
    """(the device's id, the oracle's) of one given draw."""
    row = np.ascontiguousarray(row, dtype=np.float32)
    want = O.lib().gor_sample(O.ptr(row), None, row.size, options.temperature, options.top_k,
                              options.top_p, uniform)
    sampler = DeviceSampler(torch, row.size)
    sampler.workspace.zero_()
    return sampler.sample(torch.from_numpy(row).cuda(), None, options, uniform), int(want)


@pytest.mark.parametrize("seed", [7, 11, 12, 14, 16])
def test_largest_draw_keeps_to_the_kept_candidates(torch_cuda, seed):
    """The draw 1 - 2^-53 over 1000 kept candidates that share a bin of the
    score, or fill some of them, with thousands more far below.  At these seeds
    the crowded bin's running mass rounds below the draw's target (the sums
    restated in numpy), so the place lies past every kept candidate: the
    last of them is the answer (Sampler.cpp:196-213)."""
    for spread in (0.012, 0.2):
        near = (-np.random.default_rng(seed).random(1000) * spread).astype(np.float32)
        near[0] = 0
        row = np.concatenate([near, np.full(5000, -20.0, np.float32)])
        for options in (S(1.0, top_k=1000), S(1.0, top_k=700), S(1.0, top_p=0.9),
                        S(1.0, top_k=1000, top_p=0.97)):
            for uniform in (1.0 - 2.0 ** -53, 1.0 - 2.0 ** -52, 0.0):
                got, want = drawn(torch_cuda, row, options, uniform)
                assert got == want, (spread, options, uniform)


def test_last_ranking_key_ends_the_search_range(torch_cuda):
    """More than a ranking's worth of -inf logits and, behind them all, a NaN
    with every bit set, whose ranking key has the largest upper word: the
    range of the last bin searched ends there and does not wrap.  No
    running mass is a number, so the last of the ranking is kept."""
    row = np.linspace(-3, 3, 3000).astype(np.float32)
    row[10:800] = -np.inf
    row.view(np.uint32)[5] = 0xFFFFFFFF
    sampler = DeviceSampler(torch_cuda, row.size)
    dev = torch_cuda.from_numpy(row).cuda()
    for options in (S(1.0, top_p=0.9), S(0.5, top_k=3000, top_p=0.5)):
        assert sampler.sample(dev, None, options, 0.25) == 5


@pytest.mark.parametrize("count", [1, 700])
def test_nans_behind_the_kept_candidates_weigh_nothing(torch_cuda, count):
    """NaNs with the sign set rank after every number, so a top-k that keeps
    numbers alone draws as if they were -inf; one that keeps the first of
    them has no sums that are numbers and takes its last candidate."""
    vocab = 3000
    rng = np.random.default_rng(count)
    row = rng.normal(0, 2, vocab).astype(np.float32)
    at = np.sort(rng.choice(vocab, count, replace=False))
    numbers, bits = row.copy(), row.copy()
    numbers[at] = -np.inf
    bits.view(np.uint32)[at] = 0xFFC00000
    dev = torch_cuda.from_numpy(bits).cuda()
    sampler = DeviceSampler(torch_cuda, vocab)
    for options in (S(1.0, top_k=40, seed=51), S(0.8, top_k=40, top_p=0.9, seed=52),
                    S(1.0, top_k=vocab - count, seed=53),
                    S(1.0, top_k=vocab - count, top_p=0.95, seed=54)):
        ref = O.Sampler(options.temperature, options.top_k, options.top_p, options.seed)
        for uniform in O.uniform_draws(options.seed, 20):
            assert sampler.sample(dev, None, options, uniform) == ref.sample(numbers), (options, uniform)
    if count > 1:
        for options in (S(1.0, top_k=vocab - count + 1), S(1.0, top_k=vocab - count + 1, top_p=0.5)):
            assert sampler.sample(dev, None, options, 0.25) == at[0]
    assert sampler.sample(dev, None, S(1.0, top_p=0.5), 0.25) == at[-1]
    assert sampler.sample(dev, None, S(1.0), 0.25) == vocab - 1


@pytest.mark.parametrize("vocab", [40, 3000, 60000])
def test_infinite_temperature_ranks_by_token(torch_cuda, vocab):
    """1 / temperature is zero: every score ties, whatever the logits."""
    row = np.random.default_rng(vocab).normal(0, 2, vocab).astype(np.float32)
    inf = float("inf")
    for options in (S(inf, top_k=5, seed=61), S(inf, top_k=vocab - 1, top_p=0.47, seed=62),
                    S(inf, top_p=0.9, seed=63), S(inf, seed=64)):
        got = agree(torch_cuda, row, options, draws=12)
        assert options.top_k != 5 or max(got) < 5


@pytest.mark.parametrize("spread", [0.0, 1e-5, 0.01])
def test_a_crowd_below_an_outlier(torch_cuda, spread):
    """One token 20 above the rest keeps the bins at their even width, so the
    rest crowd one or two and the search spreads them again."""
    vocab = 60000
    row = np.random.default_rng(12).random(vocab).astype(np.float32) * np.float32(spread)
    row[777] = 20.0
    for options in (S(2.0, top_k=2, seed=71), S(4.0, top_k=600, seed=72), S(4.0, top_k=30000, seed=73),
                    S(4.0, top_p=0.999, seed=74), S(4.0, top_k=50000, top_p=0.9995, seed=75)):
        agree(torch_cuda, row, options, draws=6)


@pytest.mark.parametrize("widest", [1e-44, 1e-30, 0.25, 7.9999995, 8.0, 8.000001, 16.0])
def test_rows_at_the_edges_of_the_bins_scales(torch_cuda, widest):
    vocab = 5000
    row = (-np.random.default_rng(13).random(vocab) * widest).astype(np.float32)
    row[[100, 4000]] = 0.0, -widest
    mask = (np.arange(vocab) % 3 == 0).astype(np.float32)
    mask[[100, 4000]] = 0
    for options in (S(1.0, top_k=7, seed=81), S(1.0, top_k=3000, seed=82), S(1.0, top_p=0.93, seed=83)):
        agree(torch_cuda, row, options, draws=4)
        agree(torch_cuda, row, options, draws=4, mask=mask)
