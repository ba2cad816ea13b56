"""The matrix-core pair kernels' bin lookup, evaluated on the CPU: with the high
word of a squared distance off by up to one unit (the kernels' rounding), a pair
lands in its exact bin or is marked for exact evaluation."""
import numpy as np
import pytest

from halotools_amd import _engine as E

FITS = [
    np.logspace(-1, np.log10(50), 20),
    np.logspace(-1, np.log10(30), 16),
    np.logspace(-3, 1, 30),
    np.arange(0, 41, 1.0),                    # pi edges, the first one 0
    np.linspace(1.0, 25.0, 25),
    np.array([0.0, 40.0]),
    np.array([40.0]),
    np.array([0.5, 1.0, 2.0, 4.0]),           # powers of two: edges at bucket starts
    np.array([0.0, 0.5, 1.0, 2.0, 4.0]),
]


@pytest.mark.parametrize("edges", FITS, ids=range(len(FITS)))
def test_off_by_one_high_word_is_exact_or_marked(edges):
    r2 = edges * edges
    rng = np.random.default_rng(1)
    near = [r2]
    for _ in range(4):
        near += [np.nextafter(near[-1], 0), np.nextafter(near[-1], np.inf)]
    # whole units of the high word on both sides of every edge
    hi = (r2[r2 > 0].view(np.uint64) >> np.uint64(32)).astype(np.int64)
    steps = np.concatenate([((hi + s) << 32).astype(np.uint64).view(np.float64) for s in range(-4, 5)])
    d = np.concatenate(near + [steps, steps + 1e-300, [1e-300, 1e300], rng.uniform(0, r2.max() * 1.5, 20000),
                       np.exp(rng.uniform(-30, 20, 20000))])
    d = d[d > 0]
    exact = np.searchsorted(r2, d, side="left")
    marked = 0
    for off in (-1, 0, 1):
        out, fits = E.debug_tile_lookup(r2, d, off)
        assert fits
        assert np.all((out == exact) | (out == -1))
        marked += np.count_nonzero(out[-40000:] == -1)
    assert marked < 100  # the band is narrow: random distances are hardly ever marked


def test_a_high_word_two_off_at_an_edge_is_caught():
    # the check above can fail: with the word off by three units some pair lands in a wrong bin
    r2 = np.logspace(-1, 1, 8) ** 2
    d = np.nextafter(r2, np.inf)
    out, _ = E.debug_tile_lookup(r2, d, -3)
    assert np.any((out != np.searchsorted(r2, d, side="left")) & (out != -1))


@pytest.mark.parametrize("edges", [np.array([1.0, 1.0 + 1e-12, 2.0]), np.array([0.0, 0.0]),
                                   np.linspace(0.001, 0.3, 400),
                                   np.nextafter(np.array([0.5, 1.0, 2.0, 4.0]), 0)])  # edges that end a bucket
def test_edges_that_share_a_bucket_do_not_fit(edges):
    assert not E.debug_tile_lookup(edges * edges, np.array([0.5]))[1]


@pytest.mark.parametrize("edges", FITS, ids=range(len(FITS)))
def test_words_beyond_every_number_take_the_row_past_the_last_edge(edges):
    # a coordinate that is not a number reaches the kernels (they report it): the row its
    # pairs are added to must be one of the histogram's
    d = np.array([np.inf, np.nan, np.finfo(float).max])
    out, fits = E.debug_tile_lookup(edges * edges, d)
    assert fits and np.array_equal(out, np.full(3, len(edges)))
