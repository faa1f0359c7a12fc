"""The batch autotuner's choice from measured times (no GPU)."""
import itertools

from rk_amd.autotune import choose_tile


def test_ties_do_not_change_the_choice():
    """Times of the 512-instance batch that differ by less than they repeat: any
    order of them gives the same shape."""
    close = [8.60, 8.66, 8.69, 8.74, 8.89]
    shapes = [(2, 64), (2, 96), (2, 128), (2, 160), (2, 192)]
    for t in itertools.permutations(close):
        times = dict(zip(shapes, t))
        times.update({(1, 64): 9.15, (4, 64): 9.55, (4, 128): 9.60})
        assert choose_tile(times) == (2, 192)


def test_clear_winner():
    assert choose_tile({(1, 64): 1.0, (2, 64): 1.05, (2, 192): 1.3}) == (1, 64)
    assert choose_tile({(2, 128): 1.0, (4, 128): 0.97}) == (4, 128)
    assert choose_tile({(4, 128): 2.0}) == (4, 128)
