"""Which steps the delta rule walks by tiles: by measured times (us) of both walks, wherever one is a tenth faster than the other."""
import pytest

from swiftllm_amd.worker.kernels.delta_rule import worth_tiles


# heads, head size, decoded tokens beside so many portions of so many tokens: by tokens, by tiles
@pytest.mark.parametrize("heads,dim,decoded,portions,length,tokens,tiles", [
    (8, 128, 0, 1, 48, 25.3, 14.7), (8, 128, 30, 1, 48, 43.6, 33.7), (8, 128, 30, 1, 1000, 378.4, 98.2),
    (8, 128, 200, 1, 48, 108.9, 130.8), (8, 128, 200, 4, 64, 118.6, 135.8), (8, 128, 200, 1, 100, 152.6, 133.8),
    (16, 128, 100, 1, 48, 108.6, 131.2), (16, 128, 100, 4, 48, 119.1, 134.5), (16, 128, 100, 1, 100, 154.7, 134.5),
    (16, 128, 200, 1, 100, 219.7, 244.9), (16, 128, 200, 16, 48, 212.9, 276.9), (16, 128, 200, 1, 200, 291.2, 253.5),
    (32, 128, 0, 50, 64, 430.4, 292.3), (32, 128, 30, 50, 64, 521.9, 383.2), (32, 128, 200, 50, 64, 708.1, 798.4),
    (32, 128, 200, 1, 200, 438.1, 516.8), (16, 64, 100, 50, 64, 126.7, 95.6), (16, 64, 200, 1, 200, 130.1, 97.8),
    (4, 128, 200, 50, 64, 133.4, 111.5), (8, 64, 0, 64, 16, 19.9, 25.0), (8, 128, 100, 1, 24, 61.4, 74.4)])
def test_the_faster_walk(heads, dim, decoded, portions, length, tokens, tiles):
    assert max(tokens, tiles) >= 1.1 * min(tokens, tiles)
    assert worth_tiles(length, decoded + portions, decoded + portions * length, heads, dim) == (tiles < tokens)


def test_steps_of_no_or_unknown_length():
    """Captured decode steps and hand-made ones carry no length: token by token."""
    assert not worth_tiles(0, 1, 1, 1, 16) and not worth_tiles(1, 32, 32, 8, 128) and not worth_tiles(0, 0, 0, 8, 128)
