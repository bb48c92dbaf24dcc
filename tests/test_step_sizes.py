"""The token counts that steps are padded to, at the edges of their rule."""
import pytest

from kubeai_amd.engine.runner import _bucket


@pytest.mark.parametrize("n,padded", [
    (1, 8), (8, 8), (9, 16), (48, 48), (49, 64), (97, 128), (769, 1024), (1024, 1024),
    (1025, 1280), (1280, 1280), (1281, 1536), (5174, 5376), (16383, 16384),
    (16384, 16384),
    (16385, 16385), (20001, 20001),  # beyond the largest, steps run as they are
])
def test_padded_size(n, padded):
    assert _bucket(n) == padded


def test_never_less_and_stable():
    sizes = [_bucket(n) for n in range(1, 17000)]
    assert all(p >= n for n, p in enumerate(sizes, 1))
    assert all(a <= b for a, b in zip(sizes, sizes[1:]))
    assert all(_bucket(p) == p for p in set(sizes))
