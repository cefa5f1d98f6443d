"""Read-backs of up to 2 MiB by a kernel whose workgroups each copy a run of the words: every word, wherever the runs end and the view
begins, again and again."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 3, 256, 4095, 4096, 8191, 8192, 8197, 12289, 49152, 151936, 262143, 262147, 300001, 524287, 524288, 524289])
@pytest.mark.parametrize("skip", [0, 1, 4])
def test_every_word(hip, n, skip):
    rng = np.random.default_rng(n)
    for _ in range(3):
        a = rng.integers(0, 2 ** 32, n + skip, dtype=np.uint32)
        x = hip.from_numpy(a)
        np.testing.assert_array_equal(hip.to_numpy(hip.slice(x, 0, skip, n)), a[skip:])
