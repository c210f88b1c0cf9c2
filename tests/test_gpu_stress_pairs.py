"""As many sampled pairs as the set-up takes: the pairs of one search end within a grid stride of
2^31, so that a 32-bit counter of them would pass its range."""
import numpy as np
import pytest

from gpugraphlayout_amd import Engine, GFA2Error

pytestmark = pytest.mark.gpu


def test_pairs_up_to_the_limit():
    """A star of 1,025 nodes (every pair is reached): 1,024 sources in one search with 2^21 - 1
    targets each are counted one and all; a target more each is refused."""
    print("case stress 1024 x (2^21 - 1) pairs", flush=True)
    n = 1025
    eng = Engine(n, np.zeros(n - 1, np.int32), np.arange(1, n, dtype=np.int32))
    with pytest.raises(GFA2Error):
        eng.stress_setup(1024, 1 << 21, seed=3)
    assert eng.stress_setup(1024, (1 << 21) - 1, seed=3) == 1024 * ((1 << 21) - 1)
    eng.close()
