"""Environment alias tables at the edges of the one-wave-per-row build: rows shorter than, equal to and
just past its 64-item windows and its summation tile, rows of only light or only heavy items, one heavy
item feeding a whole row, long runs of heavy items, black rows and a single row.  The sweep's operation
order is fixed, so the tables are the oracle's bit for bit."""
import numpy as np
import pytest

import oracle as O
import pathed_capi as P

pytestmark = pytest.mark.gpu


def _rows(w, rng):
    """Rows of w weights: each a way the two lists can run out."""
    ramp = np.arange(1, w + 1, dtype=np.float64)
    one = np.full(w, 1e-3)
    one[w // 2] = 1e6
    ends = np.full(w, 5.0)
    ends[: w // 2] = 0.01
    alternating = np.where(np.arange(w) % 2 == 0, 0.1, 3.0)
    return np.stack([np.ones(w), ramp, ramp[::-1], one, ends, ends[::-1], alternating, np.zeros(w), rng.lognormal(0, 2, w),
                     rng.lognormal(0, 0.01, w)])


@pytest.mark.parametrize("w", [1, 2, 63, 64, 65, 127, 128, 129, 511, 512, 513, 1025, 3000])
def test_env_tables_equal_the_oracle_at_window_edges(w):
    print(f"case: env tables, rows of {w}", flush=True)
    rng = np.random.default_rng(w)
    wts = _rows(w, rng)
    for rows in (wts, wts[:1], np.repeat(wts, 7, axis=0)):
        e = np.zeros((rows.shape[0], w, 4), np.float32)
        e[..., :3] = rows[..., None]
        for a, b in zip(P.env_tables(e), O.env_alias(e)):
            assert np.array_equal(a, b)
