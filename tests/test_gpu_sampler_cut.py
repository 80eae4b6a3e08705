"""The sampler's cut of a long candidate list: rows whose candidates do not
fit LDS give the oracle's tokens and states, over flat and peaked rows, ties
of values around the cut, temperatures, top-k / top-p limits and rows that
start unaligned."""
import numpy as np
import pytest

import lbt_oracle as orc
from conftest import announce

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("V", [4097, 5001, 40000, 128256])
@pytest.mark.parametrize("scale", [0.3, 2.5, 6.0])
def test_cut_rows_match_oracle(ctx, V, scale):
    rng = np.random.default_rng(V + int(10 * scale))
    rows = 3
    lg = (rng.standard_normal((rows, V)) * scale).astype(np.float32)
    lg[1] = np.round(lg[1] * 2) / 2  # a few dozen values, each held by many
    lg[2, rng.integers(0, V, 30)] += 8.0
    for t, p, k in ((0.8, 0.95, 0), (1.0, 1.0, 0), (0.7, 0.5, 40), (1.3, 1.0, 3000), (2.5, 0.999, 0), (1e30, 0.9, 0),
                    (0.8, 0.0, 0)):
        announce(f"sampler cut V={V} scale={scale} t={t} top_p={p} top_k={k}")
        states = rng.integers(1, 1 << 62, rows).astype(np.uint64)
        want, after = [], []
        for r in range(rows):
            s = orc.Sampler(t, p, k, int(states[r]))
            want.append(s.sample(lg[r]))
            after.append(s.state.value)
        got = ctx.sample(lg, t, p, k, states)
        assert list(got) == want
        assert [int(x) for x in states] == after
