"""The batched commit kernel over many commits: every workgroup finds its own row of the table."""

from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CHUNK = 1 << 16


@pytest.mark.parametrize("sizes", [[CHUNK], [CHUNK - 1, CHUNK, CHUNK + 1, 2 * CHUNK], [4] * 1100 + [3 * CHUNK + 7],
                                   [1 + 977 * k % (5 * CHUNK) for k in range(300)]], ids=["one", "edges", "past-the-first-table", "mixed"])
def test_every_commit_lands_whole(hipdev, sizes):
    rng = np.random.default_rng(len(sizes))
    pairs = []
    for n in sizes:
        t, v = hipdev.alloc(n), hipdev.alloc(n)
        data = rng.integers(0, 256, size=n, dtype=np.uint8)
        hipdev.copyin(v, data)
        hipdev.commit(t, v)
        pairs.append((t, data))
    hipdev.finish()
    for t, data in pairs:
        np.testing.assert_array_equal(hipdev.copyout(t), data)
