"""MaterialMap.override against distinct rows found by brute force: ids,
table order and bits of every property, for each choice of given properties,
few and many distinct values, NaN, signed zeros and strided input."""
import itertools

import numpy as np
import pytest

from rfx_amd.materials import MaterialMap


@pytest.mark.parametrize("shape, k", [((5, 4, 3), 3), ((1, 1, 1), 1), ((23, 17, 11), 4000)])
def test_override_equals_brute_force(shape, k):
    rng = np.random.default_rng(k)
    for given in itertools.product((False, True), repeat=3):
        m = MaterialMap(shape)
        ids = [0] + [m.get_id(1.0 + q, 0.1 * (q % 2), 1.0 + q % 3, q) for q in range(4)]
        m.ids = rng.choice(ids, size=shape).astype(np.uint16)
        pool = rng.uniform(1, 9, k).astype(np.float32)
        pool[:min(k, 3)] = np.array([np.nan, -0.0, 0.0], np.float32)[:min(k, 3)]
        new = [rng.choice(pool, size=shape[::-1]).T if g else None for g in given]
        old = [p[m.ids] for p in m.props()]
        want = [o if n is None else np.ascontiguousarray(n) for o, n in zip(old[:3], new)] + [old[3]]
        bits = np.stack([w.view(np.uint32).ravel() for w in want], axis=1).astype(np.int64)
        m.override(*new)
        rows = [r for r in np.unique(bits, axis=0).tolist()
                if r != [0x3F800000, 0, 0x3F800000, 0]]
        table = np.stack([p.view(np.uint32) for p in m.props()], axis=1).astype(np.int64)
        assert table.tolist() == [[0x3F800000, 0, 0x3F800000, 0]] + rows
        assert np.array_equal(table[m.ids.ravel()], bits)
        assert m.ids.dtype == np.uint16 and m.ids.shape == shape
