"""The Morton keys' kernel against the tensor form on the CPU: the same
permutation, at batch sizes around a workgroup and every number of columns,
constant columns and tied keys among them."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 255, 257, 5000])
@pytest.mark.parametrize("d", [1, 2, 3, 5, 9, 12])
def test_same_permutation(n, d):
    import torch
    from cubie_amd.batchsolving.kernel import CompileOnly, _compile_only
    if _compile_only():
        raise CompileOnly("no generated kernel")
    from cubie_amd.batchsolving.ordering import morton_order
    rng = np.random.default_rng(100 * n + d)
    cols = []
    for k in range(d):
        x = rng.normal(size=n) * 10.0 ** rng.integers(-3, 4) + rng.normal()
        if k % 4 == 1:
            x = np.round(x, 1)              # ties
        if k % 4 == 2:
            x = np.full(n, 1.5)             # constant
        cols.append(torch.from_numpy(x.astype(np.float32 if k % 3 == 0 else np.float64)))
    want = morton_order(cols).numpy()
    got = morton_order([c.cuda() for c in cols]).cpu().numpy()
    assert sorted(want.tolist()) == list(range(n))
    assert np.array_equal(got, want)
