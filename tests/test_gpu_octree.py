"""The emission of child keys (four particles per thread, grid-stride) at its remainders, with split
nodes of many levels at one particle, and past one turn of its largest grid, against the oracle."""
import numpy as np
import pytest
import torch

import oracle

pytestmark = pytest.mark.gpu
CPU = oracle.Cpu("oracle")


@pytest.fixture(scope="module")
def ctx():
    from sphexa_amd import hydro

    c = hydro.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("n,bucket", [(n, 1) for n in (1, 2, 3, 4, 5, 6, 7, 8, 9, 1023, 1024, 1025)] +
                         [(1026, 3), (2 ** 21 + 2, 16), (2 ** 21 + 1027, 1)])
@pytest.mark.parametrize("kind", ["spread", "close"])
def test_octree_emission(ctx, n, bucket, kind):
    from sphexa_amd import hydro

    print("case octree emission", n, bucket, kind, flush=True)
    rng = np.random.default_rng(n)
    keys = np.sort(rng.integers(0, 2 ** 63 if kind == "spread" else max(64, 4 * n), n, dtype=np.uint64))
    leaves, counts = CPU.compute_octree(keys, bucket)
    got = hydro.compute_octree(ctx, torch.from_numpy(keys.view(np.int64)).to("cuda"), bucket)
    assert np.array_equal(got[0].cpu().numpy().view(np.uint64), leaves)
    assert np.array_equal(got[1].cpu().numpy().view(np.uint32), counts)
