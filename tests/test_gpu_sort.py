"""sphx_sort_by_key and the octree's sorts at the edges of their forms: one workgroup, tiles with
and without the column scan launch, the prefix sort; against numpy's stable sort, bit for bit."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from sphexa_amd import hydro

    c = hydro.Context(0)
    yield c
    c.close()


def make_keys(kind, n, rng):
    if kind == "random":  # all digits vary
        return rng.integers(0, 1 << 63, n, dtype=np.uint64)
    if kind == "one_digit":  # a single digit varies, many equal keys
        return (rng.integers(0, 5, n).astype(np.uint64) << np.uint64(24)) + np.uint64(7)
    if kind == "equal":
        return np.full(n, 0x0123456789ABCDEF, np.uint64)
    if kind == "runs":  # equal top 32 bits in runs, reversed below
        return (np.arange(n, dtype=np.uint64) // np.uint64(50) << np.uint64(32)) + np.uint64(n) - np.arange(n, dtype=np.uint64)
    return np.sort(rng.integers(0, 1 << 62, n, dtype=np.uint64))[::-1].copy()  # descending


@pytest.mark.parametrize("n", [2, 63, 64, 65, 704, 705, 1024, 6143, 6144, 6145, 11264, 11265, 98304, 98305])
@pytest.mark.parametrize("kind", ["random", "one_digit", "equal", "runs", "descending"])
@pytest.mark.parametrize("entry", ["alloc", "noalloc"])
def test_sort_forms_bit_exact(ctx, n, kind, entry):
    from sphexa_amd import hydro

    print("case sort", n, kind, entry, flush=True)
    keys = make_keys(kind, n, np.random.default_rng(n))
    k = torch.from_numpy(keys.view(np.int64).copy()).to("cuda")
    v = torch.arange(n, dtype=torch.int32, device="cuda") + 3
    if entry == "alloc":
        hydro.sort_by_key(ctx, k, v)
    else:
        import ctypes as C

        ctx.check(ctx.lib.sphx_sort_by_key_noalloc(ctx.h, C.c_void_p(k.data_ptr()), C.c_void_p(v.data_ptr()), C.c_uint64(n)))
    order = np.argsort(keys, kind="stable")
    assert np.array_equal(k.cpu().numpy().view(np.uint64), keys[order])
    assert np.array_equal(v.cpu().numpy(), order.astype(np.int32) + 3)
