"""The two-level grouping, the key index and the trilinear weights at the sizes where they can go wrong."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def mods():
    from torchsparse_amd import backend
    from torchsparse_amd.nn import functional as F
    return backend, F


@pytest.mark.parametrize("m,groups,skew", [
    (1, 1, 0), (4095, 63, 0), (4097, 65, 0), (5000, 1, 0), (40000, 64, 1),     # one bucket and its edges
    (100003, 65537, 0), (300000, 1 << 16, 1), (70000, 1 << 21, 0),             # the widest low digits
    (20000, (1 << 21) + 1, 0), (30011, 1000, 2)])                              # the library sort; one group only
def test_grouping_is_a_stable_sort(mods, m, groups, skew):
    backend, _ = mods
    rng = np.random.default_rng(m)
    idx = rng.integers(-2, groups + 2, m)
    if skew == 1:
        idx[m // 3:] = np.minimum(idx[m // 3:] % 7, groups - 1)
    if skew == 2:
        idx[:] = groups - 1
    idx = idx.astype(np.int32)
    order, starts = (t.cpu().numpy() for t in backend.group_by_index(torch.from_numpy(idx).cuda(), groups))
    valid = np.flatnonzero((idx >= 0) & (idx < groups))
    want = valid[np.argsort(idx[valid], kind="stable")]
    np.testing.assert_array_equal(order[:len(want)], want)
    np.testing.assert_array_equal(starts, np.searchsorted(idx[want], np.arange(groups + 1)))


@pytest.mark.parametrize("n,how", [(0, ""), (1, ""), (17, ""), (1025, "zero"), (200003, ""), (5000, "repeated"),
                                   ((1 << 20) - 1, ""), (1 << 20, "")])  # (with bits of the hash, without)
def test_key_index_finds_every_key(mods, n, how):
    _, F = mods
    rng = np.random.default_rng(n)
    keys = np.unique(rng.integers(-2**62, 2**62, 2 * n + 8))
    keys = rng.permutation(keys)[:n]
    if how == "zero" and n:
        keys[7] = 0
    if how == "repeated":
        keys[1000:] = keys[rng.integers(0, 1000, n - 1000)]
    queries = np.concatenate([rng.permutation(keys)[:4000], rng.integers(-2**62, 2**62, 501)])
    refs = torch.from_numpy(keys).cuda()
    for _ in range(2):  # (built, then kept)
        got = F.sphashquery(torch.from_numpy(queries).cuda(), refs).cpu().numpy()
        present = np.isin(queries, keys)
        assert got.dtype == np.int32 and ((got >= 0) == present).all()
        np.testing.assert_array_equal(keys[got[present]], queries[present])
    if n:
        refs[0] = 12345  # a changed tensor is indexed again
        assert F.sphashquery(refs[:1].clone(), refs).item() == 0


@pytest.mark.parametrize("n,scale,wide,dtype", [(0, 1, False, torch.int32), (1, 1, True, torch.int64),
                                                (257, 2, True, torch.int32), (5000, 3, False, torch.int64)])
def test_trilinear_weights_are_the_operations_of_the_definition(mods, n, scale, wide, dtype):
    _, F = mods
    gen = torch.Generator().manual_seed(n)
    points = torch.rand(n, 4, generator=gen) * 50 - 10
    index = torch.randint(-1, 5, (8, n), generator=gen).to(dtype)
    if n > 10:
        index[:, 3] = -1
    points = points[:, 1:] if wide else points[:, 1:].contiguous()
    want = F.calc_ti_weights(points, index.t(), scale)           # element-wise operations, on the host
    got = F.calc_ti_weights(points.cuda() if not wide else torch.nn.functional.pad(points, (1, 0)).cuda()[:, 1:],
                            index.cuda().t(), scale)
    assert got.shape == (n, 8) and torch.allclose(got.cpu(), want, rtol=2e-5, atol=1e-6)
