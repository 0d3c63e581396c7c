"""GPU parity of the router's and the token sort's schedules where they change: one launch up to
16 tokens, routing ahead of the sort past them, four or sixteen logits per lane, one-launch sorts
of 2 to 32 chunks of 1024 routes.  Ids and sort tables are exact against the oracle, weights
within a few binary32 ulps."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,E,topk", [(16, 256, 8), (17, 256, 8), (16, 257, 8), (17, 1, 1), (20, 64, 64), (33, 65, 3),
                                      (1025, 256, 1), (1639, 20, 20)])
@pytest.mark.parametrize("renorm", [True, False])
def test_router_schedules(pkg, oracle_mod, dev, T, E, topk, renorm):
    g = torch.Generator().manual_seed(T + E)
    x = torch.randn(T, E, generator=g)
    x[1] = 1.0                                                   # every logit ties
    x[2, ::2], x[2, 1::2] = 0.0, -0.0
    x[3] = x[3].round()                                          # ties of some
    x[4, 1:], x[4, 0] = float("-inf"), -3e38
    w, ids, s, o, inv = torch.ops.mach_amd.moe_router(x.to(dev), topk, renorm)
    rw, rids, rs, ro, rinv = oracle_mod.moe_router(x.numpy(), topk, renorm)
    assert np.array_equal(ids.cpu().numpy(), rids)
    assert np.array_equal(o.cpu().numpy(), ro)
    assert np.array_equal(s.cpu().numpy(), rs) and np.array_equal(inv.cpu().numpy(), rinv)
    # binary32 exp, sum and quotient: a few ulps (2^-24 each) of the largest weight
    assert np.abs(w.double().cpu().numpy() - rw).max() <= 4e-6 * np.abs(rw).max()


@pytest.mark.parametrize("R,E", [(1025, 1024), (2048, 3), (9000, 256), (32768, 256), (32769, 256)])
def test_route_sort_with_dropped_ids(pkg, oracle_mod, dev, R, E):
    """Ids outside [0, E) are dropped in whatever chunk they fall."""
    ids = torch.randint(-2, E + 2, (R, 1), generator=torch.Generator().manual_seed(R), dtype=torch.int32)
    s, o, inv = torch.ops.mach_amd.moe_route(ids.to(dev), E)
    rs, ro, rinv = oracle_mod.moe_route(ids.numpy(), E)
    n = int(ro[-1])
    assert np.array_equal(o.cpu().numpy(), ro) and np.array_equal(inv.cpu().numpy(), rinv)
    assert np.array_equal(s.cpu().numpy()[:n], rs[:n])


@pytest.mark.parametrize("T,E,topk", [(8, 256, 8), (40, 300, 4), (1030, 64, 2)])
@pytest.mark.parametrize("renorm", [True, False])
def test_router_orders_nan_logits_by_their_bits(pkg, oracle_mod, dev, T, E, topk, renorm):
    """A NaN without sign lies above every logit, one with it below, an all-ones one lowest of all (its order key
    is 0, what a taken logit's becomes): ids and tables by that order, weights of the other rows as without."""
    g = torch.Generator().manual_seed(T)
    x = torch.randn(T, E, generator=g)
    bits = x.view(torch.int32)
    bits[1, 3], bits[1, E - 1] = 0x7FC00000, 0x7F800001
    bits[2, ::2] = -1
    bits[3] = -1
    bits[4, 0], bits[4, 5] = -0x400000, 0x7FFFFFFF               # 0xFFC00000
    w, ids, s, o, inv = torch.ops.mach_amd.moe_router(x.to(dev), topk, renorm)
    with np.errstate(invalid="ignore"):
        rw, rids, rs, ro, rinv = oracle_mod.moe_router(x.numpy(), topk, renorm)
    assert np.array_equal(ids.cpu().numpy(), rids)
    assert np.array_equal(o.cpu().numpy(), ro) and np.array_equal(s.cpu().numpy(), rs)
    assert np.array_equal(inv.cpu().numpy(), rinv)
    plain = [0] + list(range(5, T))
    assert np.abs(w.double().cpu().numpy()[plain] - rw[plain]).max() <= 4e-6
    assert bool(w[1].isnan().all())
