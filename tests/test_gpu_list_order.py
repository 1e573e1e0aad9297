"""Weight gradients that leave in the order of the inverse lists (large tables whose lists reach far) against those written to
their slots one by one, and which tables take which way."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def gradients(table, n, k, f, mean_and_max, shift=0):
    """with scratch memory (the rule decides) and without (always slot by slot)"""
    from hgcalml_amd import ops
    from hgcalml_amd._lib import check, lib, p, stream, workspace
    gen = torch.Generator(device=DEV).manual_seed(n + f)
    dist = torch.rand(n, k, device=DEV, generator=gen) * 0.5
    feat = torch.randn(n, f, device=DEV, generator=gen)
    g = torch.randn(n, 2 * f if mean_and_max else f, device=DEV, generator=gen)
    _, arg, slots, w = torch.ops.hgcalml.accumulate_knn_exp_slots(dist, feat, table, 0, mean_and_max)
    off, inv = ops.inverse_neighbour_index(table)
    moved = torch.empty(inv.numel() + 4, dtype=torch.int32, device=DEV)
    inv_at = moved[shift:shift + inv.numel()]
    inv_at.copy_(inv)
    need = lib.hgc_accumulate_knn_grad_scratch_bytes(n, k, f, int(mean_and_max))
    results = []
    for ws in (workspace(need, DEV), None):
        gw, gx = torch.full((n, k), 7.0, device=DEV), torch.empty(n, f, device=DEV)
        if ws is not None:
            ws.fill_(0x5a)  # (what is read of it has been written before)
        check(lib.hgc_accumulate_knn_grad_scratch(p(g), p(w), p(feat), p(arg), p(slots) if mean_and_max else None, p(table), p(off),
                                                  p(inv_at), None, p(gw), p(gx), n, k, f, g.shape[1], int(mean_and_max), 1, p(ws),
                                                  need if ws is not None else 0, stream()))
        results.append((gw, gx))
    return need, results


# every point far from and near to the vertices that name it, with padded rows; the size's line; a misaligned list
@pytest.mark.parametrize("n,k,f,window,listed", [(250000, 64, 64, 2000, True), (250001, 64, 64, 100, True), (249000, 64, 64, 2000, False),
                                                 (400013, 40, 100, 3000, True)])
@pytest.mark.parametrize("mean_and_max", [True, False])
def test_both_ways_give_the_same_bits(n, k, f, window, listed, mean_and_max):
    gen = torch.Generator(device=DEV).manual_seed(k)
    stratum = 2 * window // k
    off = torch.arange(k, device=DEV, dtype=torch.int32) * stratum - window
    table = torch.empty(n, k, dtype=torch.int32, device=DEV)
    for s in range(0, n, 1 << 16):
        rows = torch.arange(s, min(n, s + (1 << 16)), device=DEV, dtype=torch.int32)[:, None]
        table[s:s + len(rows)] = (rows + off + torch.randint(0, stratum, (len(rows), k), device=DEV, generator=gen, dtype=torch.int32)) % n
    table[::7, k - 3:] = -1
    table[n // 2] = -1
    quotients = 0 if k & (k - 1) == 0 else (n * f * 4 + 255) // 256 * 256
    for shift in (0, 1):
        need, ((gw, gx), (gw_one, gx_one)) = gradients(table, n, k, f, mean_and_max, shift)
        assert need == quotients + ((n * k * 4 + 255) // 256 * 256 + 256 if listed and mean_and_max else 0)
        assert torch.equal(gw, gw_one) or not quotients == 0 and torch.allclose(gw, gw_one, rtol=1e-4, atol=1e-6)
        assert torch.equal(gx, gx_one)
        assert (gw[table < 0] == 0).all()


# near lists, lists beyond an XCD's L2, and those far beyond it in tables that fit the cache behind it and that do not
@pytest.mark.parametrize("n,k,f,window,listed", [(250000, 64, 64, 100, False), (250000, 64, 64, 2000, True), (250000, 64, 64, 3300, True),
                                                 (250000, 64, 64, 20000, False), (250000, 64, 64, None, False), (400013, 40, 100, 2000, True),
                                                 (400013, 40, 100, 20000, False), (950000, 24, 64, 16000, False), (950000, 24, 64, None, True)])
def test_which_tables_take_which_way(n, k, f, window, listed):
    """read out of the scratch memory: the device's answer and the list behind the quotients. A list that starts off a 16-byte boundary
    goes slot by slot, with the quotients, and has the same bits."""
    from hgcalml_amd import ops
    from hgcalml_amd._lib import check, lib, p, stream, workspace
    gen = torch.Generator(device=DEV).manual_seed(n + k)
    if window is None:
        table = torch.randint(0, n, (n, k), device=DEV, generator=gen, dtype=torch.int32)
    else:
        stratum = 2 * window // k
        off = torch.arange(k, device=DEV, dtype=torch.int32) * stratum - window
        rows = torch.arange(n, device=DEV, dtype=torch.int32)[:, None]
        table = (rows + off + torch.randint(0, stratum, (n, k), device=DEV, generator=gen, dtype=torch.int32)) % n
    table[::11, k - 2:] = -1
    dist, feat, g = (torch.rand(*shape, device=DEV, generator=gen) for shape in ((n, k), (n, f), (n, 2 * f)))
    _, arg, slots, w = torch.ops.hgcalml.accumulate_knn_exp_slots(dist, feat, table, 0, True)
    off, inv = ops.inverse_neighbour_index(table)
    need = lib.hgc_accumulate_knn_grad_scratch_bytes(n, k, f, 1)
    list_at, flag_at = (need - 256 - n * k * 4) // 256 * 256, need - 256
    moved = torch.empty(inv.numel() + 4, dtype=torch.int32, device=DEV)
    results = []
    for shift in (0, 1):
        at = moved[shift:shift + inv.numel()]
        at.copy_(inv)
        ws = workspace(need, DEV)
        ws.fill_(0x5a)
        gw, gx = torch.full((n, k), 7.0, device=DEV), torch.empty(n, f, device=DEV)
        check(lib.hgc_accumulate_knn_grad_scratch(p(g), p(w), p(feat), p(arg), p(slots), p(table), p(off), p(at), None, p(gw), p(gx), n,
                                                  k, f, 2 * f, 1, 1, p(ws), need, stream()))
        untouched = bool((ws[list_at:flag_at] == 0x5a).all())
        flag = ws[flag_at:flag_at + 4].view(torch.int32).item()
        assert (flag, untouched) == ((0x5a5a5a5a, True) if shift else (int(listed), not listed))
        results.append((gw, gx))
    assert all(torch.equal(a, b) for a, b in zip(*results))


@pytest.mark.parametrize("n,k,f", [(250000, 64, 64), (400013, 40, 100)])
def test_scratch_of_the_quotients_alone(n, k, f):
    """slot by slot, with the same bits"""
    from hgcalml_amd import ops
    from hgcalml_amd._lib import check, lib, p, stream, workspace
    gen = torch.Generator(device=DEV).manual_seed(n)
    rows = torch.arange(n, device=DEV, dtype=torch.int32)[:, None]
    table = (rows + torch.arange(k, device=DEV, dtype=torch.int32) * (4000 // k) - 2000) % n
    w, feat, g = (torch.rand(*shape, device=DEV, generator=gen) for shape in ((n, k), (n, f), (n, 2 * f)))
    _, arg, slots = torch.ops.hgcalml.accumulate_knn_slots(w, feat, table, 0, True)
    off, inv = ops.inverse_neighbour_index(table)
    full = lib.hgc_accumulate_knn_grad_scratch_bytes(n, k, f, 1)
    quotients = 0 if k & (k - 1) == 0 else (n * f * 4 + 255) // 256 * 256
    results = []
    for size in (full, quotients):
        ws = workspace(full, DEV)
        ws.fill_(0x5a)
        gw, gx = torch.empty(n, k, device=DEV), torch.empty(n, f, device=DEV)
        check(lib.hgc_accumulate_knn_grad_scratch(p(g), p(w), p(feat), p(arg), p(slots), p(table), p(off), p(inv), None, p(gw), p(gx),
                                                  n, k, f, 2 * f, 1, 0, p(ws), size, stream()))
        assert bool((ws[quotients:] == 0x5a).all()) == (size < full)
        results.append((gw, gx))
    assert all(torch.equal(a, b) for a, b in zip(*results))


@pytest.mark.parametrize("kind,n,k,asked", [("ordered", 250000, 64, 0), ("ordered", 400013, 40, 1), ("clone", 250000, 64, 2), ("block", 250000, 64, 0),
                                            ("block", 400013, 40, 1)])
def test_memory_is_asked_for_where_it_is_used(kind, n, k, asked, monkeypatch):
    """tables with a processing order and the block's (which reads the index of the whole table) have room for the quotients (1)
    or none (0), and only a table without an order has more (2); 64 features"""
    from hgcalml_amd import AccumulateKnn, BinnedSelectKnn, RaggedGravNet, ops
    torch.manual_seed(3)
    sizes, real = [], ops.workspace
    rs = torch.tensor([0, n], dtype=torch.int32, device=DEV)
    if kind == "block":
        out = RaggedGravNet(8, k, 3, 8, 64).to(DEV)(torch.rand(n, 8, device=DEV), rs)[0]
    else:
        idx, dist = BinnedSelectKnn(k, torch.rand(n, 3, device=DEV), rs)
        out, _ = AccumulateKnn(dist, torch.rand(n, 64, device=DEV, requires_grad=True), idx.clone() if kind == "clone" else idx)
    monkeypatch.setattr(ops, "workspace", lambda size, dev: sizes.append(size) or real(size, dev))
    out.sum().backward()
    full, quotients = ops.lib.hgc_accumulate_knn_grad_scratch_bytes(n, k, 64, 1), (n * 64 * 4 + 255) // 256 * 256
    assert (full in sizes, quotients in sizes) == (asked == 2, asked == 1)
