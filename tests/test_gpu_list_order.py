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
