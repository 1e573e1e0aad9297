"""Noise hits as condensation points of their own, inside the library: whole numbers equal to the per-event loop, at the
borders of the parts of 1024 hits the counts are taken over, with empty events, without noise and with nothing else."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.mark.parametrize("splits,noise_share", [
    ([0, 1], 1.0), ([0, 1], 0.0), ([0, 0, 5, 5, 5, 70, 70], 0.5), ([0, 1023], 0.3), ([0, 1024], 0.3), ([0, 1025], 0.9),
    ([0, 1024, 2048, 2049], 0.5), ([0, 700, 700, 1500, 3072], 0.97), ([0, 2500, 5000], 0.0), ([0, 2500, 5000], 1.0),
    (list(range(0, 3001, 3)), 0.4), ([0, 1200000], 0.6)])
def test_keep_noise_in_the_library(splits, noise_share):
    from hgcalml_amd._lib import check, lib, p, stream, workspace
    from test_oracle_pins import merge_noise_per_event_loop
    rng = np.random.default_rng(len(splits) + splits[-1])
    n, rows = splits[-1], len(splits) - 1
    a, asso = np.full(n, -1, np.int32), np.full(n, -1, np.int32)
    is_cond, alpha, ncond = np.zeros(n, bool), [], [0]
    for lo, hi in zip(splits[:-1], splits[1:]):
        hits = lo + np.flatnonzero(rng.random(hi - lo) >= noise_share)
        points = rng.permutation(hits)[:max(1, len(hits) // 7)] if len(hits) else hits
        if len(hits):
            a[hits] = rng.integers(0, len(points), len(hits))
            a[points] = np.arange(len(points))
            asso[hits] = points[a[hits]]
            is_cond[points] = True
        alpha += list(points)
        ncond.append(ncond[-1] + len(points))
    rs, ncond = np.array(splits, np.int32), np.array(ncond, np.int32)
    want = merge_noise_per_event_loop(a[:, None], asso, np.array(alpha, np.int32), is_cond[:, None], ncond, rs)

    def t(x):
        return torch.from_numpy(np.ascontiguousarray(x)).to(DEV)

    room = np.full(n, -7, np.int32)
    room[:len(alpha)] = alpha
    ta, tasso, tcond, tncond = t(a), t(asso), t(is_cond), t(ncond)
    out_alpha = torch.full((2 * n,), -9, dtype=torch.int32, device=DEV)
    out_ncond, total = torch.empty_like(tncond), torch.empty(1, dtype=torch.int32, device=DEV)
    ws = workspace(lib.hgc_keep_noise_condensates_workspace_bytes(n, rows), DEV)
    tr, troom = t(rs), t(room)
    check(lib.hgc_keep_noise_condensates(p(tr), n, rows, p(troom), p(tncond), p(ta), p(tasso), p(tcond), p(out_alpha),
                                         p(out_ncond), p(total), p(ws), ws.numel(), stream()))
    count = int(total)
    got = (ta.cpu().numpy(), tasso.cpu().numpy(), out_alpha[:count].cpu().numpy(),
           tcond.cpu().numpy(), out_ncond.cpu().numpy())
    for g, w in zip(got, want):
        assert g.shape == np.asarray(w).shape and (g == w).all()
    assert (out_alpha[count:].cpu().numpy() == -9).all()
