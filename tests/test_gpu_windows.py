"""GPU parity of the window forward (k_win_fwd: three ticks per launch, a workgroup per range of
posts and batch entry) at the sizes where it can go wrong, against the C oracle: deterministic mode
bit for bit (spikes, voltages, final state), event mode within 1e-5 / 1e-6 as long as the trains agree.

* rollouts of 1 to 8 ticks (windows of one, two and three ticks, the single last one, carried on
  from a state), posts around the 64-lane wave and the range, delays within one and over two
  groups of 8;
* a network that spikes so much that segments hold more spikes than their digest, a launch more
  visits than it lists at a time and more events than it links at a time;
* a network with 64 delays, whose row offsets outgrow their bound: a launch per tick.
"""
import dataclasses

import numpy as np
import pytest

from oracle.cpu import OracleCell
from tests.helpers import tiny_config
from v1_glif_model_amd import synthetic as sy
from v1_glif_model_amd.tables import build_cell_tables

pytestmark = pytest.mark.gpu

KW = dict(gauss_std=0.5, damp=0.5, rd=0.5, vgd=0.5, pseudo_gauss=True)
CKW = dict(gauss_std=0.5, dampening_factor=0.5, pseudo_gauss=True)


def _check(cell, net, lgn, bkg, mode, min_rate=0.0):
    oz, ov, _, ost = OracleCell(build_cell_tables(net), **KW).forward(lgn, bkg)
    assert oz.mean() >= min_rate, oz.mean()
    T = len(lgn)
    cut = (T + 1) // 2   # in two pieces, the second from the carried state
    z0, v0, st = cell.rollout(lgn[:cut], bkg[:cut], mode=mode)
    z, v = z0.cpu().numpy(), v0.cpu().numpy()
    if cut < T:
        z1, v1, st = cell.rollout(lgn[cut:], bkg[cut:], state=st, mode=mode)
        z, v = np.concatenate([z, z1.cpu().numpy()]), np.concatenate([v, v1.cpu().numpy()])
    if mode == "deterministic":
        np.testing.assert_array_equal(z.astype(np.uint8), oz)
        np.testing.assert_array_equal(v.view(np.uint32), ov.view(np.uint32))
        for i, k in enumerate(("zbuf", "v", "r", "asc", "psc_rise", "psc")):
            np.testing.assert_array_equal(st[i].cpu().numpy().astype(ost[k].dtype), ost[k], err_msg=k)
        return
    diff = np.nonzero(np.any(z.astype(np.uint8) != oz, axis=(1, 2)))[0]
    end = int(diff[0]) if diff.size else T
    assert end >= min(T, 3)   # a spike reaches a voltage three ticks later
    err = np.abs(v[:end].astype(np.float64) - ov[:end])
    assert np.all(err <= 1e-5 * np.abs(ov[:end]) + 1e-6), float(err.max())


@pytest.mark.parametrize("mode", ["deterministic", "event"])
@pytest.mark.parametrize("n,D,T,B,nb", [(1, 1, 1, 1, 1), (63, 2, 2, 3, 5), (64, 8, 3, 1, 2), (65, 9, 4, 2, 3),
                                        (128, 3, 5, 1, 6), (129, 17, 7, 2, 5), (769, 4, 8, 1, 8)])
def test_window_edges(n, D, T, B, nb, mode):
    from v1_glif_model_amd.models import V1Column
    fan = min(6, n)
    cfg = dataclasses.replace(tiny_config(n=n, fanin=fan, delays=D, n_lgn=70, lgn_fanin=6, n_bkg=6, bkg_fanin=3, rs=2.0,
                                          ins=6.0, lgn_p=0.3), n_basis=nb, n_syn_types=nb + 1, fanin_mean=fan,
                              fanin_sigma=None)
    net = sy.make_network(cfg, seed=n + D, dense_basis=True)
    net["network"]["synapses"]["delays"][0] = D   # every slot of the ring exists
    lgn, bkg = sy.make_inputs(cfg, seed=T, seq_len=T, batch=B)
    print(n, D, T, B, nb, mode, flush=True)
    _check(V1Column(net, **CKW), net, lgn, bkg, mode)


@pytest.mark.parametrize("mode", ["deterministic", "event"])
def test_window_dense_activity(mode):
    from v1_glif_model_amd.models import V1Column
    cfg = dataclasses.replace(tiny_config(n=1500, fanin=60, delays=3, n_lgn=600, lgn_fanin=30, n_bkg=6, bkg_fanin=3,
                                          rs=0.5, ins=20.0, lgn_p=0.3), n_basis=4, n_syn_types=6, fanin_mean=60,
                              fanin_sigma=None)
    net = sy.make_network(cfg, seed=4, dense_basis=True)
    # one post that half of the network reaches: its lists are long
    syn = net["network"]["synapses"]
    hub = np.unique(np.stack([np.zeros(750, np.int64), np.arange(0, 1500, 2)], -1), axis=0)
    keep = syn["indices"][:, 0] != 0
    for k, new in (("weights", np.full(750, 0.01, np.float32)), ("delays", np.ones(750, np.float32)),
                   ("syn_ids", np.zeros(750, np.uint8))):
        syn[k] = np.concatenate([new, syn[k][keep]]).astype(syn[k].dtype)
    syn["indices"] = np.concatenate([hub, syn["indices"][keep]])
    lgn, bkg = sy.make_inputs(cfg, seed=2, seq_len=25, batch=2)
    _check(V1Column(net, **CKW), net, lgn, bkg, mode, min_rate=0.1)


@pytest.mark.parametrize("mode", ["deterministic", "event"])
def test_per_tick_path(mode):
    """165,000 neurons with 64 delays: 8 delay groups x 165,000 rows x 215 ranges of offsets."""
    from v1_glif_model_amd.models import V1Column
    cfg = dataclasses.replace(tiny_config(n=165000, fanin=2, delays=64, n_lgn=80, lgn_fanin=4, n_bkg=6, bkg_fanin=3,
                                          rs=3.0, ins=20.0, lgn_p=0.2), n_basis=2, n_syn_types=2, fanin_mean=2,
                              fanin_sigma=None)
    net = sy.make_network(cfg, seed=6)
    lgn, bkg = sy.make_inputs(cfg, seed=3, seq_len=18, batch=1)
    _check(V1Column(net, **CKW), net, lgn, bkg, mode)
