"""GPU parity of the window forward (k_win_fwd: three ticks per launch, a workgroup per range of
posts and batch entry) at the sizes where it can go wrong, against the C oracle: deterministic mode
bit for bit (spikes, voltages, final state), event mode within 1e-5 / 1e-6 as long as the trains agree.

* rollouts of 1 to 26 ticks (windows of one, two and three ticks, the single last one, carried on
  from a state) from a spike history of every delay, posts around the 64-lane wave and the range, delays
  within one and over two and three groups of 8, rollouts shorter and longer than the longest;
* the same with the recurrent currents summed from the posts' rows (win_dense) wherever its history allows, over
  rows of none to 1400 hits in three ticks (more than a wave's queue holds), its history in LDS and gathered
  from memory, one batch entry over the line and another below it;
* a network that spikes so much that segments hold more spikes than their digest, a launch more
  visits than it lists at a time and more events than it links at a time;
* a network with 64 delays, whose row offsets outgrow their bound: a launch per tick.
"""
import dataclasses

import numpy as np
import pytest

from oracle.cpu import OracleCell
from tests.helpers import tiny_config
from tests.test_gpu_params import _state_dev
from v1_glif_model_amd import synthetic as sy
from v1_glif_model_amd.tables import build_cell_tables

pytestmark = pytest.mark.gpu

KW = dict(gauss_std=0.5, damp=0.5, rd=0.5, vgd=0.5, pseudo_gauss=True)
CKW = dict(gauss_std=0.5, dampening_factor=0.5, pseudo_gauss=True)


def _check(cell, net, lgn, bkg, mode, min_rate=0.0, history=None):
    oc = OracleCell(build_cell_tables(net), **KW)
    first = oc.zero_state(lgn.shape[1])
    if history is not None:
        first["zbuf"] = history
    oz, ov, _, ost = oc.forward(lgn, bkg, state=first)
    assert oz.mean() >= min_rate, oz.mean()
    T = len(lgn)
    cut = (T + 1) // 2   # in two pieces, the second from the carried state
    z0, v0, st = cell.rollout(lgn[:cut], bkg[:cut], state=_state_dev(cell, first), mode=mode)
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


def _small(n, D, T, B, nb, p=0.3):
    """A network of n posts with every delay up to D, its inputs, and a spike history of every delay."""
    fan = min(6, n)
    cfg = dataclasses.replace(tiny_config(n=n, fanin=fan, delays=D, n_lgn=70, lgn_fanin=6, n_bkg=6, bkg_fanin=3, rs=4.0,
                                          ins=150.0, lgn_p=0.3), n_basis=nb, n_syn_types=nb + 1, fanin_mean=fan,
                              fanin_sigma=None)
    net = sy.make_network(cfg, seed=n + D, dense_basis=True)
    net["network"]["synapses"]["delays"][0] = D   # every slot of the ring exists
    lgn, bkg = sy.make_inputs(cfg, seed=T, seq_len=T, batch=B)
    history = (np.random.default_rng(T).random((B, D * n)) < (1.0 if n == 1 else p)).astype(np.float32)
    return net, lgn, bkg, history


def _recurrent_counts(net, lgn, bkg, history):
    """That the recurrent events reach the currents: without them the final state is another."""
    ends = []
    for scale in (1.0, 0.0):
        other = dict(net, network=dict(net["network"], synapses=dict(net["network"]["synapses"])))
        other["network"]["synapses"]["weights"] = net["network"]["synapses"]["weights"] * np.float32(scale)
        oc = OracleCell(build_cell_tables(other), **KW)
        oz, _, _, st = oc.forward(lgn, bkg, state=dict(oc.zero_state(lgn.shape[1]), zbuf=history))
        ends.append((oz, st["psc_rise"]))
    assert not np.array_equal(ends[0][1], ends[1][1])
    return ends[0][0]


EDGES = [(1, 1, 1, 1, 1), (63, 2, 2, 3, 5), (64, 8, 3, 1, 2), (65, 9, 4, 2, 3), (128, 3, 5, 1, 6), (129, 17, 7, 2, 5),
         (769, 4, 8, 1, 8), (129, 9, 13, 2, 4), (200, 17, 22, 1, 3), (130, 24, 26, 2, 2)]


@pytest.mark.parametrize("mode", ["deterministic", "event"])
@pytest.mark.parametrize("n,D,T,B,nb", EDGES)
def test_window_edges(n, D, T, B, nb, mode):
    from v1_glif_model_amd.models import V1Column
    net, lgn, bkg, history = _small(n, D, T, B, nb)
    oz = _recurrent_counts(net, lgn, bkg, history)
    assert T < 7 or oz[:(T + 1) // 2].any()   # spikes of its own before the split too
    print(n, D, T, B, nb, mode, flush=True)
    cell = V1Column(net, **CKW)
    cell.set_forward(row_spikes=2 ** 31 - 2)
    _check(cell, net, lgn, bkg, mode, history=history)


@pytest.mark.parametrize("mode", ["deterministic", "event"])
@pytest.mark.parametrize("n,D,T,B,nb", [(1, 1, 14, 1, 1), (63, 2, 13, 3, 5), (64, 6, 14, 1, 2), (65, 5, 15, 2, 3), (128, 3, 16, 1, 6),
                                        (769, 4, 17, 2, 8), (129, 6, 18, 2, 4), (300, 1, 14, 32, 7), (130, 7, 14, 2, 4)])
def test_row_sums(n, D, T, B, nb, mode):
    """Seven delays are one too many for the history: the spikes' entries, whatever the setting."""
    from v1_glif_model_amd.models import V1Column
    net, lgn, bkg, history = _small(n, D, T, B, nb)
    _recurrent_counts(net, lgn, bkg, history)
    print(n, D, T, B, nb, mode, flush=True)
    cell = V1Column(net, **CKW)
    cell.set_forward(row_spikes=0)
    _check(cell, net, lgn, bkg, mode, history=history)


@pytest.mark.parametrize("mode", ["deterministic", "event"])
def test_row_sums_gathered(mode):
    """Too many neurons for a history in LDS."""
    from v1_glif_model_amd.models import V1Column
    cfg = dataclasses.replace(tiny_config(n=150011, fanin=3, delays=6, n_lgn=80, lgn_fanin=4, n_bkg=6, bkg_fanin=3,
                                          rs=3.0, ins=20.0, lgn_p=0.2), n_basis=2, n_syn_types=2, fanin_mean=3,
                              fanin_sigma=None)
    net = sy.make_network(cfg, seed=7)
    lgn, bkg = sy.make_inputs(cfg, seed=3, seq_len=14, batch=2)
    cell = V1Column(net, **CKW)
    cell.set_forward(row_spikes=0)
    _check(cell, net, lgn, bkg, mode, history=(np.random.default_rng(8).random((2, 6 * 150011)) < 0.2).astype(np.float32))


@pytest.mark.parametrize("mode", ["deterministic", "event"])
def test_row_sums_by_batch_entry(mode):
    """The line is drawn for each batch entry: the first one's inputs are silent."""
    from v1_glif_model_amd.models import V1Column
    net, lgn, bkg, history = _small(600, 4, 20, 3, 5)
    history[0] = lgn[:, 0] = bkg[:, 0] = 0
    oz = OracleCell(build_cell_tables(net), **KW).forward(lgn, bkg)[0]
    three = np.stack([oz[t:t + 3].sum(axis=(0, 2)) for t in range(len(oz) - 2)])
    line = int(three[:, 1:].max()) // 2
    assert line > 0 and three[:, 0].max() < line < three[:, 1:].max()
    cell = V1Column(net, **CKW)
    cell.set_forward(row_spikes=line)
    _check(cell, net, lgn, bkg, mode, history=history)


@pytest.mark.parametrize("row_spikes", [2 ** 31 - 2, 0])
@pytest.mark.parametrize("mode", ["deterministic", "event"])
def test_window_dense_activity(mode, row_spikes):
    from v1_glif_model_amd.models import V1Column
    cfg = dataclasses.replace(tiny_config(n=1500, fanin=60, delays=3, n_lgn=600, lgn_fanin=30, n_bkg=6, bkg_fanin=3,
                                          rs=0.5, ins=20.0, lgn_p=0.3), n_basis=4, n_syn_types=6, fanin_mean=60,
                              fanin_sigma=None)
    net = sy.make_network(cfg, seed=4, dense_basis=True)
    # two posts of one wave that half of the network and nearly all of it reach: their lists are long, and the
    # second one's hits are more than a queue holds; and a post without synapses between them
    syn = net["network"]["synapses"]
    pre = [np.arange(0, 1500, 2), np.arange(0, 1400)]
    hub = np.concatenate([np.stack([np.full(len(c), p, np.int64), c], -1) for p, c in zip((0, 2), pre)])
    keep = syn["indices"][:, 0] > 2
    for k, new in (("weights", np.full(len(hub), 0.01, np.float32)), ("delays", np.ones(len(hub), np.float32)),
                   ("syn_ids", np.zeros(len(hub), np.uint8))):
        syn[k] = np.concatenate([new, syn[k][keep]]).astype(syn[k].dtype)
    syn["indices"] = np.concatenate([hub, syn["indices"][keep]])
    lgn, bkg = sy.make_inputs(cfg, seed=2, seq_len=25, batch=2)
    history = (np.random.default_rng(3).random((2, 3 * 1500)) < 0.8).astype(np.float32)
    cell = V1Column(net, **CKW)
    cell.set_forward(row_spikes=row_spikes)
    _check(cell, net, lgn, bkg, mode, min_rate=0.1, history=history)


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
