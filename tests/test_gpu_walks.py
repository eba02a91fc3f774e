"""GPU parity of the cell backward's grouped walk against the C oracle at each row length (4, 8, 16 and
32 floats), with a column group on one, two and four lane groups (few, twice as many and four times as
many waves), in windows of three ticks up to the widest batch that takes them and of one above:
gradients within 1e-5 of the largest plus 1e-6."""
import dataclasses

import numpy as np
import pytest
import torch

from oracle.cpu import OracleCell
from tests.helpers import tiny_config
from v1_glif_model_amd import synthetic as sy
from v1_glif_model_amd.tables import build_cell_tables

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,D,B", [(301, 3, 1), (301, 3, 2), (299, 3, 6), (302, 3, 7), (300, 3, 10), (301, 3, 11),
                                   (297, 3, 17), (33001, 8, 1), (66001, 8, 1), (33001, 4, 2), (66001, 4, 2),
                                   (33001, 4, 3), (33001, 1, 10), (66001, 1, 10)])
def test_walk(n, D, B):
    from v1_glif_model_amd.models import V1Column
    big = n > 1000
    cfg = dataclasses.replace(tiny_config(n=n, fanin=2 if big else 9, delays=D, n_lgn=60, lgn_fanin=5, n_bkg=6,
                                          bkg_fanin=3, rs=3.0, ins=60.0, lgn_p=0.08),
                              n_basis=4, n_syn_types=5, fanin_mean=2 if big else 9, fanin_sigma=None)
    net = sy.make_network(cfg, seed=n + B, dense_basis=True)
    net["network"]["synapses"]["delays"][0] = D
    T = 9 if big else 19
    lgn, bkg = sy.make_inputs(cfg, seed=B, seq_len=T, batch=B)
    print(n, D, B, flush=True)
    oc = OracleCell(build_cell_tables(net), gauss_std=0.5, damp=0.5, rd=0.5, vgd=0.5, pseudo_gauss=True)
    oz, ov, oref, _ = oc.forward(lgn, bkg)
    assert oz.sum() > 0
    cell = V1Column(net, mode="deterministic", gauss_std=0.5, dampening_factor=0.5, recurrent_dampening_factor=0.5,
                    voltage_gradient_dampening=0.5, pseudo_gauss=True)
    z, _, _ = cell.rollout(lgn, bkg)
    np.testing.assert_array_equal(z.cpu().numpy().astype(np.uint8), oz)
    gz = np.random.default_rng(B).normal(0, 1, oz.shape).astype(np.float32)
    g = cell.backward(gz=torch.tensor(gz, device="cuda"))
    og = oc.backward(lgn, bkg, oz, oref, ov, gz_loss=gz)
    for k in ("rec", "lgn", "bkg"):
        a, e = g[k].cpu().numpy(), og[k]
        scale = np.max(np.abs(e))
        assert scale > 0, k
        assert np.max(np.abs(a - e)) <= 1e-5 * scale + 1e-6, k


def test_wide_windows_where_their_rows_fit():
    """A batch of 6 takes windows of three ticks, whose 32-float rows outgrow 4 GiB from 33.6 million
    rows on (here 141,000 neurons, 240 types, type by type): windows of one tick there, with both G layouts on
    one rollout."""
    from v1_glif_model_amd.models import V1Column
    n, B, T = 141_000, 6, 9
    cfg = dataclasses.replace(tiny_config(n=n, fanin=2, delays=1, n_lgn=60, lgn_fanin=3, n_bkg=6, bkg_fanin=2,
                                          rs=3.0, ins=60.0, lgn_p=0.1),
                              n_basis=2, n_syn_types=240, fanin_mean=2, fanin_sigma=None)
    net = sy.make_network(cfg, seed=5, dense_basis=True)
    lgn, bkg = sy.make_inputs(cfg, seed=6, seq_len=T, batch=B)
    oc = OracleCell(build_cell_tables(net), gauss_std=0.5, damp=0.5, rd=0.5, vgd=0.5, pseudo_gauss=True)
    oz, ov, oref, _ = oc.forward(lgn, bkg)
    gz = np.random.default_rng(B).normal(0, 1, oz.shape).astype(np.float32)
    og = oc.backward(lgn, bkg, oz, oref, ov, gz_loss=gz)
    cell = V1Column(net, mode="deterministic", gauss_std=0.5, dampening_factor=0.5, recurrent_dampening_factor=0.5,
                    voltage_gradient_dampening=0.5, pseudo_gauss=True)
    assert cell.g_layout()[1]
    cell.set_g_layout(False)
    ws = cell.workspace(B, T)
    cell.set_g_layout(True)
    z, _, _ = cell.rollout(lgn, bkg, ws=ws)
    np.testing.assert_array_equal(z.cpu().numpy().astype(np.uint8), oz)
    for compact in (True, False):
        cell.set_g_layout(compact)
        print("compact", compact, flush=True)
        g = cell.backward(gz=torch.tensor(gz, device="cuda"))
        for k in ("rec", "lgn", "bkg"):
            a, e = g[k].cpu().numpy(), og[k]
            scale = np.max(np.abs(e))
            assert scale > 0, k
            assert np.max(np.abs(a - e)) <= 1e-5 * scale + 1e-6, (compact, k)
