"""Which copies of its synapses a table keeps, and that their weights are the ones set last.

* the spike-major rows of the window forward (12 bytes per synapse and their offsets) come with the
  cell that reads them, for its recurrent and LGN tables, not with a table;
* they carry the weights that the tables held before the cell was made, and later ones, gathered at once
  (small tables) or in two passes (over a million synapses)."""
import dataclasses

import numpy as np
import pytest
import torch

from oracle.cpu import OracleCell
from tests.helpers import tiny_config
from tests.test_gpu_params import _state_dev
from v1_glif_model_amd import synthetic as sy
from v1_glif_model_amd.tables import build_cell_tables

pytestmark = pytest.mark.gpu


def _used():
    torch.cuda.synchronize()
    free, total = torch.cuda.mem_get_info()
    return total - free


def test_spike_rows_come_with_the_cell(monkeypatch):
    from v1_glif_model_amd import _lib, models
    cfg = dataclasses.replace(tiny_config(n=12000, fanin=150, delays=2, n_lgn=500, lgn_fanin=50, n_bkg=10, bkg_fanin=5),
                              n_basis=5, n_syn_types=5, fanin_mean=150, fanin_sigma=None)
    net = sy.make_network(cfg, seed=1)
    made = {}
    create = _lib.lib().glif_cell_create

    class Lib:
        def __getattr__(self, name):
            return getattr(_lib.lib(), name)

        def glif_cell_create(self, *args):
            before = _used()
            rc = create(*args)
            made["cell"] = _used() - before
            return rc
    monkeypatch.setattr(models, "lib", lambda: Lib())
    cell = models.V1Column(net)
    n = cell.rec_table.n_syn + cell.lgn_table.n_syn
    print(n, made, flush=True)
    assert made["cell"] >= 12 * n   # 2.4 million synapses: 29 MB, of 2 MB pages
    tb = build_cell_tables(net)
    lgn, bkg = sy.make_inputs(cfg, seed=3, seq_len=7, batch=2)
    oc = OracleCell(tb, gauss_std=0.5, damp=0.5, rd=0.5, vgd=0.5, pseudo_gauss=True)
    first = oc.zero_state(2)
    first["zbuf"] = (np.random.default_rng(4).random(first["zbuf"].shape) < 0.02).astype(np.float32)
    for scale in (1.0, 3.0):   # the second weights reach the rows too
        with torch.no_grad():
            cell.recurrent_weight_values.copy_(torch.tensor(tb.rec.weight * np.float32(scale)))
        other = dataclasses.replace(tb, rec=dataclasses.replace(tb.rec, weight=tb.rec.weight * np.float32(scale)))
        _, ov, _, ost = OracleCell(other, gauss_std=0.5, damp=0.5, rd=0.5, vgd=0.5, pseudo_gauss=True).forward(lgn, bkg, state=first)
        _, v, st = cell.rollout(lgn, bkg, state=_state_dev(cell, first), mode="deterministic")
        np.testing.assert_array_equal(v.cpu().numpy().view(np.uint32), ov.view(np.uint32))
        np.testing.assert_array_equal(st[4].cpu().numpy(), ost["psc_rise"])


def test_spike_rows_take_the_weights_already_set(monkeypatch):
    from v1_glif_model_amd import models
    cfg = dataclasses.replace(tiny_config(n=300, fanin=20, delays=3, rs=2.0, ins=5.0, lgn_p=0.2), n_basis=3,
                              n_syn_types=4, fanin_mean=20, fanin_sigma=None)
    net = sy.make_network(cfg, seed=2, dense_basis=True)
    tb = build_cell_tables(net)
    pops = iter((tb.rec, tb.lgn, tb.bkg))

    class Table(models.SynapseTable):
        def __init__(self, *args, **kw):
            super().__init__(*args, **kw)
            self.set_weights(torch.tensor(next(pops).weight, device="cuda"))
    monkeypatch.setattr(models, "SynapseTable", Table)
    cell = models.V1Column(net, mode="deterministic", gauss_std=0.5, dampening_factor=0.5, pseudo_gauss=True)
    cell.refresh_weights = lambda force=False: None
    lgn, bkg = sy.make_inputs(cfg, seed=3, seq_len=30, batch=2)
    oz, ov, _, _ = OracleCell(tb, gauss_std=0.5, damp=0.5, rd=0.5, vgd=0.5, pseudo_gauss=True).forward(lgn, bkg)
    assert oz.mean() > 0.01
    z, v, _ = cell.rollout(lgn, bkg)
    np.testing.assert_array_equal(z.cpu().numpy().astype(np.uint8), oz)
    np.testing.assert_array_equal(v.cpu().numpy().view(np.uint32), ov.view(np.uint32))
