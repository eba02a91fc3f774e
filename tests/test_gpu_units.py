"""GPU parity of the op's backward over work units and over the split column walk, of the counts
pull over the padded rows and of the event push with a lane per receptor, against the C oracle, at the sizes where they can go wrong: batches around
the padded row lengths (1 to 32), columns of no, one and a few synapses, around a unit's 256 synapses
and over many of them, runs of more columns than a wave has lane groups, counts and spikes.  The
forward bit for bit (also where a count is infinite), dz and dW within 1e-5 of each element's sum of
absolute terms + 1e-6 (a sum of at most a few thousand float32 terms is off by far less)."""
import numpy as np
import pytest
import torch

from oracle import cpu as orc
from oracle import dense
from v1_glif_model_amd.tables import SynapseTable as Tab

pytestmark = pytest.mark.gpu

N = 2200
LENGTHS = {
    # a column beyond 2048 synapses: always the units
    "long": [0, 1, 2, 255, 256, 257, 512, 513, 2100, 0, 3] + [1] * 130 + [7] * 40 + [100, 156, 1, 0],
    # runs of short columns: units up to 8 batch entries, the walk above
    "short": [0, 5, 9, 1, 3, 0, 2, 4] * 17 + [300, 1, 0],
    # middling columns: units at every batch
    "middle": [97, 130, 256, 300, 0, 64, 511] * 5,
    # columns of many units, whose sums several lanes add
    "tall": [20000, 300, 0, 12345, 1],
}
# rows that pad well: the counts pull, one and two, four, eight batch entries a lane by the number of posts
POSTS = {"tall": 20000, "even 5000": 5000, "even 33000": 33000}


def _table(kind, rng):
    if kind.startswith("even"):   # 10 of 100 inputs each, the last posts fewer
        n = POSTS.get(kind, N)
        pairs = [np.stack([np.full(k, p), np.sort(rng.permutation(100)[:k])], -1)
                 for p in range(n) for k in [10 if p < n - 3 else n - p]]
        ind, n_cols = np.concatenate(pairs), 100
    else:
        cols = [np.stack([rng.permutation(POSTS.get(kind, N))[:k], np.full(k, c)], -1) for c, k in enumerate(LENGTHS[kind])]
        ind, n_cols = np.concatenate(cols), len(LENGTHS[kind])
        ind = ind[np.lexsort((ind[:, 1], ind[:, 0]))]
    n = len(ind)
    return Tab(ind[:, 0].astype(np.int64), ind[:, 1].astype(np.int64), rng.normal(0, 1, n).astype(np.float32),
               rng.integers(0, 5, n).astype(np.uint8), POSTS.get(kind, N), n_cols), ind


@pytest.mark.parametrize("counts", [False, True])
@pytest.mark.parametrize("kind", ["long", "short", "middle", "even", "even 5000", "even 33000", "tall"])
@pytest.mark.parametrize("B", [1, 4, 5, 9, 16, 17, 32])
def test_units(B, kind, counts):
    from v1_glif_model_amd.ops import SynapseTable
    rng = np.random.default_rng(B)
    tab, ind = _table(kind, rng)
    basis = rng.random((5, 4)).astype(np.float32)
    print(B, kind, counts, flush=True)
    t = SynapseTable(ind, tab.syn_id, (tab.n_post, tab.n_cols), basis)
    t.set_weights(torch.tensor(tab.weight, device="cuda"))
    z = (rng.random((B, tab.n_cols)) < 0.3).astype(np.float32)
    if counts:
        z *= rng.integers(1, 4, z.shape).astype(np.float32)
    dy = rng.normal(0, 1, (B * tab.n_post, 4)).astype(np.float32)
    on = lambda a: torch.tensor(a, device="cuda")
    rdz, rdw = orc.syn_bwd(tab, z, basis, dy, use_count=counts)
    _, _, dz_abs, dw_abs = dense.syn_bwd_f64(tab, z, basis, dy, use_count=counts)
    for want_dz, want_dw in ((True, True), (True, False), (False, True)):   # together and alone
        dz, dw = t.backward(on(z), on(dy), counts=counts, want_dz=want_dz, want_dw=want_dw)
        if want_dz:
            assert np.max(np.abs(dz.cpu().numpy() - rdz) - 1e-5 * dz_abs) <= 1e-6
        if want_dw:
            assert np.max(np.abs(dw.cpu().numpy() - rdw) - 1e-5 * dw_abs) <= 1e-6
    if not counts:
        return
    for infinite in (False, True):
        if infinite:
            z[B // 2, 0] = np.inf
        with np.errstate(invalid="ignore"):
            ref = orc.syn_fwd(tab, z, basis, use_count=True)
        got = t.forward(torch.tensor(z, device="cuda"), counts=True, mode="deterministic").cpu().numpy()
        np.testing.assert_array_equal(got, ref)
        if kind.startswith("even"):   # pulled in event mode too
            ev = t.forward(torch.tensor(z, device="cuda"), counts=True, mode="event").cpu().numpy()
            np.testing.assert_array_equal(ev, ref)


@pytest.mark.parametrize("counts", [False, True])
@pytest.mark.parametrize("nb", [1, 2, 3, 4, 5, 8])
@pytest.mark.parametrize("n_cols", [129, 131073])   # over the work units; by the column scan
def test_push_receptors(n_cols, nb, counts):
    from v1_glif_model_amd.ops import SynapseTable
    rng = np.random.default_rng(nb)
    n_post, B = 701, 3
    cols = [(0, 1), (1, 17), (2, 64), (3, 65), (100, 200), (n_cols - 1, 130)]   # (column, synapses)
    ind = np.concatenate([np.stack([rng.permutation(n_post)[:k], np.full(k, c)], -1) for c, k in cols])
    ind = ind[np.lexsort((ind[:, 1], ind[:, 0]))]
    n = len(ind)
    tab = Tab(ind[:, 0].astype(np.int64), ind[:, 1].astype(np.int64), rng.normal(0, 1, n).astype(np.float32),
              rng.integers(0, 7, n).astype(np.uint8), n_post, n_cols)
    basis = rng.normal(0, 1, (7, nb)).astype(np.float32)
    basis[rng.random(basis.shape) < 0.2] = 0.0
    z = np.zeros((B, n_cols), np.float32)
    for c, _ in cols:
        z[:, c] = rng.integers(0, 3, B) if counts else rng.integers(0, 2, B)
    print(n_cols, nb, counts, flush=True)
    t = SynapseTable(ind, tab.syn_id, (n_post, n_cols), basis)
    t.set_weights(torch.tensor(tab.weight, device="cuda"))
    ev = t.forward(torch.tensor(z, device="cuda"), counts=counts, mode="event").cpu().numpy()
    ref = orc.syn_fwd(tab, z, basis, use_count=counts)
    assert np.max(np.abs(ev - ref) - 1e-5 * dense.syn_fwd_abs(tab, z, basis, use_count=counts)) <= 1e-6
