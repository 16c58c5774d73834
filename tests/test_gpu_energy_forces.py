"""The node sweeps from one call each (mlcg_energy_forces, mlcg_energy_forces_grad)
against the same launches made one by one: energies, forces and parameter gradients are equal
bit for bit, since kernels, operands and order are the same."""

import pytest
import torch

from tests.helpers import make_cfg, make_model
from oracle import schnet_ref as R

pytestmark = pytest.mark.gpu


# blocks (seven pass a launch's 30 weight images), widths, activations, one and
# many frames, filters pair by pair and through their tables, in fp32 and fp16
@pytest.mark.parametrize("blocks,hidden,act,basis,frames,beads,table,f16", [
    (1, 32, "tanh", "gaussian", 1, 2, False, False),
    (2, 128, "ssp", "expnormal", 3, 17, False, False),
    (3, 64, "tanh", "gaussian", 5, 35, True, False),
    (3, 64, "ssp", "gaussian", 2, 40, False, True),
    (7, 64, "ssp", "gaussian", 2, 23, True, False),
])
def test_one_call_matches_separate_launches(blocks, hidden, act, basis, frames, beads, table,
                                            f16, monkeypatch):
    from mlcg_amd import _lib, nn, ops, synthetic
    from mlcg_amd.nn import _fused

    cfg = make_cfg(num_blocks=blocks, act=act, basis=basis, num_rbf=20)
    model = make_model(cfg, R.random_state_dict(cfg, seed=3, out_widths=(hidden,)),
                       out_widths=(hidden,))
    model.fp16_filters = f16
    data = synthetic.config1(frames, beads).to_torch("cuda")
    monkeypatch.setattr(_fused, "_FILTER_TABLE", table)
    sweeps = []
    for name in ("energy_forces", "energy_forces_grad"):
        fn = getattr(ops, name)
        monkeypatch.setattr(ops, name, lambda *a, f=fn, n=name: sweeps.append(n) or f(*a))

    def run(native):
        # a timer on the sweeps' launches asks for them one by one
        old = _lib.set_timer(None if native else _lib.LaunchTimer(None))
        try:
            gm = nn.GradientsOut(model).train(not f16)
            model.zero_grad()
            out = gm(data.clone()).out[model.name]
            if not f16:
                (out["forces"].square().sum() + out["energy"].sum()).backward()
        finally:
            _lib.set_timer(old)
        return [out["energy"].detach(), out["forces"].detach(),
                *[p.grad for p in model.parameters() if p.grad is not None]]

    got = run(True)
    assert sweeps == ["energy_forces"] + ([] if f16 else ["energy_forces_grad"])
    ref = run(False)
    assert len(sweeps) == (1 if f16 else 2)
    assert len(got) == len(ref) and (f16 or len(got) > 2)
    for a, b in zip(got, ref):
        assert torch.isfinite(b).all() and torch.equal(a, b)


def _grads(model, data, native, loss):
    """Energies, forces and parameter gradients by the native sweeps or by
    separate launches (which a launch timer asks for)."""
    from mlcg_amd import _lib, nn

    old = _lib.set_timer(None if native else _lib.LaunchTimer(None))
    try:
        training = loss is not None
        gm = nn.GradientsOut(model).train(training)
        model.zero_grad()
        out = gm(data.clone()).out[model.name]
        if training:
            loss(out).backward()
    finally:
        _lib.set_timer(old)
    return [out["energy"].detach(), out["forces"].detach(),
            *[p.grad for p in model.parameters() if p.grad is not None]]


@pytest.mark.parametrize("table", [False, True])
@pytest.mark.parametrize("loss", ["energy", "forces", "expanded"])
def test_losses_on_one_output(loss, table, monkeypatch):
    """A loss on the energies alone goes back through the separate launches
    after a native first sweep, one on the forces alone (its gradient dense, or
    one value expanded) through both native sweeps."""
    from mlcg_amd import synthetic
    from mlcg_amd.nn import _fused

    monkeypatch.setattr(_fused, "_FILTER_TABLE", table)
    cfg = make_cfg(num_blocks=2, num_rbf=20)
    model = make_model(cfg, R.random_state_dict(cfg, seed=5))
    fn = {"energy": lambda o: o["energy"].sum(), "forces": lambda o: o["forces"].square().sum(),
          "expanded": lambda o: o["forces"].sum()}[loss]
    data = synthetic.config1(3, 20).to_torch("cuda")
    got, ref = (_grads(model, data, native, fn) for native in (True, False))
    assert len(got) == len(ref) > 2
    for a, b in zip(got, ref):
        assert torch.isfinite(b).all() and torch.equal(a, b)


@pytest.mark.parametrize("table", [False, True])
def test_capacity_without_live_pairs(table, monkeypatch):
    """A graph of fixed capacity none of whose pairs is within the cutoff."""
    from mlcg_amd import synthetic
    from mlcg_amd.nn import _fused

    monkeypatch.setattr(_fused, "_FILTER_TABLE", table)
    cfg = make_cfg(num_blocks=2, num_rbf=20, rc=5.0)
    model = make_model(cfg, R.random_state_dict(cfg, seed=6))
    model.graph_capacity = 256
    data = synthetic.config1(3, 20).to_torch("cuda")
    data.pos = data.pos * 100.0
    got, ref = (_grads(model, data, native, lambda o: o["forces"].square().sum()
                       + o["energy"].square().sum()) for native in (True, False))
    assert int(model.last_graph.n_pairs_dev) == 0 and bool((got[1] == 0).all())
    for a, b in zip(got, ref):
        assert torch.isfinite(b).all() and torch.equal(a, b)


def test_linears_without_a_bias():
    """Energies and forces of a model whose block linears were replaced by ones
    without a bias: nothing to add, not an error."""
    from mlcg_amd import synthetic

    cfg = make_cfg(num_blocks=2, num_rbf=20)
    model = make_model(cfg, R.random_state_dict(cfg, seed=7))
    data = synthetic.config1(3, 20).to_torch("cuda")
    with torch.no_grad():
        for block in model.interaction_blocks:
            for lin in (block.lin, block.conv.lin2):
                lin.bias.zero_()
    ref = _grads(model, data, False, None)
    for block in model.interaction_blocks:
        for lin in (block.lin, block.conv.lin2):
            lin.bias = None
    for native in (True, False):
        for a, b in zip(_grads(model, data, native, None)[:2], ref):
            assert torch.equal(a, b)
