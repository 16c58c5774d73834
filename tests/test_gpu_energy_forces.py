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
