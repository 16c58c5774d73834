"""The filters' table over the pair distance: ordering of the pairs,
interpolated rows, the reverse onto the table's nodes and the gate that sends
a model whose filters the table cannot hold to the pair-by-pair kernels.

Tolerances: rows and gradients against float64.  A row is a sum of four table
values (each within the fp32 evaluation's 1e-6 of the largest, weights summing
to at most 1.7 in magnitude, where a cell has no node on one side) plus an
interpolation error below 2.5e-7 of it: 2e-6 of the largest value, 4e-6 for
derivatives.  Gradients are sums over the
pairs of fp32 products: 3e-6 of each tensor's norm.
"""

import math

import pytest
import torch

from tests.helpers import make_cfg, make_model, rel_err
from oracle import schnet_ref as R

pytestmark = pytest.mark.gpu

RC = 12.0


def _model(basis="gaussian", act="tanh", num_rbf=50, seed=3, trainable=False, blocks=1, scale=1.0):
    cfg = make_cfg(num_blocks=blocks, rc=RC, num_rbf=num_rbf, basis=basis, act=act)
    sd = R.random_state_dict(cfg, seed=seed)
    for k in sd:
        if k.endswith("filter_network.layers.0.weight"):
            sd[k] = sd[k] * scale
    return make_model(cfg, sd, trainable_basis=trainable)


def _pairs(dist):
    """A pair list with the given distances: pair p joins nodes 2p and 2p + 1."""
    from mlcg_amd import ops

    n = dist.numel()
    pos = torch.zeros(2 * n, 3)
    pos[1::2, 0] = dist
    ids = torch.arange(2 * n, dtype=torch.int32)
    graph = ops.PairGraph(edge_index=None, rowptr=None, col=None,
                          pair_ij=torch.stack([ids[0::2], ids[1::2]]).contiguous().cuda(),
                          pairptr=torch.tensor([n], dtype=torch.int32).cuda(), eid2pair=None,
                          frame_ptr=None, num_nodes=0, num_edges=2 * n, num_pairs=n)
    return pos.cuda(), graph


def _distances(n, h, seed=0):
    """Spread distances with the places where an index can go wrong: zero, the
    first and last cells, nodes themselves, the cutoff and its neighbours, and
    a third of the pairs at one bond length."""
    g = torch.Generator().manual_seed(seed)
    d = torch.rand(n, generator=g) * RC
    rc = torch.tensor(RC)
    edge = torch.tensor([0.0, h, 1.5 * h, 2 * h, 3.5 * h, RC - h, RC - 2.5 * h, RC / 2, RC,
                         float(torch.nextafter(rc, torch.zeros(()))), 0.3 * h])
    d[:min(n, edge.numel())] = edge[:n]
    d[n - n // 3:] = 3.8
    return d


def _filters64(model, d):
    """W, dW/dd [P, F] in float64."""
    p = {k: v.detach().double().cpu() for k, v in model.state_dict().items()}
    act = torch.tanh if isinstance(model.interaction_blocks[0].activation, torch.nn.Tanh) else (
        lambda x: torch.nn.functional.softplus(x) - math.log(2.0))
    net = "interaction_blocks.0.conv.filter_network.layers."

    def f(t):
        cut = (0.5 * (torch.cos(t * math.pi / RC) + 1.0) * (t < RC)).unsqueeze(1)
        if "rbf_layer.coeff" in p:
            g = torch.exp(p["rbf_layer.coeff"] * (t.unsqueeze(1) - p["rbf_layer.offset"]) ** 2)
        else:
            x = torch.exp(-5.0 / RC * t).unsqueeze(1)
            g = torch.exp(-p["rbf_layer.betas"] * (x - p["rbf_layer.means"]) ** 2)
        h = act(g * cut @ p[net + "0.weight"].t() + p[net + "0.bias"])
        return h @ p[net + "2.weight"].t() * cut

    t = d.double()
    return torch.func.jvp(f, (t,), (torch.ones_like(t),))


def _setup(model, dist, open_gate=True):
    from mlcg_amd import ops

    spec, P = model.fused_spec(), model.fused_params()
    grid = ops.filter_grid(spec.filt, torch.device("cuda:0"))
    pos, graph = _pairs(dist)
    b = P.blocks[0]
    tables, gates = ops.filter_tables(grid, spec.filt, [(b.W1, b.b1, b.W2)])
    assert ops.filter_tables_serve(gates).tolist() == [open_gate]
    return spec, b, grid, pos, graph, tables, gates, ops.pair_bins(pos, graph, grid)


@pytest.mark.parametrize("n", [1, 63, 64, 65, 1025, 20000])
def test_pairs_in_stencil_order(n):
    from mlcg_amd import ops

    model = _model()
    grid = ops.filter_grid(model.fused_spec().filt, torch.device("cuda:0"))
    dist = _distances(n, grid.h)
    pos, graph = _pairs(dist)
    bins = ops.pair_bins(pos, graph, grid)
    assert torch.equal(bins.dist.cpu(), dist)
    u = (dist.double() / grid.h * 2 ** 18).long()
    u[dist >= RC] = 2 ** 32 - 1
    key = ((u >> 18) - 1).clamp(0, grid.nodes - 4)
    order = torch.sort(key, stable=True).indices
    counts = torch.bincount(key, minlength=grid.nodes - 3)
    assert torch.equal(bins.records[:, 0].cpu().long(), order)
    assert torch.equal(bins.records[:, 2].cpu().long(), 2 * order + 1)
    assert torch.equal(bins.records[:, 3].cpu().long() & 0xffffffff, u[order])
    start = torch.cat([torch.zeros(1, dtype=torch.long), counts.cumsum(0)])
    runs = torch.cat([torch.zeros(1, dtype=torch.long), ((counts + 63) // 64).cumsum(0)])
    assert torch.equal(bins.start.cpu().long(), start)
    assert torch.equal(bins.runs.cpu().long(), runs)


@pytest.mark.parametrize("basis,act,num_rbf,n", [
    ("gaussian", "tanh", 50, 1), ("gaussian", "tanh", 50, 3001), ("gaussian", "ssp", 33, 3001),
    ("gaussian", "tanh", 100, 257), ("expnormal", "tanh", 64, 3001), ("expnormal", "ssp", 20, 65)])
def test_rows_match_float64(basis, act, num_rbf, n):
    from mlcg_amd import ops

    model = _model(basis, act, num_rbf)
    dist = _distances(n, ops.filter_grid_shape(model.fused_spec().filt)[1])
    spec, b, grid, pos, graph, tables, gates, bins = _setup(model, dist)
    for dt, rel in ((torch.float32, 1.0), (torch.float16, 600.0)):  # fp16: 2^-11 = 4.9e-4
        out, = ops.filter_rows(grid, bins, pos, graph, spec.filt, [(b.W1, b.b1, b.W2)], tables,
                               gates, f16=dt == torch.float16)
        assert out[0].dtype == dt
        for got, ref, tol in zip(out, _filters64(model, dist), (2e-6, 4e-6)):
            # the scale is the function's, not that of the few sampled pairs
            d = torch.linspace(0, RC, 4001)
            big = _filters64(model, d)[0 if tol == 2e-6 else 1].abs().max()
            err = (got.double().cpu() - ref).abs().max()
            assert err <= tol * rel * big, (dt, float(err / big))
    assert bool((out[0][dist.cuda() >= RC] == 0).all())


@pytest.mark.parametrize("n,one", [(1, False), (65, False), (5000, False), (3000, True)])
@pytest.mark.parametrize("tangent,ydot", [(True, True), (True, False), (False, False)])
def test_reverse_matches_pairwise_gradients(n, one, tangent, ydot):
    from mlcg_amd import ops

    model = _model("expnormal" if n == 65 else "gaussian")
    h = ops.filter_grid_shape(model.fused_spec().filt)[1]
    dist = torch.full((n,), 3.8) if one else _distances(n, h, seed=n)
    spec, b, grid, pos, graph, _, gates, bins = _setup(model, dist)
    g = torch.Generator("cuda").manual_seed(n)
    g2, y, g1, yd = (torch.randn(2 * n, 128, device="cuda", generator=g) for _ in range(4))
    dd = torch.randn(n, device="cuda", generator=g)
    args = (g2, y, g1 if tangent else None, yd if ydot else None, dd if tangent else None)

    def run():
        slots = ops.filter_table_slots(grid, graph, 1)
        ops.filter_table_reverse(grid, bins, graph, *args, gates[0], slots[0])
        wbar, wdbar = ops.filter_table_combine(grid, bins, graph, tangent, gates, slots)
        grads = ops.filter_grads(spec.filt, "cuda")
        ops.filter_bwd_blocks(grid.pos, grid.graph, spec.filt, [(b.W1, b.b1, b.W2)],
                              [(wbar[0], wdbar[0])], [grads], gates, 1)
        return grads

    got = run()
    assert all(torch.equal(x, z) for x, z in zip(got, run()))
    # float64: the pair adjoints through the network
    i, j = graph.pair_ij.long().cpu()
    g2, y, g1, yd, dd = (t.double().cpu() for t in (g2, y, g1, yd, dd))
    Wb = g2[i] * y[j] + g2[j] * y[i]
    Wdb = torch.zeros_like(Wb)
    if tangent:
        Wdb = dd.unsqueeze(1) * (g1[i] * y[j] + g1[j] * y[i])
        if ydot:
            Wb = Wb + g1[i] * yd[j] + g1[j] * yd[i]
    m64 = {k: v.detach().double().cpu() for k, v in model.state_dict().items()}
    net = "interaction_blocks.0.conv.filter_network.layers."
    W = [m64[net + k].requires_grad_(True) for k in ("0.weight", "0.bias", "2.weight")]
    t = dist.double()

    def basis(t):
        cut = (0.5 * (torch.cos(t * math.pi / RC) + 1.0) * (t < RC)).unsqueeze(1)
        if "rbf_layer.coeff" in m64:
            return torch.exp(m64["rbf_layer.coeff"]
                             * (t.unsqueeze(1) - m64["rbf_layer.offset"]) ** 2) * cut
        x = torch.exp(-5.0 / RC * t).unsqueeze(1)
        return torch.exp(-m64["rbf_layer.betas"] * (x - m64["rbf_layer.means"]) ** 2) * cut

    G, Gd = torch.func.jvp(basis, (t,), (torch.ones_like(t),))
    cut = (0.5 * (torch.cos(t * math.pi / RC) + 1.0) * (t < RC)).unsqueeze(1)
    dcut = (-0.5 * math.pi / RC * torch.sin(t * math.pi / RC) * (t < RC)).unsqueeze(1)
    H = torch.tanh(G @ W[0].t() + W[1])
    Q, Qd = H @ W[2].t(), ((1 - H * H) * (Gd @ W[0].t())) @ W[2].t()
    ref = torch.autograd.grad((Wb * Q * cut).sum() + (Wdb * (Qd * cut + Q * dcut)).sum(), W)
    for name, x, r in zip(("W1", "b1", "W2"), got, ref):
        assert rel_err(x, r) <= 3e-6, (name, rel_err(x, r))


def _batch(frames=40, beads=20):
    import numpy as np

    from mlcg_amd import synthetic

    rng = np.random.default_rng(5)
    pos = synthetic.self_avoiding_walk(frames, beads, rng)
    types = rng.integers(1, 21, size=(frames, beads))
    forces = rng.standard_normal((frames * beads, 3)).astype(np.float32)
    return synthetic._flatten(pos, types, 5, forces).to_torch("cuda")


def _step(model, table, open_gates=None):
    """A force-matching step by the given route; open_gates: of each block, as
    the step's own check left them (all, by default)."""
    from mlcg_amd import nn, ops
    from mlcg_amd.nn import _fused

    saved, _fused._FILTER_TABLE = _fused._FILTER_TABLE, table
    make, gates = ops.filter_tables, []

    def tables(*args, **kw):
        out = make(*args, **kw)
        gates.append(out[1])
        return out

    ops.filter_tables = tables
    try:
        model.zero_grad(set_to_none=True)
        gm = nn.GradientsOut(model).train()
        d = gm(_batch())
        out = d.out["SchNet"]
        torch.nn.functional.mse_loss(out["forces"], d.forces).backward()
        assert len(gates) == int(table)
        if table:
            want = open_gates or [True] * len(model.interaction_blocks)
            assert ops.filter_tables_serve(gates[0]).tolist() == want
        return [out["energy"].detach(), out["forces"].detach()] + [
            p.grad.clone() for p in model.parameters()]
    finally:
        _fused._FILTER_TABLE = saved
        ops.filter_tables = make


@pytest.mark.parametrize("basis,trainable", [("gaussian", False), ("gaussian", True),
                                             ("expnormal", True)])
def test_step_through_table_matches_pairwise(basis, trainable):
    """A whole step on both routes: the two differ by the roundings of the
    filters (4e-7) and their derivatives, 1e-5 of each tensor's norm."""
    model = _model(basis, trainable=trainable, blocks=2)
    for a, b in zip(_step(model, True), _step(model, False)):
        assert rel_err(a, b) <= 1e-5, rel_err(a, b)


@pytest.mark.parametrize("poison", ["sharp", "inf", "nan"])
def test_closed_gate_gives_the_pairwise_result(poison):
    """A filter the grid cannot hold (first-layer weights of several hundred, a
    non-finite weight) takes the pair-by-pair kernels: energies and forces bit
    for bit, gradients up to the order of the workgroups' partial sums (each
    rounding 6e-8, 1e-5 of a tensor's norm where its terms cancel)."""
    model = _model(blocks=2, scale=400.0 if poison == "sharp" else 1.0)
    if poison != "sharp":
        with torch.no_grad():
            model.interaction_blocks[1].conv.filter_network.layers[2].weight[3, 5] = float(poison)
    table = _step(model, True, [False, False] if poison == "sharp" else [True, False])
    direct = _step(model, False)
    assert torch.equal(table[0].nan_to_num(7.0), direct[0].nan_to_num(7.0))
    assert torch.equal(table[1].nan_to_num(7.0), direct[1].nan_to_num(7.0))
    for a, b in zip(table[2:], direct[2:]):
        assert torch.equal(a.isnan(), b.isnan())
        assert rel_err(a.nan_to_num(7.0), b.nan_to_num(7.0)) <= 1e-5
    from mlcg_amd import ops
    ops.numerics_flags("cuda", clear=True)  # the poisoned weights raise them on both routes


def test_gate_is_the_blocks_own():
    """One block's filters are too sharp for the grid, the other's are not."""
    from mlcg_amd import ops

    model = _model(blocks=10)  # more blocks than one launch takes
    with torch.no_grad():
        model.interaction_blocks[0].conv.filter_network.layers[0].weight.mul_(400.0)
    for a, b in zip(_step(model, True, [False] + [True] * 9), _step(model, False)):
        assert rel_err(a, b) <= 1e-5, rel_err(a, b)
    ops.numerics_flags("cuda", clear=True)


@pytest.mark.parametrize("n", [15, 700, 20001])
@pytest.mark.parametrize("closed", [(0,), (1,), (0, 2), (0, 1, 2)])
def test_closed_blocks_share_the_launch(n, closed):
    """Of a three-block launch for the blocks whose gate is closed, those take
    all the workgroups: the gradients equal, bit for bit, those of a launch of
    the closed blocks alone, and the others' stay untouched.  The same for the
    launch on the open ones."""
    from mlcg_amd import ops

    model = _model(blocks=3)
    spec, P = model.fused_spec(), model.fused_params()
    weights = [(b.W1, b.b1, b.W2) for b in P.blocks]
    pos, graph = _pairs(_distances(n, 0.01, seed=n))
    g = torch.Generator("cuda").manual_seed(n)
    adj = [tuple(torch.randn(n, 128, device="cuda", generator=g) for _ in range(2))
           for _ in range(3)]
    gates = torch.zeros(3, ops.GATE_WORDS, dtype=torch.int32, device="cuda")
    for k in closed:
        gates[k, 8] = 0x7f800000  # a pre-activation's change per node: infinite
    for want, blocks in ((0, closed), (1, [k for k in range(3) if k not in closed])):
        def run(which):
            grads = [tuple(t.fill_(7.0) for t in ops.filter_grads(spec.filt, "cuda"))
                     for _ in which]
            ops.filter_bwd_blocks(pos, graph, spec.filt, [weights[k] for k in which],
                                  [adj[k] for k in which], grads,
                                  gates[list(which)].contiguous(), want)
            return grads

        got = run(range(3))
        alone = dict(zip(blocks, run(blocks))) if blocks else {}
        for k in range(3):
            for x, y in zip(got[k], alone.get(k, (7.0, 7.0, 7.0))):
                assert torch.equal(x, y) if k in alone else bool((x == y).all()), (want, k)


@pytest.mark.parametrize("table", [True, False])
def test_one_block_of_first_layer_adjoints_at_a_time(table, monkeypatch):
    """With a trainable basis the [P, F] first-layer adjoints of one block are
    alive at a time, on either route."""
    import weakref

    from mlcg_amd import ops

    make, alive, most = ops._pair_adjoint_outputs, [], [0]

    def outputs(want, cap, F, dev):
        out = make(want, cap, F, dev)
        if want and cap > 10000:  # the pairs', not the grid nodes'
            alive.extend(weakref.ref(t) for t in out)
            most[0] = max(most[0], sum(r() is not None for r in alive))
        return out

    monkeypatch.setattr(ops, "_pair_adjoint_outputs", outputs)
    model = _model("expnormal", trainable=True, blocks=3)
    model.graph_capacity = 40000  # past the number of nodes
    _step(model, table)
    assert most[0] == 2


@pytest.mark.parametrize("basis", ["gaussian", "expnormal"])
def test_narrow_basis_between_nodes_closes_the_gate(basis):
    """Trained basis functions of a fiftieth of the grid's spacing, centred
    between nodes: every node sees a smooth filter (the functions are e^-300
    there), the pairs at the centres do not, so they go pair by pair.  A
    centre's float rounding (1e-6 A, a fortieth of the width) takes 3e-4 off a
    peak: 1e-2 of the largest value."""
    from mlcg_amd import ops

    model = _model(basis, num_rbf=50, trainable=True)
    h = ops.filter_grid_shape(model.fused_spec().filt)[1]
    d = ((torch.arange(50).double() * RC / 50 / h).floor() + 0.5) * h
    alpha = 5.0 / RC
    with torch.no_grad():
        if basis == "gaussian":
            model.rbf_layer.coeff.fill_(-0.5 / (0.02 * h) ** 2)
            model.rbf_layer.offset.copy_(d)
        else:
            slope = alpha * torch.exp(-alpha * d)
            model.rbf_layer.betas.copy_(0.5 / (0.02 * h * slope) ** 2)
            model.rbf_layer.means.copy_(torch.exp(-alpha * d))
    dist = d.float()
    spec, b, grid, pos, graph, tables, gates, bins = _setup(model, dist, open_gate=False)
    out, = ops.filter_rows(grid, bins, pos, graph, spec.filt, [(b.W1, b.b1, b.W2)], tables, gates)
    ref = _filters64(model, dist)[0]
    assert (out[0].double().cpu() - ref).abs().max() <= 1e-2 * ref.abs().max()
    ops.numerics_flags("cuda", clear=True)


def _cut64(cutoff, t):
    if cutoff.kind_id == 0:
        return torch.ones_like(t).unsqueeze(1)
    hi = cutoff.cutoff_upper
    return (0.5 * (torch.cos(t * math.pi / hi) + 1.0) * (t < hi)).unsqueeze(1)


@pytest.mark.parametrize("rc,num_rbf,basis", [(15.0, 40, "gaussian"), (12.0, 50, "gaussian"),
                                              (18.5, 50, "expnormal"), (2.0, 5, "gaussian")])
@pytest.mark.parametrize("rbf_cut,conv_hi", [("cosine", 1.0), ("cosine", 1.3),
                                             ("cosine", None), ("identity", None)])
def test_rows_in_the_first_and_last_cells(rc, num_rbf, basis, rbf_cut, conv_hi):
    """Rows of pairs within two cells of zero distance and of the cutoff, also
    where the filter does not vanish there, against float64: the fp32 sums of
    the nodes' values (3e-7 of the largest) times the weights' sum (1.6) and the
    interpolation (2.5e-7) make 7.5e-7, for derivatives 1.5e-6."""
    from mlcg_amd import nn, ops

    torch.manual_seed(5)
    cut = nn.CosineCutoff(0.0, rc) if rbf_cut == "cosine" else nn.IdentityCutoff(0.0, rc)
    conv = nn.IdentityCutoff(0.0, rc) if conv_hi is None else nn.CosineCutoff(0.0, conv_hi * rc)
    make = nn.GaussianBasis if basis == "gaussian" else nn.ExpNormalBasis
    model = nn.StandardSchNet(make(cut, num_rbf=num_rbf), conv, [64], num_interactions=1).cuda()
    spec, b = model.fused_spec(), model.fused_params().blocks[0]
    with torch.no_grad():
        b.b1.normal_(0.0, 0.1)
    grid = ops.filter_grid(spec.filt, torch.device("cuda:0"))
    x = torch.rand(600, generator=torch.Generator().manual_seed(1)) * 2 * grid.h
    dist = torch.cat([x, rc - x, torch.tensor([rc])])
    pos, graph = _pairs(dist)
    tables, gates = ops.filter_tables(grid, spec.filt, [(b.W1, b.b1, b.W2)])
    assert ops.filter_tables_serve(gates).all()
    bins = ops.pair_bins(pos, graph, grid)
    out, = ops.filter_rows(grid, bins, pos, graph, spec.filt, [(b.W1, b.b1, b.W2)], tables, gates)
    p = {k: v.detach().double().cpu() for k, v in model.state_dict().items()}

    def f(t):
        u = t.unsqueeze(1)
        if basis == "gaussian":
            g = torch.exp(p["rbf_layer.coeff"] * (u - p["rbf_layer.offset"]) ** 2)
        else:
            g = torch.exp(-p["rbf_layer.betas"]
                          * (torch.exp(-model.rbf_layer.alpha * u) - p["rbf_layer.means"]) ** 2)
        a = torch.tanh((g * _cut64(cut, t)) @ b.W1.detach().double().cpu().t()
                       + b.b1.detach().double().cpu())
        return (a @ b.W2.detach().double().cpu().t()) * _cut64(conv, t)

    def both(t):
        t = t.double()
        return torch.func.jvp(f, (t,), (torch.ones_like(t),))

    wide = both(torch.linspace(0, rc, 4001))
    for got, ref, big, tol in zip(out, both(dist), wide, (7.5e-7, 1.5e-6)):
        err = ((got.double().cpu() - ref).abs().max() / big.abs().max()).item()
        assert err <= tol, err


@pytest.mark.parametrize("basis,act,num_rbf", [("gaussian", "tanh", 50), ("expnormal", "ssp", 64),
                                               ("gaussian", "ssp", 100)])
@pytest.mark.parametrize("mode", ["split", "strict", "fp16"])
def test_blocks_forward_equals_the_single_one(basis, act, num_rbf, mode):
    """filter_fwd_blocks, which the model calls, gives every block filter_fwd's
    rows bit for bit: what is shown of the one holds for the other."""
    from mlcg_amd import ops

    model = _model(basis, act, num_rbf, blocks=9)  # more than one launch takes
    spec, P = model.fused_spec(), model.fused_params()
    pos, graph = _pairs(_distances(2001, 0.01))
    kw = dict(f16=mode == "fp16", strict_fp32=mode == "strict")
    weights = [(b.W1, b.b1, b.W2) for b in P.blocks]
    rows, dist = ops.filter_fwd_blocks(pos, graph, spec.filt, weights, **kw)
    for w, (W, Wd) in zip(weights, rows):
        ref = ops.filter_fwd(pos, graph, spec.filt, *w, **kw)
        assert torch.equal(W, ref[0]) and torch.equal(Wd, ref[1]) and torch.equal(dist, ref[2])
