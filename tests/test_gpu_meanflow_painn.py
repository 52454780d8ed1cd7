"""The PaiNN meanflow denoiser (learned-dynamics_amd/meanflow_painn.py, mirror of archs/meanflow_painn8.py:127-217) and
the samplers / rollout loop of rollout.py against the oracle's restatement (oracle/models.py) with the same weights
and the same normal draws: forward passes, a pos_mutable stack (the graph is rebuilt after every block), three
rollout frames of the one-call meanflow sampler and of the reverse-diffusion loop."""
import importlib

import pytest
import torch

from oracle import models as OM
from parity import assert_parity

pytestmark = pytest.mark.gpu


def _system(B, N, box, seed):
    g = torch.Generator().manual_seed(seed)
    steps = torch.randn(B, N, 3, generator=g)
    x = (3.8 * steps / steps.norm(dim=-1, keepdim=True)).cumsum(1) + torch.rand(B, 1, 3, generator=g) * box
    one_hot = torch.nn.functional.one_hot(torch.randint(0, 20, (N,), generator=g), 20).float()
    i = torch.arange(N - 1)
    return x, one_hot, torch.cat([i, i + 1]), torch.cat([i + 1, i])


def _model(n, N, blks, r0, mutate_pos, seed):
    mp = importlib.import_module("learned-dynamics_amd.meanflow_painn")
    torch.manual_seed(seed)
    model = mp.SE3ITO(r0, n, N, blks_0=blks[0], blks_1=blks[1], mutate_pos=mutate_pos).cuda().eval()
    with torch.no_grad():
        for name, p in model.named_parameters():
            if name.endswith("gn.gamma") or name.endswith("gn.beta"):
                p.copy_(torch.randn_like(p) * (1.0 if name.endswith("gamma") else 0.1))
            if name.endswith("lin_push_pos.W"):
                p.mul_(0.05)
    sd = {k: v.detach().cpu() for k, v in model.state_dict().items()}
    return mp, model, sd


@pytest.mark.parametrize("mutate_pos", [False, True])
def test_se3ito_forward_against_oracle(pkg, mutate_pos):
    B, N, n, r0, L = 2, 256, 32, 6.0, 40.0
    box = (L, L, L)
    mp, model, sd = _model(n, N, (1, 2), r0, mutate_pos, seed=0x947 + 6)
    x0, one_hot, bs, bd = _system(B, N, L, seed=3)
    x1 = x0 + 0.4 * torch.randn(B, N, 3, generator=torch.Generator().manual_seed(4))
    s, t = torch.tensor([0.1, 0.0]), torch.tensor([0.6, 1.0])
    topo = mp.Topology(one_hot.cuda(), bs.cuda(), bd.cuda())
    with torch.no_grad():
        v = model((s.cuda(), t.cuda()), x0.cuda(), x1.cuda(), box, topo)
    ref = {dt: OM.se3ito(sd, (s, t), x0, x1, box, one_hot, bs, bd, r0, n, 1, 2, dt) for dt in (torch.float32, torch.float64)}
    assert_parity(v, ref[torch.float32], ref[torch.float64], f"SE3ITO forward, mutate_pos={mutate_pos}")
    if not mutate_pos:
        assert not bool(v[1].any())            # (s, t) = (0, 1) with positions left in place: identically zero


@pytest.mark.parametrize("n, N", [(64, 150), (128, 371)])
def test_a_step_that_moves_positions_rounds_its_additions(pkg, monkeypatch, n, N):
    """Value and derivative of a mutate_pos step with the layers' inputs added inside their kernels against additions of their own:
    the same bits.  The output subtracts moved positions from the old ones, so that one rounding less in the layer below is whole
    spacings of the positions in it."""
    diff = importlib.import_module("learned-dynamics_amd.differentiable")
    mp, model, _ = _model(n, N, (1, 2), 5.0, True, seed=0x947 + n)
    x0, one_hot, bs, bd = _system(1, N, 25.0, seed=5)
    x0 = x0.cuda()
    z, v = x0 + 0.3 * torch.randn_like(x0), torch.randn_like(x0)
    topo = mp.Topology(one_hot.cuda(), bs.cuda(), bd.cuda())
    s, t = torch.zeros(1).cuda(), torch.full((1,), 0.02).cuda()

    def step():
        return [o.detach() for o in diff.jvp(lambda z, t: model((s, t), x0, z, (40.0,) * 3, topo), (z, t), (v, torch.ones_like(t)))]

    inside, calls = step(), []
    for name in ("painn_message", "painn_update"):
        def outside(layer, *args, residual=False, own=getattr(diff, name)):
            calls.append(layer)
            args, residual = (args[:-1], args[-1]) if isinstance(args[-1], bool) else (args, residual)
            x_a, x_v = [a for a in args if torch.is_tensor(a)][:2]
            out = own(layer, *args)
            return tuple(diff.add(x, d) for x, d in zip((x_a, x_v), out)) if residual else out
        monkeypatch.setattr(diff, name, outside)
    for a, b in zip(inside, step()):
        assert torch.equal(a, b), float((a - b).norm() / b.norm())
    assert len(calls) == 9


@pytest.mark.parametrize("n, N, B, together", [(64, 150, 1, 6), (128, 130, 2, 6), (128, 400, 8, 3)])
def test_filters_of_all_blocks_together(pkg, monkeypatch, n, N, B, together):
    """A stack whose blocks' filters (of every edge, of grids, of some of both) are evaluated ahead against its blocks called one by one
    (a hook on the stack that changes nothing): rows of the same arithmetic, reduced in two orders, 2^-22 of a row each, through
    two or three blocks.  together: the filters in the one evaluation, those of both graphs of three blocks or of the bonds alone."""
    r0, box = 5.0, (40.0,) * 3
    mp, model, _ = _model(n, N, (1, 3), r0, False, seed=0x947 + n)
    x0, one_hot, bs, bd = _system(B, N, 25.0, seed=3)
    x1 = x0 + 0.4 * torch.randn(B, N, 3, generator=torch.Generator().manual_seed(4))
    topo = mp.Topology(one_hot.cuda(), bs.cuda(), bd.cuda())
    st = (torch.zeros(B).cuda(), torch.full((B,), 0.4).cuda())
    stack = model.cpainn_1
    graph_bond = mp.get_bond_graph(B, topo, torch.device("cuda"))
    flat = x1.cuda().reshape(-1, 3)
    r_bond = (flat[graph_bond.dst] - flat[graph_bond.src]).contiguous()
    x_a, x_v = torch.randn(B, N, n).cuda(), torch.randn(B, N, n, 3).cuda()
    painn, asked = importlib.import_module("learned-dynamics_amd.painn"), []
    real = painn.ops.filter_grids
    monkeypatch.setattr(painn.ops, "filter_grids", lambda *jobs: asked.append([j[0].shape[0] for j in jobs]) or real(*jobs))
    with torch.no_grad():
        got = stack(x1.cuda(), graph_bond, r_bond, x_a, x_v, box, topo)
        assert [len(rows) for rows in asked] == [together] and r_bond.shape[0] in asked[0], asked
        hook = stack.blocks.register_forward_hook(lambda *a: None)
        want = stack(x1.cuda(), graph_bond, r_bond, x_a, x_v, box, topo)
        hook.remove()
        assert torch.isfinite(model(st, x0.cuda(), x1.cuda(), box, topo)).all()
    for y, z in zip(got[1:], want[1:]):
        assert float((y - z).norm()) <= 2e-6 * float(z.norm())


def test_meanflow_rollout_against_oracle(pkg):
    """Three frames of ModelPredictor.predict around Meanflow.generate with pos_mutable blocks (otherwise the
    network's output at (0, 1) is zero and the frames are just accumulated noise), the normal draws shared."""
    ro = importlib.import_module("learned-dynamics_amd.rollout")
    B, N, n, r0, L, sigma_0, frames = 2, 256, 32, 6.0, 40.0, 0.3, 3
    box = (L, L, L)
    mp, model, sd = _model(n, N, (1, 1), r0, True, seed=0x947 + 7)
    x, one_hot, bs, bd = _system(B, N, L, seed=5)
    topo = mp.Topology(one_hot.cuda(), bs.cuda(), bd.cuda())
    dn = lambda st, x0, z1: model(st, x0, z1, box, topo)
    gen = torch.Generator("cuda").manual_seed(11)
    state = x.cuda().clone()
    traj = ro.rollout(lambda s: ro.meanflow_generate(dn, s, sigma_0, generator=gen), frames, state)
    # the same draws, in the order the sampler takes them
    gen2 = torch.Generator("cuda").manual_seed(11)
    noises = [torch.randn(B, N, 3, device="cuda", generator=gen2).cpu() for _ in range(frames)]
    refs = {}
    for dt in (torch.float32, torch.float64):
        dn_o = lambda st, x0, z1: OM.se3ito(sd, st, x0, z1, box, one_hot, bs, bd, r0, n, 1, 1, dt)
        refs[dt] = OM.rollout(lambda k, xx: OM.meanflow_generate(dn_o, xx, sigma_0, noises[k].to(dt)), frames, x.to(dt))
    assert float((refs[torch.float64][-1] - (x + sigma_0 * sum(noises)).double()).abs().max()) > 1e-3    # the network moved atoms
    for k in range(frames):
        # rel 1e-4 of the frame's scale after up to three network calls fed with their own outputs
        assert_parity(traj[k], refs[torch.float32][k], refs[torch.float64][k], f"meanflow rollout frame {k}",
                      rtol=1e-4, atol=1e-4)


def test_diffusion_rollout_against_oracle(pkg):
    """Two frames of the 4-step reverse-diffusion sampler (archs/diffuser_atoms15.py:536-555) around a denoiser that
    returns (epsilon_pred, x1_pred) built from the SE3ITO output, draws shared."""
    ro = importlib.import_module("learned-dynamics_amd.rollout")
    B, N, n, r0, L, sigma_max, zeta, steps, frames = 1, 256, 32, 6.0, 40.0, 2.0, 0.5, 4, 2
    box = (L, L, L)
    mp, model, sd = _model(n, N, (1, 1), r0, False, seed=0x947 + 8)
    x, one_hot, bs, bd = _system(B, N, L, seed=6)
    topo = mp.Topology(one_hot.cuda(), bs.cuda(), bd.cuda())

    def dn(t, x0, noised):
        tt = t.expand(x0.shape[0])
        eps = model((torch.zeros_like(tt), 0.5 * tt), x0, noised, box, topo)
        return eps, noised - 0.5 * eps
    gen = torch.Generator("cuda").manual_seed(21)
    state = x.cuda().clone()
    traj = ro.rollout(lambda s: ro.diffusion_generate(dn, s, sigma_max, zeta, steps=steps, generator=gen), frames, state)
    gen2 = torch.Generator("cuda").manual_seed(21)
    noises = [[torch.randn(B, N, 3, device="cuda", generator=gen2).cpu() for _ in range(steps + 1)] for _ in range(frames)]
    refs = {}
    for dt in (torch.float32, torch.float64):
        def dn_o(t, x0, noised, dt=dt):
            tt = t.expand(x0.shape[0])
            eps = OM.se3ito(sd, (torch.zeros_like(tt), 0.5 * tt), x0, noised, box, one_hot, bs, bd, r0, n, 1, 1, dt)
            return eps, noised - 0.5 * eps
        refs[dt] = OM.rollout(lambda k, xx: OM.diffusion_generate(dn_o, xx, sigma_max, zeta, steps,
                                                                  [z.to(dt) for z in noises[k]]), frames, x.to(dt))
    for k in range(frames):
        assert_parity(traj[k], refs[torch.float32][k], refs[torch.float64][k], f"diffusion rollout frame {k}",
                      rtol=1e-4, atol=1e-4)
