"""Gradients of the layers on the GPU against the oracle's autograd (the same formulas on the CPU in float64):
first derivatives with respect to inputs, edge vectors and weights for the PaiNN Message / Update and the rank-0/1/2
Messages / SelfTensProds; the differentiable path against the fused inference path; second-order use as the meanflow
loss makes it (torch.autograd.functional.jvp with create_graph=True followed by a backward pass,
archs/meanflow_painn8.py:274-296) through TensLinear, the 13 products, gathers and segment sums and through the whole
PaiNN meanflow denoiser; and the weight gradient's run-to-run reproducibility."""
import importlib

import pytest
import torch
import torch.autograd.forward_ad as fwAD

from oracle import layers as OL
from oracle import models as OM
from oracle import products as OP

pytestmark = pytest.mark.gpu
F64 = torch.float64


def _mlp_w(mlp, dt=F64):
    L = mlp.layers
    return {"W1": L[0].weight.detach().cpu().to(dt), "b1": L[0].bias.detach().cpu().to(dt),
            "W2": L[2].weight.detach().cpu().to(dt), "b2": L[2].bias.detach().cpu().to(dt),
            "W3": L[4].weight.detach().cpu().to(dt), "b3": L[4].bias.detach().cpu().to(dt)}


def _close(got, ref, what, tol=2e-5):
    got, ref = got.detach().cpu().double(), ref.detach().double()
    scale = max(1.0, float(ref.abs().max()))
    err = float((got - ref).abs().max())
    assert err <= tol * scale, f"{what}: max err {err:.3g} at scale {scale:.3g}"


def _ring(N, k, gen):
    src = torch.arange(N).repeat_interleave(k)
    dst = (src + torch.randint(1, N, (N * k,), generator=gen)) % N
    return src, dst


def test_painn_message_and_update_gradients(pkg):
    painn = importlib.import_module("learned-dynamics_amd.painn")
    gl = importlib.import_module("learned-dynamics_amd.graph_layers")
    torch.manual_seed(3)
    n, n_rbf, N, r0 = 16, 8, 40, 5.0
    gen = torch.Generator().manual_seed(4)
    src, dst = _ring(N, 6, gen)
    msg, upd = painn.Message(r0, n, n_rbf).cuda(), painn.Update(n).cuda()
    with torch.no_grad():
        upd.gn.gamma.normal_(); upd.gn.beta.normal_()
    x_a = torch.randn(1, N, n, generator=gen)
    x_v = torch.randn(1, N, n, 3, generator=gen)
    r = torch.randn(len(src), 3, generator=gen) * 2
    ca, cv = torch.randn(1, N, n, generator=gen), torch.randn(1, N, n, 3, generator=gen)
    graph = gl.Graph(src.cuda(), dst.cuda(), None, 1, N)
    # device
    xa_d, xv_d, r_d = (t.cuda().requires_grad_(True) for t in (x_a, x_v, r))
    da, dv = msg(graph, xa_d, xv_d, r_d)
    ua, uv = upd(xa_d + da, xv_d + dv)
    loss = (ua * ca.cuda()).sum() + (uv * cv.cuda()).sum() + (da ** 2).sum()
    loss.backward()
    # oracle, float64
    xa_o, xv_o, r_o = (t.double().requires_grad_(True) for t in (x_a, x_v, r))
    wd, wa = _mlp_w(msg.mlp_dist), _mlp_w(msg.mlp_actv)
    for w in (wd, wa):
        for v in w.values():
            v.requires_grad_(True)
    wu = {"W_l": upd.lin_l.W.detach().cpu().double().requires_grad_(True), "W_r": upd.lin_r.W.detach().cpu().double().requires_grad_(True),
          "W_v": upd.lin_v.W.detach().cpu().double().requires_grad_(True), "mlp": _mlp_w(upd.mlp),
          "gn_gamma": upd.gn.gamma.detach().cpu().double().requires_grad_(True), "gn_beta": upd.gn.beta.detach().cpu().double().requires_grad_(True)}
    for v in wu["mlp"].values():
        v.requires_grad_(True)
    oa, ov = OL.painn_message(src, dst, 1, N, xa_o, xv_o, r_o, wd, wa, r0, n, n_rbf)
    qa, qv = OL.painn_update(xa_o + oa, xv_o + ov, wu, n)
    ((qa * ca.double()).sum() + (qv * cv.double()).sum() + (oa ** 2).sum()).backward()
    _close(da, oa, "forward dx_a"); _close(uv, qv, "forward update v")
    _close(xa_d.grad, xa_o.grad, "d/dx_a"); _close(xv_d.grad, xv_o.grad, "d/dx_v"); _close(r_d.grad, r_o.grad, "d/dr_ij")
    _close(msg.mlp_dist.layers[0].weight.grad, wd["W1"].grad, "d/dW1 of mlp_dist")
    _close(msg.mlp_actv.layers[4].bias.grad, wa["b3"].grad, "d/db3 of mlp_actv")
    _close(upd.lin_r.W.grad, wu["W_r"].grad, "d/dW_r"); _close(upd.gn.gamma.grad, wu["gn_gamma"].grad, "d/dgamma")
    _close(upd.mlp.layers[2].weight.grad, wu["mlp"]["W2"].grad, "d/dW2 of the update MLP")
    # and the differentiable path gives what the fused inference path gives
    with torch.no_grad():
        fa, fv = msg(graph, x_a.cuda(), x_v.cuda(), r.cuda())
    _close(da, fa.cpu(), "differentiable vs fused dx_a", 5e-6); _close(dv, fv.cpu(), "differentiable vs fused dx_v", 5e-6)


def test_bee_layers_gradients(pkg):
    bee = importlib.import_module("learned-dynamics_amd.bee_layers")
    gl = importlib.import_module("learned-dynamics_amd.graph_layers")
    torch.manual_seed(5)
    dims, chan, N, r0 = (12, 8, 4), 16, 30, 6.0
    gen = torch.Generator().manual_seed(6)
    src, dst = _ring(N, 5, gen)
    msg, prod = bee.Messages(r0, *dims, chan).cuda(), bee.SelfTensProds(*dims, chan, groups=2).cuda()
    xs = [torch.randn(1, N, dims[0], generator=gen), torch.randn(1, N, dims[1], 3, generator=gen),
          torch.randn(1, N, dims[2], 3, 3, generator=gen)]
    r = torch.randn(len(src), 3, generator=gen) * 2
    cs = [torch.randn_like(t) for t in xs]
    graph = gl.Graph(src.cuda(), dst.cuda(), None, 1, N)
    xd = [t.cuda().requires_grad_(True) for t in xs]
    r_d = r.cuda().requires_grad_(True)
    B = msg(graph, r_d, *xd)
    Y = prod(*[x + b for x, b in zip(xd, B)])
    sum((y * c.cuda()).sum() for y, c in zip(Y, cs)).backward()
    dd = lambda p: p.detach().cpu().double().requires_grad_(True)
    Lm = msg.mlp_a.layers
    w = {"L0": dd(msg.L0.W), "L1": dd(msg.L1.W), "L2": dd(msg.L2.W), "Y": {lab: dd(getattr(msg, f"Y_{lab}").W) for lab in OP.BEE_ORDER},
         "enc_W": dd(msg.lin_enc.weight), "enc_b": dd(msg.lin_enc.bias),
         "mlp_a": {"W_direct": dd(msg.mlp_a.lin_direct.weight), "W1": dd(Lm[0].weight), "b1": dd(Lm[0].bias), "W2": dd(Lm[2].weight),
                   "b2": dd(Lm[2].bias), "W3": dd(Lm[4].weight), "b3": dd(Lm[4].bias)}}
    ws = {k: dd(getattr(prod, k).W) for k in ("L0", "R0", "L1", "R1", "L2", "R2")}
    ws["Y"] = {lab: dd(getattr(prod, f"Y_{lab}").W) for lab in OP.BEE_ORDER}
    ws.update(gn_a=dd(prod.gn_a.gamma), gn_v=dd(prod.gn_v.gamma), gn_d=dd(prod.gn_d.gamma))
    xo = [t.double().requires_grad_(True) for t in xs]
    r_o = r.double().requires_grad_(True)
    Bo = OL.bee_messages(src, dst, 1, N, r_o, *xo, w, r0)
    Yo = OL.self_tens_prods(*[x + b for x, b in zip(xo, Bo)], ws, groups=2)
    sum((y * c.double()).sum() for y, c in zip(Yo, cs)).backward()
    for k in range(3):
        _close(Y[k], Yo[k], f"forward rank {k}")
        _close(xd[k].grad, xo[k].grad, f"d/dx rank {k}")
    _close(r_d.grad, r_o.grad, "d/dr_ij")
    _close(msg.Y_212.W.grad, w["Y"]["212"].grad, "d/dY_212 (Messages)")
    _close(msg.lin_enc.weight.grad, w["enc_W"].grad, "d/d lin_enc")
    _close(msg.mlp_a.layers[2].weight.grad, w["mlp_a"]["W2"].grad, "d/dW2 of mlp_a")
    _close(prod.R1.W.grad, ws["R1"].grad, "d/dR1"); _close(prod.Y_111.W.grad, ws["Y"]["111"].grad, "d/dY_111 (SelfTensProds)")
    _close(prod.gn_d.gamma.grad, ws["gn_d"].grad, "d/d gn_d.gamma")


def test_displacement_tensors_gradients(pkg):
    """DisplacementTensors under autograd (archs/diffuser_atoms15.py:206-225): outputs, the gradients for the edge
    vectors and every parameter against the oracle's autograd in float64; the same tangent in forward mode as from
    nested backward passes."""
    bee = importlib.import_module("learned-dynamics_amd.bee_layers")
    gl = importlib.import_module("learned-dynamics_amd.graph_layers")
    diff = importlib.import_module("learned-dynamics_amd.differentiable")
    torch.manual_seed(0x947 + 59)
    dims, N, r0 = (24, 12, 6), 60, 6.0
    gen = torch.Generator().manual_seed(7)
    src, dst = _ring(N, 7, gen)
    mod = bee.DisplacementTensors(r0, *dims).cuda()
    r = torch.randn(len(src), 3, generator=gen) * 2.5
    graph = gl.Graph(src.cuda(), dst.cuda(), None, 1, N)
    cs = [torch.randn(1, N, dims[0], generator=gen), torch.randn(1, N, dims[1], 3, generator=gen),
          torch.randn(1, N, dims[2], 3, 3, generator=gen)]
    r_d = r.cuda().requires_grad_(True)
    out = mod(graph, r_d)
    sum((y * c.cuda()).sum() for y, c in zip(out, cs)).backward()
    dd = lambda p: p.detach().cpu().double().requires_grad_(True)
    L = mod.mlp_radial[1].layers
    w = {"lin_W": dd(mod.mlp_radial[0].weight), "lin_b": dd(mod.mlp_radial[0].bias),
         "mlp": {"W_direct": dd(mod.mlp_radial[1].lin_direct.weight), "W1": dd(L[0].weight), "b1": dd(L[0].bias),
                 "W2": dd(L[2].weight), "b2": dd(L[2].bias), "W3": dd(L[4].weight), "b3": dd(L[4].bias)},
         "readout_v": dd(mod.readout_v.W), "readout_d": dd(mod.readout_d.W)}
    r_o = r.double().requires_grad_(True)
    ref = OL.displacement_tensors(src, 1, N, r_o, w, r0)
    sum((y * c.double()).sum() for y, c in zip(ref, cs)).backward()
    for k in range(3):
        _close(out[k], ref[k], f"A rank {k}")
    _close(r_d.grad, r_o.grad, "d/dr_ij")
    _close(mod.mlp_radial[0].weight.grad, w["lin_W"].grad, "d/d first linear")
    _close(mod.mlp_radial[1].layers[2].weight.grad, w["mlp"]["W2"].grad, "d/dW2 of the radial MLP")
    _close(mod.mlp_radial[1].lin_direct.weight.grad, w["mlp"]["W_direct"].grad, "d/d direct")
    _close(mod.readout_v.W.grad, w["readout_v"].grad, "d/d readout_v")
    _close(mod.readout_d.W.grad, w["readout_d"].grad, "d/d readout_d")
    f = lambda rr: mod(graph, rr)[2]
    u = torch.randn(len(src), 3, generator=gen).cuda()
    _, t_fw = diff.jvp(f, (r.cuda(),), (u,))
    _, t_bw = torch.autograd.functional.jvp(f, (r.cuda(),), (u,), create_graph=True)
    _close(t_fw, t_bw.double().cpu(), "tangent of A_d", 1e-5)


def test_norm_and_sigmoid_modules_under_autograd(pkg):
    """ScalGroupNorm, TensGroupNorm, TensSigmoid / tens_sigmoid called as modules with inputs that want a gradient
    (managan/layers_common.py:201-223, managan/tensor_products.py:167-232): outputs and gradients against the oracle's
    formulas in float64; without a gradient the same modules run the fused kernels and agree."""
    tp = importlib.import_module("learned-dynamics_amd.tensor_products")
    lc = importlib.import_module("learned-dynamics_amd.layers_common")
    g = torch.Generator().manual_seed(0x947 + 61)
    B, N, chan = 2, 50, 16
    sn, tn = lc.ScalGroupNorm(chan, 4, epsilon=0.5).cuda(), tp.TensGroupNorm(1, chan, 4).cuda()
    with torch.no_grad():
        sn.gamma.normal_(); sn.beta.normal_(); tn.gamma.normal_()
    x = torch.randn(B, N, chan, generator=g)
    v = torch.randn(B, N, chan, 3, generator=g)
    c_x, c_v = torch.randn(B, N, chan, generator=g), torch.randn(B, N, chan, 3, generator=g)
    xd, vd = x.cuda().requires_grad_(), v.cuda().requires_grad_()
    ys, yt, yg = sn(xd), tn(vd), tp.TensSigmoid(1)(vd)
    assert ys.grad_fn is not None and yt.grad_fn is not None and yg.grad_fn is not None
    ((ys * c_x.cuda()).sum() + (yt * c_v.cuda()).sum() + (yg * c_v.cuda()).sum()).backward()
    xo, vo = x.double().requires_grad_(), v.double().requires_grad_()
    dd = lambda p: p.detach().cpu().double().requires_grad_()
    gam_s, bet_s, gam_t = dd(sn.gamma), dd(sn.beta), dd(tn.gamma)
    rs = OL.scal_group_norm(xo, 4, gam_s, bet_s, 0.5)
    rt = OL.tens_group_norm(1, vo, 4, gam_t, 1e-5)
    rg = OL.tens_sigmoid(1, vo)
    ((rs * c_x.double()).sum() + (rt * c_v.double()).sum() + (rg * c_v.double()).sum()).backward()
    _close(ys, rs, "ScalGroupNorm"); _close(yt, rt, "TensGroupNorm"); _close(yg, rg, "TensSigmoid")
    _close(xd.grad, xo.grad, "d/dx"); _close(vd.grad, vo.grad, "d/dv")
    _close(sn.gamma.grad, gam_s.grad, "d/d gamma (scalar)"); _close(sn.beta.grad, bet_s.grad, "d/d beta")
    _close(tn.gamma.grad, gam_t.grad, "d/d gamma (tensor)")
    with torch.no_grad():
        _close(sn(x.cuda()), rs, "ScalGroupNorm, fused"); _close(tn(v.cuda()), rt, "TensGroupNorm, fused")
        _close(tp.tens_sigmoid(1, v.cuda()), rg, "tens_sigmoid, fused")


def test_second_order_through_linear_products_gather_and_scatter(pkg):
    """jvp(create_graph=True) of f(x) = scatter(Y(Bee(L x, R gather(x)))) and a backward pass through the result,
    against the same thing on the oracle's functions."""
    tp = importlib.import_module("learned-dynamics_amd.tensor_products")
    cg = importlib.import_module("learned-dynamics_amd.codegen_tensor_products")
    gl = importlib.import_module("learned-dynamics_amd.graph_layers")
    gen = torch.Generator().manual_seed(7)
    N, C = 12, 8
    src, dst = _ring(N, 3, gen)
    graph = gl.Graph(src.cuda(), dst.cuda(), None, 1, N)
    W = [torch.randn(C, C, generator=gen) * 0.4 for _ in range(7)]
    xs = [torch.randn(1, N, C, generator=gen), torch.randn(1, N, C, 3, generator=gen), torch.randn(1, N, C, 3, 3, generator=gen)]
    vs = [torch.randn_like(t) for t in xs]

    def f_dev(Wd):
        def f(a, v, d):
            l = [tp.tensor_linear(k, Wd[k], t.reshape(N, C, *([3] * k))) for k, t in enumerate((a, v, d))]
            r = [gl.edges_read_dst(graph, tp.tensor_linear(k, Wd[3 + k], t).contiguous()) for k, t in enumerate((a, v, d))]
            l = [t[src.cuda()] for t in l]
            prods = cg.Bee.apply(*l, *r)
            y = tp.tensor_linear(1, Wd[6], prods[11]) + prods[5] + prods[3] + prods[4] + prods[6]   # 111 (chiral), 121, 011, 101, 211
            return gl.edges_reduce_src(graph, y)
        return f

    def f_ref(Wr):
        def f(a, v, d):
            l = [OP.tensor_linear(k, Wr[k], t.reshape(N, C, *([3] * k)))[src] for k, t in enumerate((a, v, d))]
            r = [OL.edges_read_dst(dst, OP.tensor_linear(k, Wr[3 + k], t), 1, N) for k, t in enumerate((a, v, d))]
            prods = OP.bee(*l, *r)
            y = OP.tensor_linear(1, Wr[6], prods[11]) + prods[5] + prods[3] + prods[4] + prods[6]
            return OL.edges_reduce_src(src, y, 1, N)
        return f

    Wd = [w.cuda().requires_grad_(True) for w in W]
    xd = tuple(t.cuda().requires_grad_(True) for t in xs)
    out_d, jvp_d = torch.autograd.functional.jvp(f_dev(Wd), xd, tuple(v.cuda() for v in vs), create_graph=True)
    (jvp_d ** 2).sum().backward()
    Wr = [w.double().requires_grad_(True) for w in W]
    xr = tuple(t.double().requires_grad_(True) for t in xs)
    out_r, jvp_r = torch.autograd.functional.jvp(f_ref(Wr), xr, tuple(v.double() for v in vs), create_graph=True)
    (jvp_r ** 2).sum().backward()
    _close(out_d, out_r, "f"); _close(jvp_d, jvp_r, "jvp")
    for k in range(3):
        _close(xd[k].grad, xr[k].grad, f"d(jvp^2)/dx rank {k}", 1e-4)
    for k in range(7):
        _close(Wd[k].grad, Wr[k].grad, f"d(jvp^2)/dW[{k}]", 1e-4)


def _meanflow_case():
    """A small PaiNN meanflow denoiser with positions that move, its float64 copy for the oracle, and one batch."""
    mp = importlib.import_module("learned-dynamics_amd.meanflow_painn")
    torch.manual_seed(0x947 + 9)
    B, N, n, r0, L = 1, 48, 8, 5.0, 30.0
    box = (L, L, L)
    model = mp.SE3ITO(r0, n, N, blks_0=1, blks_1=1, mutate_pos=True).cuda()
    with torch.no_grad():
        for name, p in model.named_parameters():
            if name.endswith("lin_push_pos.W"):
                p.mul_(0.05)
    sd = {k: v.detach().cpu().double().requires_grad_(True) for k, v in model.state_dict().items()}
    gen = torch.Generator().manual_seed(2)
    steps = torch.randn(B, N, 3, generator=gen)
    x_prev = (2.0 * steps / steps.norm(dim=-1, keepdim=True)).cumsum(1) + 0.5 * L
    z_0 = x_prev + 0.2 * torch.randn(B, N, 3, generator=gen)
    z_1 = x_prev + 0.5 * torch.randn(B, N, 3, generator=gen)
    t, s = torch.tensor([0.7]), torch.tensor([0.2])
    one_hot = torch.nn.functional.one_hot(torch.randint(0, 20, (N,), generator=gen), 20).float()
    i = torch.arange(N - 1)
    bs, bd = torch.cat([i, i + 1]), torch.cat([i + 1, i])
    topo = mp.Topology(one_hot.cuda(), bs.cuda(), bd.cuda())
    on_device = lambda st, x0, z: model(st, x0, z, box, topo)
    oracle = lambda st, x0, z: OM.se3ito(sd, st, x0, z, box, one_hot.double(), bs, bd, r0, n, 1, 1, F64)
    return model, sd, on_device, oracle, (x_prev, z_0, z_1, t, s)


def _meanflow_loss(dn, to, batch, jvp_of):
    """archs/meanflow_painn8.py:283-296 up to the mean over the batch.  jvp_of(f, primals, tangents) -> (f(primals)
    or None, jvp); when the first is None the model is evaluated again for v_pred, as the reference does."""
    x_prev, z_0, z_1, t, s = batch
    z_t = to(t)[:, None, None] * to(z_1) + (1 - to(t)[:, None, None]) * to(z_0)
    v = to(z_1) - to(z_0)
    f = lambda zz, tt: dn((to(s), tt), to(x_prev), zz)
    v_pred, jvp = jvp_of(f, (z_t, to(t)), (v, torch.ones_like(to(t))))
    v_target = v - (to(t) - to(s))[:, None, None] * jvp
    if v_pred is None:
        v_pred = dn((to(s), to(t)), to(x_prev), z_t)
    return ((v_pred - v_target) ** 2).mean(), jvp


def _nested_backward_jvp(f, primals, tangents):
    return None, torch.autograd.functional.jvp(f, primals, tangents, create_graph=True)[1]


def _check_meanflow_gradients(model, sd, loss_d, jvp_d, loss_r, jvp_r):
    _close(jvp_d, jvp_r, "jvp of the denoiser", 1e-4)
    assert abs(float(loss_d.detach()) - float(loss_r.detach())) <= 1e-4 * max(1.0, abs(float(loss_r.detach())))
    checked = 0
    for name, p in model.named_parameters():
        if p.grad is None:
            continue
        ref = sd[name].grad
        assert ref is not None, name
        _close(p.grad, ref, f"d loss / d {name}", 5e-4)
        checked += 1
    assert checked >= 40


def test_meanflow_loss_through_the_painn_denoiser(pkg):
    """v_target = v - (t - s) jvp, loss = mean (v_pred - v_target)^2, loss.backward(): the reference's training step
    (archs/meanflow_painn8.py:274-296) on a small PaiNN meanflow denoiser with positions that move, against the oracle."""
    model, sd, on_device, oracle, batch = _meanflow_case()
    loss_d, jvp_d = _meanflow_loss(on_device, lambda a: a.cuda(), batch, _nested_backward_jvp)
    loss_d.backward()
    loss_r, jvp_r = _meanflow_loss(oracle, lambda a: a.double(), batch, _nested_backward_jvp)
    loss_r.backward()
    _check_meanflow_gradients(model, sd, loss_d, jvp_d, loss_r, jvp_r)


def test_meanflow_loss_with_the_jvp_in_forward_mode(pkg):
    """The same loss and gradients with the Jacobian-vector product taken in forward mode (differentiable.jvp: one
    pass gives v_pred and the jvp) against the oracle, which keeps the reference's nested backward passes."""
    diff = importlib.import_module("learned-dynamics_amd.differentiable")
    model, sd, on_device, oracle, batch = _meanflow_case()
    loss_d, jvp_d = _meanflow_loss(on_device, lambda a: a.cuda(), batch, diff.jvp)
    assert jvp_d.grad_fn is not None
    loss_d.backward()
    loss_r, jvp_r = _meanflow_loss(oracle, lambda a: a.double(), batch, _nested_backward_jvp)
    loss_r.backward()
    _check_meanflow_gradients(model, sd, loss_d, jvp_d, loss_r, jvp_r)
    # forward mode leaves nothing behind on the inputs or the parameters
    assert all(not diff.has_tangent(p) for p in model.parameters())


def test_forward_mode_rules_agree_with_nested_backward(pkg, ops):
    """differentiable.jvp against torch.autograd.functional.jvp on each autograd function that has a forward-mode
    rule (linear with and without bias and with emitted row bounds, SiLU, gather, segment sum, the PaiNN combine, the
    13 products alone and with the edge filters and gathers folded in, one bare product),
    and a backward pass through the tangent against one through the nested-backward result."""
    diff = importlib.import_module("learned-dynamics_amd.differentiable")
    gl = importlib.import_module("learned-dynamics_amd.graph_layers")
    tp = importlib.import_module("learned-dynamics_amd.tensor_products")
    g = torch.Generator().manual_seed(0x947 + 31)
    rnd = lambda *shape: torch.randn(*shape, generator=g).cuda()
    nodes, n = 40, 16
    src = torch.sort(torch.randint(0, nodes, (300,), generator=g)).values
    dst = torch.randint(0, nodes, (300,), generator=g)
    graph = gl.Graph(src.cuda(), dst.cuda(), None, 1, nodes)
    W, W1, b = rnd(24, n).requires_grad_(), rnd(8, n).requires_grad_(), rnd(24).requires_grad_()
    torch.manual_seed(5)
    lin, lin2 = torch.nn.Linear(n, 24).cuda(), torch.nn.Linear(24, 24).cuda()

    def linear_chain(x, xv):
        y, bound = diff.linear(lin, x, want_bound=True)
        z = diff.linear(lin2, diff.silu(y), x_bound=bound)
        return z.sum(-1, keepdim=True) * tp.tensor_linear(1, W1, xv)[..., 0, :] + tp.tensor_linear(0, W, x, bias=b)[:, :3]

    def graph_ops(x):
        x_src, x_dst = gl.edges_read(graph, x[None])
        return gl.edges_reduce_src(graph, diff.silu(x_src) * x_dst)

    def combine(dist, actv, v, r):
        direction = r / torch.sqrt(0.01 + (r ** 2).sum(-1, keepdim=True))
        out_v, out_a = diff.painn_combine(graph, dist, actv[None], v[None], direction)
        return out_v.sum(-2) * out_a[..., :3]

    bee = importlib.import_module("learned-dynamics_amd.bee_layers")
    dims = (12, 8, 4)
    msg, prod = bee.Messages(6.0, *dims, 16).cuda(), bee.SelfTensProds(*dims, 16, groups=2).cuda()
    bare = tp.TensorProdBare(1, 2, 1)

    def rank012_block(r, a, v, d):
        B = msg(graph, r, a[None], v[None], d[None])
        ya, yv, yd = prod(a[None] + B[0], v[None] + B[1], d[None] + B[2])
        return ya.sum(-1)[..., None] + bare(yv.sum(-2, keepdim=True), yd.sum(-3, keepdim=True))[..., 0, :]

    cases = [("linear chain", linear_chain, (rnd(50, n), rnd(50, n, 3)),
              [W, W1, b] + list(lin.parameters()) + list(lin2.parameters())),
             ("gather / segment sum", graph_ops, (rnd(nodes, 12),), []),
             ("painn combine", combine, (rnd(300, 4 * n), rnd(nodes, 4 * n), rnd(nodes, n, 3), rnd(300, 3)), []),
             ("Messages, SelfTensProds and one bare product", rank012_block,
              (2.0 * rnd(300, 3), rnd(nodes, dims[0]), rnd(nodes, dims[1], 3), rnd(nodes, dims[2], 3, 3)),
              list(msg.parameters()) + list(prod.parameters()))]
    for name, f, primals, params in cases:
        tangents = tuple(rnd(*p.shape) for p in primals)
        leaves = [p.requires_grad_() for p in primals] + params
        value, tangent = diff.jvp(f, primals, tangents)
        grads = torch.autograd.grad((tangent ** 2).sum() + value.sum(), leaves, allow_unused=True)
        value_n, tangent_n = torch.autograd.functional.jvp(f, primals, tangents, create_graph=True)
        grads_n = torch.autograd.grad((tangent_n ** 2).sum() + value_n.sum(), leaves, allow_unused=True)
        _close(value, value_n.double().cpu(), f"{name}: value", 1e-5)
        _close(tangent, tangent_n.double().cpu(), f"{name}: tangent", 1e-4)
        for k, (a, r) in enumerate(zip(grads, grads_n)):
            assert (a is None) == (r is None), (name, k)
            if a is not None:
                _close(a, r.double().cpu(), f"{name}: gradient {k}", 1e-4)


def test_rank012_denoiser_in_forward_mode(pkg):
    """The whole rank-0/1/2 denoiser (neighbour search, time embedding, two blocks of Messages + SelfTensProds, readout)
    under differentiable.jvp against torch.autograd.functional.jvp(create_graph=True) on the device: value, tangent and
    the gradients of a function of both for every parameter."""
    den = importlib.import_module("learned-dynamics_amd.denoiser")
    diff = importlib.import_module("learned-dynamics_amd.differentiable")
    torch.manual_seed(0x947 + 51)
    B, N, box = 2, 200, (30.0, 30.0, 30.0)
    model = den.Denoiser(6.0, dim_a=32, dim_v=16, dim_d=8, chan=32, blocks=2).cuda()
    g = torch.Generator().manual_seed(1)
    x1 = (torch.rand(B, N, 3, generator=g) * 30).cuda()
    x0 = x1 + 0.3 * torch.randn(B, N, 3, generator=g).cuda()
    one_hot = torch.nn.functional.one_hot(torch.randint(0, 20, (B, N), generator=g), 20).float().cuda()
    s, t = torch.zeros(B).cuda(), torch.rand(B, generator=g).cuda()
    v = torch.randn(B, N, 3, generator=g).cuda()
    f = lambda xx, tt: model((s, tt), x0, xx, one_hot, box)
    params = list(model.parameters())
    value, tangent = diff.jvp(f, (x1, t), (v, torch.ones_like(t)))
    got = torch.autograd.grad((tangent ** 2).sum() + value.sum(), params, allow_unused=True)
    value_n, tangent_n = torch.autograd.functional.jvp(f, (x1, t), (v, torch.ones_like(t)), create_graph=True)
    ref = torch.autograd.grad((tangent_n ** 2).sum() + f(x1, t).sum(), params, allow_unused=True)
    _close(value, value_n.double().cpu(), "value", 1e-5)
    _close(tangent, tangent_n.double().cpu(), "tangent", 1e-5)
    checked = 0
    for (name, _), a, r in zip(model.named_parameters(), got, ref):
        assert (a is None) == (r is None), name
        if a is not None:
            _close(a, r.double().cpu(), f"gradient for {name}", 1e-4)
            checked += 1
    assert checked >= 80


def test_weight_gradient_is_reproducible(ops):
    g = torch.Generator().manual_seed(8)
    dy, x = torch.randn(30000, 96, 3, generator=g).cuda(), torch.randn(30000, 64, 3, generator=g).cuda()
    a = ops.tensor_linear_wgrad(1, dy, x)
    for _ in range(3):
        assert torch.equal(ops.tensor_linear_wgrad(1, dy, x), a)
    ref = torch.einsum("rot,rit->oi", dy.double().cpu(), x.double().cpu())
    torch.testing.assert_close(a.cpu().double(), ref, rtol=1e-5, atol=2e-5 * float(ref.abs().max()))


@pytest.mark.parametrize("lro", [(1, 1, 0), (0, 1, 1), (1, 1, 2), (1, 2, 1), (2, 2, 2)])
def test_tensor_prods_module_trains(lro):
    """TensorProds (managan/tensor_products.py:109-121) with gradients: first derivatives for both operands and the
    three weights, and a second derivative (gradient of a gradient norm), against autograd through the oracle."""
    tp = importlib.import_module("learned-dynamics_amd.tensor_products")
    il, ir, io = lro
    torch.manual_seed(11 + sum(lro))
    mod = tp.TensorProds(il, ir, io, 24, 40, 16, 32).cuda()
    g = torch.Generator().manual_seed(12)
    x_l = torch.randn(7, 5, 24, *([3] * il), generator=g)
    x_r = torch.randn(7, 5, 40, *([3] * ir), generator=g)
    cot = torch.randn(7, 5, 16, *([3] * io), generator=g)

    def run(W, xl, xr, c):
        return (OP.tensor_prods(il, ir, io, *W, xl, xr) * c).sum()

    Wd = [p.detach().cpu().double().requires_grad_() for p in (mod.lin_l.W, mod.lin_r.W, mod.lin_o.W)]
    xl_d, xr_d = x_l.double().requires_grad_(), x_r.double().requires_grad_()
    ref = torch.autograd.grad(run(Wd, xl_d, xr_d, cot.double()), [xl_d, xr_d, *Wd], create_graph=True)
    ref2 = torch.autograd.grad(sum((r ** 2).sum() for r in ref[:2]), [xl_d, xr_d, *Wd])

    xl_g, xr_g = x_l.cuda().requires_grad_(), x_r.cuda().requires_grad_()
    params = [mod.lin_l.W, mod.lin_r.W, mod.lin_o.W]
    y = mod(xl_g, xr_g)
    assert y.requires_grad
    got = torch.autograd.grad((y * cot.cuda()).sum(), [xl_g, xr_g, *params], create_graph=True)
    got2 = torch.autograd.grad(sum((r ** 2).sum() for r in got[:2]), [xl_g, xr_g, *params])
    for a, r in zip(list(got) + list(got2), list(ref) + list(ref2)):
        torch.testing.assert_close(a.detach().cpu().double(), r.detach(), rtol=2e-4, atol=2e-5 * float(r.abs().max()) + 1e-9)


@pytest.mark.parametrize("lro", [(0, 0, 0), (1, 1, 0), (2, 2, 0), (0, 1, 1), (1, 0, 1), (1, 2, 1), (2, 1, 1),
                                 (0, 2, 2), (2, 0, 2), (1, 1, 2), (2, 2, 2)])
def test_one_product_autograd_function(lro):
    """TensorProdBare with gradients (one product kernel per gradient, tensor_products._ProdBareFn): first derivatives
    for both operands and the gradient of a gradient norm, against autograd through the oracle's einsum in float64 and
    against the route through the 13-product function."""
    tp = importlib.import_module("learned-dynamics_amd.tensor_products")
    il, ir, io = lro
    g = torch.Generator().manual_seed(40 + 9 * il + 3 * ir + io)
    x_l = torch.randn(5, 6, 24, *([3] * il), generator=g)
    x_r = torch.randn(5, 6, 24, *([3] * ir), generator=g)
    cot = torch.randn(5, 6, 24, *([3] * io), generator=g)
    ld, rd = x_l.double().requires_grad_(), x_r.double().requires_grad_()
    ref = torch.autograd.grad((OP.tensor_prod_bare(il, ir, io, ld, rd) * cot.double()).sum(), [ld, rd], create_graph=True)
    ref2 = torch.autograd.grad(sum((r ** 2).sum() for r in ref), [ld, rd])
    outs = []
    for route in (tp.TensorProdBare(il, ir, io), lambda a, b: tp._prod_with_grad((il, ir, io), a, b)):
        lg, rg = x_l.cuda().requires_grad_(), x_r.cuda().requires_grad_()
        y = route(lg, rg)
        got = torch.autograd.grad((y * cot.cuda()).sum(), [lg, rg], create_graph=True)
        got2 = torch.autograd.grad(sum((t ** 2).sum() for t in got), [lg, rg])
        outs.append([y, *got, *got2])
        for a, r in zip(list(got) + list(got2), list(ref) + list(ref2)):
            torch.testing.assert_close(a.detach().cpu().double(), r.detach(), rtol=1e-5, atol=2e-6 * float(r.abs().max()) + 1e-9)
    for a, b in zip(*outs):
        torch.testing.assert_close(a, b, rtol=1e-5, atol=2e-6 * float(b.abs().max()) + 1e-9)


@pytest.mark.parametrize("E,n", [(1000, 128), (257, 4), (3001, 32), (130, 256)])
def test_painn_combine_against_plain_arithmetic(pkg, E, n):
    """The fused elementwise middle of the PaiNN message (archs/meanflow_painn8.py:91-100: the gathers by destination
    and the sums over the edges of a source node included) and its fused gradient against the same lines in float64
    tensor arithmetic; and the gradient of a gradient (which takes the plain arithmetic path) against float64 as
    well."""
    diff = importlib.import_module("learned-dynamics_amd.differentiable")
    gl = importlib.import_module("learned-dynamics_amd.graph_layers")
    g = torch.Generator().manual_seed(E + n)
    N = max(3, E // 7)
    src = torch.sort(torch.randint(0, N, (E,), generator=g)).values
    dst = torch.randint(0, N, (E,), generator=g)
    graph = gl.Graph(src.cuda(), dst.cuda(), None, 1, N)
    shapes = [(E, 4 * n), (1, N, 4 * n), (1, N, n, 3), (E, 3)]
    cpu = [torch.randn(*s, generator=g, dtype=F64).requires_grad_() for s in shapes]
    gpu = [t.detach().float().cuda().requires_grad_() for t in cpu]

    m_ref, a_ref = diff._painn_combine_plain(cpu[0], cpu[1][0, dst], cpu[2][0, dst], cpu[3])
    ref = (torch.zeros(N, n, 3, dtype=F64).index_add(0, src, m_ref)[None],
           torch.zeros(N, n, dtype=F64).index_add(0, src, a_ref)[None])
    got = diff.painn_combine(graph, *gpu)
    assert got[0].grad_fn is not None
    _close(got[0], ref[0], "sums of m")
    _close(got[1], ref[1], "sums of a")
    wm, wa = torch.randn(1, N, n, 3, generator=g, dtype=F64), torch.randn(1, N, n, generator=g, dtype=F64)

    loss_ref = (ref[0] * wm).sum() + (ref[1] * wa).sum()
    loss_got = (got[0] * wm.float().cuda()).sum() + (got[1] * wa.float().cuda()).sum()
    g_ref = torch.autograd.grad(loss_ref, cpu, create_graph=True)
    g_fused = torch.autograd.grad(loss_got, gpu, retain_graph=True)               # the fused gradient kernel
    g_got = torch.autograd.grad(loss_got, gpu, create_graph=True)                 # recorded: plain arithmetic
    for a, b, c, name in zip(g_fused, g_got, g_ref, ("dist", "actv", "v", "direction")):
        _close(a, c, f"fused gradient of {name}")
        _close(b, c, f"recorded gradient of {name}")
    # second order: gradient of |gradient|^2
    s_ref = sum((t ** 2).sum() for t in g_ref)
    s_got = sum((t ** 2).sum() for t in g_got)
    for a, c, name in zip(torch.autograd.grad(s_got, gpu), torch.autograd.grad(s_ref, cpu), ("dist", "actv", "v", "direction")):
        _close(a, c, f"second-order gradient of {name}", tol=1e-4)


@pytest.mark.parametrize("rows,cols,E", [(512, 512, 9000), (64, 16, 700), (2048, 128, 3000), (8, 1024, 50)])
def test_table_interpolation_kernels_against_float64(pkg, ops, rows, cols, E):
    """Interpolating a periodic grid at the edge lengths, and the adjoint (gradients for the grid and the lengths),
    against the same 4-point Lagrange formula in float64 tensor arithmetic; empty grid rows, lengths beyond one
    period, and the same bits on a second run."""
    diff = importlib.import_module("learned-dynamics_amd.differentiable")
    g = torch.Generator().manual_seed(rows + cols)
    period = 8.0        # a power of two: d * rows / period is exact in float32, so both sides interpolate at the same t
    table = torch.randn(rows, cols, generator=g, dtype=F64).requires_grad_()
    d = (torch.rand(E, generator=g, dtype=F64) * 0.5 * period)          # (the upper half of the grid stays empty)
    d[:5] += period                                                       # wrapped
    d = d.float().double().requires_grad_()
    w = torch.randn(E, cols, generator=g, dtype=F64)
    ref = diff._table_interp_plain(table, d, period)
    ref_t, ref_d = torch.autograd.grad((ref * w).sum(), (table, d))
    tab32, d32, w32 = table.detach().float().cuda(), d.detach().float().cuda(), w.float().cuda()
    out = ops.painn_table_interp_fwd(tab32, d32, period)
    _close(out, ref, "interpolated rows")
    perm, bucket_ptr = ops.painn_table_sorted_edges(d32, rows, period)
    assert int(bucket_ptr[-1]) == E and sorted(perm.tolist()) == list(range(E))
    d_table, dd = ops.painn_table_interp_bwd(w32, tab32, d32, period, perm, bucket_ptr)
    _close(d_table, ref_t, "grid gradient", 2e-5)
    _close(dd, ref_d, "length gradient", 1e-4)
    again, _ = ops.painn_table_interp_bwd(w32, tab32, d32, period, perm, bucket_ptr, want_length_grad=False)
    assert torch.equal(again, d_table)

    # the autograd functions over these kernels, recorded: first derivatives again, and a second-order gradient
    # (derivative orders 1 and 2 of the interpolation weights) against float64
    tab_g, d_g = tab32.clone().requires_grad_(), d32.clone().requires_grad_()
    out_g = diff.table_interp(tab_g, d_g, period)
    g1 = torch.autograd.grad((out_g * w32).sum(), (tab_g, d_g), create_graph=True)
    _close(g1[0], ref_t, "recorded grid gradient", 2e-5)
    _close(g1[1], ref_d, "recorded length gradient", 1e-4)
    ref = diff._table_interp_plain(table, d, period)
    r1 = torch.autograd.grad((ref * w).sum(), (table, d), create_graph=True)
    v_t, v_d = torch.randn(rows, cols, generator=g, dtype=F64), torch.randn(E, generator=g, dtype=F64)
    s_ref = (r1[0] * v_t).sum() + (r1[1] * v_d).sum() + (r1[1] ** 2).sum()
    s_got = (g1[0] * v_t.float().cuda()).sum() + (g1[1] * v_d.float().cuda()).sum() + (g1[1] ** 2).sum()
    for a, c, name in zip(torch.autograd.grad(s_got, (tab_g, d_g)), torch.autograd.grad(s_ref, (table, d)),
                          ("grid", "lengths")):
        _close(a, c, f"second-order gradient for the {name}", 2e-4)


def test_painn_filter_from_its_grid(pkg):
    """The differentiable filter through the grid (Message.table_rows accepts 512 rows for these weights) against the
    filter MLP on every edge (archs/meanflow_painn8.py:92): values, gradients for the MLP's parameters, the recorded
    backward pass and a second-order gradient.  Edge vectors that require a gradient keep the MLP on every edge (the
    interpolant's derivative amplifies the rounding noise of the grid values); the grid functions' own length
    gradient is tested against float64 in test_table_interpolation_kernels_against_float64."""
    diff = importlib.import_module("learned-dynamics_amd.differentiable")
    painn = importlib.import_module("learned-dynamics_amd.painn")
    torch.manual_seed(0x947 + 12)
    msg = painn.Message(5.0, 32, n_rbf=16).cuda()
    g = torch.Generator().manual_seed(3)
    E = 6000
    u = torch.randn(E, 3, generator=g)
    r_ij = (u / u.norm(dim=-1, keepdim=True) * (0.4 + 4.6 * torch.rand(E, 1, generator=g))).cuda()
    w = torch.randn(E, 4 * msg.n, generator=g).cuda()
    params = list(msg.mlp_dist.parameters())
    assert msg.table_rows() == 512

    f_moving = diff.painn_filter(msg, r_ij.clone().requires_grad_())
    assert not type(f_moving.grad_fn).__name__.startswith("_TableInterp")
    f_grid = diff.painn_filter(msg, r_ij)
    assert type(f_grid.grad_fn).__name__.startswith("_TableInterp")
    msg.use_table = False
    try:
        f_edge = diff.painn_filter(msg, r_ij)
        g_edge = torch.autograd.grad((f_edge * w).sum(), params)
    finally:
        msg.use_table = True
    scale = float(f_edge.abs().max())
    assert float((f_grid - f_edge).abs().max()) <= 1e-5 * scale
    assert torch.equal(f_moving.detach(), f_edge.detach())
    g_grid = torch.autograd.grad((f_grid * w).sum(), params, retain_graph=True)
    g_rec = torch.autograd.grad((f_grid * w).sum(), params, create_graph=True)
    for a, b, c, p in zip(g_grid, g_rec, g_edge, params):
        s = float(c.abs().max())
        assert float((a - c).abs().max()) <= 2e-5 * s, (tuple(p.shape), float((a - c).abs().max()), s)
        assert float((b - a).abs().max()) <= 2e-5 * s
    second = torch.autograd.grad(sum((t ** 2).sum() for t in g_rec), params, allow_unused=True)
    assert all(t is None or bool(torch.isfinite(t).all()) for t in second)


@pytest.mark.parametrize("n, rows", [(32, 512), (128, 512), (8, 2048)])
def test_combine_gradient_with_the_filter_interpolated_inside(ops, n, rows):
    """mg_painn_combine_bwd_grid against mg_painn_table_interp_fwd followed by mg_painn_combine_bwd on a smooth grid
    (the two kernels may round the position inside a grid cell differently, by an ulp of length x rows / period: the
    compiler is free to contract the subtraction of the floor into the product), with outputs left out as well."""
    g = torch.Generator().manual_seed(0x947 + 43 + n)
    E, nodes, period = 3000, 200, 10.0
    phase = 2 * torch.pi * torch.arange(rows)[:, None] / rows
    table = (torch.sin(phase * torch.randint(1, 4, (1, 4 * n), generator=g) + torch.rand(1, 4 * n, generator=g))
             * torch.randn(1, 4 * n, generator=g)).cuda()
    d = (torch.rand(E, generator=g) * period * 0.999).cuda()
    actv, v = torch.randn(nodes, 4 * n, generator=g).cuda(), torch.randn(nodes, n, 3, generator=g).cuda()
    direction = torch.nn.functional.normalize(torch.randn(E, 3, generator=g), dim=-1).cuda()
    dm, da = torch.randn(nodes, n, 3, generator=g).cuda(), torch.randn(nodes, n, generator=g).cuda()
    node = torch.randint(0, nodes, (E,), generator=g).int().cuda()
    grad_row = torch.randint(0, nodes, (E,), generator=g).int().cuda()
    dist = ops.painn_table_interp_fwd(table, d, period, 0)
    for want in ((True, True, True, True), (True, False, True, False), (False, True, False, False)):
        ref = ops.painn_combine_bwd(dist, actv, v, direction, dm, da, node=node, grad_row=grad_row, want=want)
        got = ops.painn_combine_bwd_grid(table, period, d, actv, v, direction, dm, da, node, grad_row, want=want)
        for k in range(4):
            assert (got[k] is None) == (not want[k]) and (ref[k] is None) == (not want[k])
            if want[k]:
                _close(got[k], ref[k].double().cpu(), f"gradient {k} with outputs {want}", 2e-6)


@pytest.mark.parametrize("n, E, nodes", [(32, 3000, 200), (128, 5000, 64), (4, 700, 900), (256, 2500, 7), (64, 1, 300)])
def test_combine_gradient_summed_per_row_inside_the_kernel(ops, n, E, nodes):
    """mg_painn_combine_bwd_rows (the gradients of actv and v summed over the edges that read a row, inside the kernel)
    against mg_painn_combine_bwd followed by segment sums, with the filter stored and with the filter interpolated
    from its grid; rows that no edge reads; a subset of the outputs; and float64 for the sums."""
    g = torch.Generator().manual_seed(0x947 + 47 + n)
    rows, period = 512, 10.0
    phase = 2 * torch.pi * torch.arange(rows)[:, None] / rows
    table = (torch.sin(phase * torch.randint(1, 4, (1, 4 * n), generator=g) + torch.rand(1, 4 * n, generator=g))
             * torch.randn(1, 4 * n, generator=g)).cuda()
    d = (torch.rand(E, generator=g) * period * 0.999).cuda()
    actv, v = torch.randn(nodes, 4 * n, generator=g).cuda(), torch.randn(nodes, n, 3, generator=g).cuda()
    direction = torch.nn.functional.normalize(torch.randn(E, 3, generator=g), dim=-1).cuda()
    dm, da = torch.randn(nodes, n, 3, generator=g).cuda(), torch.randn(nodes, n, generator=g).cuda()
    node = torch.randint(0, nodes, (E,), generator=g).int().cuda()
    grad_row = torch.randint(0, nodes, (E,), generator=g).int().cuda()
    order = torch.sort(node.long(), stable=True).indices.int().contiguous()
    row_ptr = ops.segment_row_ptr(node[order.long()].contiguous(), nodes)
    dist = ops.painn_table_interp_fwd(table, d, period, 0)
    ref = ops.painn_combine_bwd(dist, actv, v, direction, dm, da, node=node, grad_row=grad_row)
    sums = [torch.zeros(nodes, *t.shape[1:], dtype=F64).index_add_(0, node.long().cpu(), t.double().cpu()) for t in ref[1:3]]
    for name, kw in (("stored filter", dict(dist=dist)), ("grid", dict(dist=None, table=table, period=period, d=d))):
        filt = kw.pop("dist")
        for want in ((True, True, True, True), (False, True, True, False), (True, False, True, False)):
            got = ops.painn_combine_bwd_rows(filt, actv, v, direction, dm, da, row_ptr, order, grad_row, want=want, **kw)
            for k in range(4):
                assert (got[k] is None) == (not want[k])
            if want[0]:
                _close(got[0], ref[0].double().cpu(), f"{name}: d_dist", 2e-6)
            if want[3]:
                _close(got[3], ref[3].double().cpu(), f"{name}: d_dir", 2e-6)
            if want[1]:
                _close(got[1], sums[0], f"{name}: d_actv per row", 4e-6)
            _close(got[2], sums[1], f"{name}: dv per row", 4e-6)
    # edges already sorted by the row they read: no order array
    node_sorted = node[order.long()].contiguous()
    pick = lambda t: t[order.long()].contiguous()
    got = ops.painn_combine_bwd_rows(pick(dist), actv, v, pick(direction), dm, da, row_ptr, None, pick(grad_row))
    _close(got[1], sums[0], "sorted edges: d_actv per row", 4e-6)
    _close(got[0], pick(ref[0]).double().cpu(), "sorted edges: d_dist", 2e-6)
    assert int(node_sorted[0]) <= int(node_sorted[-1])


@pytest.mark.parametrize("n, E, nodes, terms", [(32, 3000, 200, 15), (128, 4000, 50, 15), (4, 500, 700, 6), (256, 900, 5, 3)])
def test_combine_summed_per_source_row_inside_the_kernel(ops, n, E, nodes, terms):
    """mg_painn_combine_fwd_rows against mg_painn_combine_fwd followed by sums over the edges of a source node in
    float64 (edges sorted by source; rows without edges give zeros)."""
    g = torch.Generator().manual_seed(0x947 + 53 + n)
    src = torch.sort(torch.randint(0, nodes, (E,), generator=g)).values.int().cuda()
    row_ptr = ops.segment_row_ptr(src, nodes)
    dist, actv = torch.randn(E, 4 * n, generator=g).cuda(), torch.randn(nodes, 4 * n, generator=g).cuda()
    v = torch.randn(nodes, n, 3, generator=g).cuda()
    direction = torch.nn.functional.normalize(torch.randn(E, 3, generator=g), dim=-1).cuda()
    node = torch.randint(0, nodes, (E,), generator=g).int().cuda()
    m, a = ops.painn_combine_fwd(dist, actv, v, direction, node=node, terms=terms)
    ref_v = torch.zeros(nodes, n, 3, dtype=F64).index_add_(0, src.long().cpu(), m.double().cpu())
    ref_a = torch.zeros(nodes, n, dtype=F64).index_add_(0, src.long().cpu(), a.double().cpu())
    out_v, out_a = ops.painn_combine_fwd_rows(dist, actv, v, direction, node, row_ptr, nodes, terms=terms)
    _close(out_v, ref_v, "out_v", 4e-6)
    _close(out_a, ref_a, "out_a", 4e-6)


def test_painn_message_through_its_grid_in_one_forward_kernel(pkg):
    """Message under autograd with edge vectors that are not differentiated: the forward pass is the inference kernel
    on the grid (differentiable._PainnGridMessage) and the backward pass interpolates the filter again.  Values and
    every gradient against the unfused formulation (interpolated filter stored, painn_combine), the recorded backward
    pass and a second-order gradient likewise; the unfused formulation has its own tests against float64."""
    diff = importlib.import_module("learned-dynamics_amd.differentiable")
    painn = importlib.import_module("learned-dynamics_amd.painn")
    gl = importlib.import_module("learned-dynamics_amd.graph_layers")
    torch.manual_seed(0x947 + 41)
    n, N = 32, 400
    msg = painn.Message(5.0, n, n_rbf=16).cuda()
    g = torch.Generator().manual_seed(5)
    src, dst = _ring(N, 16, g)
    E = len(src)
    u = torch.randn(E, 3, generator=g)
    r_ij = (u / u.norm(dim=-1, keepdim=True) * (0.4 + 4.6 * torch.rand(E, 1, generator=g))).cuda()
    graph = gl.Graph(src.cuda(), dst.cuda(), None, 1, N)
    x_a = torch.randn(1, N, n, generator=g).cuda().requires_grad_()
    x_v = torch.randn(1, N, n, 3, generator=g).cuda().requires_grad_()
    c_a, c_v = torch.randn(1, N, n, generator=g).cuda(), torch.randn(1, N, n, 3, generator=g).cuda()
    params = list(msg.parameters())
    assert msg.table_rows() == 512 and E >= 4 * 512

    def unfused():
        dist = diff.painn_filter(msg, r_ij)
        out_v, out_a = diff.painn_combine(graph, dist, diff.mlp_silu(msg.mlp_actv, x_a), x_v,
                                          diff._unit_vectors(r_ij, msg.epsilon))
        return out_a, out_v

    ops = importlib.import_module("learned-dynamics_amd.ops")
    calls, kernels = [], (ops.painn_table_message, ops.painn_table_message_sliced)
    ops.painn_table_message = lambda *a, **k: (calls.append("caches"), kernels[0](*a, **k))[1]
    ops.painn_table_message_sliced = lambda *a, **k: (calls.append("lds"), kernels[1](*a, **k))[1]
    try:
        da, dv = msg(graph, x_a, x_v, r_ij)
    finally:
        ops.painn_table_message, ops.painn_table_message_sliced = kernels
    assert calls == ["lds"]                              # the forward pass was the inference kernel (grid in LDS)
    ra, rv = unfused()
    _close(da, ra.double().cpu(), "out_a"); _close(dv, rv.double().cpu(), "out_v")
    leaves = [x_a, x_v] + params
    loss = lambda a, v: (a * c_a).sum() + (v * c_v).sum()
    got = torch.autograd.grad(loss(da, dv), leaves, allow_unused=True)
    ref = torch.autograd.grad(loss(ra, rv), leaves, allow_unused=True)
    for k, (a, r) in enumerate(zip(got, ref)):
        assert (a is None) == (r is None), k
        if a is not None:
            _close(a, r.double().cpu(), f"gradient {k}", 3e-5)
    # the recorded backward pass and a gradient of its result
    da, dv = msg(graph, x_a, x_v, r_ij)
    ra, rv = unfused()
    g1 = torch.autograd.grad(loss(da, dv), [x_a, x_v], create_graph=True)
    r1 = torch.autograd.grad(loss(ra, rv), [x_a, x_v], create_graph=True)
    second = lambda gs: sum((t ** 2).sum() for t in gs)
    got2 = torch.autograd.grad(second(g1), leaves, allow_unused=True)
    ref2 = torch.autograd.grad(second(r1), leaves, allow_unused=True)
    for k, (a, r) in enumerate(zip(got2, ref2)):
        assert (a is None) == (r is None), k
        if a is not None:
            _close(a, r.double().cpu(), f"second-order gradient {k}", 1e-4)
    # inputs with a forward-mode tangent take the unfused formulation
    value, tangent = diff.jvp(lambda a, v: msg(graph, a, v, r_ij)[0], (x_a.detach(), x_v.detach()),
                              (torch.randn_like(x_a), torch.randn_like(x_v)))
    _close(value, ra.double().cpu(), "value in forward mode")
    assert bool(torch.isfinite(tangent).all())


def test_message_products_with_folded_gathers(pkg):
    """The 13 products of Messages with the node operands read through the destination index and the gradients of the
    summed products through the source index (chan = 256, the width the folded kernels take), against the plain
    formulation (filters, gather, products, sums) on the unfused kernels: the indexed forward bit for bit, the
    inference kernel as forward (filters from the 8 radial functions inside it) and the first gradients to fp32
    rounding of the sums, and the recorded backward pass."""
    diff = importlib.import_module("learned-dynamics_amd.differentiable")
    gl = importlib.import_module("learned-dynamics_amd.graph_layers")
    g = torch.Generator().manual_seed(21)
    N, E, C = 37, 500, 256
    src = torch.sort(torch.randint(0, N, (E,), generator=g)).values
    dst = torch.randint(0, N, (E,), generator=g)
    graph = gl.Graph(src.cuda(), dst.cuda(), None, 1, N)
    enc8 = torch.randn(E, 8, generator=g).cuda()
    W, b = (torch.randn(C, 8, generator=g) / 3).cuda(), torch.randn(C, generator=g).cuda()
    shapes = [(1, N, C), (1, N, C, 3), (1, N, C, 3, 3)]
    xs = [torch.randn(*s, generator=g).cuda().requires_grad_() for s in shapes]
    xs += [(enc8 @ W.t() + b).requires_grad_(), torch.randn(E, 3, generator=g).cuda().requires_grad_()]
    flat = [gl._flat_nodes(graph, t) for t in xs[:3]]

    ref = diff._message_products_plain(*flat, *xs[3:], graph.by_dst, graph.by_src)
    got = diff.message_products(graph, *xs)
    fused = diff.message_products(graph, *xs, enc_source=(enc8, W, b))
    assert type(got[0].grad_fn).__name__.startswith("_MessageProducts")
    for a, f, r in zip(got, fused, ref):
        assert torch.equal(a, r)
        assert float((f - r).abs().max()) <= 1e-5 * float(r.abs().max())
    ws = [torch.randn(*t.shape, generator=g).cuda() for t in ref]
    loss = lambda out: sum((o * w).sum() for o, w in zip(out, ws))
    g_ref = torch.autograd.grad(loss(ref), xs)
    g_got = torch.autograd.grad(loss(fused), xs, retain_graph=True)
    g_rec = torch.autograd.grad(loss(fused), xs, create_graph=True)
    for a, r_, c in zip(g_got, g_rec, g_ref):
        scale = float(c.abs().max())
        assert float((a - c).abs().max()) <= 1e-5 * scale
        assert float((r_ - c).abs().max()) <= 1e-5 * scale
    second = torch.autograd.grad(sum((t ** 2).sum() for t in g_rec), xs)
    assert all(bool(torch.isfinite(t).all()) for t in second)


@pytest.mark.parametrize("N,E,C", [(1, 1, 64), (5, 3, 192), (37, 500, 128), (9, 2000, 256), (700, 4096, 64)])
def test_gradients_of_the_rank012_message_products(pkg, ops, N, E, C):
    """ops.bee_message_bwd against the products of rank 0-2 differentiated in float64: one edge, one slice of 64 channels and
    several, a last workgroup that is not full, nodes without edges on either side, odd and even numbers of edges at a
    destination; each gradient alone gives what all together give.  Tolerance: the node gradients are sums over an edge's 63 and
    a destination's terms, those of rh over an edge's 63 terms and all channels: 2^-24 sqrt(terms) of the largest entry, with a factor 8."""
    gl = importlib.import_module("learned-dynamics_amd.graph_layers")
    g = torch.Generator().manual_seed(0x947 + E)
    src = torch.sort(torch.randint(0, N, (E,), generator=g)).values
    dst = torch.randint(0, max(1, N - 1), (E,), generator=g)
    rnd = lambda *shape: torch.randn(*shape, generator=g)
    graph = gl.Graph(src.cuda(), dst.cuda(), None, 1, N)
    left, enc, rh = [rnd(N, C, *([3] * k)) for k in range(3)], rnd(E, C), rnd(E, 3)
    dys = [rnd(N if k else E, C, *([3] * k)) for k in (0, 0, 0, 1, 1, 1, 1, 2, 2, 2, 2, 1, 2)]
    xs = [t.double().requires_grad_() for t in (*left, enc, rh)]
    phi_v = xs[3][..., None] * xs[4][:, None]
    phi_d = phi_v[..., None] * xs[4][:, None, None]
    prods = OP.bee(*[t[dst] for t in xs[:3]], xs[3], phi_v, phi_d)
    # (the gradient of an edge's product is the gradient of its source node's sum)
    total = sum((p * (d.double() if d.dim() == 2 else d.double()[src])).sum() for p, d in zip(prods, dys))
    ref = torch.autograd.grad(total, xs)
    args = ([t.cuda() for t in left], enc.cuda(), rh.cuda(), [t.cuda() for t in dys], graph.by_src, graph.by_dst)
    d_left, d_enc, d_rh = ops.bee_message_bwd(*args, True, True, True)
    for name, x, y, terms in zip(("l_0", "l_1", "l_2", "enc", "rh"), (*d_left, d_enc, d_rh), ref, (63 * E, 63 * E, 63 * E, 63, 63 * C)):
        err = float((x.cpu().double() - y).abs().max() / y.abs().max())
        assert err <= 8 * 2 ** -24 * terms ** 0.5, f"{name}: {err:.3g}"
    alone = ops.bee_message_bwd(*args, True, False, False)
    assert all(torch.equal(a, b) for a, b in zip(alone[0], d_left)) and alone[1] is None and alone[2] is None
    assert torch.equal(ops.bee_message_bwd(*args, False, True, False)[1], d_enc)
    assert torch.equal(ops.bee_message_bwd(*args, False, False, True)[2], d_rh)
    if ops.bee_indexed_supported(C):                                    # the same one edge at a time
        phi = ops.bee_edge_filters_fwd(enc.cuda(), rh.cuda())
        per_edge = ops.bee_bwd_indexed(0, enc.cuda(), *phi, None, args[3], graph.by_src.index, E)
        for x, y, z in zip(per_edge, d_left, ref):
            x = torch.zeros_like(z).index_add_(0, dst, x.cpu().double())
            assert float((x - y.cpu()).abs().max()) <= 8 * 2 ** -24 * (63 * E) ** 0.5 * float(z.abs().max())


@pytest.mark.parametrize("E,C", [(300, 256), (17, 40), (1000, 64), (5, 700)])
def test_edge_filters_against_broadcasting_arithmetic(pkg, E, C):
    """phi_v = enc (x) rh and phi_d = enc (x) rh (x) rh of Messages (archs/diffuser_atoms15.py:241-243) as one kernel:
    bit for bit the broadcasting products, and the adjoint kernel / the recorded backward pass against float64."""
    diff = importlib.import_module("learned-dynamics_amd.differentiable")
    g = torch.Generator().manual_seed(E + C)
    enc64, rh64 = torch.randn(E, C, generator=g, dtype=F64).requires_grad_(), torch.randn(E, 3, generator=g, dtype=F64).requires_grad_()
    enc, rh = enc64.detach().float().cuda().requires_grad_(), rh64.detach().float().cuda().requires_grad_()
    w_v, w_d = torch.randn(E, C, 3, generator=g, dtype=F64), torch.randn(E, C, 3, 3, generator=g, dtype=F64)
    got = diff._EdgeFilters.apply(enc, rh)
    same = diff._edge_filters_plain(enc.detach(), rh.detach())
    assert torch.equal(got[0], same[0]) and torch.equal(got[1], same[1])
    ref = diff._edge_filters_plain(enc64, rh64)
    loss_ref = (ref[0] * w_v).sum() + (ref[1] * w_d).sum()
    loss_got = (got[0] * w_v.float().cuda()).sum() + (got[1] * w_d.float().cuda()).sum()
    g_ref = torch.autograd.grad(loss_ref, (enc64, rh64))
    g_got = torch.autograd.grad(loss_got, (enc, rh), retain_graph=True)
    g_rec = torch.autograd.grad(loss_got, (enc, rh), create_graph=True)
    for a, b, c, name in zip(g_got, g_rec, g_ref, ("enc", "rh")):
        _close(a, c, f"gradient of {name}")
        _close(b, c, f"recorded gradient of {name}")
    assert all(bool(torch.isfinite(t).all()) for t in torch.autograd.grad(sum((t ** 2).sum() for t in g_rec), (enc, rh)))


def test_silu_family_against_float64_derivatives(pkg, ops):
    """SiLU and its first four derivatives (one kernel each) against autograd in float64 through F.silu, as values
    (ops.silu_order, with and without the fused factor) and through the closed autograd family: the plain backward
    pass and three recorded ones."""
    diff = importlib.import_module("learned-dynamics_amd.differentiable")
    g = torch.Generator().manual_seed(77)
    z64 = torch.cat([torch.linspace(-30, 30, 1203, dtype=F64), 4 * torch.randn(5000, generator=g, dtype=F64)]).requires_grad_()
    ders = [torch.nn.functional.silu(z64)]
    for _ in range(4):
        ders.append(torch.autograd.grad(ders[-1].sum(), z64, create_graph=True)[0])
    z = z64.detach().float().cuda()
    m = torch.randn(z.shape, generator=g).cuda()
    for k in range(5):
        _close(ops.silu_order(z, k), ders[k], f"SiLU derivative {k}", tol=2e-6)
        _close(ops.silu_order(z, k, mul=m), ders[k] * m.cpu().double(), f"SiLU derivative {k} times a factor", tol=2e-6)
    with pytest.raises(RuntimeError):
        ops.silu_order(z, 5)
    # through autograd: w . silu(z), its gradient without recording, and the chain of recorded gradients
    zg = z.clone().requires_grad_()
    w = torch.randn(z.shape, generator=g, dtype=F64)
    w32 = w.float().cuda()
    y = diff.silu(zg)
    _close(y, ders[0], "silu")
    _close(torch.autograd.grad((y * w32).sum(), zg, retain_graph=True)[0], ders[1] * w, "gradient")
    cur = (y * w32).sum()
    for k in range(1, 4):
        grad, = torch.autograd.grad(cur, zg, create_graph=True)
        _close(grad, ders[k] * w, f"recorded gradient {k}", tol=2e-5)
        cur = grad.sum()
    # an odd length takes the scalar tail
    _close(ops.silu_order(z[:1001].contiguous(), 2), ders[2][:1001], "tail", tol=2e-6)


def test_fused_training_functions_on_a_graph_without_edges(pkg):
    """No edges at all: the folded functions return zero sums and zero gradients for the node operands."""
    diff = importlib.import_module("learned-dynamics_amd.differentiable")
    gl = importlib.import_module("learned-dynamics_amd.graph_layers")
    N, n, C = 5, 8, 256
    empty = torch.empty(0, dtype=torch.long).cuda()
    graph = gl.Graph(empty, empty, None, 1, N)
    actv = torch.randn(1, N, 4 * n).cuda().requires_grad_()
    v = torch.randn(1, N, n, 3).cuda().requires_grad_()
    out_v, out_a = diff.painn_combine(graph, torch.empty(0, 4 * n).cuda(), actv, v, torch.empty(0, 3).cuda())
    assert tuple(out_v.shape) == (1, N, n, 3) and float(out_v.abs().max()) == 0.0 and float(out_a.abs().max()) == 0.0
    ga, gv = torch.autograd.grad(out_v.sum() + out_a.sum(), (actv, v))
    assert float(ga.abs().max()) == 0.0 and float(gv.abs().max()) == 0.0
    nodes = [torch.randn(1, N, C, *([3] * k)).cuda().requires_grad_() for k in range(3)]
    prods = diff.message_products(graph, *nodes, torch.empty(0, C).cuda(), torch.empty(0, 3).cuda())
    assert len(prods) == 13 and all(float(p.abs().sum()) == 0.0 for p in prods)
    grads = torch.autograd.grad(sum(p.sum() for p in prods), nodes, allow_unused=True)
    assert all(g is None or float(g.abs().max()) == 0.0 for g in grads)


@pytest.mark.parametrize("B,N,n,n_rbf,degree", [(1, 1, 4, 4, 1), (2, 65, 8, 12, 3), (3, 64, 32, 16, 5), (1, 700, 128, 128, 4)])
def test_painn_layers_of_values_and_tangents(pkg, B, N, n, n_rbf, degree):
    """Message and Update as the fused functions run them under differentiation: values, forward-mode tangents, the gradients
    of a function of both for every input and parameter, and (values alone) the gradients without tangents, against the
    oracle's layers in float64.  Sizes around the pieces of the kernels: one node, a node past a piece of 64, rows of one lane
    up to a wave, one and several pieces of the group norm's statistics, products of 4 and of 1024 gradient rows.  Tolerance: a gradient
    here is a chain of at most ten sums of up to 700 terms, 10 sqrt(700) 2^-24 = 1.6e-5 of the largest entry."""
    painn = importlib.import_module("learned-dynamics_amd.painn")
    gl = importlib.import_module("learned-dynamics_amd.graph_layers")
    diff = importlib.import_module("learned-dynamics_amd.differentiable")
    torch.manual_seed(0x947 + n)
    gen = torch.Generator().manual_seed(7 + N)
    r0 = 5.0
    rnd = lambda *shape: torch.randn(*shape, generator=gen)
    src = torch.arange(B * N).repeat_interleave(degree)
    if N > 1:
        src = src[src % N != 1]                                          # (a node without edges)
    dst = (src // N) * N + torch.randint(0, N, (len(src),), generator=gen)
    msg, upd = painn.Message(r0, n, n_rbf).cuda(), painn.Update(n).cuda()
    with torch.no_grad():
        upd.gn.gamma.normal_(); upd.gn.beta.normal_()
    graph = gl.Graph(src.cuda(), dst.cuda(), None, B, N)
    x = [rnd(B, N, n), rnd(B, N, n, 3), 2 * rnd(len(src), 3)]
    t = [rnd(*a.shape) for a in x]
    c = [rnd(B, N, n), rnd(B, N, n, 3), rnd(B, N, n), rnd(B, N, n, 3)]

    def layers(msg_f, upd_f):
        def f(xa, xv, r):
            da, dv = msg_f(xa, xv, r)
            return upd_f(xa + da, xv + dv)
        return f

    wd, wa, wu_mlp = _mlp_w(msg.mlp_dist), _mlp_w(msg.mlp_actv), _mlp_w(upd.mlp)
    copy = lambda p: p.detach().cpu().double().requires_grad_(True)
    wu = {"W_l": copy(upd.lin_l.W), "W_r": copy(upd.lin_r.W), "W_v": copy(upd.lin_v.W), "mlp": wu_mlp,
          "gn_gamma": copy(upd.gn.gamma), "gn_beta": copy(upd.gn.beta)}
    params_o = []
    for w in (wd, wa, wu_mlp):
        for k in ("W1", "b1", "W2", "b2", "W3", "b3"):
            params_o.append(w[k].requires_grad_(True))
    params_o += [wu[k] for k in ("W_l", "W_r", "W_v", "gn_gamma", "gn_beta")]
    params_d = [p for m in (msg.mlp_dist, msg.mlp_actv, upd.mlp) for k in (0, 2, 4) for p in (m.layers[k].weight, m.layers[k].bias)]
    params_d += [upd.lin_l.W, upd.lin_r.W, upd.lin_v.W, upd.gn.gamma, upd.gn.beta]
    f_d = layers(lambda xa, xv, r: msg(graph, xa, xv, r), upd)
    f_o = layers(lambda xa, xv, r: OL.painn_message(src, dst, B, N, xa, xv, r, wd, wa, r0, n, n_rbf),
                 lambda xa, xv: OL.painn_update(xa, xv, wu, n))
    x_d, x_o = [a.cuda().requires_grad_() for a in x], [a.double().requires_grad_() for a in x]
    t_d, t_o = tuple(a.cuda() for a in t), tuple(a.double() for a in t)
    value_d, tangent_d = diff.jvp(f_d, tuple(x_d), t_d)
    value_o, tangent_o = torch.autograd.functional.jvp(f_o, tuple(x_o), t_o, create_graph=True)
    for k, name in enumerate(("a", "v")):
        _close(value_d[k], value_o[k], f"value {name}", 1.6e-5)
        _close(tangent_d[k], tangent_o[k], f"tangent {name}", 1.6e-5)
    total = lambda vs, to: sum((v * to(w)).sum() for v, w in zip(vs, c))
    g_d = torch.autograd.grad(total((*value_d, *tangent_d), lambda w: w.cuda()), x_d + params_d)
    g_o = torch.autograd.grad(total((*value_o, *tangent_o), lambda w: w.double()), x_o + params_o)
    for k, (a, b) in enumerate(zip(g_d, g_o)):
        _close(a, b, f"gradient {k} through value and tangent", 1.6e-5)
    g_d = torch.autograd.grad(total(f_d(*x_d), lambda w: w.cuda()), x_d + params_d)
    g_o = torch.autograd.grad(total(f_o(*x_o), lambda w: w.double()), x_o + params_o)
    for k, (a, b) in enumerate(zip(g_d, g_o)):
        _close(a, b, f"gradient {k}", 1.6e-5)


@pytest.mark.parametrize("r_grad", [False, True])
def test_what_the_fused_painn_layers_keep_passes_the_saved_tensor_hooks(pkg, r_grad):
    """Message (its filter from the grid, or the MLP on every edge where the edge vectors are differentiated) and Update keep
    the rows of their hidden layers through save_for_backward: hooks such as save_on_cpu see them, a graph that has been
    backpropagated holds none of them, and the gradients are the same ones."""
    painn = importlib.import_module("learned-dynamics_amd.painn")
    gl = importlib.import_module("learned-dynamics_amd.graph_layers")
    torch.manual_seed(0x947)
    n, N, E = 32, 60, 2400 if r_grad else 9000
    src, dst = torch.sort(torch.randint(0, N, (E,))).values, torch.randint(0, N, (E,))
    graph = gl.Graph(src.cuda(), dst.cuda(), None, 1, N)
    msg, upd = painn.Message(5.0, n, 16).cuda(), painn.Update(n).cuda()
    x_a, x_v, r = torch.randn(1, N, n).cuda(), torch.randn(1, N, n, 3).cuda(), torch.randn(E, 3).cuda()
    leaves = [x_a.requires_grad_(), x_v.requires_grad_()] + ([r.requires_grad_()] if r_grad else [])
    leaves += list(msg.parameters()) + list(upd.parameters())

    def loss():
        da, dv = msg(graph, x_a, x_v, r)
        ya, yv = upd(x_a + da, x_v + dv)
        return (ya ** 2).sum() + (yv ** 2).sum()

    want = torch.autograd.grad(loss(), leaves)
    packed = []

    def pack(t):
        packed.append(tuple(t.shape))
        return t.detach().cpu()

    with torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t.cuda()):
        value = loss()
    got = torch.autograd.grad(value, leaves)
    for mlp, rows in ((msg.mlp_actv, N), (upd.mlp, N)) + (((msg.mlp_dist, E),) if r_grad else ()):
        assert packed.count((rows, mlp.layers[0].out_features)) >= 4, "two hidden layers, before and after the activation"
    for k, (a, b) in enumerate(zip(got, want)):
        torch.testing.assert_close(a, b, rtol=1e-5, atol=1e-5 * float(b.abs().max()), msg=f"gradient {k}")


@pytest.mark.parametrize("n,rows,N,E,seed", [(16, 4, 3, 40, 0), (32, 64, 50, 3000, 1), (128, 512, 700, 20000, 2), (256, 512, 33, 5, 3),
                                            (128, 512, 40, 500000, 4)])
def test_gradients_of_the_message_from_its_grid(pkg, ops, n, rows, N, E, seed):
    """painn_grid_message_bwd against the unfused formulation differentiated in float64: grids from 4 rows to what LDS holds, one
    slice of channels and sixteen, fewer edges than a step of a wave, rows without edges, several pieces per grid row.
    Tolerance: a gradient is a sum of at most E products rounded to 2^-24 each, 8 2^-24 sqrt(E) of the largest entry, and the
    fraction of an edge between grid rows carries rows 2^-24."""
    g = torch.Generator().manual_seed(0x947 + seed)
    period, eps = 10.0, 0.1
    src = torch.sort(torch.randint(0, N, (E,), generator=g)).values
    dst = torch.randint(0, max(1, N - 1), (E,), generator=g)
    u = torch.randn(E, 3, generator=g)
    r = (u / u.norm(dim=-1, keepdim=True) * (0.05 + 4.9 * torch.rand(E, 1, generator=g)))
    k = torch.arange(rows)[:, None] / rows * 2 * torch.pi
    table = torch.randn(1, 4 * n, generator=g) * torch.cos(k + torch.randn(1, 4 * n, generator=g))      # smooth along the grid
    actv, v = torch.randn(N, 4 * n, generator=g), torch.randn(N, n, 3, generator=g)
    g_v, g_a = torch.randn(N, n, 3, generator=g), torch.randn(N, n, generator=g)
    gl = importlib.import_module("learned-dynamics_amd.graph_layers")
    graph = gl.Graph(src.cuda(), dst.cuda(), None, 1, N)
    order, ordered = ops.sort_by_key(graph.dst32, N)
    assert torch.equal(order.cpu().long(), torch.sort(dst, stable=True).indices) and torch.equal(ordered.cpu().long(), torch.sort(dst).values)
    T, A, V = (t.double().requires_grad_() for t in (table, actv, v))
    rd = r.double()
    diff = importlib.import_module("learned-dynamics_amd.differentiable")
    f = diff._table_interp_plain(T, rd.norm(dim=-1), period)
    m, a = diff._painn_combine_plain(f, A[dst], V[dst], rd / torch.sqrt(eps + (rd ** 2).sum(-1, keepdim=True)))
    ref = torch.autograd.grad((m * g_v.double()[src]).sum() + (a * g_a.double()[src]).sum(), (T, A, V))
    perm = ops.painn_slice_permutation(n, "cuda")
    got = ops.painn_grid_message_bwd(table.cuda(), actv.cuda(), actv.cuda()[:, perm].contiguous(), v.cuda(), r.cuda(), g_v.cuda(),
                                     g_a.cuda(), graph.src32, graph.dst32, graph.by_dst.row_ptr, graph.by_dst.perm, None, period,
                                     eps, True, True, True)
    for name, x, y in zip(("grid", "actv", "v"), got, ref):
        err = float((x.cpu().double() - y).abs().max() / y.abs().max())
        assert err <= 2 ** -24 * (8 * E ** 0.5 + rows), f"{name}: {err:.3g}"


@pytest.mark.parametrize("E", [5, 40, 3000])
@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_gradient_of_the_grid_reads_only_nodes_that_have_edges(pkg, ops, E, bad):
    """A node without edges (padding) may hold anything, the first one too, whose rows stand in for the edges that a step of
    the kernel lacks: its gradients are zeros, the others bit for bit those with zeros there.  Grid rows
    with fewer edges than a step of a wave, with several steps, and without any."""
    gl = importlib.import_module("learned-dynamics_amd.graph_layers")
    gen = torch.Generator().manual_seed(0x947 + E)
    n, rows, N = 32, 64, 50
    src = torch.sort(torch.randint(1, N, (E,), generator=gen)).values
    dst = torch.randint(1, N, (E,), generator=gen)
    graph = gl.Graph(src.cuda(), dst.cuda(), None, 1, N)
    rnd = lambda *shape: torch.randn(*shape, generator=gen).cuda()
    table, actv, v, r, g_v, g_a = rnd(rows, 4 * n), rnd(N, 4 * n), rnd(N, n, 3), 2 * rnd(E, 3), rnd(N, n, 3), rnd(N, n)
    perm = ops.painn_slice_permutation(n, "cuda")

    def gradients(first):
        args = [t.clone() for t in (actv, v, g_v, g_a)]
        for t in args:
            t[0] = first
        a, x_v, gv, ga = args
        return ops.painn_grid_message_bwd(table, a, a[:, perm].contiguous(), x_v, r, gv, ga, graph.src32, graph.dst32,
                                          graph.by_dst.row_ptr, graph.by_dst.perm, None, 10.0, 0.1, True, True, True)

    got, want = gradients(bad), gradients(0.0)
    for a, b in zip(got, want):
        assert torch.equal(a, b) and bool(torch.isfinite(a).all())
    for a in got[1:]:
        assert float(a[0].abs().max()) == 0.0


def test_update_under_autograd_of_more_boxes_than_a_grid_dimension(pkg):
    """70 001 boxes of two nodes: values, tangents and gradients against the oracle in float64.  Tolerance: 1.6e-5 of the
    largest entry as for other sizes; parameters sum 140 002 rows and their tangents, 10 sqrt(280 004) 2^-24 = 3.2e-4."""
    painn = importlib.import_module("learned-dynamics_amd.painn")
    diff = importlib.import_module("learned-dynamics_amd.differentiable")
    torch.manual_seed(0x947)
    B, N, n = 70001, 2, 8
    upd = painn.Update(n).cuda()
    copy = lambda p: p.detach().cpu().double().requires_grad_(True)
    wu = {"W_l": copy(upd.lin_l.W), "W_r": copy(upd.lin_r.W), "W_v": copy(upd.lin_v.W), "mlp": _mlp_w(upd.mlp),
          "gn_gamma": copy(upd.gn.gamma), "gn_beta": copy(upd.gn.beta)}
    mlp = [wu["mlp"][k].requires_grad_(True) for k in ("W1", "b1", "W2", "b2", "W3", "b3")]
    params_o = [*mlp, *(wu[k] for k in ("W_l", "W_r", "W_v", "gn_gamma", "gn_beta"))]
    params_d = [p for k in (0, 2, 4) for p in (upd.mlp.layers[k].weight, upd.mlp.layers[k].bias)]
    params_d += [upd.lin_l.W, upd.lin_r.W, upd.lin_v.W, upd.gn.gamma, upd.gn.beta]
    x, t = ([torch.randn(B, N, n), torch.randn(B, N, n, 3)] for _ in range(2))
    c = [torch.randn(B, N, n), torch.randn(B, N, n, 3), torch.randn(B, N, n), torch.randn(B, N, n, 3)]
    x_d, x_o = [a.cuda().requires_grad_() for a in x], [a.double().requires_grad_() for a in x]
    value_d, tangent_d = diff.jvp(lambda a, v: upd(a, v), tuple(x_d), tuple(a.cuda() for a in t))
    value_o, tangent_o = torch.autograd.functional.jvp(lambda a, v: OL.painn_update(a, v, wu, n), tuple(x_o),
                                                       tuple(a.double() for a in t), create_graph=True)
    for k, name in enumerate(("a", "v")):
        _close(value_d[k], value_o[k], f"value {name}", 1.6e-5)
        _close(tangent_d[k], tangent_o[k], f"tangent {name}", 1.6e-5)
    g_d = torch.autograd.grad(sum((v * w.cuda()).sum() for v, w in zip((*value_d, *tangent_d), c)), x_d + params_d)
    g_o = torch.autograd.grad(sum((v * w.double()).sum() for v, w in zip((*value_o, *tangent_o), c)), x_o + params_o)
    for k, (a, b) in enumerate(zip(g_d, g_o)):
        _close(a, b, f"gradient {k}", 1.6e-5 if k < 2 else 3.2e-4)


@pytest.mark.parametrize("dual", [False, True])
def test_edge_encoding_with_epsilon_zero(pkg, dual):
    """Unit vectors without the offset under the root, for edges of positive length: values, tangents and gradients against the
    formulas in float64 (an entry is a sum of at most 12 products of sines and cosines of phases below 30: 40 2^-24)."""
    diff = importlib.import_module("learned-dynamics_amd.differentiable")
    gen = torch.Generator().manual_seed(0x947)
    E, n, rmax = 77, 12, 5.0
    r, r_t = torch.randn(E, 3, generator=gen), torch.randn(E, 3, generator=gen)
    xs = [r] + ([r_t] if dual else [])
    d, o = [t.cuda().requires_grad_() for t in xs], [t.double().requires_grad_() for t in xs]
    got = diff._EdgeEncode.apply(d[0], d[1] if dual else None, n, rmax, 0.0)[:-1]
    pieces = lambda x: (diff.radial_encode_painn(x, n, rmax), diff._unit_vectors(x, 0.0))
    if dual:
        values, tangents = torch.autograd.functional.jvp(pieces, o[0], o[1], create_graph=True)
        want = (values[0], tangents[0], values[1], tangents[1])
    else:
        want = pieces(o[0])
    weights = [torch.randn(*w.shape, generator=gen) for w in want]
    g_d = torch.autograd.grad(sum((a * w.cuda()).sum() for a, w in zip(got, weights)), d)
    g_o = torch.autograd.grad(sum((a * w.double()).sum() for a, w in zip(want, weights)), o)
    for a, b in zip((*got, *g_d), (*want, *g_o)):
        _close(a, b, "edge encoding", 40 * 2 ** -24)


@pytest.mark.parametrize("R", [100, 2500, 5000])
def test_bias_gradient_of_values_beside_an_infinite_tangent(pkg, R):
    """The bias of an MLP's last layer gets the sum of the value's gradient rows; the rows of the tangent's gradient lie behind
    them in the same array and do not count, whatever they hold (sums of R terms: 8 sqrt(R) 2^-24 of the largest entry)."""
    diff = importlib.import_module("learned-dynamics_amd.differentiable")
    painn = importlib.import_module("learned-dynamics_amd.painn")
    torch.manual_seed(0x947)
    mlp = painn.MLP(64, 64).cuda()
    params = diff._mlp_parameters(mlp)
    y, y_t = diff._MlpSilu.apply(torch.randn(R, 64, device="cuda"), torch.randn(R, 64, device="cuda"), None, *params)
    g, g_t = torch.randn_like(y), torch.randn_like(y)
    g_t[R // 2, 5], g_t[0, 7] = float("inf"), float("nan")
    got, = torch.autograd.grad((y, y_t), params[-1:], (g, g_t))
    want = g.double().sum(0)
    assert float((got.double() - want).abs().max() / want.abs().max()) <= 8 * R ** 0.5 * 2 ** -24


@pytest.mark.parametrize("N,E,extra", [(1, 7, 0), (255, 40, 0), (257, 3000, 13), (5000, 60000, 0), (70000, 9000, 300)])
def test_grid_gradient_with_the_edges_in_the_order_of_the_nodes(pkg, ops, N, E, extra):
    """Every edge once, source by source in any order of the nodes (nodes without edges, more nodes than one block of the scan,
    edges behind the last row): what reaches the grid is the sum as without an order, up to the order of its terms."""
    L = importlib.import_module("learned-dynamics_amd._lib")
    import ctypes
    gen = torch.Generator().manual_seed(0x947 + N)
    n, rows, period = 16, 64, 10.0
    src = torch.sort(torch.randint(0, N, (E,), generator=gen)).values.cuda().int()
    row_ptr = ops.segment_row_ptr(src, N)
    order = torch.randperm(N, generator=gen).cuda().int()
    total = E + extra
    r = 2 * torch.randn(total, 3, generator=gen).cuda()
    lib, p = L.load(), lambda t: ctypes.c_void_p(t.data_ptr())
    key, plain, edge = (torch.full((total,), -1, dtype=torch.int32, device="cuda") for _ in range(3))
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    size = ctypes.c_size_t(0)
    L.check(lib.mg_painn_grid_rows_by_node_workspace_bytes(N, ctypes.byref(size)))
    ws = torch.empty(size.value, dtype=torch.uint8, device="cuda")
    L.check(lib.mg_painn_grid_rows_by_node(p(r), total, p(row_ptr), p(order), N, rows, period, p(ws), p(key), p(edge), stream))
    L.check(lib.mg_painn_grid_rows(p(r), total, rows, period, p(plain), stream))
    degree = (row_ptr[1:] - row_ptr[:-1]).long()
    want = torch.cat([torch.repeat_interleave(row_ptr[:-1].long()[order.long()], degree[order.long()]) + _within(degree[order.long()]),
                      torch.arange(E, total, device="cuda")])
    assert torch.equal(edge.long(), want) and torch.equal(key, plain[want])
    if extra:
        return
    rnd = lambda *shape: torch.randn(*shape, generator=gen).cuda()
    table, actv, v, g_v, g_a = rnd(rows, 4 * n), rnd(N, 4 * n), rnd(N, n, 3), rnd(N, n, 3), rnd(N, n)
    dst = torch.randint(0, N, (E,), generator=gen).cuda().int()
    gl = importlib.import_module("learned-dynamics_amd.graph_layers")
    graph = gl.Graph(src, dst, None, 1, N)
    args = (table, actv, actv[:, ops.painn_slice_permutation(n, "cuda")].contiguous(), v, r, g_v, g_a, src, dst, graph.by_dst.row_ptr,
            graph.by_dst.perm)
    a = ops.painn_grid_message_bwd(*args, order, period, 0.1, True, True, True, src_row_ptr=row_ptr)
    b = ops.painn_grid_message_bwd(*args, None, period, 0.1, True, True, True)
    for x, y in zip(a, b):
        assert float((x - y).abs().max() / y.abs().max()) <= 2 ** -24 * 8 * E ** 0.5


def _within(counts):
    """0 .. c - 1 for every c in turn."""
    ends = counts.cumsum(0)
    return torch.arange(int(counts.sum()), device=counts.device) - torch.repeat_interleave(ends - counts, counts)


@pytest.mark.parametrize("chan, dims, N, E", [(256, (64, 32, 16), 37, 500), (256, (32, 5, 3), 300, 700), (192, (64, 32, 16), 70, 300)])
def test_rank012_layers_on_stacked_products(pkg, chan, dims, N, E):
    """Messages (from 256 channels) and SelfTensProds under autograd take the products of a rank side by side, component by
    component, and apply their output linears as one.  Against the route with one product and one linear at a time, which a module
    with a hook on one of them takes: values, first gradients, second gradients and forward mode.  Tolerance: both routes sum the
    same terms in another order, in fp32 or from pieces of 22 bits: 1e-5 of the largest entry as for the products above."""
    bee, gl, diff = (importlib.import_module(f"learned-dynamics_amd.{m}") for m in ("bee_layers", "graph_layers", "differentiable"))
    g = torch.Generator().manual_seed(chan + N)
    src = torch.sort(torch.randint(0, N, (E,), generator=g)).values
    graph = gl.Graph(src.cuda(), torch.randint(0, N, (E,), generator=g).cuda(), None, 1, N)
    torch.manual_seed(7)
    msg, prods = bee.Messages(6.0, *dims, chan).cuda(), bee.SelfTensProds(*dims, chan, groups=1).cuda()
    r_ij = (4 * torch.randn(E, 3, generator=g)).clamp(-3, 3).cuda()
    xs = [torch.randn(1, N, d, *([3] * k), generator=g).cuda().requires_grad_() for k, d in enumerate(dims)]
    ts = [torch.randn(x.shape, generator=g).cuda() for x in xs]
    ws = [torch.randn(x.shape, generator=g).cuda() for x in xs]

    def results(layer, module):
        f = lambda *x: layer(*x)
        ys = f(*xs)
        loss = sum((y * w).sum() for y, w in zip(ys, ws))
        inputs = xs + list(module.parameters())
        first = torch.autograd.grad(loss, inputs, retain_graph=True, allow_unused=True)
        recorded = torch.autograd.grad(loss, inputs, create_graph=True, allow_unused=True)
        second = torch.autograd.grad(sum((x * t).sum() for x, t in zip(recorded[:3], ts)), inputs, allow_unused=True)
        value, tangent = diff.jvp(f, tuple(x.detach() for x in xs), tuple(ts))
        return [*ys, *first, *recorded, *second, *value, *tangent]

    for layer, module in ((lambda a, v, d: msg(graph, r_ij, a, v, d), msg), (prods, prods)):
        got = results(layer, module)
        hook = module.Y_110.register_forward_hook(lambda *a: None)
        ref = results(layer, module)
        hook.remove()
        assert len(got) == len(ref)
        for k, (x, y) in enumerate(zip(got, ref)):
            assert (x is None) == (y is None), k
            if x is not None:
                assert x.shape == y.shape
                assert float((x - y).abs().max()) <= 1e-5 * max(float(y.abs().max()), 1e-3), (type(module).__name__, k)


def _by_rank(x, rank):
    return x if rank == 0 else x.reshape(-1, 3 ** rank, x.shape[1]).transpose(1, 2).reshape(-1, x.shape[1], *[3] * rank).contiguous()


@pytest.mark.parametrize("rank, C, O, N", [(0, 256, 64, 100), (0, 256, 256, 5000), (0, 192, 5, 4100), (1, 256, 64, 100), (1, 192, 64, 1500),
                                           (1, 256, 96, 11000), (2, 256, 16, 500), (2, 256, 64, 3700), (2, 24, 3, 600), (2, 512, 64, 500)])
def test_linears_side_by_side_of_any_magnitude(pkg, ops, rank, C, O, N):
    """Tensor linears whose operands lie side by side, each 1e-3 to 1e-8 as large as the first, forward and in the gradient of
    the operands, against float64 and against the linears one after the other.  Tolerance: pieces of 22 bits
    of the largest of a row (of a weight, of a gradient) leave 2^-22 of it per term, 2^-21 in a product of two, and the terms' errors
    are as independent as the terms: 2^-21 of the 2-norm; sums in fp32 in chains of K = C add 2^-24 sqrt(K)."""
    diff = importlib.import_module("learned-dynamics_amd.differentiable")
    g = torch.Generator().manual_seed(N)
    sizes = (1.0, 1e-3, 1e-8) if rank == 0 else (1.0, 1e-3, 1e-5, 1e-6, 1e-8)
    R, G = N * 3 ** rank, len(sizes)
    x = torch.cat([m * torch.randn(R, C, generator=g) for m in sizes], dim=1).cuda()
    W = [torch.randn(O, C, generator=g).cuda().requires_grad_() for _ in sizes]
    dy = torch.randn(R, O, generator=g).cuda()
    x.requires_grad_()
    y = diff._RowLinears.apply(rank, True, x, *W)
    dx, = torch.autograd.grad(y, [x], dy)
    tol = 2 ** -21 + 2 ** -24 * C ** 0.5
    rel = lambda a, b: float((a.double() - b).norm() / b.norm())
    x64, dy64 = x.detach().double(), dy.double()
    assert rel(y.detach(), sum(x_k @ w.detach().double().t() for x_k, w in zip(x64.split(C, 1), W))) <= tol
    assert rel(dx, dy64 @ torch.cat([w.detach().double() for w in W], dim=1)) <= tol
    for k in range(G):
        # and one linear by itself
        alone = diff._RowLinears.apply(rank, True, x.detach()[:, k * C:(k + 1) * C].contiguous(), W[k].detach())
        ref = diff.tensor_linear(rank, W[k].detach(), _by_rank(x.detach()[:, k * C:(k + 1) * C], rank), sequential=True)
        assert rel(alone, diff._component_rows(ref).double() if rank else ref.double()) <= 2 * tol
    for k in range(1, G):                                    # the larger ones without a weight
        few = [torch.zeros_like(w) if j < k else w.detach() for j, w in enumerate(W)]
        assert rel(diff._RowLinears.apply(rank, True, x.detach(), *few),
                   sum(x_j @ w.double().t() for x_j, w in zip(x64.split(C, 1), few))) <= tol, k


@pytest.mark.parametrize("rank, C, O, N, groups", [(0, 256, 64, 4096, 3), (0, 60, 8, 5000, 5), (0, 256, 64, 9000, 1), (1, 256, 64, 1500, 5),
                                                   (1, 192, 132, 3000, 5), (2, 256, 16, 3001, 5), (2, 20, 12, 500, 4), (1, 256, 64, 500, 5)])
def test_weight_gradients_side_by_side_of_any_magnitude(pkg, ops, rank, C, O, N, groups):
    """The gradient of each weight by itself where the operands of the linears are 1 to 1e-8 in size.  Tolerance: dy and each x_k in
    pieces of 22 bits of their own largest, M times their rms, leave an error of 2^-22 M rms / 2 per element at most, independent from
    element to element; sums in fp32 in runs of 256, 64 such runs at most on the way to the result, add 2^-24 (16 + 8)."""
    diff = importlib.import_module("learned-dynamics_amd.differentiable")
    g = torch.Generator().manual_seed(N + C)
    sizes = (1e-3, 1.0, 1e-5, 1e-6, 1e-8)[:groups]
    R = N * 3 ** rank
    x = torch.cat([m * torch.randn(R, C, generator=g) for m in sizes], dim=1).cuda()
    W = [torch.randn(O, C, generator=g).cuda().requires_grad_() for _ in sizes]
    dy = torch.randn(R, O, generator=g).cuda()
    y = diff._RowLinears.apply(rank, True, x, *W)
    dW = torch.autograd.grad(y, W, dy)
    spread = lambda t: float(t.abs().max() / t.double().pow(2).mean().sqrt())
    for k, (d, x_k) in enumerate(zip(dW, x.split(C, 1))):
        want = dy.double().t() @ x_k.double()
        tol = 2 ** -23 * (spread(dy) + spread(x_k)) + 2 ** -24 * 24
        assert float((d.double() - want).norm() / want.norm()) <= tol, k


@pytest.mark.parametrize("rank, C, O, N", [(1, 64, 256, 300), (1, 256, 64, 10922), (2, 256, 64, 3640), (2, 256, 16, 8000)])
def test_component_rows_below_the_line_stay_in_fp32(pkg, rank, C, O, N):
    """Linears on component rows keep fp32 operands below 32 768 rows and for fewer than 64 outputs, like the linears of
    tensors: an entry 2^-30 as large as its row's largest, whose weight is zero, keeps its 24 bits (pieces of fp16 would leave it 9)."""
    diff = importlib.import_module("learned-dynamics_amd.differentiable")
    g = torch.Generator().manual_seed(C)
    R = N * 3 ** rank
    x, W = 2.0 ** -30 * torch.randn(R, C, generator=g), torch.randn(O, C, generator=g)
    x[:, 0], W[:, 0] = 1.0, 0.0
    y = diff._RowLinears.apply(rank, True, x.cuda(), W.cuda()).double().cpu()
    want = x.double() @ W.double().t()
    assert float((y - want).norm() / want.norm()) <= 2 ** -24 * (2 + C ** 0.5)


@pytest.mark.parametrize("N,E,C", [(5, 3, 64), (37, 500, 192)])
def test_message_gradients_by_product_and_by_component(pkg, ops, N, E, C):
    """ops.bee_message_bwd, operands and products one by one and by channel, and ops.bee_message_grad, component-major and side
    by side: one kernel in two layouts, the same sums in the same order."""
    gl = importlib.import_module("learned-dynamics_amd.graph_layers")
    g = torch.Generator().manual_seed(E)
    rnd = lambda *shape: torch.randn(*shape, generator=g).cuda()
    src = torch.sort(torch.randint(0, N, (E,), generator=g)).values
    graph = gl.Graph(src.cuda(), torch.randint(0, N, (E,), generator=g).cuda(), None, 1, N)
    left, enc, rh = [rnd(N, C, *([3] * k)) for k in range(3)], rnd(E, C), rnd(E, 3)
    dys = [rnd(E if lab[2] == "0" else N, C, *([3] * int(lab[2]))) for lab in ops.BEE_ORDER]
    by_comp = [left[0]] + [t.flatten(2).transpose(1, 2).contiguous() for t in left[1:]]
    d_left, *rest = ops.bee_message_bwd(left, enc, rh, dys, graph.by_src, graph.by_dst, True, True, True)
    d_rows, *rest_rows = ops.bee_message_grad(by_comp, enc, rh, ops.stack_products(dys), graph.by_src, graph.by_dst, True, True, True)
    for a, b in zip(d_left, d_rows):
        assert torch.equal(a.flatten(2).transpose(1, 2) if a.dim() > 2 else a, b)
    assert all(torch.equal(a, b) for a, b in zip(rest, rest_rows))


@pytest.mark.parametrize("what", ["by product", "rows", "node products"])
def test_recorded_backward_without_any_gradient(pkg, what):
    """The functions of the rank-0/1/2 products behind one whose backward returns no gradient: autograd calls them with None for
    every result, and a recorded backward pass gives zeros, as the plain one does."""
    diff, gl = (importlib.import_module(f"learned-dynamics_amd.{m}") for m in ("differentiable", "graph_layers"))
    g = torch.Generator().manual_seed(3)
    N, E, C = 9, 20, 256
    src = torch.sort(torch.randint(0, N, (E,), generator=g)).values
    graph = gl.Graph(src.cuda(), torch.randint(0, N, (E,), generator=g).cuda(), None, 1, N)
    rnd = lambda *shape: torch.randn(*shape, generator=g).cuda().requires_grad_()
    rows = lambda: [rnd(N, C), rnd(N, 3, C), rnd(N, 9, C)]
    if what == "node products":
        leaves = rows() + rows()
        out = diff._NodeProducts.apply(*leaves)
    else:
        leaves = (rows() if what == "rows" else [rnd(N, C, *[3] * k) for k in range(3)]) + [rnd(E, C), rnd(E, 3)]
        out = diff._MessageProducts.apply(*leaves, graph.by_dst, graph.by_src, None, what == "by product")

    class Drop(torch.autograd.Function):
        @staticmethod
        def forward(ctx, *ts):
            return sum(t.sum() for t in ts)

        @staticmethod
        def backward(ctx, g):
            return (None,) * len(out)

    dropped = Drop.apply(*out)
    for recorded in (False, True):
        grads = torch.autograd.grad(dropped, leaves, retain_graph=True, create_graph=recorded)
        assert all(float(t.abs().max()) == 0.0 for t in grads)


@pytest.mark.parametrize("what", ["mlp", "linears of rank 0", "linears of rank 2"])
def test_tangent_of_an_incoming_gradient(pkg, what):
    """A gradient that carries a forward-mode tangent through the backward passes that are kernels: they are linear in it, so the
    tangent of the result is the gradient of the tangent (the same sums in another kernel: fp16 pieces leave 2^-21 per factor, four
    factors deep, against entries of order one)."""
    import torch.autograd.forward_ad as fwAD
    diff, bee = (importlib.import_module(f"learned-dynamics_amd.{m}") for m in ("differentiable", "bee_layers"))
    torch.manual_seed(5)
    if what == "mlp":
        x = torch.randn(600, 64, device="cuda", requires_grad=True)
        y = diff.mlp_leaky(bee.MLP(64).cuda().requires_grad_(False), x)
        assert "MlpLeaky" in type(y.grad_fn.next_functions[0][0]).__name__ + type(y.grad_fn).__name__
    else:
        rank = int(what[-1])
        x = torch.randn(100 * 3 ** rank, 5 * 64, device="cuda", requires_grad=True)
        y = diff._RowLinears.apply(rank, True, x, *(torch.randn(64, 64, device="cuda") / 8 for _ in range(5)))
    g, g_t = torch.randn_like(y), torch.randn_like(y)
    want, want_t = (torch.autograd.grad(y, x, t, retain_graph=True)[0] for t in (g, g_t))
    with fwAD.dual_level():
        dx, = torch.autograd.grad(y, x, fwAD.make_dual(g, g_t))
        dx, dx_t = fwAD.unpack_dual(dx)
    assert not dx.requires_grad
    for a, b in ((dx, want), (dx_t, want_t)):
        assert float((a - b).norm() / b.norm()) <= 4 * 2 ** -21


def test_tangent_through_the_gradient_of_node_products_is_refused(pkg):
    """Their derivative kernels have no rule for forward mode: an error, and not a gradient without its tangent."""
    import torch.autograd.forward_ad as fwAD
    diff = importlib.import_module("learned-dynamics_amd.differentiable")
    leaves = [torch.randn(9, *shape, device="cuda", requires_grad=True) for shape in 2 * [(64,), (3, 64), (9, 64)]]
    out = diff._NodeProducts.apply(*leaves)
    with fwAD.dual_level():
        dual = [fwAD.make_dual(torch.ones_like(o), torch.ones_like(o)) for o in out]
        with pytest.raises(RuntimeError, match="orward AD|forward mode"):
            torch.autograd.grad(out, leaves, dual)


@pytest.mark.parametrize("inds, chan, groups, batch, nodes", [(0, 256, 8, 4, 100), (1, 64, 8, 1, 1), (2, 16, 8, 3, 333), (0, 8, 8, 2, 65), (1, 300, 4, 5, 64), (2, 33, 1, 33, 7)])
def test_tensor_norm_and_its_adjoint_as_kernels(pkg, inds, chan, groups, batch, nodes):
    """Values and gradients against the formula in float64: sums in float64, a handful of float32 roundings a result.  The same through
    a recorded backward pass, in forward mode and under vmap, which take the formula; groups that a workgroup has a part of."""
    tp = importlib.import_module("learned-dynamics_amd.tensor_products")
    torch.manual_seed(chan + nodes)
    norm = tp.TensGroupNorm(inds, chan, groups).cuda()
    with torch.no_grad():
        norm.gamma.normal_()
    x = (torch.randn(batch, nodes, chan, *[3] * inds) * torch.rand(batch, 1, chan, *[1] * inds).exp2()).cuda().requires_grad_()
    dy = torch.randn_like(x)
    gd, xd = norm.gamma.detach().double().requires_grad_(), x.detach().double().requires_grad_()
    xg = xd.reshape(batch, nodes, groups, -1, 3 ** inds)
    ref = (xg / (xg.pow(2).sum(-1, keepdim=True).mean([1, 3], keepdim=True) + norm.epsilon).sqrt()).reshape(x.shape) * gd
    want = torch.autograd.grad(ref, (xd, gd), dy.double(), create_graph=True)
    y = norm(x)
    got = torch.autograd.grad(y, (x, norm.gamma), dy, retain_graph=True)
    for name, a, r in (("y", y, ref), ("dx", got[0], want[0]), ("dgamma", got[1], want[1])):
        assert a.shape == r.shape and float((a.double() - r).norm()) <= 4 * 2.0 ** -24 * float(r.norm()) + 1e-12, name
    # (a result per channel: its own sums, whose terms cancel)
    assert torch.equal(torch.autograd.grad(norm(x), x, dy)[0], got[0])
    recorded = torch.autograd.grad(norm(x), (x, norm.gamma), dy, create_graph=True)
    second, = torch.autograd.grad(recorded[0], x, dy)
    second_ref, = torch.autograd.grad(want[0], xd, dy.double())
    assert float((recorded[0].double() - want[0]).norm()) <= 1e-6 * float(want[0].norm())
    assert float((second.double() - second_ref).norm()) <= 1e-5 * float(second_ref.norm()) + 1e-9
    value, tangent = torch.func.jvp(norm, (x.detach(),), (dy,))
    assert float((value - y).norm()) <= 1e-6 * float(y.norm()) and torch.isfinite(tangent).all()
    many = torch.func.vmap(lambda t: norm(t[None])[0], randomness="error")(x.detach())
    assert float((many - y).norm()) <= 1e-6 * float(y.norm())
    strided = x.detach().transpose(0, 1).contiguous().transpose(0, 1).requires_grad_()
    assert torch.equal(torch.autograd.grad(norm(strided), strided, dy)[0], got[0])


@pytest.mark.parametrize("residual", [False, True])
@pytest.mark.parametrize("E,n,missing", [(1, 4, ()), (700, 128, ()), (701, 64, ("dist", "dir")), (90, 256, ("actv", "v"))])
def test_messages_with_tangents_two_or_four_channels_a_lane(pkg, E, n, missing, residual):
    """Message sums and their tangents and the gradients of both against the formula in float64: a handful of float32 roundings a term,
    in sums over the edges of a row.  Rows of no edge, of one, of many; tangents that are left out; the node's own row added to the
    sums, whose gradient the adjoint adds."""
    diff = importlib.import_module("learned-dynamics_amd.differentiable")
    gl = importlib.import_module("learned-dynamics_amd.graph_layers")
    g = torch.Generator().manual_seed(E + n)
    N = max(3, E // 9)
    src = torch.sort(torch.randint(0, N, (E,), generator=g)).values
    dst = torch.randint(0, max(1, N - 1), (E,), generator=g)
    graph = gl.Graph(src.cuda(), dst.cuda(), None, 1, N)
    shapes = dict(dist=(E, 4 * n), actv=(N, 4 * n), v=(N, n, 3), dir=(E, 3))
    pairs = {k: [torch.randn(s, generator=g, dtype=F64).float(), torch.randn(s, generator=g, dtype=F64).float()] for k, s in shapes.items()}
    if residual:
        pairs["x"] = [torch.randn(N, n, generator=g, dtype=F64).float(), torch.randn(N, n, generator=g, dtype=F64).float()]
    for k in missing:
        pairs[k][1] = None
    flat = [t for p in pairs.values() for t in p]
    cpu = [None if t is None else t.double().requires_grad_() for t in flat]
    gpu = [None if t is None else t.cuda().requires_grad_() for t in flat]

    def sums(dist, actv, v, direction, x=None):
        m, a = diff._painn_combine_plain(dist, actv[dst], v[dst], direction)
        first = (v, x) if residual else (torch.zeros(N, n, 3, dtype=F64), torch.zeros(N, n, dtype=F64))
        return first[0].index_add(0, src, m), first[1].index_add(0, src, a)

    values, tangents = tuple(cpu[0::2]), tuple(torch.zeros_like(c) if t is None else t for c, t in zip(cpu[0::2], cpu[1::2]))
    ref, ref_t = torch.autograd.functional.jvp(sums, values, tangents, create_graph=True)
    want = (*ref, *ref_t)
    got = diff._PainnCombineDual.apply(graph.by_dst, graph.by_src, *(gpu[8:] or (None, None)), *gpu[:8])
    weights = [torch.randn(w.shape, generator=g, dtype=F64).float() for w in want]
    live = [i for i, t in enumerate(gpu) if t is not None]
    g_want = torch.autograd.grad(sum((w * k.double()).sum() for w, k in zip(want, weights)), [cpu[i] for i in live])
    g_got = torch.autograd.grad(sum((o.reshape(k.shape) * k.cuda()).sum() for o, k in zip(got, weights)), [gpu[i] for i in live])
    for what, a, r in [("sums", a, r) for a, r in zip(got, want)] + [("gradients", a, r) for a, r in zip(g_got, g_want)]:
        err = float((a.detach().cpu().double().reshape(r.shape) - r.detach()).norm())
        assert err <= 8 * 2.0 ** -24 * float(r.detach().norm()) + 1e-12, (what, err, float(r.detach().norm()))


@pytest.mark.parametrize("count", [1, 64, 511, 513, 2 ** 17 + 1, 2 ** 18 + 1, 2 ** 19 + 1, 2 ** 20 + 7])
def test_sort_by_key_in_chunks_of_every_length(ops, count):
    """The stable order of keys of one, two and three digits, at counts around a chunk and past each change of its length."""
    g = torch.Generator().manual_seed(count)
    for limit in (1, 512, 513, 2 ** 18 + 3):
        keys = torch.randint(0, limit, (count,), generator=g, dtype=torch.int32)
        order, ordered = ops.sort_by_key(keys.cuda(), limit)
        want = torch.sort(keys, stable=True)
        assert torch.equal(order.cpu().long(), want.indices) and torch.equal(ordered.cpu(), want.values), limit


@pytest.mark.parametrize("count, sized_for", [(2 ** 17, 2 ** 17 + 1), (2 ** 18, 2 ** 18 + 1), (2 ** 19, 2 ** 19 + 1), (513, 100000)])
def test_sort_by_key_in_the_workspace_of_a_larger_count(ops, count, sized_for):
    """More chunks than the count that the workspace was sized for has: nothing behind it is written."""
    import ctypes
    L = importlib.import_module("learned-dynamics_amd._lib")
    lib, size = L.load(), ctypes.c_size_t(0)
    L.check(lib.mg_sort_by_key_workspace_bytes(sized_for, ctypes.byref(size)))
    keys = torch.randint(0, 2 ** 18, (count,), generator=torch.Generator().manual_seed(count), dtype=torch.int32)
    on_device, workspace = keys.cuda(), torch.full((size.value // 4 + 2 ** 18,), -7, dtype=torch.int32, device="cuda")
    order, ordered = torch.empty_like(on_device), torch.empty_like(on_device)
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    L.check(lib.mg_sort_by_key(p(on_device), count, 2 ** 18, p(workspace), p(order), p(ordered),
                               ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
    want = torch.sort(keys, stable=True)
    assert torch.equal(order.cpu().long(), want.indices) and torch.equal(ordered.cpu(), want.values)
    assert bool((workspace[size.value // 4:] == -7).all())


@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
def test_row_pointers_of_long_runs_of_empty_rows(ops, dtype):
    """Runs of rows without an edge, before, between and behind the rows that have one, in one wave of edges and across waves."""
    cases = [([], 5), ([0], 1), ([700], 1000), ([3] * 64 + [4], 5), ([0, 3, 4, 9, 1000, 1000, 1005, 5000], 9000),
             ([*range(0, 64 * 40, 40), *range(3000, 3200)], 3200), ([5] * 255 + [4000, 4000], 4001)]
    for rows, n in cases:
        index = torch.tensor(rows, dtype=dtype)
        want = torch.searchsorted(index, torch.arange(n + 1, dtype=dtype))
        assert torch.equal(ops.segment_row_ptr(index.cuda(), n).cpu().long(), want), (rows[:4], n)


@pytest.mark.parametrize("E,n", [(30000, 64), (600, 64), (600, 24)])
def test_layers_that_add_their_input(pkg, E, n):
    """Message and Update of training with residual=True against the same layers with the input added outside: filters from their
    grid, from the MLP on every edge, and in pieces (n no power of two); values, values with tangents, gradients, recorded gradients.
    The additions are the same ones: results to a rounding, gradients to the order in which two of their terms are added."""
    painn = importlib.import_module("learned-dynamics_amd.painn")
    gl = importlib.import_module("learned-dynamics_amd.graph_layers")
    diff = importlib.import_module("learned-dynamics_amd.differentiable")
    g = torch.Generator().manual_seed(E + n)
    torch.manual_seed(n)
    N = 300
    src = torch.sort(torch.randint(0, N, (E,), generator=g)).values
    dst = torch.randint(0, N, (E,), generator=g)
    graph = gl.Graph(src.cuda(), dst.cuda(), None, 1, N)
    message, update = painn.Message(5.0, n).cuda(), painn.Update(n).cuda()
    r = torch.randn(E, 3, generator=g).cuda()
    x_a, x_v, t_a, t_v = (torch.randn(*s, generator=g).cuda() for s in [(1, N, n), (1, N, n, 3)] * 2)
    x_a, x_v = x_a.requires_grad_(), x_v.requires_grad_()
    w = [torch.randn(1, N, n, generator=g).cuda(), torch.randn(1, N, n, 3, generator=g).cuda()]

    def outside(f):
        return lambda a, v: tuple(diff.add(x, d) for x, d in zip((a, v), f(a, v, False)))

    for layer in (lambda a, v, res: message(graph, a, v, r, residual=res), lambda a, v, res: update(a, v, residual=res)):
        inside = lambda a, v: layer(a, v, True)
        ways = []
        for f in (outside(layer), inside):
            out = f(x_a, x_v)
            first = torch.autograd.grad(out, (x_a, x_v), w, retain_graph=True)
            recorded = torch.autograd.grad(out, (x_a, x_v), w, create_graph=True)
            value, tangent = diff.jvp(f, (x_a, x_v), (t_a, t_v))
            both = torch.autograd.grad((*value, *tangent), (x_a, x_v), w + w)
            only_a = torch.autograd.grad(f(x_a, x_v)[0].sum(), (x_a, x_v), allow_unused=True)
            ways.append([*out, *first, *recorded, *value, *tangent, *both, *only_a])
        for k, (a, b) in enumerate(zip(*ways)):
            assert (a is None) == (b is None), k
            if a is not None:
                err, size = float((a.detach() - b.detach()).norm()), float(a.detach().norm())
                assert err <= 2e-6 * size, (k, err, size)


@pytest.mark.parametrize("residual", [False, True])
def test_message_with_tangents_on_the_weights_of_its_node_mlp(pkg, residual):
    """Forward mode over mlp_actv's weights alone, the inputs without tangents, on as many edges as the filter is read from its grid
    for: the derivative that the message with the filter MLP on every edge gives, not none."""
    painn = importlib.import_module("learned-dynamics_amd.painn")
    gl = importlib.import_module("learned-dynamics_amd.graph_layers")
    g = torch.Generator().manual_seed(0x947)
    torch.manual_seed(0x947)
    N, E, n = 300, 30000, 64
    src = torch.sort(torch.randint(0, N, (E,), generator=g)).values
    graph = gl.Graph(src.cuda(), torch.randint(0, N, (E,), generator=g).cuda(), None, 1, N)
    msg = painn.Message(5.0, n).cuda()
    assert 0 < msg.table_rows() <= E // 4
    r, x_a, x_v = (torch.randn(*s, generator=g).cuda() for s in ((E, 3), (1, N, n), (1, N, n, 3)))
    names = [f"mlp_actv.layers.{k}.{w}" for k in (0, 4) for w in ("weight", "bias")]
    params = dict(msg.named_parameters())
    tangents = {k: torch.randn(params[k].shape, generator=g).cuda() for k in names}
    ways = []
    for msg.use_table in (True, False):
        with fwAD.dual_level():
            duals = {k: fwAD.make_dual(params[k], t) for k, t in tangents.items()}
            out = torch.func.functional_call(msg, duals, (graph, x_a, x_v, r), dict(residual=residual))
            ways.append([fwAD.unpack_dual(o) for o in out])
    for (p, t), (p_ref, t_ref) in zip(*ways):
        assert t is not None and t_ref is not None and float(t_ref.detach().norm()) > 0
        for a, b in ((p, p_ref), (t, t_ref)):
            assert float((a - b).detach().norm()) <= 1e-5 * float(b.detach().norm())


@pytest.mark.parametrize("batch, nodes, chan, inds", [(3, 1, 16, 1), (2, 4, 16, 2), (70, 20, 64, 0), (2, 253, 16, 1), (2, 257, 16, 1),
                                                      (1, 1030, 32, 0)])
def test_tensor_norm_gradient_in_a_workspace_of_the_boxes_size(ops, batch, nodes, chan, inds):
    """Chunks of a box by its nodes: gradients against float64, nothing written behind the workspace, which for small boxes is smaller
    than what x takes."""
    import ctypes
    L = importlib.import_module("learned-dynamics_amd._lib")
    diff = importlib.import_module("learned-dynamics_amd.differentiable")
    lib, groups, comps = L.load(), 4, 3 ** inds
    g = torch.Generator().manual_seed(nodes)
    x, dy = (torch.randn(batch, nodes, chan, *[3] * inds, generator=g).cuda() for _ in range(2))
    gamma = torch.randn(chan, *[1] * inds, generator=g).cuda()
    y, kept = ops.tens_norm_fwd(x, gamma, groups, 1e-5)
    size, any_nodes = ctypes.c_size_t(0), ctypes.c_size_t(0)
    L.check(lib.mg_tensor_norm_grad_workspace_bytes_of(batch, nodes, chan, groups, comps, ctypes.byref(size)))
    L.check(lib.mg_tensor_norm_grad_workspace_bytes(batch, chan, groups, comps, ctypes.byref(any_nodes)))
    assert size.value <= any_nodes.value and (nodes >= 253 or size.value <= 8 * batch * (chan * comps * (nodes + 7) // 4 + chan + groups))
    workspace = torch.full((size.value // 4 + 4096,), -7, dtype=torch.int32, device="cuda")
    dx, dgamma = torch.empty_like(x), torch.empty_like(gamma)
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    L.check(lib.mg_tensor_norm_grad(p(dy), p(x), batch, nodes, chan, groups, comps, 1e-5, p(gamma), p(kept), p(workspace), p(dx), p(dgamma),
                                    ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
    assert bool((workspace[size.value // 4:] == -7).all())
    leaves = [t.double().cpu().requires_grad_() for t in (x, gamma)]
    want = torch.autograd.grad(diff._tens_norm_plain(*leaves, groups, 1e-5), leaves, dy.double().cpu())
    for a, b in zip((dx, dgamma), want):                                 # (a handful of roundings to fp32 of sums in fp64)
        assert float((a.double().cpu() - b).norm()) <= 4 * 2.0 ** -24 * float(b.norm())


def test_tensor_norm_with_a_batch_of_gradients(pkg):
    """torch.autograd.grad(.., is_grads_batched=True), whose gradients have no memory that a kernel could read, against one at a time."""
    tp = importlib.import_module("learned-dynamics_amd.tensor_products")
    g = torch.Generator().manual_seed(7)
    norm = tp.TensGroupNorm(1, 16, 4).cuda()
    x = torch.randn(2, 50, 16, 3, generator=g).cuda().requires_grad_()
    dys = torch.randn(3, 2, 50, 16, 3, generator=g).cuda()
    y = norm(x)
    together = torch.autograd.grad(y, (x, norm.gamma), dys, is_grads_batched=True, retain_graph=True)
    for k, dy in enumerate(dys):
        for a, b in zip(together, torch.autograd.grad(y, (x, norm.gamma), dy, retain_graph=True)):
            assert float((a[k] - b).norm()) <= 1e-6 * float(b.norm())


@pytest.mark.parametrize("rows, chan", [(1, 32), (37, 96), (300, 256)])
def test_node_products_whose_rank_two_leads_nowhere(rows, chan):
    """Without a gradient of P2 the operands' gradients are those with zeros for it, to the bit; a gradient that is missing for another
    product is zeros as before."""
    diff, ops = (importlib.import_module(f"learned-dynamics_amd.{m}") for m in ("differentiable", "ops"))
    g = torch.Generator().manual_seed(rows)
    shapes = 2 * [(rows, chan), (rows, 3, chan), (rows, 9, chan)]
    leaves = [torch.randn(s, generator=g).cuda().requires_grad_() for s in shapes]
    P0, P1, P2 = diff._NodeProducts.apply(*leaves)
    d0, d1 = torch.randn(P0.shape, generator=g).cuda(), torch.randn(P1.shape, generator=g).cuda()
    for outs, dys in (((P0, P1), (d0, d1)), ((P1,), (d1,))):
        got = torch.autograd.grad(outs, leaves, dys, retain_graph=True)
        zeros = ops.bee_node_products_grad([t.detach() for t in leaves], [
            (d0 if len(dys) == 2 else torch.zeros_like(d0)).view(rows, 3, chan), d1.view(rows, 3, 5, chan), torch.zeros(rows, 9, 5, chan).cuda()])
        assert all(torch.equal(a, b) for a, b in zip(got, zeros))
