"""The layers as the reference writes them, out of differentiable pieces: what the modules run when a gradient is
asked for (training, or the Jacobian-vector product of the meanflow loss, archs/meanflow_painn8.py:274-282).

The fused inference kernels have no backward pass.  Every heavy operation here is an autograd function of this
package whose forward AND backward passes are HIP kernels (tensor_linear with its weight / input gradients, the 13
products with their two gradient kernels, gather and segment sum, which are each other's adjoints) and whose
backward is itself differentiable; the elementwise glue in between (activations, norms, the radial encodings, the
cross product, the periodic wrap) is plain torch arithmetic on the device, which autograd differentiates as it does
for the reference.  Results equal the fused path up to fp32 summation order (tests/test_gpu_autograd.py).

Forward mode: the functions that a forward pass runs also carry jvp rules, written with the same functions, so `jvp`
below returns a value and its derivative along a direction from one pass on dual tensors, both differentiable
afterwards; add / sub / mul are the arithmetic to use where only one operand can carry a tangent.
"""
import math

import torch
import torch.autograd.forward_ad as fwAD
import torch.nn.functional as F
import torch.nn.modules.module as _nn_module

from . import graph_layers as gl
from . import ops
from .codegen_tensor_products import Bee
from .tensor_products import TensLinear, tensor_linear


def has_tangent(t):
    """True for a tensor that carries a forward-mode tangent (inside jvp below)."""
    if t is None or getattr(fwAD, "_current_level", 0) < 0:       # (no dual level is open: nothing to unpack)
        return False
    return fwAD.unpack_dual(t).tangent is not None


def differentiated(t):
    """True when a derivative with respect to t is being taken, in either mode."""
    return t is not None and ((torch.is_grad_enabled() and t.requires_grad) or has_tangent(t))


def wants_grad(module, *tensors):
    """True when a gradient could flow to an input or a parameter (autograd is recording), or an input carries a
    forward-mode tangent: the cases the fused inference kernels do not serve."""
    if any(has_tangent(t) for t in tensors):
        return True
    if not torch.is_grad_enabled():
        return False
    if any(t is not None and t.requires_grad for t in tensors):
        return True
    return any(p.requires_grad for p in module.parameters())


def plain_call(module, cls):
    """True when calling the module runs cls.forward and nothing else: not a subclass or another module in its place, no
    hooks, no compiled call.  What the fused functions, which read a submodule's parameters and enqueue, may stand for."""
    own = module.__dict__
    return (type(module) is cls and "forward" not in own and own.get("_compiled_call_impl") is None
            and not (own["_forward_hooks"] or own["_forward_pre_hooks"] or own["_backward_hooks"] or own["_backward_pre_hooks"]
                     or _nn_module._global_forward_hooks or _nn_module._global_forward_pre_hooks
                     or _nn_module._global_backward_hooks or _nn_module._global_backward_pre_hooks))


def _one_sided(a, b):
    """(the operand with a tangent, the other, whether they were exchanged) when exactly one of a, b carries a
    forward-mode tangent, else None."""
    ta, tb = torch.is_tensor(a) and has_tangent(a), torch.is_tensor(b) and has_tangent(b)
    if ta == tb:
        return None
    return (b, a, True) if tb else (a, b, False)


def add(a, b):
    """a + b.  When only one operand carries a forward-mode tangent the tangent passes through unchanged: torch's own
    rule forms a symbolic zero for the other operand (a number or a parameter has none) and adds it through a slow
    path (Python meta kernels, 0.15 ms of host time per call).  Outside forward mode this is a + b."""
    one = _one_sided(a, b)
    if one is None:
        return a + b
    p, t = fwAD.unpack_dual(one[0])
    out = p + one[1]
    return fwAD.make_dual(out, t if t.shape == out.shape else t.expand(out.shape))


def sub(a, b):
    """a - b, in forward mode as add."""
    one = _one_sided(a, b)
    if one is None:
        return a - b
    p, t = fwAD.unpack_dual(one[0])
    out, t = (one[1] - p, -t) if one[2] else (p - one[1], t)
    return fwAD.make_dual(out, t if t.shape == out.shape else t.expand(out.shape))


def mul(a, b):
    """a * b, in forward mode as add: the tangent is the one operand's tangent times the other operand."""
    one = _one_sided(a, b)
    if one is None:
        return a * b
    p, t = fwAD.unpack_dual(one[0])
    return fwAD.make_dual(p * one[1], t * one[1])


def div(a, b):
    """a / b for a b without a tangent, in forward mode as add."""
    if not (torch.is_tensor(a) and has_tangent(a)) or (torch.is_tensor(b) and has_tangent(b)):
        return a / b
    p, t = fwAD.unpack_dual(a)
    return fwAD.make_dual(p / b, t / b)


def jvp(f, primals, tangents, create_graph=True, strict=False):
    """(f(*primals), the derivative of f at primals along tangents) in forward mode: every autograd function of this
    package that a forward pass runs has a jvp rule made of the package's differentiable functions, so the pair costs
    about two forward passes and both results can be differentiated afterwards (loss.backward()).
    torch.autograd.functional.jvp(f, primals, tangents, create_graph=True), which the reference's meanflow loss calls
    (archs/meanflow_painn8.py:274-282), gets the same derivative out of two nested backward passes, and the loss then
    differentiates all three; its first result is the same f(*primals) that the loss evaluates again as v_pred
    (archs/meanflow_painn8.py:291-292), so one call here stands for both.  The signature and the order of the results
    are functional.jvp's, so the name is the only change at a call site; create_graph and strict are accepted for that
    and change nothing (both results are always recorded when autograd is recording; without it, under no_grad, neither
    is).  primals and tangents may be single tensors."""
    if torch.is_tensor(primals):
        primals, tangents = (primals,), (tangents,)
    def unpack(out):
        value, tangent = fwAD.unpack_dual(out)
        return value, (tangent if tangent is not None else torch.zeros_like(value))

    with fwAD.dual_level():
        out = f(*(fwAD.make_dual(p, t) for p, t in zip(primals, tangents)))
        if isinstance(out, (tuple, list)):               # several results: (values, tangents), like functional.jvp
            pairs = [unpack(o) for o in out]
            return tuple(v for v, _ in pairs), tuple(t for _, t in pairs)
        return unpack(out)


def linear(lin, x, x_bound=None, want_bound=False, sequential=True):
    """nn.Linear through the tensor_linear kernels (weight and input gradients are kernels too).  x_bound / want_bound:
    row maxima handed from one layer to the next (tensor_products.tensor_linear).  sequential: see _TensorLinearFn."""
    lead = x.shape[:-1]
    out = tensor_linear(0, lin.weight, x.reshape(-1, x.shape[-1]).contiguous(), bias=lin.bias, x_bound=x_bound,
                        want_bound=want_bound, sequential=sequential)
    if want_bound:
        return out[0].reshape(*lead, -1), out[1]
    return out.reshape(*lead, -1)


class _SiluOrder(torch.autograd.Function):
    """SiLU^(order)(z).  Its derivative is the next member of the same family times the incoming gradient, so the
    family is closed under differentiation: every derivative order of an MLP costs one kernel per activation (plus one
    product while a higher derivative is still being recorded) instead of autograd's chain of elementwise formulas for
    the derivative of SiLU's derivative."""

    @staticmethod
    def forward(ctx, z, order):
        ctx.save_for_backward(z)
        ctx.save_for_forward(z)
        ctx.order = order
        return ops.silu_order(z.contiguous(), order)

    @staticmethod
    def jvp(ctx, z_t, _):
        z, = ctx.saved_tensors
        return z_t * _silu_order(z, ctx.order + 1)

    @staticmethod
    def backward(ctx, g):
        z, = ctx.saved_tensors
        if not torch.is_grad_enabled():
            return ops.silu_order(z.contiguous(), ctx.order + 1, mul=g.contiguous()), None
        return g * _silu_order(z, ctx.order + 1), None


def _silu_order(z, order):
    if order > ops.SILU_MAX_ORDER:
        raise RuntimeError(f"SiLU is differentiable {ops.SILU_MAX_ORDER} times here")
    return _SiluOrder.apply(z, order)


def silu(z):
    """nn.SiLU on a CUDA float32 tensor, differentiable up to ops.SILU_MAX_ORDER times."""
    if z.is_cuda and z.dtype == torch.float32:
        return _silu_order(z, 0)
    return F.silu(z)


def _unpack(x):
    """(value, forward-mode tangent or None) of a tensor."""
    if getattr(fwAD, "_current_level", 0) < 0:
        return x, None
    p, t = fwAD.unpack_dual(x)
    return p, t


def _dual(p, t):
    return p if t is None else fwAD.make_dual(p, t)


def _dense(t):
    return t if t is None else t.contiguous()


def _as_pair(f, x, x_t):
    """(value, tangent) of f, which maps one tensor to one tensor, from the plain tensors (x, x_t); x_t may be None."""
    if x_t is None:
        return (f(x),)
    if getattr(fwAD, "_current_level", 0) >= 0:
        return fwAD.unpack_dual(f(fwAD.make_dual(x, x_t)))
    with fwAD.dual_level():
        return tuple(fwAD.unpack_dual(f(fwAD.make_dual(x, x_t))))


def _recorded_gradients(f, inputs, needed, grads):
    """The gradients of f's outputs for `inputs`, recorded so that they can be differentiated again: what the fused
    functions below fall back on inside a recorded backward pass.  f is the same layer out of differentiable pieces."""
    with torch.enable_grad():
        leaves = [t if t is None or t.requires_grad or not need else t.detach().requires_grad_()
                  for t, need in zip(inputs, needed)]
        pairs = [(o, g) for o, g in zip(f(*leaves), grads) if g is not None and o is not None and o.requires_grad]
        wanted = [t for t, need in zip(leaves, needed) if need]
        found = iter(torch.autograd.grad([o for o, _ in pairs], wanted, [g for _, g in pairs], create_graph=True,
                                         allow_unused=True) if wanted and pairs else [None] * len(wanted))
    return tuple(next(found) if need else None for need in needed)


def _gradients_in_pieces(f, inputs, needed, grads):
    """_recorded_gradients if the backward pass is recorded or an incoming gradient or a saved tensor carries a forward-mode
    tangent, which the kernels of a backward pass know nothing of: the pieces have rules of their own for it, or refuse.  Else None."""
    if torch.is_grad_enabled():
        return _recorded_gradients(f, inputs, needed, grads)
    if any(has_tangent(t) for t in (*inputs, *grads)):
        pairs = [(None, None) if g is None else _unpack(g) for g in _recorded_gradients(f, inputs, needed, grads)]
        return tuple(p if p is None else _dual(p.detach(), t if t is None else t.detach()) for p, t in pairs)
    return None


class _MlpSilu(torch.autograd.Function):
    """painn.MLP on rows, values alone or values and tangents: one call into the C++ binding for each direction (three
    linear maps and two activations; three weight gradients, two or three input gradients, two activations).  The
    value and its tangent are two arguments and two results: forward mode is spelled out here, not left to jvp rules.
    bound: row maxima of |x| (and of the tangent's rows) if the caller holds them."""

    @staticmethod
    def forward(ctx, x, x_t, bound, *params):
        train = any(ctx.needs_input_grad)
        y, y_t, rows = ops.mlp_silu_fwd(x, x_t, bound, params[0::2], params[1::2], train)
        ctx.save_for_backward(x, x_t, *params, *(rows if train else ()))
        ctx.set_materialize_grads(False)
        return y if x_t is None else (y, y_t)

    @staticmethod
    def backward(ctx, g, g_t=None):
        x, x_t, *saved = ctx.saved_tensors
        params, rows = saved[:6], saved[6:]
        need = list(ctx.needs_input_grad)
        if g is None and g_t is None:
            return (None,) * len(need)
        if torch.is_grad_enabled():
            outs = _recorded_gradients(lambda x, x_t, *p: _as_pair(lambda z: _mlp_rows(p, z), x, x_t), (x, x_t, *params),
                                       need[:2] + need[3:], (g, g_t))
            return outs[:2] + (None,) + outs[2:]
        # (a result that nothing depends on leaves what only it depends on without a gradient, as separate functions would)
        if g is None:
            g, need[8] = torch.zeros_like(g_t), False                       # the last bias
        if x_t is not None and g_t is None:
            g_t, need[1] = torch.zeros_like(g), False
        g_x, g_xt, d_params = ops.mlp_silu_bwd(g.contiguous(), _dense(g_t), x, x_t, params[0::2], rows,
                                               need[0] or need[1], any(need[3:]))
        return (g_x if need[0] else None, g_xt if need[1] else None, None) \
            + tuple(d if nd else None for d, nd in zip(d_params, need[3:]))


def _mlp_rows(params, x):
    """Linear, SiLU, Linear, SiLU, Linear out of differentiable pieces.  |SiLU(z)| <= |z|: the row maxima that a layer's
    kernel emits for z bound the next layer's input."""
    W0, b0, W1, b1, W2, b2 = params
    lead, x = x.shape[:-1], x.reshape(-1, x.shape[-1])
    z, b = tensor_linear(0, W0, x, bias=b0, want_bound=True)
    z, b = tensor_linear(0, W1, silu(z), bias=b1, x_bound=b, want_bound=True)
    return tensor_linear(0, W2, silu(z), bias=b2, x_bound=b).reshape(*lead, -1)


def _mlp_parameters(mlp):
    L = mlp.layers
    return [p for k in (0, 2, 4) for p in (L[k].weight, L[k].bias)]


def _fused(params, *tensors):
    """Whether the fused functions take these: float32 on the device, rows of whole 16-byte pieces, no tangents on the
    parameters."""
    return (all(t is None or (t.is_cuda and t.dtype == torch.float32 and t.data_ptr() % 16 == 0 and t.numel() > 0) for t in tensors)
            and all(p is not None and p.is_cuda and p.dtype == torch.float32 and p.is_contiguous() and p.shape[0] % 4 == 0 for p in params)
            and not any(has_tangent(p) for p in params))


def mlp_silu(mlp, x):
    """painn.MLP: Linear, SiLU, Linear, SiLU, Linear (archs/meanflow_painn8.py:38-51)."""
    params = _mlp_parameters(mlp)
    p, t = _unpack(x)
    p, t = p.contiguous(), _dense(t)
    if not (_fused(params, p, t) and p.shape[-1] % 4 == 0):
        return _mlp_rows(params, x)
    out = _MlpSilu.apply(p, t, None, *params)
    return out if t is None else fwAD.make_dual(*out)


def _mlp_silu_pair(mlp, x):
    """mlp_silu's (value, tangent or None) for a caller that takes them apart: a dual tensor would copy the tangent."""
    params = _mlp_parameters(mlp)
    p, t = (_dense(z) for z in _unpack(x))
    if not (_fused(params, p, t) and p.shape[-1] % 4 == 0):
        return _unpack(_mlp_rows(params, x))
    out = _MlpSilu.apply(p, t, None, *params)
    return (out, None) if t is None else out


class _MlpLeaky(torch.autograd.Function):
    """bee_layers.MLP on rows: the layers as one kernel each way, the direct map added to their result.  params: weight and bias of
    the three layers, then the direct map's weight.  residual: of x + y, added where the kernels write y and the gradient of x."""

    @staticmethod
    def forward(ctx, residual, x, *params):
        ctx.residual = residual
        y, rows = ops.mlp_leaky_fwd(x, params[0:6:2] + params[6:], params[1:6:2], residual)
        ctx.save_for_backward(x, *params, *(rows if any(ctx.needs_input_grad) else ()))
        ctx.set_materialize_grads(False)
        return y

    @staticmethod
    def backward(ctx, g):
        x, *saved = ctx.saved_tensors
        params, rows = saved[:7], saved[7:]
        need, residual = ctx.needs_input_grad[1:], ctx.residual
        if g is None:
            return (None,) * (1 + len(need))
        pieces = _gradients_in_pieces(lambda x, *p: (x + _mlp_leaky_rows(p, x) if residual else _mlp_leaky_rows(p, x),), (x, *params),
                                      need, (g,))
        if pieces is not None:
            return (None, *pieces)
        g = g.contiguous()
        if g.data_ptr() % 16:
            g = g.clone()
        g_x, d_params = ops.mlp_leaky_bwd(g, x, params[0:6:2] + params[6:], rows, need[0], any(need[1:]), residual)
        return (None, g_x if need[0] else None) + tuple(d if nd else None for d, nd in zip(d_params or [None] * 7, need[1:]))


def _mlp_leaky_rows(params, x):
    """The same out of differentiable pieces."""
    W0, b0, W1, b1, W2, b2, Wd = params
    z, b = tensor_linear(0, W0, x, bias=b0, want_bound=True, sequential=True)
    z, b = tensor_linear(0, W1, F.leaky_relu(z, 0.1), bias=b1, x_bound=b, want_bound=True, sequential=True)
    return tensor_linear(0, Wd, x, sequential=True) + tensor_linear(0, W2, F.leaky_relu(z, 0.1), bias=b2, x_bound=b, sequential=True)


def mlp_leaky(mlp, x, residual=False):
    """bee_layers.MLP: lin_direct(x) + layers(x) with LeakyReLU(0.1) (archs/diffuser_atoms15.py:98-110); x + that with residual."""
    params = [*_mlp_parameters(mlp), mlp.lin_direct.weight]
    lead, rows = x.shape[:-1], x.reshape(-1, x.shape[-1]).contiguous()
    fused = (mlp.lin_direct.bias is None and not any(t is None or has_tangent(t) for t in (rows, *params))
             and ops.mlp_leaky_takes(rows, params[0:6:2] + params[6:], params[1:6:2]))
    if fused:
        inside = residual and params[4].shape[0] == rows.shape[1]
        y = _MlpLeaky.apply(inside, rows, *params).reshape(*lead, -1)
        return x + y if residual and not inside else y
    y = _mlp_leaky_rows(params, rows)
    if mlp.lin_direct.bias is not None:
        y = y + mlp.lin_direct.bias
    y = y.reshape(*lead, -1)
    return x + y if residual else y


def radial_encode_painn(r, n, rmax):
    """archs/meanflow_painn8.py:25-35"""
    hn = (n + 1) // 2
    coeffs = (math.pi / rmax) * (1 + torch.arange(0, hn, device=r.device) // 2)
    phase = mul(torch.linalg.vector_norm(r, dim=-1)[..., None], coeffs)
    return torch.cat([torch.cos(phase), torch.sin(phase[..., :(n - hn)])], dim=-1)


_JACOBI = {}


def _jacobi_matrix(device):
    """Coefficients of the shifted Jacobi polynomials P_i^(1,0)(2x - 1), i < 8 (managan/jacobi_radenc.py:8-22)."""
    key = str(device)
    if key not in _JACOBI:
        A = torch.zeros(8, 9, dtype=torch.float64)
        for n in range(8):
            for s in range(n + 1):
                w = math.comb(n + 1, n - s) * math.comb(n, s)
                for k in range(s + 1):
                    A[n, k + n - s] += w * math.comb(s, k) * (-1.0) ** (s - k)
        _JACOBI[key] = A.to(device)
    return _JACOBI[key]


def radial_encode_8(r, rmax):
    """managan/jacobi_radenc.py:24-37; the polynomials are evaluated in float64 (Horner) like the inference kernel:
    their monomial form in fp32 loses three digits."""
    z = div(torch.linalg.vector_norm(r, dim=-1), rmax)[..., None].double()
    A = _jacobi_matrix(r.device)
    acc = A[:, 8].expand(*z.shape[:-1], 8)
    for k in range(7, -1, -1):
        acc = add(mul(acc, z), A[:, k])
    return (acc * torch.relu(sub(1.0, z))).to(r.dtype)


def tens_sigmoid(inds, x):
    dims = tuple(-(1 + n) for n in range(inds))
    xx = (x ** 2).sum(dims, keepdim=True) if inds > 0 else x ** 2
    return x / torch.sqrt(add(xx, 1.0))


def scal_group_norm(gn, x, gamma=None, beta=None):
    """managan/layers_common.py:201-223"""
    gamma, beta = gn.gamma if gamma is None else gamma, gn.beta if beta is None else beta
    B, N, chan = x.shape
    xg = x.reshape(B, N, gn.groups, -1)
    sh = xg - xg.mean([1, 3], keepdim=True)
    var = (sh ** 2).mean([1, 3], keepdim=True)
    return add(mul((sh / torch.sqrt(add(var, gn.epsilon))).reshape(B, N, chan), gamma), beta)


def _tens_norm_plain(x, gamma, groups, eps):
    """managan/tensor_products.py:215-232"""
    B, N = x.shape[:2]
    xg = x.reshape(B, N, groups, -1, math.prod(x.shape[3:]))
    m2 = (xg ** 2).sum(-1, keepdim=True).mean([1, 3], keepdim=True)
    return mul((xg / torch.sqrt(add(m2, eps))).reshape(x.shape), gamma)


class _TensNorm(torch.autograd.Function):
    """TensGroupNorm: two passes each way and one between them, sums in float64."""

    @staticmethod
    def forward(ctx, x, gamma, groups, eps):
        y, sums = ops.tens_norm_fwd(x, gamma, groups, eps)
        ctx.save_for_backward(x, gamma, sums)
        ctx.groups, ctx.eps = groups, eps
        ctx.set_materialize_grads(False)
        return y

    @staticmethod
    def backward(ctx, dy):
        x, gamma, sums = ctx.saved_tensors
        need = ctx.needs_input_grad[:2]
        if dy is None:
            return None, None, None, None
        f = lambda x, g: (_tens_norm_plain(x, g, ctx.groups, ctx.eps),)
        if not torch._C._has_storage(dy):                                   # (a batch of gradients under vmap: is_grads_batched)
            return _recorded_gradients(f, (x, gamma), need, (dy,)) + (None, None)
        pieces = _gradients_in_pieces(f, (x, gamma), need, (dy,))
        if pieces is not None:
            return pieces + (None, None)
        dx, dgamma = ops.tens_norm_bwd(dy.contiguous(), x, gamma, sums, ctx.groups, ctx.eps)
        return dx if need[0] else None, dgamma if need[1] else None, None, None


def tens_group_norm(gn, x):
    """managan/tensor_products.py:215-232"""
    gamma = gn.gamma
    fused = (x.is_cuda and x.dtype == gamma.dtype == torch.float32 and gamma.is_cuda and gamma.is_contiguous() and x.numel() > 0
             and x.shape[0] <= 65535 and tuple(x.shape[2:]) == (gn.chan, *[3] * gn.inds)
             and not has_tangent(x) and not has_tangent(gamma) and torch._C._functorch.peek_interpreter_stack() is None)
    return _TensNorm.apply(x.contiguous(), gamma, gn.groups, gn.epsilon) if fused else _tens_norm_plain(x, gamma, gn.groups, gn.epsilon)


def edge_vectors(graph, pos, box):
    """boxwrap(box, pos[dst] - pos[src]) with a gradient for pos (archs/meanflow_painn8.py:167-172)."""
    pos_src, pos_dst = gl.edges_read(graph, pos)
    tbox = torch.tensor(box, device=pos.device, dtype=pos.dtype)
    delta = pos_dst - pos_src
    if has_tangent(delta):
        # the wrap shifts by a locally constant multiple of the box: its Jacobian is the identity
        p, t = fwAD.unpack_dual(delta)
        return fwAD.make_dual(gl.boxwrap(tbox, p), t)
    return gl.boxwrap(tbox, delta)


def _painn_combine_plain(dist, actv, v, direction):
    """archs/meanflow_painn8.py:94-100, as the reference writes it"""
    n = v.size(1)
    prod = dist * actv
    cross = torch.linalg.cross(v, direction[:, None].expand_as(v))
    m = v * prod[..., :n, None] + cross * prod[..., n:2 * n, None] + direction[:, None] * prod[..., 2 * n:3 * n, None]
    return m, prod[..., 3 * n:]


_TERMS_ALL, _TERMS_V, _TERMS_DIR = 15, 3, 6      # the four terms of the message; those that contain v; those with the direction


def _sum_opt(parts):
    parts = [p for p in parts if p is not None]
    return sum(parts[1:], parts[0]) if parts else None


class _PainnCombine(torch.autograd.Function):
    """Lines 94-100 of archs/meanflow_painn8.py as one kernel with the graph operations on either side folded in:
    actv and v come per node and the kernel reads the destination's row (by_dst); m and a are summed over the edges
    of their source node (by_src).  Returns (out_v (nodes, n, 3), out_a (nodes, n)).  `terms` masks the four terms of
    the message.  The pairing sum (G_v . out_v + G_a . out_a) is linear in (G_v, G_a), in dist and in actv, and in v
    and the direction once restricted to the terms that contain them: every derivative of this function and of
    _PainnCombineGrad is one of the two with a cotangent in one argument's place and that argument's mask, so the
    pair is closed under differentiation and recorded backward passes run on the same two kernels."""

    @staticmethod
    def forward(ctx, dist, actv_node, v_node, direction, by_dst, by_src, terms):
        ctx.by_dst, ctx.by_src, ctx.terms = by_dst, by_src, terms
        ctx.save_for_backward(dist, actv_node, v_node, direction)
        ctx.save_for_forward(dist, actv_node, v_node, direction)
        ctx.set_materialize_grads(False)
        # (the edges are sorted by their source node: its CSR is the row pointer of the sums)
        return ops.painn_combine_fwd_rows(dist.contiguous(), actv_node.contiguous(), v_node.contiguous(),
                                          direction.contiguous(), by_dst.index, by_src.row_ptr, by_src.n_rows, terms=terms)

    @staticmethod
    def jvp(ctx, dist_t, actv_t, v_t, dir_t, *_):
        """The function is linear in each argument within the terms that contain it: the tangent is the sum of the
        function itself with one argument's tangent in that argument's place."""
        dist, actv, v, direction = ctx.saved_tensors
        idx, t = (ctx.by_dst, ctx.by_src), ctx.terms
        slots = [(dist_t, (dist_t, actv, v, direction), t), (actv_t, (dist, actv_t, v, direction), t),
                 (v_t, (dist, actv, v_t, direction), t & _TERMS_V), (dir_t, (dist, actv, v, dir_t), t & _TERMS_DIR)]
        pairs = [_PainnCombine.apply(*args, *idx, mask) for x_t, args, mask in slots if x_t is not None and mask]
        return _sum_opt([p[0] for p in pairs]), _sum_opt([p[1] for p in pairs])

    @staticmethod
    def backward(ctx, g_v, g_a):
        if g_v is None or g_a is None:
            ref_v, ref_a = ctx.saved_tensors[2], ctx.saved_tensors[1]
            nodes = ctx.by_src.n_rows
            g_v = g_v if g_v is not None else ref_v.new_zeros(nodes, ref_v.size(1), 3)
            g_a = g_a if g_a is not None else ref_a.new_zeros(nodes, ref_v.size(1))
        want = tuple(ctx.needs_input_grad[:4])
        grads = _PainnCombineGrad.apply(g_v, g_a, *ctx.saved_tensors, ctx.by_dst, ctx.by_src, ctx.terms, want)
        return tuple(g if need else None for g, need in zip(grads, want)) + (None, None, None)


class _PainnCombineGrad(torch.autograd.Function):
    """(g_v, g_a, dist, actv, v, direction) -> the gradients of _PainnCombine's four inputs: d_dist (edges, 4n),
    d_actv (nodes, 4n), dv (nodes, n, 3), d_direction (edges, 3): one kernel; the gradient rows of an edge's source
    node are read through the source index, the gradients of actv and v are summed over the edges of a destination
    inside it (mg_painn_combine_bwd_rows)."""

    @staticmethod
    def forward(ctx, g_v, g_a, dist, actv_node, v_node, direction, by_dst, by_src, terms, want):
        """want: which of the four gradients to compute (the others come back as empty tensors)."""
        ctx.by_dst, ctx.by_src, ctx.terms, ctx.want = by_dst, by_src, terms, want
        ctx.save_for_backward(g_v, g_a, dist, actv_node, v_node, direction)
        args = (dist.contiguous(), actv_node.contiguous(), v_node.contiguous(), direction.contiguous(), g_v.contiguous(),
                g_a.contiguous())
        if want[1] or want[2]:
            # the gradients of actv and v are summed over the edges of a destination inside the kernel
            d_dist, d_actv, dv, d_dir = ops.painn_combine_bwd_rows(*args, by_dst.row_ptr, by_dst.perm, by_src.index,
                                                                   terms=terms, want=want)
        else:
            d_dist, d_actv, dv, d_dir = ops.painn_combine_bwd(*args, node=by_dst.index, grad_row=by_src.index,
                                                              terms=terms, want=want)
        outs = [d_dist, d_actv, dv, d_dir]
        for k in range(4):
            if outs[k] is None:
                outs[k] = dist.new_empty(0)
                ctx.mark_non_differentiable(outs[k])
        return tuple(outs)

    @staticmethod
    def backward(ctx, h_dist, h_actv, h_v, h_dir):
        g_v, g_a, dist, actv, v, direction = ctx.saved_tensors
        idx, t = (ctx.by_dst, ctx.by_src), ctx.terms
        need = ctx.needs_input_grad
        # one entry per cotangent: the four arguments with the cotangent in its own argument's place, and the mask
        slots = [(h_dist, (h_dist, actv, v, direction), t), (h_actv, (dist, h_actv, v, direction), t),
                 (h_v, (dist, actv, h_v, direction), t & _TERMS_V), (h_dir, (dist, actv, v, h_dir), t & _TERMS_DIR)]
        slots = [(k, args, mask) for k, (h, args, mask) in enumerate(slots) if h is not None and ctx.want[k]]
        out_g_v = out_g_a = None
        if need[0] or need[1]:
            pairs = [_PainnCombine.apply(*args, *idx, mask) for _, args, mask in slots]
            out_g_v, out_g_a = _sum_opt([p[0] for p in pairs]), _sum_opt([p[1] for p in pairs])
        grads = [[], [], [], []]
        for k, args, mask in slots:
            # (output k of such a call would be the derivative in the cotangent itself: not wanted)
            want = tuple(bool(need[2 + j]) and j != k for j in range(4))
            if any(want):
                outs = _PainnCombineGrad.apply(g_v, g_a, *args, *idx, mask, want)
                for j in range(4):
                    if want[j]:
                        grads[j].append(outs[j])
        return ((out_g_v, out_g_a) + tuple(_sum_opt(g) if nd else None for g, nd in zip(grads, need[2:6]))
                + (None, None, None, None))


class _PainnCombineDual(torch.autograd.Function):
    """_PainnCombine of values and tangents at once: (dist, dist_t, actv, actv_t, v, v_t, direction, direction_t) -> (out_v,
    out_a, out_v_t, out_a_t), any tangent None.  One kernel each way, where the rule of _PainnCombine.jvp makes one call
    for the values and one for each argument with a tangent, and as many in the backward pass.
    x, x_t: None, or the rows that out_a and its tangent are added to; v and v_t are then added to out_v and its tangent, and the
    adjoint's kernel adds both gradients of v."""

    @staticmethod
    def forward(ctx, by_dst, by_src, x, x_t, *args):
        ctx.by_dst, ctx.by_src, ctx.residual = by_dst, by_src, x is not None
        ctx.save_for_backward(*args)
        return ops.painn_combine_dual_fwd(args, by_dst.index, by_src.row_ptr, by_src.n_rows,
                                          (x, x_t, args[4], args[5]) if ctx.residual else ())

    @staticmethod
    def backward(ctx, *grads):
        args, need, residual = ctx.saved_tensors, ctx.needs_input_grad[4:], ctx.residual
        by_dst, by_src = ctx.by_dst, ctx.by_src
        past = tuple(g if nd else None for g, nd in zip((grads[1], grads[3]), ctx.needs_input_grad[2:4]))
        if torch.is_grad_enabled():
            return (None, None, *past) + _recorded_gradients(lambda *a: _combine_pairs(a, by_dst, by_src, residual), args, need, grads)
        outs = ops.painn_combine_dual_bwd(args, by_dst.row_ptr, by_dst.perm, [g.contiguous() for g in grads], by_src.index,
                                          by_src.n_rows, need, residual)
        return (None, None, *past) + tuple(o if nd else None for o, nd in zip(outs, need))


def _combine_pairs(args, by_dst, by_src, residual=False):
    """_PainnCombineDual out of calls of _PainnCombine (of the rows that results are added to, v and v_t alone)."""
    values, tangents = args[0::2], args[1::2]
    out_v, out_a = _PainnCombine.apply(*values, by_dst, by_src, _TERMS_ALL)
    pairs = [_PainnCombine.apply(*(t if j == k else v for j, v in enumerate(values)), by_dst, by_src, terms)
             for k, (t, terms) in enumerate(zip(tangents, (_TERMS_ALL, _TERMS_ALL, _TERMS_V, _TERMS_DIR))) if t is not None]
    out_vt, out_at = _sum_opt([p[0] for p in pairs]), _sum_opt([p[1] for p in pairs])
    if residual:
        out_v, out_vt = args[4] + out_v, out_vt if args[5] is None else args[5] + out_vt
    return out_v, out_a, out_vt, out_at


def painn_combine(graph, dist, actv_node, v_node, direction):
    """dist (E, 4n), direction (E, 3) per edge; actv_node (batch, nodes, 4n), v_node (batch, nodes, n, 3) per node, read
    at each edge's destination.  Returns the sums over the edges of each source node: (out_v (batch, nodes, n, 3),
    out_a (batch, nodes, n))."""
    actv_flat, v_flat = gl._flat_nodes(graph, actv_node), gl._flat_nodes(graph, v_node)
    if (ops.painn_combine_supported(v_flat.size(1)) and all(t.is_contiguous() and t.data_ptr() % 16 == 0
                                                            for t in (dist, actv_flat, v_flat, direction))):
        out_v, out_a = _PainnCombine.apply(dist, actv_flat, v_flat, direction, graph.by_dst, graph.by_src, _TERMS_ALL)
    else:
        m, a = _painn_combine_plain(dist, gl._Gather.apply(actv_flat, graph.by_dst),
                                    gl._Gather.apply(v_flat, graph.by_dst), direction)
        out_v, out_a = gl._ScatterSum.apply(m, graph.by_src), gl._ScatterSum.apply(a.contiguous(), graph.by_src)
    return (out_v.reshape(graph.batch, graph.nodes, *out_v.shape[1:]),
            out_a.reshape(graph.batch, graph.nodes, *out_a.shape[1:]))


def _table_interp_plain(table, d, period):
    """4-point Lagrange interpolation of a periodic grid in tensor arithmetic (differentiable in the grid and in d):
    the formula table_interp's kernels implement, kept as the yardstick its tests differentiate in float64."""
    rows = table.size(0)
    u = d * (float(rows) / period)
    fl = torch.floor(u).detach()
    t = (u - fl)[:, None]
    i = fl.long()
    tp, tm, tq = t + 1.0, t - 1.0, t - 2.0
    w = (-(1.0 / 6.0) * t * tm * tq, 0.5 * tp * tm * tq, -0.5 * tp * t * tq, (1.0 / 6.0) * tp * t * tm)
    return sum(w[j] * table[(i - 1 + j) % rows] for j in range(4))


class _SortedLengths:
    """The edges sorted by the grid row below their length: what the sums into the grid run by; computed on first
    use and shared by every pass over the same lengths."""

    def __init__(self, d, rows, period):
        self.d, self.rows, self.period = d, rows, period
        self._sorted = None

    def get(self):
        if self._sorted is None:
            self._sorted = ops.painn_table_sorted_edges(self.d.detach(), self.rows, self.period)
        return self._sorted


class _TableInterp(torch.autograd.Function):
    """order 0: the filter of every edge interpolated from its grid; order k: the interpolant's k-th derivative in
    the edge length (its weights are cubics: orders 0 .. 3 exist, the fourth derivative is zero).  The gradient for
    the grid is _TableScatter of the same order, the gradient for the lengths a row-wise product with _TableInterp of
    the next order: the family is closed under differentiation, so any number of nested derivatives run on these
    kernels.  Outside a recorded backward pass both gradients come from one fused call."""

    @staticmethod
    def forward(ctx, table, d, period, order, order_by):
        ctx.period, ctx.order, ctx.order_by = period, order, order_by
        ctx.save_for_backward(table, d)
        return ops.painn_table_interp_fwd(table, d, period, order)

    @staticmethod
    def backward(ctx, g):
        table, d = ctx.saved_tensors
        g = g.contiguous()
        need_t, need_d = ctx.needs_input_grad[0], ctx.needs_input_grad[1] and ctx.order < 3
        if not torch.is_grad_enabled():
            perm, bucket_ptr = ctx.order_by.get()
            d_table, dd = ops.painn_table_interp_bwd(g, table, d, ctx.period, perm, bucket_ptr, want_length_grad=need_d,
                                                     order=ctx.order)
            return (d_table if need_t else None), dd, None, None, None
        d_table = dd = None
        if need_t:
            d_table = _TableScatter.apply(g, d, ctx.period, ctx.order, table.size(0), ctx.order_by)
        if need_d:
            dd = (g * _TableInterp.apply(table, d, ctx.period, ctx.order + 1, ctx.order_by)).sum(-1)
        return d_table, dd, None, None, None


class _TableScatter(torch.autograd.Function):
    """The adjoint of _TableInterp in the grid: every edge's row g[e] added to the four grid rows around its length
    with the (order-th derivative) weights, in the order of a sort by grid row.  Linear in g; its gradients are
    _TableInterp calls."""

    @staticmethod
    def forward(ctx, g, d, period, order, rows, order_by):
        ctx.period, ctx.order, ctx.order_by = period, order, order_by
        ctx.save_for_backward(g, d)
        perm, bucket_ptr = order_by.get()
        return ops.painn_table_interp_bwd(g.contiguous(), None, d, period, perm, bucket_ptr, want_length_grad=False,
                                          order=order, table_rows=rows)[0]

    @staticmethod
    def backward(ctx, dd_table):
        g, d = ctx.saved_tensors
        dd_table = dd_table.contiguous()
        d_g = dd = None
        if ctx.needs_input_grad[0]:
            d_g = _TableInterp.apply(dd_table, d, ctx.period, ctx.order, ctx.order_by)
        if ctx.needs_input_grad[1] and ctx.order < 3:
            dd = (g * _TableInterp.apply(dd_table, d, ctx.period, ctx.order + 1, ctx.order_by)).sum(-1)
        return d_g, dd, None, None, None, None


def table_interp(table, d, period):
    """The grid `table` (rows, cols) of a function of period `period` interpolated at the lengths d (edges):
    (edges, cols), differentiable in both any number of times."""
    table, d = table.contiguous(), d.contiguous()
    return _TableInterp.apply(table, d, period, 0, _SortedLengths(d, table.size(0), period))


def _filter_grid_rows(msg, r_ij):
    """Rows of the grid the differentiable filter interpolates from, or 0 for the MLP on every edge."""
    E = r_ij.shape[0]
    rows = msg.table_rows() if (getattr(msg, "use_table", False) and E >= 4 * msg.TABLE_ROWS[0]) else 0
    if r_ij.requires_grad or has_tangent(r_ij):
        # The gradient for the edge vectors would go through the interpolant's derivative: differences of neighbouring
        # grid rows divided by the spacing, which amplifies the fp32-level noise of the grid values (1e-6 of their size
        # from the GEMMs that evaluate them) by rows / period: 4e-5 of the largest gradient entry at 2048 rows, 2e-4 at
        # 512 (where the interpolation error of the derivative dominates), against 7e-7 for the MLP on every edge.
        # A grid evaluated in float64 does not help (3e-5 at 2048 rows): the float32 differences themselves cancel
        # that many digits.  Positions that are differentiated (the meanflow loss, blocks that move them) keep the
        # per-edge MLP.
        return 0
    return rows if rows and E >= 4 * rows and ops.painn_table_interp_supported(rows, 4 * msg.n) else 0


def painn_filter(msg, r_ij):
    """mlp_dist(radial_encode(r_ij)) (archs/meanflow_painn8.py:92), (edges, 4n).  The filter is a smooth periodic
    function of the edge length: when the module's grid test accepts a grid for the current weights (the test the
    inference path uses, Message.table_rows) the MLP runs on the grid's rows and every edge interpolates, so that the
    backward pass differentiates the MLP on a few hundred rows instead of on every edge.  Only when the edge vectors
    need no gradient (_filter_grid_rows)."""
    rows = _filter_grid_rows(msg, r_ij)
    if rows:
        table = mlp_silu(msg.mlp_dist, msg._grid_encoding(rows, 0.0, r_ij.device))
        d = torch.linalg.vector_norm(r_ij, dim=-1).contiguous()
        return table_interp(table, d, 2.0 * msg.r0)
    return mlp_silu(msg.mlp_dist, radial_encode_painn(r_ij, msg.n_rbf, msg.r0))


def _unit_vectors(r_ij, epsilon):
    return r_ij / torch.sqrt(add((r_ij ** 2).sum(-1, keepdim=True), epsilon))


class _EdgeEncode(torch.autograd.Function):
    """Edge vectors -> (radial_encode, unit vectors, row bounds of the encoding) and, with tangents, (radial_encode, its
    tangent, unit vectors, their tangent, row bounds): one kernel each way."""

    @staticmethod
    def forward(ctx, r, r_t, n, rmax, epsilon):
        ctx.save_for_backward(r, r_t)
        ctx.shape_args = (n, rmax, epsilon)
        enc, enc_t, bound, direction, direction_t = ops.painn_edge_encode_fwd(r, r_t, n, rmax, epsilon)
        ctx.mark_non_differentiable(bound)
        return (enc, direction, bound) if r_t is None else (enc, enc_t, direction, direction_t, bound)

    @staticmethod
    def backward(ctx, *grads):
        r, r_t = ctx.saved_tensors
        n, rmax, epsilon = ctx.shape_args
        need = ctx.needs_input_grad[:2]
        if torch.is_grad_enabled():
            def pieces(r, r_t):
                enc = _as_pair(lambda x: radial_encode_painn(x, n, rmax), r, r_t)
                return enc + _as_pair(lambda x: _unit_vectors(x, epsilon), r, r_t)
            return _recorded_gradients(pieces, (r, r_t), need, grads[:-1]) + (None, None, None)
        g = [g.contiguous() for g in grads[:-1]]
        g_enc, g_enc_t, g_dir, g_dir_t = (g[0], None, g[1], None) if r_t is None else g
        g_r, g_rt = ops.painn_edge_encode_bwd(r, r_t, n, rmax, epsilon, g_enc, g_enc_t, g_dir, g_dir_t)
        return g_r if need[0] else None, g_rt if need[1] else None, None, None, None


def _message_edges(msg, graph, actv, x_v, r_ij, x_a=None):
    """The message with the filter MLP on every edge, or None where the fused functions do not take it.  actv: value and tangent."""
    params, n = _mlp_parameters(msg.mlp_dist), msg.n
    (r, r_t), (a, a_t), (v, v_t) = _unpack(r_ij), actv, _unpack(x_v)
    r, r_t = r.contiguous(), _dense(r_t)
    flat = [_dense(t if t is None else gl._flat_nodes(graph, t)) for t in (a, a_t, v, v_t)]
    if not (ops.painn_combine_supported(n) and msg.n_rbf % 4 == 0 and _fused(params, r, r_t, *flat)):
        return None
    if r_t is None:
        enc, direction, bound = _EdgeEncode.apply(r, None, msg.n_rbf, msg.r0, msg.epsilon)
        dist, dist_t, direction_t = _MlpSilu.apply(enc, None, bound, *params), None, None
    else:
        enc, enc_t, direction, direction_t, bound = _EdgeEncode.apply(r, r_t, msg.n_rbf, msg.r0, msg.epsilon)
        dist, dist_t = _MlpSilu.apply(enc, enc_t, bound, *params)
    return _combine_flat(graph, dist, dist_t, *flat, direction, direction_t, x_a, x_v)


def _combine_flat(graph, dist, dist_t, a, a_t, v, v_t, direction, direction_t, x_a=None, x_v=None):
    """(out_a, out_v), with tangents where an operand has one, from operands per edge and per flat node; added to x_a and x_v (v is
    x_v by flat nodes) unless x_a is None."""
    x = x_t = None
    if all(t is None for t in (dist_t, a_t, v_t, direction_t)):
        pairs = [(o, None) for o in _PainnCombine.apply(dist, a, v, direction, graph.by_dst, graph.by_src, _TERMS_ALL)]
    else:
        if x_a is not None:
            x, x_t = (_dense(t if t is None else gl._flat_nodes(graph, t)) for t in _unpack(x_a))
            rows = graph.by_src.n_rows
            if not (v.shape[0] == rows and all(t is None or (t.dtype == v.dtype and t.shape == (rows, v.shape[1]) and t.data_ptr() % 16 == 0)
                                               for t in (x, x_t))):
                x = x_t = None
        o_v, o_a, o_vt, o_at = _PainnCombineDual.apply(graph.by_dst, graph.by_src, x, x_t, dist, dist_t, a, a_t, v, v_t, direction,
                                                       direction_t)
        pairs = [(o_v, o_vt), (o_a, o_at)]
    out_v, out_a = (_dual(*(t if t is None else t.reshape(graph.batch, graph.nodes, *t.shape[1:]) for t in pair))
                    for pair in pairs)
    return (add(x_a, out_a), add(x_v, out_v)) if x_a is not None and x is None else (out_a, out_v)


_SLICE_PERMUTATIONS = {}


def _slice_permutation(n, device):
    key = (n, str(device))
    if key not in _SLICE_PERMUTATIONS:
        _SLICE_PERMUTATIONS[key] = ops.painn_slice_permutation(n, device)
    return _SLICE_PERMUTATIONS[key]


class _PainnGridMessage(torch.autograd.Function):
    """(grid (rows, 4n), actv (nodes, 4n), v (nodes, n, 3)) -> (out_v, out_a) of the message for edge vectors that are
    not differentiated, with the filter interpolated from the grid.  Forward: the inference kernel of the layer
    (mg_painn_table_message: lengths, directions, interpolation, the lines 94-100 of archs/meanflow_painn8.py and the
    sum over the edges of a node in one pass; no per-edge filter is stored).  Backward: where the grid fits in LDS, one
    kernel for the gradients of actv and v and one, over the edges sorted by grid row, for the grid's
    (mg_painn_grid_node_grad, mg_painn_grid_table_grad: nothing per edge is stored); for larger grids the gradient kernel of
    the unfused formulation with the filter of every edge interpolated again inside it (mg_painn_combine_bwd_rows), then
    the scatter into the grid.  A recorded backward pass differentiates the unfused formulation instead.
    x (nodes, n): None, or the rows that out_a is added to; v is then added to out_v, and the kernel that writes the gradient of v
    adds that of out_v."""

    @staticmethod
    def forward(ctx, table, actv, v, r_ij, x, graph, period, epsilon):
        ctx.graph, ctx.period, ctx.epsilon, ctx.residual = graph, period, epsilon, x is not None
        table, actv, v = table.contiguous(), actv.contiguous(), v.contiguous()
        res = () if x is None else (x.contiguous(), v)
        actv_s = None
        n = v.size(1)
        if table.size(0) <= ops.PAINN_SLICED_MAX_ROWS and n % ops.PAINN_SLICE == 0:
            # the grid fits in LDS: the kernel that holds it there takes actv with its columns grouped slice by slice
            actv_s = actv[:, _slice_permutation(n, actv.device)].contiguous()
            out_a, out_v = ops.painn_table_message_sliced(graph.row_ptr, graph.dst32, r_ij, table, period, actv_s, v, epsilon, *res,
                                                          node_order=getattr(graph, "cell_order", None))
        else:
            out_a, out_v = ops.painn_table_message(graph.row_ptr, graph.dst32, r_ij, table, period, actv, v, epsilon, *res)
        ctx.save_for_backward(table, actv, v, r_ij, actv_s if ctx.needs_input_grad[0] else None)
        return out_v, out_a

    @staticmethod
    def backward(ctx, g_v, g_a):
        table, actv, v, r_ij, actv_s = ctx.saved_tensors
        graph, need, residual = ctx.graph, ctx.needs_input_grad, ctx.residual
        past = (None, g_a if need[4] else None, None, None, None)
        if torch.is_grad_enabled():
            with torch.enable_grad():
                leaves = [t if t.requires_grad else t.detach().requires_grad_() for t in (table, actv, v)]
                out = _grid_message_unfused(*leaves, r_ij, graph, ctx.period, ctx.epsilon)
                if residual:
                    out = (out[0] + leaves[2], out[1])
                grads = torch.autograd.grad(out, leaves, (g_v, g_a), create_graph=True, allow_unused=True)
            return tuple(g if nd else None for g, nd in zip(grads, need)) + past
        by_dst, by_src = graph.by_dst, graph.by_src
        if ops.painn_grid_grad_supported(table.size(0), v.size(1)) and all(t.data_ptr() % 16 == 0 for t in (table, v, actv)):
            # (the sliced rows are read for the grid's gradient only)
            grads = ops.painn_grid_message_bwd(table, actv, actv if actv_s is None else actv_s, v, r_ij, g_v.contiguous(),
                                               g_a.contiguous(), graph.src32, graph.dst32, by_dst.row_ptr, by_dst.perm,
                                               getattr(graph, "cell_order", None), ctx.period, ctx.epsilon, need[0], need[1],
                                               need[2], graph.row_ptr, residual)
            return (*grads, *past)
        d = torch.linalg.vector_norm(r_ij, dim=-1).contiguous()
        want = (bool(need[0]), bool(need[1]), bool(need[2]), False)
        # (actv and v are read at an edge's destination: their gradients are summed over a destination's edges inside)
        d_dist, d_actv, dv, _ = ops.painn_combine_bwd_rows(None, actv, v, _unit_vectors(r_ij, ctx.epsilon).contiguous(),
                                                           g_v.contiguous(), g_a.contiguous(), by_dst.row_ptr, by_dst.perm,
                                                           by_src.index, terms=_TERMS_ALL, want=want, table=table,
                                                           period=ctx.period, d=d)
        d_table = None
        if need[0]:
            rows = table.size(0)
            perm, bucket_ptr = ops.painn_table_sorted_edges(d, rows, ctx.period)
            d_table = ops.painn_table_interp_bwd(d_dist, None, d, ctx.period, perm, bucket_ptr, want_length_grad=False,
                                                 order=0, table_rows=rows)[0]
        dv = (dv + g_v.reshape(dv.shape) if residual else dv) if need[2] else None
        return (d_table, d_actv if need[1] else None, dv, *past)


def _grid_message_unfused(table, actv, v, r_ij, graph, period, epsilon):
    d = torch.linalg.vector_norm(r_ij, dim=-1).contiguous()
    return _PainnCombine.apply(table_interp(table, d, period), actv, v, _unit_vectors(r_ij, epsilon).contiguous(),
                               graph.by_dst, graph.by_src, _TERMS_ALL)


def painn_message(msg, graph, x_a, x_v, r_ij, residual=False):
    """archs/meanflow_painn8.py:85-100; (x_a + da, x_v + dv) with residual.  The kernels that sum over a node's edges then add the node's
    own row, and their adjoints the gradient that goes past the message (a step of three blocks on 4
    systems of 1024 atoms, 128 channels, values and tangents: 99 launches and 260 us less, with the copies of the tangents)."""
    # the MLP acts on rows, so it commutes with the gather: N rows go through it, not E (the reference gathers first),
    # and the gathers themselves are folded into the combining kernel
    actv = _mlp_silu_pair(msg.mlp_actv, x_a)
    rows = _filter_grid_rows(msg, r_ij)
    n = x_v.size(-2)
    # (actv has a tangent without x_a where its MLP's weights have one)
    if (rows and n % 4 == 0 and ops.painn_combine_supported(n) and actv[1] is None and not any(has_tangent(t) for t in (x_a, x_v))
            and r_ij.is_contiguous() and not getattr(graph, "padded", False)):
        table = mlp_silu(msg.mlp_dist, msg._grid_encoding(rows, 0.0, r_ij.device))
        flat_v, flat_a = gl._flat_nodes(graph, x_v), gl._flat_nodes(graph, x_a) if residual else None
        inside = residual and all(t.data_ptr() % 16 == 0 for t in (flat_a, flat_v))
        out_v, out_a = _PainnGridMessage.apply(table, gl._flat_nodes(graph, actv[0]), flat_v, r_ij, flat_a if inside else None, graph,
                                               2.0 * msg.r0, msg.epsilon)
        out_a, out_v = (t.reshape(graph.batch, graph.nodes, *t.shape[1:]) for t in (out_a, out_v))
        return (add(x_a, out_a), add(x_v, out_v)) if residual and not inside else (out_a, out_v)
    x = x_a if residual else None
    if not rows and not getattr(graph, "padded", False):
        out = _message_edges(msg, graph, actv, x_v, r_ij, x)
        if out is not None:
            return out
    dist, direction = painn_filter(msg, r_ij), _unit_vectors(r_ij, msg.epsilon)
    if ops.painn_combine_supported(n) and (actv[1] is not None or has_tangent(x_v)) and not has_tangent(dist):
        flat = [_dense(t if t is None else gl._flat_nodes(graph, t)) for t in (*actv, *_unpack(x_v))]
        if all(t is None or t.data_ptr() % 16 == 0 for t in (*flat, dist)):
            return _combine_flat(graph, dist.contiguous(), None, *flat, direction.contiguous(), None, x, x_v)
    out_v, out_a = painn_combine(graph, dist, _dual(*actv), x_v, direction)
    return (add(x_a, out_a), add(x_v, out_v)) if residual else (out_a, out_v)


class _PainnUpdate(torch.autograd.Function):
    """painn.Update, values alone or values and tangents: one call into the C++ binding for each direction.
    residual: the results are added to x_a and x_v, and the gradients of these are the sums of both."""

    @staticmethod
    def forward(ctx, upd, residual, x_a, x_at, x_v, x_vt, *params):
        ctx.upd, ctx.residual = upd, residual
        outs, rows = ops.painn_update_train_fwd(x_a, x_at, x_v, x_vt, params[:3], params[5::2], params[6::2], upd.gn.groups,
                                                params[3], params[4], upd.gn.epsilon, residual)
        ctx.save_for_backward(x_a, x_at, x_v, x_vt, *params, *(rows if any(ctx.needs_input_grad) else ()))
        ctx.set_materialize_grads(False)
        return tuple(outs)

    @staticmethod
    def backward(ctx, g_a, g_v, g_at=None, g_vt=None):
        upd, residual, need = ctx.upd, ctx.residual, list(ctx.needs_input_grad[1:])
        x_a, x_at, x_v, x_vt, *saved = ctx.saved_tensors
        params, rows = saved[:11], saved[11:]
        if all(g is None for g in (g_a, g_v, g_at, g_vt)):
            return (None,) * (1 + len(need))
        if torch.is_grad_enabled():
            def pieces(x_a, x_at, x_v, x_vt, *params):
                if x_vt is None:
                    return _update_pieces(upd, params, x_a, x_v, residual=residual)
                split = lambda: tuple(zip(*(fwAD.unpack_dual(o) for o in _update_pieces(upd, params, _dual(x_a, x_at), _dual(x_v, x_vt),
                                                                                        residual=residual))))
                if getattr(fwAD, "_current_level", 0) >= 0:
                    return sum(split(), ())
                with fwAD.dual_level():
                    return sum(split(), ())
            return (None, None) + _recorded_gradients(pieces, (x_a, x_at, x_v, x_vt, *params), need[1:], (g_a, g_v, g_at, g_vt))
        # (a result that nothing depends on leaves what only it depends on without a gradient, as separate functions would)
        if g_a is None and g_at is None:
            need[5] = need[8] = need[9] = False                             # the map l, gamma, beta
        if g_v is None and g_vt is None:
            need[7] = False                                                 # the map v
        if g_a is None:
            need[9] = False
        zeros = lambda g, like: torch.zeros_like(like) if g is None else g.contiguous()
        g_a, g_v = zeros(g_a, x_a), zeros(g_v, x_v)
        if x_vt is not None:
            g_at, g_vt = zeros(g_at, x_a), zeros(g_vt, x_v)
        g_x, d_params = ops.painn_update_train_bwd(g_a, g_at, g_v, g_vt, params[5::2], upd.gn.groups, params[3], rows, residual)
        grads = list(g_x) + list(d_params)
        return (None, None) + tuple(g if nd else None for g, nd in zip(grads, need[1:]))


def _update_pieces(upd, params, x_a, x_v, maps=None, residual=False):
    """painn.Update out of differentiable pieces; params: gamma, beta and the MLP's behind the three maps' weights, which
    `maps` (callables) stand in for."""
    n = upd.n
    x_v = x_v.contiguous()
    lin_l, lin_r, lin_v = maps or [lambda x, W=W: tensor_linear(1, W, x) for W in params[:3]]
    v_l, v_r = lin_l(x_v), lin_r(x_v)
    ip = (v_l * v_r).sum(-1)
    y = _mlp_rows(params[-6:], torch.cat([x_a, torch.linalg.vector_norm(v_r, dim=-1)], dim=-1))
    v = lin_v(x_v) * y[..., :n, None]
    a = scal_group_norm(upd.gn, ip * y[..., n:2 * n], params[-8], params[-7]) + y[..., 2 * n:]
    v = v / torch.sqrt(add((v ** 2).sum(-1, keepdim=True), 1.))
    return (add(x_a, a), add(x_v, v)) if residual else (a, v)


def painn_update(upd, x_a, x_v, residual=False):
    """archs/meanflow_painn8.py:63-75; (x_a + da, x_v + dv) with residual, as painn_message."""
    maps = (upd.lin_l, upd.lin_r, upd.lin_v)
    params = [upd.gn.gamma, upd.gn.beta, *_mlp_parameters(upd.mlp)]
    if not all(plain_call(lin, TensLinear) for lin in maps):
        return _update_pieces(upd, params, x_a, x_v, maps, residual)
    params = [lin.W for lin in maps] + params
    pairs = [tuple(_dense(t) for t in _unpack(x)) for x in (x_a, x_v)]
    (a, a_t), (v, v_t) = pairs
    if a_t is not None and v_t is None:
        v_t = torch.zeros_like(v)
    if not (x_a.dim() == 3 and upd.n <= 256 and _fused(params, a, a_t, v, v_t)):
        return _update_pieces(upd, params, x_a, x_v, residual=residual)
    outs = _PainnUpdate.apply(upd, residual, a, a_t, v, v_t, *params)
    return outs if v_t is None else tuple(fwAD.make_dual(p, t) for p, t in zip(outs[:2], outs[2:]))


def apply_tens_prod_submodules(module, prods):
    """archs/diffuser_atoms15.py:52-57"""
    from .ops import BEE_ORDER
    out = [None, None, None]
    for lab, p in zip(BEE_ORDER, prods):
        y = getattr(module, f"Y_{lab}")(p)
        k = int(lab[2])
        out[k] = y if out[k] is None else out[k] + y
    return tuple(out)


def _message_products_plain(a_node, v_node, d_node, enc, rh, by_dst, by_src):
    """The 13 products of the gathered node operands with the edge filters (enc, enc (x) rh, enc (x) rh (x) rh); those
    of rank 1 and 2 summed over the edges of their source node (archs/diffuser_atoms15.py:241-252 with the sum moved
    before the output linears).  Built from functions that are differentiable any number of times."""
    from .ops import BEE_ORDER
    phi_v, phi_d = _EdgeFilters.apply(enc, rh)
    prods = Bee.apply(gl._Gather.apply(a_node, by_dst), gl._Gather.apply(v_node, by_dst), gl._Gather.apply(d_node, by_dst),
                      enc.contiguous(), phi_v, phi_d)
    return tuple(p if lab[2] == "0" else gl._ScatterSum.apply(p.contiguous(), by_src) for lab, p in zip(BEE_ORDER, prods))


def _by_component(*tensors):
    """(rows, chan, 3, ..) as (rows, 3^rank, chan)"""
    return tuple(t.flatten(2).transpose(1, 2).contiguous() if t.dim() > 2 else t.contiguous() for t in tensors)


def _by_channel(*tensors):
    """(rows, 3, chan) or (rows, 9, chan) as (rows, chan, 3, ..)"""
    return tuple(t if t.dim() == 2 else t.transpose(1, 2).reshape(t.shape[0], -1, *([3] if t.shape[1] == 3 else [3, 3])).contiguous()
                 for t in tensors)


def _as_rows(P0, S1, S2):
    """P0, S1, S2 as plain rows, one per (row, component)"""
    return P0.flatten(1), S1.reshape(-1, 5 * S1.shape[-1]), S2.reshape(-1, 5 * S2.shape[-1])


class _MessageProducts(torch.autograd.Function):
    """The same with everything between the node operands and the per-node sums folded into kernels.  by_label: operands
    and 13 results as in the plain formulation; else v_node (nodes, 3, chan), d_node (nodes, 9, chan) and the results as the plain
    rows of P0, S1, S2 (ops.bee_message), which the output linears of a rank read side by side.
    Forward: the inference kernel of the layer (mg_bee_message: filters formed in registers, node rows gathered at the destination,
    products summed over the edges of a node; only the three scalar products are stored per edge) when `enc_source`
    = (the 8 radial functions, weight and bias of the encoding linear) is given, else the indexed product kernel and
    segment sums.  Backward: one kernel walks the edges of a source node with the gradients of its sums in registers and
    yields the gradients of enc and rh and, per edge, of the node operands, which a second one sums by destination.  A recorded backward pass (create_graph=True)
    differentiates the plain formulation instead."""

    @staticmethod
    def forward(ctx, a_node, v_node, d_node, enc, rh, by_dst, by_src, enc_source, by_label):
        ctx.by_dst, ctx.by_src, ctx.by_label = by_dst, by_src, by_label
        ctx.set_materialize_grads(False)
        a_node, v_node, d_node, enc, rh = (t.contiguous() for t in (a_node, v_node, d_node, enc, rh))
        ctx.save_for_backward(a_node, v_node, d_node, enc, rh)
        ctx.save_for_forward(a_node, v_node, d_node, enc, rh)
        N, C = a_node.shape
        left = a_node, v_node, d_node
        if enc_source is not None:
            enc8, W, b = enc_source
            b = b if b is not None else torch.zeros(C, dtype=torch.float32, device=enc.device)
            operands = by_src.row_ptr, by_dst.index, rh, enc8.contiguous(), *(_by_component(*left) if by_label else left)
            stacked = ops.bee_message(*operands, W.detach().contiguous(), b.detach().contiguous())
            if by_label:
                return ops.unstack_products(*stacked)
        else:
            phi_v, phi_d = ops.bee_edge_filters_fwd(enc, rh)
            prods = ops.bee_fwd_indexed(*(left if by_label else (t.contiguous() for t in _by_channel(*left))), by_dst.index, enc,
                                        phi_v, phi_d)
            prods = tuple(p if lab[2] == "0" else ops.segment_sum_csr(p, by_src.row_ptr, by_src.n_rows)
                          for lab, p in zip(ops.BEE_ORDER, prods))
            if by_label:
                return prods
            stacked = ops.stack_products(prods)
        return _as_rows(*stacked)

    @staticmethod
    def jvp(ctx, a_t, v_t, d_t, enc_t, rh_t, *_):
        """Forward mode through the plain formulation: the products are bilinear in (node operands, edge filters), so
        the tangent is P(gathered tangents, filters) + P(gathered operands, the filters' tangent), summed per node
        like the products themselves."""
        *left, enc, rh = ctx.saved_tensors
        left_t = [torch.zeros_like(t) if g is None else g for g, t in zip((a_t, v_t, d_t), left)]
        enc_t, rh_t = (torch.zeros_like(t) if g is None else g for g, t in zip((enc_t, rh_t), (enc, rh)))
        by_dst, by_src, by_label = ctx.by_dst, ctx.by_src, ctx.by_label
        gather = lambda ts: [gl._Gather.apply(t.contiguous(), by_dst) for t in (ts if by_label else _by_channel(*ts))]
        phi_v, phi_d = _EdgeFilters.apply(enc, rh)
        phi_v_t, phi_d_t = _edge_filters_tangent(enc, rh, enc_t, rh_t)
        prods = [a + b for a, b in zip(Bee.apply(*gather(left_t), enc, phi_v, phi_d),
                                       Bee.apply(*gather(left), enc_t.contiguous(), phi_v_t.contiguous(), phi_d_t.contiguous()))]
        prods = tuple(p if lab[2] == "0" else gl._ScatterSum.apply(p.contiguous(), by_src) for lab, p in zip(ops.BEE_ORDER, prods))
        return prods if by_label else _as_rows(*ops.stack_products(prods))

    @staticmethod
    def backward(ctx, *dys):
        saved, by_dst, by_src, by_label = ctx.saved_tensors, ctx.by_dst, ctx.by_src, ctx.by_label
        need = ctx.needs_input_grad
        if torch.is_grad_enabled():
            with torch.enable_grad():
                leaves = [t if t.requires_grad else t.detach().requires_grad_() for t in saved]
                out = _message_products_plain(*(leaves[:3] if by_label else _by_channel(*leaves[:3])), *leaves[3:], by_dst, by_src)
                out = out if by_label else _as_rows(*ops.stack_products(out))
                dys = [torch.zeros_like(o) if g is None else g for o, g in zip(out, dys)]
                grads = torch.autograd.grad(out, leaves, dys, create_graph=True)
            return tuple(g if nd else None for g, nd in zip(grads, need)) + (None, None, None, None)
        *left, enc, rh = saved
        N, C, E = left[0].shape[0], left[0].shape[1], enc.shape[0]
        if by_label:
            run = ops.bee_message_bwd
            shapes = [(by_src.n_rows if lab[2] != "0" else E, C, *[3] * int(lab[2])) for lab in ops.BEE_ORDER]
        else:
            run, shapes = ops.bee_message_grad, ((E, 3, C), (by_src.n_rows, 3, 5, C), (by_src.n_rows, 9, 5, C))
        dys = [enc.new_zeros(sh) if g is None else g.contiguous().reshape(sh) for g, sh in zip(dys, shapes)]
        d_l, d_enc, d_rh = run(left, enc, rh, dys, by_src, by_dst, any(need[:3]), need[3], need[4])
        return tuple(d_l[k] if need[k] else None for k in range(3)) + (d_enc, d_rh, None, None, None, None)


class _NodeProducts(torch.autograd.Function):
    """The 13 products of operands (rows, chan), (rows, 3, chan), (rows, 9, chan) as the plain rows of P0, P1, P2
    (ops.bee_node_products).  A recorded backward pass differentiates the product function instead, forward mode is the
    product rule."""

    @staticmethod
    def forward(ctx, *operands):
        operands = tuple(t.contiguous() for t in operands)
        ctx.save_for_backward(*operands)
        ctx.save_for_forward(*operands)
        ctx.set_materialize_grads(False)
        return _as_rows(*ops.bee_node_products(*operands))

    @staticmethod
    def jvp(ctx, *tangents):
        operands = ctx.saved_tensors
        tangents = [torch.zeros_like(x) if t is None else t for t, x in zip(tangents, operands)]
        left, right = _NodeProducts.apply(*tangents[:3], *operands[3:]), _NodeProducts.apply(*operands[:3], *tangents[3:])
        return tuple(a + b for a, b in zip(left, right))

    @staticmethod
    def backward(ctx, *dys):
        operands, need = ctx.saved_tensors, ctx.needs_input_grad
        pieces = _gradients_in_pieces(lambda *t: _as_rows(*ops.stack_products(Bee.apply(*_by_channel(*t)))), operands, (True,) * 6, dys)
        if pieces is not None:
            grads = [torch.zeros_like(x) if g is None else g for g, x in zip(pieces, operands)]
        else:
            N, C = operands[0].shape
            shapes = (N, 3, C), (N, 3, 5, C), (N, 9, 5, C)
            # (without a gradient of P2, 45 of a node's 63, none is written as zeros to be read)
            grads = ops.bee_node_products_grad(operands, [g if g is None and k == 2 else operands[0].new_zeros(sh) if g is None else g.contiguous()
                                                          for k, (g, sh) in enumerate(zip(dys, shapes))])
        return tuple(g if nd else None for g, nd in zip(grads, need))


def _component_rows(x):
    """(.., chan, 3, ..) of rank 1 or 2 as plain rows, one per (row, component)"""
    return x.flatten(2).transpose(1, 2).reshape(-1, x.shape[1])


def _rows_of_rank(x, rank):
    """(rows, chan, 3, ..) from plain rows (rows 3^rank, chan)"""
    return x if rank == 0 else x.reshape(-1, 3 ** rank, x.shape[-1]).transpose(1, 2).reshape(-1, x.shape[-1], *[3] * rank)


class _RowLinears(torch.autograd.Function):
    """sum_k W_k x_k for x = [x_1 | x_2 | ..] on plain rows, one per (row, component) of tensors of a rank: tensor linears that
    lie side by side.  The arithmetic, its fp32 line included, is that of one linear after the other (see _TensorLinearFn): the
    x_k may differ in magnitude by any factor, so each has scales of its own."""

    @staticmethod
    def forward(ctx, rank, sequential, x, *W):
        x = x.contiguous()
        y, x_max = ops.row_linears_fwd(x, W, 3 ** rank, sequential)
        ctx.rank = rank
        ctx.save_for_backward(x, x_max, *W)
        ctx.save_for_forward(x, x_max, *W)
        ctx.set_materialize_grads(False)
        return y

    @staticmethod
    def jvp(ctx, _rank, _sequential, x_t, *W_t):
        x, _, *W = ctx.saved_tensors
        parts = [] if x_t is None else [_RowLinears.apply(ctx.rank, False, x_t, *W)]
        if any(t is not None for t in W_t):
            parts.append(_RowLinears.apply(ctx.rank, False, x, *(torch.zeros_like(w) if t is None else t for w, t in zip(W, W_t))))
        return sum(parts[1:], parts[0]) if parts else None

    @staticmethod
    def backward(ctx, dy):
        x, x_max, *W = ctx.saved_tensors
        need = ctx.needs_input_grad
        if dy is None:
            return (None,) * len(need)
        pieces = _gradients_in_pieces(lambda x, *W: (_row_linears_plain(ctx.rank, x, W),), (x, *W), need[2:], (dy,))
        if pieces is not None:
            return (None, None) + pieces
        dy = dy.contiguous()
        dx, dW = ops.row_linears_bwd(dy, x, W, x_max, 3 ** ctx.rank, need[2], any(need[3:]))
        return (None, None, dx) + tuple(d if nd else None for d, nd in zip(dW or [None] * len(W), need[3:]))


def _row_linears_plain(rank, x, W):
    """The same as linears one after the other."""
    y = [tensor_linear(rank, w, _rows_of_rank(x_k, rank)) for w, x_k in zip(W, x.split(W[0].shape[1], dim=1))]
    y = sum(y[1:], y[0])
    return y if rank == 0 else _component_rows(y)


def _linear_by_component(lin, rank, rows):
    """A TensLinear of rank 0, 1 or 2 on the plain rows of x -> (rows of x, chan) or (rows of x, 3^rank, chan)."""
    if rank == 0:
        return tensor_linear(0, lin.W, rows, sequential=torch.is_grad_enabled())
    y = _RowLinears.apply(rank, torch.is_grad_enabled(), rows, lin.W)
    return y.reshape(-1, 3 ** rank, y.shape[-1])


def _linears_of_rank(mod, rank, P):
    """The output linears of one rank on the plain rows P of their products, summed: (rows, dim), (rows, dim, 3) or
    (rows, dim, 3, 3)."""
    return _rows_of_rank(_RowLinears.apply(rank, torch.is_grad_enabled(), P, *(getattr(mod, f"Y_{lab}").W for lab in ops.STACKED[rank])),
                         rank)


def _plain_linears(mod, operands):
    """True when calling the module's tensor linears (the operands' and Y_*) does what TensLinear.forward does and nothing else."""
    return all(plain_call(getattr(mod, name), TensLinear) for name in (*operands, *(f"Y_{lab}" for lab in ops.BEE_ORDER)))


def message_products(graph, a_node, v_node, d_node, enc, rh, enc_source=None):
    """a_node (batch, nodes, chan), v_node (.., chan, 3), d_node (.., chan, 3, 3): the node operands, read at each
    edge's destination; enc (edges, chan), rh (edges, 3): what the edge filters are made of.  Returns the 13 products
    in ops.BEE_ORDER: those of rank 0 per edge, those of rank 1 and 2 summed over the edges of their source node
    ((batch * nodes, chan, ...)).  enc_source: see _MessageProducts."""
    flat = [gl._flat_nodes(graph, t) for t in (a_node, v_node, d_node)]
    enc, rh = enc.contiguous(), rh.contiguous()
    if ops.bee_indexed_supported(enc.size(1)) and all(t.data_ptr() % 16 == 0 for t in flat + [enc]):
        return _MessageProducts.apply(*flat, enc, rh, graph.by_dst, graph.by_src, enc_source, True)
    return _message_products_plain(*flat, enc, rh, graph.by_dst, graph.by_src)


def _edge_filters_plain(enc, rh):
    """archs/diffuser_atoms15.py:241-243"""
    return enc[..., None] * rh[..., None, :], enc[..., None, None] * rh[..., None, None, :] * rh[..., None, :, None]


def _edge_filters_tangent(enc, rh, enc_t, rh_t):
    """The derivative of _edge_filters_plain along (enc_t, rh_t): the product rule on its two and three factors."""
    phi_v_t = enc_t[..., None] * rh[..., None, :] + enc[..., None] * rh_t[..., None, :]
    rr = rh[..., None, None, :] * rh[..., None, :, None]
    rr_t = rh_t[..., None, None, :] * rh[..., None, :, None] + rh[..., None, None, :] * rh_t[..., None, :, None]
    return phi_v_t, enc_t[..., None, None] * rr + enc[..., None, None] * rr_t


class _EdgeFilters(torch.autograd.Function):
    """phi_v = enc (x) rh and phi_d = enc (x) rh (x) rh as one kernel, and their adjoint as another; a recorded
    backward pass differentiates the broadcasting arithmetic instead."""

    @staticmethod
    def forward(ctx, enc, rh):
        ctx.save_for_backward(enc, rh)
        ctx.save_for_forward(enc, rh)
        return ops.bee_edge_filters_fwd(enc.contiguous(), rh.contiguous())

    @staticmethod
    def jvp(ctx, enc_t, rh_t):
        return _edge_filters_tangent(*ctx.saved_tensors, enc_t, rh_t)

    @staticmethod
    def backward(ctx, g_v, g_d):
        enc, rh = ctx.saved_tensors
        if torch.is_grad_enabled():
            with torch.enable_grad():
                leaves = [t if t.requires_grad else t.detach().requires_grad_() for t in (enc, rh)]
                grads = torch.autograd.grad(_edge_filters_plain(*leaves), leaves, (g_v, g_d), create_graph=True)
            return tuple(g if nd else None for g, nd in zip(grads, ctx.needs_input_grad))
        d_enc, d_rh = ops.bee_edge_filters_bwd(enc.contiguous(), rh.contiguous(), g_v.contiguous(), g_d.contiguous())
        return (d_enc if ctx.needs_input_grad[0] else None), (d_rh if ctx.needs_input_grad[1] else None)


def bee_messages(msg, graph, r_ij, x_a, x_v, x_d):
    """archs/diffuser_atoms15.py:238-253"""
    if differentiated(r_ij) or not (r_ij.is_cuda and r_ij.dtype == torch.float32):
        enc8, rh = radial_encode_8(r_ij, msg.r0), tens_sigmoid(1, mul(r_ij, 7. / msg.r0))
    else:
        enc8, rh = ops.bee_edge_geometry(r_ij.contiguous(), msg.r0)            # (two dozen of torch's passes over the edges)
    enc = linear(msg.lin_enc, enc8)
    # The output linears of the vector and rank-2 channels have no bias and nothing nonlinear follows them before the
    # sum over edges, so they commute with it: the products are summed per node first and the ten linears run on N
    # rows, not E (the reference applies them per edge).  The scalar channel goes through an MLP per edge.
    B, N = x_a.shape[:2]
    if _plain_linears(msg, ("L0", "L1", "L2")) and ops.bee_indexed_supported(enc.size(1)):
        a, v, d = (gl._flat_nodes(graph, t) for t in (x_a, x_v, x_d))
        nodes = [_linear_by_component(lin, k, x)
                 for k, (lin, x) in enumerate(zip((msg.L0, msg.L1, msg.L2), (a, _component_rows(v), _component_rows(d))))]
        P0, S1, S2 = _MessageProducts.apply(*nodes, enc, rh, graph.by_dst, graph.by_src,
                                            (enc8.detach(), msg.lin_enc.weight, msg.lin_enc.bias), False)
        psi_a, *sums = (_linears_of_rank(msg, k, P) for k, P in enumerate((P0, S1, S2)))
        psi_a = mlp_leaky(msg.mlp_a, psi_a, residual=True)
        return (mul(gl.edges_reduce_src(graph, psi_a), 0.1), *(mul(t.reshape(B, N, *t.shape[1:]), 0.1) for t in sums))
    prods = message_products(graph, msg.L0(x_a), msg.L1(x_v), msg.L2(x_d), enc, rh,
                             enc_source=(enc8.detach(), msg.lin_enc.weight, msg.lin_enc.bias))
    from .ops import BEE_ORDER
    psi_a, sums = None, [None, None, None]
    for lab, p in zip(BEE_ORDER, prods):
        k = int(lab[2])
        y = getattr(msg, f"Y_{lab}")(p if k == 0 else p.reshape(graph.batch, graph.nodes, *p.shape[1:]))
        if k == 0:
            psi_a = y if psi_a is None else psi_a + y
        else:
            sums[k] = y if sums[k] is None else sums[k] + y
    psi_a = mlp_leaky(msg.mlp_a, psi_a, residual=True)
    return mul(gl.edges_reduce_src(graph, psi_a), 0.1), mul(sums[1], 0.1), mul(sums[2], 0.1)


def displacement_tensors(mod, graph, r_ij):
    """archs/diffuser_atoms15.py:216-225 out of differentiable pieces: the radial MLP per edge, the edge filters
    rad (x) u and rad (x) u (x) u as one kernel (their adjoint another), sums over the edges of a source node, the two
    readouts on node rows."""
    first = mod.mlp_radial[0]
    rad = mlp_leaky(mod.mlp_radial[1], linear(first, radial_encode_8(r_ij, mod.r0)))
    u = tens_sigmoid(1, mul(r_ij, 7. / mod.r0))
    phi_v, phi_d = _EdgeFilters.apply(rad.contiguous(), u.contiguous())
    A_a, A_v, A_d = (gl.edges_reduce_src(graph, t) for t in (rad, phi_v, phi_d))
    return A_a, mod.readout_v(A_v), mod.readout_d(A_d)


def self_tens_prods(mod, x_a, x_v, x_d):
    """archs/diffuser_atoms15.py:75-95"""
    *rest, dim_a = x_a.shape
    dim_v, dim_d = x_v.shape[-2], x_d.shape[-3]
    a, v, d = x_a.reshape(-1, dim_a), x_v.reshape(-1, dim_v, 3), x_d.reshape(-1, dim_d, 3, 3)
    if _plain_linears(mod, ("L0", "L1", "L2", "R0", "R1", "R2")):
        rows = a, _component_rows(v), _component_rows(d)
        operands = [_linear_by_component(lin, k, x) for side in ((mod.L0, mod.L1, mod.L2), (mod.R0, mod.R1, mod.R2))
                    for k, (lin, x) in enumerate(zip(side, rows))]
        y_a, y_v, y_d = (_linears_of_rank(mod, k, P) for k, P in enumerate(_NodeProducts.apply(*operands)))
    else:
        prods = Bee.apply(mod.L0(a), mod.L1(v), mod.L2(d), mod.R0(a), mod.R1(v), mod.R2(d))
        y_a, y_v, y_d = apply_tens_prod_submodules(mod, prods)
    return (tens_group_norm(mod.gn_a, y_a.reshape(*rest, dim_a)), tens_group_norm(mod.gn_v, y_v.reshape(*rest, dim_v, 3)),
            tens_group_norm(mod.gn_d, y_d.reshape(*rest, dim_d, 3, 3)))
