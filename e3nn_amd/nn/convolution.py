"""Equivariant point convolution of the reference's ``v2106`` model family
(``e3nn/nn/models/v2106/points_convolution.py:19-113``), every step on the HIP kernels of this package:

    self-connection, lin1, lin2, alpha   FullyConnectedTensorProduct(features, node_attr)   uvw kernels
    radial network                        FullyConnectedNet(edge_scalars)                     uvw + gate kernels
    message                               scatter(tp(x[src], edge_attr, w), dst)              fused uvu kernel

``node_features[edge_src]`` and the per-edge messages are never materialised.
"""
import torch

from .. import _lib
from ..o3.irreps import Irrep, Irreps
from ..o3.tensor_product import _OUT, FullyConnectedTensorProduct, TensorProduct, _permuted_weights, _slot_backward, _TpSlot
from .edges import DstSortedEdges
from .fc import FullyConnectedNet
from .message import message_instructions

# The message kernel with the radial network inside deals whole rows to 8192 workers: below about one row each it waits
# for the longest rows on a half-empty chip.  A block without gradients, 32x0e+32x1o+32x2e, 35 edges per row, network inside
# / two kernels: 60 rows 177 / 124 us, 1000 rows 250 / 152, 5003 rows 340 / 252, 8000 rows 386 / 334, 12 000 rows 420 / 429,
# 50 000 rows 1154 / 1533.  Other degrees shift the gain, not the line: at 3, 12, 120 and 400 edges per row the network inside
# takes 0.94 to 1.10, 1.07 to 1.10, 1.06 to 2.45 and 1.08 to 3.64 times as long below it, and between 0.91 and 1.10 times
# at 20 000 rows; sets that the kernel does not take (64 channels, 16 channels) run the two kernels on either side.  The two
# kernels store the weights of all edges: not beyond 1 GiB of them, and not where these do not fit the memory that is left.
_ROWS_INSIDE = 10_000
_MAX_STORED_WEIGHTS = 1 << 28


class _Mix(torch.autograd.Function):
    """``sc + (c0 + alpha * c1) * conv`` with ``c0 = (1 - m) / sqrt(n)``, ``c1 = m / n`` (reference
    points_convolution.py:110-113 with the division by sqrt(num_neighbors) moved behind lin2 and alpha): one kernel
    forward and one backward in fp32, elementwise operations elsewhere.  Under ``create_graph`` the backward pass is
    written in differentiable elementwise operations, so it can itself be differentiated."""

    @staticmethod
    def forward(ctx, sc, alpha, conv, c0, c1):
        ctx.save_for_backward(alpha, conv, c0, c1)
        if not _mix_in_one_kernel(sc, alpha, conv, c0, c1):
            return torch.addcmul(sc, torch.addcmul(c0, alpha, c1), conv)
        out = torch.empty_like(sc)
        with _lib.on_device(sc.device):
            _lib.check(_lib.lib().e3x_mix_forward(*(_lib.ptr(t) for t in (sc, alpha, conv, c0, c1, out)), *sc.shape, _lib.stream_ptr(sc.device)))
        return out

    @staticmethod
    def backward(ctx, g):
        alpha, conv, c0, c1 = ctx.saved_tensors
        need_sc, need_alpha, need_conv = ctx.needs_input_grad[:3]
        g_rows = g.contiguous()
        if not torch.is_grad_enabled() and _mix_in_one_kernel(g_rows, alpha, conv, c0, c1):
            g_alpha = torch.empty_like(alpha) if need_alpha else None
            g_conv = torch.empty_like(conv) if need_conv else None
            with _lib.on_device(g.device):
                _lib.check(_lib.lib().e3x_mix_backward(*(_lib.ptr(t) for t in (g_rows, alpha, conv, c0, c1, g_alpha, g_conv)), *conv.shape, _lib.stream_ptr(g.device)))
            return (g if need_sc else None), g_alpha, g_conv, None, None
        return _mix_gradients(ctx.saved_tensors, g, ctx.needs_input_grad)


def _mix_gradients(saved, g, needs):
    """Differentiable gradients of the mixing."""
    alpha, conv, c0, c1 = saved
    g_alpha = (g * conv * c1).sum(-1, keepdim=True) if needs[1] else None
    g_conv = g * torch.addcmul(c0, alpha, c1) if needs[2] else None
    return (g if needs[0] else None), g_alpha, g_conv, None, None


def _mix(sc, alpha, conv, c0, c1):
    out = _lib.native().mix(sc, alpha, conv, c0, c1)
    return _Mix.apply(sc, alpha, conv, c0, c1) if out is None else out


def _mix_in_one_kernel(rows, alpha, conv, c0, c1):
    return (
        rows.is_cuda and rows.dim() == 2 and rows.shape == conv.shape and alpha.shape == (rows.shape[0], 1)
        and c0.shape == c1.shape == rows.shape[1:]
        and all(t.dtype == torch.float32 and t.is_contiguous() and t.device == rows.device for t in (rows, alpha, conv, c0, c1))
    )  # fmt: skip


def _lin2_alpha_gradients(lin2, head, saved, g_conv, g_alpha, need):
    """Differentiable gradients of ``lin2`` and ``alpha``: the two products' own."""
    features, attr, w_lin2, w_alpha = saved[:4]
    k = head.irreps_in1.dim
    gf, _, gw_lin2 = _slot_backward(_TpSlot, _OUT, (features, attr, w_lin2), g_conv.contiguous(), (need[0], False, need[2]), lin2)
    gs, _, gw_alpha = _slot_backward(_TpSlot, _OUT, (features[:, :k].contiguous(), attr, w_alpha), g_alpha.contiguous(), (need[0], False, need[3]), head)
    if need[0]:
        gf = gf + torch.nn.functional.pad(gs, (0, features.shape[1] - k))
    return gf, None, gw_lin2, gw_alpha


_lib.connect({"mix_gradients": _mix_gradients, "lin2_alpha_gradients": _lin2_alpha_gradients})


def _lin2_alpha(features, attr, w_lin2, w_alpha, lin2, alpha, head):
    in_place = head._plan(features.dtype).family == "uvw_node" and features.shape[1] % 4 == 0
    reads = alpha if in_place else head
    packs = [(tp._plans.get("native") or tp._native_plans())[0] for tp in (lin2, reads, head)]
    if None not in packs:
        out = _lib.native().lin2_alpha(*packs, lin2, reads, head, alpha, head.irreps_in1.dim, in_place, features, attr, w_lin2, w_alpha)
        if out is not None:
            return out
    return _Lin2Alpha.apply(features, attr, w_lin2, w_alpha, lin2, alpha, head)


class _Lin2Alpha(torch.autograd.Function):
    """``lin2(features, attr)`` and ``alpha(features, attr)`` as one node of the autograd graph.  ``alpha`` reads only
    the leading scalars of the features (``head`` is ``alpha`` restricted to them, same weights), so its input gradient
    is added into the leading columns of lin2's instead of being written as a second zero-padded [N, features] array
    that autograd then adds to the first: three passes over an array as wide as the messages saved."""

    @staticmethod
    def forward(ctx, features, attr, w_lin2, w_alpha, lin2, alpha, head):
        dt = features.dtype
        # the node-wise kernels read the scalars where they lie; the vector-ALU kernel stages whole rows, and takes a copy
        in_place = head._plan(dt).family == "uvw_node" and features.shape[1] % 4 == 0
        scalars, ctx.reads_scalars = (features, alpha) if in_place else (features[:, : head.irreps_in1.dim].contiguous(), head)
        ctx.lin2, ctx.head = lin2, head
        ctx.save_for_backward(features, attr, w_lin2, w_alpha, scalars)
        return lin2._plan(dt).forward(features, attr, w_lin2), ctx.reads_scalars._plan(dt).forward(scalars, attr, w_alpha)

    @staticmethod
    def backward(ctx, g_conv, g_alpha):
        lin2, head = ctx.lin2, ctx.head
        features, attr, w_lin2, w_alpha, scalars = ctx.saved_tensors
        k = head.irreps_in1.dim
        g_conv, g_alpha = g_conv.contiguous(), g_alpha.contiguous()
        if torch.is_grad_enabled():
            return (*_lin2_alpha_gradients(lin2, head, ctx.saved_tensors, g_conv, g_alpha, ctx.needs_input_grad), None, None, None)
        dt = features.dtype
        g_features = gw_lin2 = gw_alpha = None
        if ctx.needs_input_grad[2]:
            gw_lin2 = lin2._plan(dt).backward_w_uvw(features, attr, g_conv, True)
        if ctx.needs_input_grad[3]:
            gw_alpha = ctx.reads_scalars._plan(dt).backward_w_uvw(scalars, attr, g_alpha, True)
        if ctx.needs_input_grad[0]:
            g_features = lin2._grad_plan("x1", dt).forward(g_conv, attr, _permuted_weights(lin2, w_lin2, (2, 1, 0)))
            g_scalars = head._grad_plan("x1", dt).forward(g_alpha, attr, _permuted_weights(head, w_alpha, (2, 1, 0)))
            g_features[:, :k] += g_scalars
        return g_features, None, gw_lin2, gw_alpha, None, None, None


class Convolution(torch.nn.Module):
    r"""Same constructor and ``forward`` arguments as the reference; ``forward`` also accepts a prebuilt
    ``edges=DstSortedEdges(...)`` so that the destination sort is paid once per graph instead of once per layer."""

    def __init__(
        self, irreps_node_input, irreps_node_attr, irreps_edge_attr, irreps_node_output, fc_neurons, num_neighbors
    ) -> None:
        super().__init__()
        self.irreps_node_input, self.irreps_node_attr = Irreps(irreps_node_input), Irreps(irreps_node_attr)
        self.irreps_edge_attr, self.irreps_node_output = Irreps(irreps_edge_attr), Irreps(irreps_node_output)
        self.num_neighbors = num_neighbors

        def node_wise(features, out):  # features (x) node attributes -> out, shared weights
            return FullyConnectedTensorProduct(features, self.irreps_node_attr, out)

        # messages carry every irrep the output asks for, plus scalars for the per-node mixing coefficient `alpha`
        wanted = {ir for _, ir in self.irreps_node_output} | {Irrep(0, 1)}
        irreps_mid, instructions = message_instructions(self.irreps_node_input, self.irreps_edge_attr, wanted)
        if irreps_mid.dim == 0:
            raise AssertionError(
                f"no product of an input irrep ({self.irreps_node_input}) with an edge irrep ({self.irreps_edge_attr}) "
                f"lies in the output irreps ({self.irreps_node_output}): there is no message to send"
            )
        # submodules in the reference's registration order (state_dict keys and the random stream of the initial weights)
        self.sc = node_wise(self.irreps_node_input, self.irreps_node_output)
        self.lin1 = node_wise(self.irreps_node_input, self.irreps_node_input)
        message = TensorProduct(
            self.irreps_node_input, self.irreps_edge_attr, irreps_mid, instructions, internal_weights=False, shared_weights=False
        )
        self.fc = FullyConnectedNet([*fc_neurons, message.weight_numel], torch.nn.functional.silu)
        self.tp = message
        self.lin2 = node_wise(irreps_mid, self.irreps_node_output)
        self.alpha = node_wise(irreps_mid, "0e")
        torch.nn.init.zeros_(self.alpha.weight)  # the block starts as its self-connection
        if self.alpha.output_mask[0] != 1.0:
            raise AssertionError(f"the messages ({irreps_mid}) and the node attributes ({self.irreps_node_attr}) cannot produce a scalar for alpha")
        # alpha restricted to the leading irreps of the messages when those are all it reads (scalar node attributes and
        # sorted messages: always): same instructions, weights and normalisation; kept out of the module tree, it has
        # no parameters and must not add keys to the state_dict
        self.__dict__["_alpha_head"] = None
        n_head = 1 + max(ins.i_in1 for ins in self.alpha.instructions)
        if irreps_mid[:n_head].dim % 4 == 0 and n_head < len(irreps_mid):
            head = FullyConnectedTensorProduct(irreps_mid[:n_head], self.irreps_node_attr, "0e", internal_weights=False, shared_weights=True)
            key = lambda tp: [(i.i_in1, i.i_in2, i.i_out, i.path_shape, i.path_weight) for i in tp.instructions]  # noqa: E731
            if key(head) == key(self.alpha) and head.weight_numel == self.alpha.weight_numel:
                self.__dict__["_alpha_head"] = head

    def forward(self, node_input, node_attr, edge_src, edge_dst, edge_attr, edge_scalars, edges=None) -> torch.Tensor:
        node_self_connection = self.sc(node_input, node_attr)
        node_features = self.lin1(node_input, node_attr)
        if edges is None:
            edges = DstSortedEdges(edge_src, edge_dst, node_input.shape[0])
        messages = None
        wants_grad = torch.is_grad_enabled() and (
            any(t.requires_grad for t in (node_features, edge_attr, edge_scalars)) or any(p.requires_grad for p in self.fc.parameters())
        )
        if not wants_grad and (edges.num_nodes >= _ROWS_INSIDE or edges.num_edges * self.tp.weight_numel > _MAX_STORED_WEIGHTS):
            # the radial network inside the message kernel: the [E, weight_numel] weights are never stored
            messages = self.tp.forward_gather_scatter_radial(node_features, edge_attr, edge_scalars, self.fc, edges)
        if messages is None:
            try:
                weight = self.fc(edge_scalars)
            except torch.OutOfMemoryError:
                # the weights of all edges do not fit the memory that is left: once more without storing them
                messages = None if wants_grad else self.tp.forward_gather_scatter_radial(node_features, edge_attr, edge_scalars, self.fc, edges)
                if messages is None:
                    raise
            else:
                messages = self.tp.forward_gather_scatter(node_features, edge_attr, weight, edges=edges)
        node_features = messages
        # lin2 and alpha are linear in the features, so the division by sqrt(num_neighbors) that the reference applies
        # to the summed messages (points_convolution.py:108) is applied to their outputs instead, which are four to a
        # thousand times narrower than the messages
        inv = 1.0 / self.num_neighbors**0.5
        if (
            self._alpha_head is not None
            and torch.is_grad_enabled()
            and node_features.requires_grad
            and not node_attr.requires_grad
            and node_features.dim() == 2
            and node_attr.shape[:-1] == node_features.shape[:-1]
            and node_features.dtype == torch.float32
        ):
            node_conv_out, alpha = _lin2_alpha(
                node_features.contiguous(), node_attr.to(node_features.dtype).contiguous(), self.lin2.weight, self.alpha.weight,
                self.lin2, self.alpha, self._alpha_head,
            )  # fmt: skip
        else:
            node_conv_out = self.lin2(node_features, node_attr)
            alpha = self.alpha(node_features, node_attr)
        m = self.sc.output_mask
        key = (m.device, m.dtype, m._version, inv)
        if self.__dict__.get("_mix_key") != key:  # the two constant rows of the mixing, once per device
            self.__dict__["_mix_key"], self.__dict__["_mix_rows"] = key, ((1 - m) * inv, m * (inv * inv))
        c0, c1 = self.__dict__["_mix_rows"]
        return _mix(node_self_connection, alpha, node_conv_out, c0, c1)
