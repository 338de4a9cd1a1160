"""GPU parity of the backward pass: gradients from the HIP kernels against torch autograd (float64) through the
CPU restatement of the reference's einsum graph (oracle/torch_cpu.py)."""
import numpy as np
import pytest
import torch

from e3nn_amd._lib import E3xError
from e3nn_amd.nn import DstSortedEdges
from oracle.torch_cpu import tp_forward_torch, tp_gather_scatter_torch
from tests import kernel_sets as ks
from tests.helpers import assert_close, oracle_spec, seeded

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _oracle_grads(fn, tensors, cot):
    ts = [t.double().clone().requires_grad_(True) for t in tensors]
    out = fn(*ts)
    out.backward(cot.double())
    return out.detach(), [t.grad for t in ts]


@pytest.mark.parametrize("maker,Z", [
    (lambda: ks.golden_tp("uvu_merged_cfg3_like_mul4"), 9), (lambda: ks.golden_tp("uvu_builderA_cfg4_like_mul2"), 7),
    (lambda: ks.cfg3(True), 130), (lambda: ks.cfg3(False), 65), (lambda: ks.cfg4("A"), 17), (ks.odd_mul, 33),
])  # fmt: skip
def test_uvu_plain_gradients(maker, Z):
    tp = maker()
    spec = oracle_spec(tp)
    x1, x2, w = seeded(Z, tp.irreps_in1.dim, seed=1), seeded(Z, tp.irreps_in2.dim, seed=2), seeded(Z, tp.weight_numel, seed=3)
    cot = seeded(Z, tp.irreps_out.dim, seed=4)
    ref_out, (r1, r2, rw) = _oracle_grads(lambda a, b, c: tp_forward_torch(spec, a, b, c), (x1, x2, w), cot)
    a, b, c = (t.to(DEV).requires_grad_(True) for t in (x1, x2, w))
    out = tp(a, b, c)
    # the weight gradient is written without a zero fill: hand the allocator a NaN-filled block of its size first,
    # so that an element the kernel skipped would show
    junk = torch.full((Z, tp.weight_numel), float("nan"), device=DEV)
    del junk
    out.backward(cot.to(DEV))
    # per-sample contractions: the benchmark's tolerance for contractions, |err| <= 1e-4 + 1e-5 |ref|
    assert_close(out, ref_out.numpy())
    assert_close(a.grad, r1.numpy(), what="d/dx1")
    assert_close(b.grad, r2.numpy(), what="d/dx2")
    assert_close(c.grad, rw.numpy(), what="d/dw")


@pytest.mark.parametrize("maker,N,E,idx", [(lambda: ks.cfg3(True), 120, 3000, torch.int64), (lambda: ks.cfg3(False), 50, 900, torch.int32),
                                           (lambda: ks.cfg4("A"), 25, 300, torch.int32),
                                           # multiplicities that leave lane groups partly filled (80, 24, 5): every
                                           # weight-gradient column must still be written (the buffer is not zero-filled)
                                           (ks.odd_mul, 40, 600, torch.int32), (ks.narrow_message, 60, 900, torch.int64),
                                           # groups of four lanes, and of eight with some of them idle
                                           (ks.message_ragged_groups, 30, 700, torch.int64), (ks.message_four_lanes, 30, 700, torch.int32)])  # fmt: skip
def test_fused_message_gradients(maker, N, E, idx):
    tp = maker()
    spec = oracle_spec(tp)
    g = torch.Generator().manual_seed(7)
    src, dst = torch.randint(0, N, (E,), generator=g), torch.randint(0, N - 2, (E,), generator=g)
    node_x, attr, w = seeded(N, tp.irreps_in1.dim, seed=1), seeded(E, tp.irreps_in2.dim, seed=2), seeded(E, tp.weight_numel, seed=3)
    cot = seeded(N, tp.irreps_out.dim, seed=4)
    ref_out, (r1, r2, rw) = _oracle_grads(lambda a, b, c: tp_gather_scatter_torch(spec, a, b, c, src, dst, N), (node_x, attr, w), cot)
    a, b, c = (t.to(DEV).requires_grad_(True) for t in (node_x, attr, w))
    edges = DstSortedEdges(src.to(idx).to(DEV), dst.to(idx).to(DEV), N)
    out = tp.forward_gather_scatter(a, b, c, edges=edges)
    junk = torch.full((E, tp.weight_numel), float("nan"), device=DEV)  # see test_uvu_plain_gradients
    del junk
    out.backward(cot.to(DEV))
    scale = lambda r: max(1.0, float(r.abs().max()))  # noqa: E731
    assert_close(out, ref_out.numpy(), atol=1e-4 * scale(ref_out))
    assert_close(a.grad, r1.numpy(), atol=1e-4 * scale(r1), what="d/dnode_x")
    # sums over the edges of a node are held to a tolerance scaled by their size (the order of summation differs
    # from scatter_add_), per-edge contractions to the benchmark's 1e-4 + 1e-5 |ref|
    assert_close(b.grad, r2.numpy(), what="d/dedge_attr")
    assert_close(c.grad, rw.numpy(), what="d/dweight")
    # only some inputs require a gradient
    a2, c2 = node_x.to(DEV).requires_grad_(True), w.to(DEV)
    tp.forward_gather_scatter(a2, attr.to(DEV), c2, edges=edges).backward(cot.to(DEV))
    # (another kernel than above where one kernel writes every gradient: the lane groups of a wavefront are combined
    # in another order, so the last bits may differ)
    assert_close(a2.grad, a.grad.cpu().numpy(), atol=1e-5 * scale(r1), what="d/dnode_x alone")
    # node features and weights but not the edge attributes (training without forces): one kernel on the transposed
    # plan writes both gradients where the instruction set fits it (a lane group owning a whole row)
    a4, c4 = node_x.to(DEV).requires_grad_(True), w.to(DEV).requires_grad_(True)
    tp.forward_gather_scatter(a4, attr.to(DEV), c4, edges=edges).backward(cot.to(DEV))
    assert_close(a4.grad, r1.numpy(), atol=1e-4 * scale(r1), what="d/dnode_x, one backward kernel")
    assert_close(c4.grad, rw.numpy(), what="d/dweight, one backward kernel")
    # negative source indices wrap in the gather; the gradient scatters onto the wrapped rows
    neg = torch.where(torch.arange(E) % 3 == 0, src - N, src)
    a3 = node_x.to(DEV).requires_grad_(True)
    tp.forward_gather_scatter(a3, attr.to(DEV), c2, edges=DstSortedEdges(neg.to(idx).to(DEV), dst.to(idx).to(DEV), N)).backward(cot.to(DEV))
    assert torch.equal(a3.grad, a2.grad)
    a5, c5 = node_x.to(DEV).requires_grad_(True), w.to(DEV).requires_grad_(True)
    tp.forward_gather_scatter(a5, attr.to(DEV), c5, edges=DstSortedEdges(neg.to(idx).to(DEV), dst.to(idx).to(DEV), N)).backward(cot.to(DEV))
    assert torch.equal(a5.grad, a4.grad) and torch.equal(c5.grad, c4.grad)


@pytest.mark.parametrize("maker", [lambda: ks.cfg4("A"), ks.ragged_wide_message])
@pytest.mark.parametrize("degrees,idx,grouped", [([0, 1, 63, 64, 65, 0, 130, 2], torch.int64, True), ([3, 0, 0, 129], torch.int32, False), ([1], torch.int64, True),
                                                # rows around one, two and three pieces of 128 edges
                                                ([129, 0, 127, 300, 128, 0], torch.int32, True), ([5, 257, 0, 400], torch.int64, False)])
def test_message_gradients_grouped_by_destination(maker, degrees, idx, grouped):
    # messages much wider than the node features: rows without edges, one edge, around the blocks of 64 edges, an odd
    # and an even number of them; sources without edges get exact zeros
    tp = maker()
    spec = oracle_spec(tp)
    N, E, n_src = len(degrees), sum(degrees), 9
    dst = torch.repeat_interleave(torch.arange(N), torch.tensor(degrees))
    src = torch.randint(1, n_src, (E,), generator=torch.Generator().manual_seed(3))
    if not grouped:
        dst = dst[torch.randperm(E, generator=torch.Generator().manual_seed(4))]
    node_x, attr, w = seeded(n_src, tp.irreps_in1.dim, seed=1), seeded(E, tp.irreps_in2.dim, seed=2), seeded(E, tp.weight_numel, seed=3)
    cot = seeded(N, tp.irreps_out.dim, seed=4)
    _, (r1, r2, rw) = _oracle_grads(lambda a, b, c: tp_gather_scatter_torch(spec, a, b, c, src, dst, N), (node_x, attr, w), cot)
    edges = DstSortedEdges(src.to(idx).to(DEV), dst.to(idx).to(DEV), N, n_src)
    plan = tp._plan(torch.float32)
    x, a, ww, g = (t.to(DEV) for t in (node_x, attr, w, cot))
    for want_x2 in (True, False):
        junk = torch.full((E, tp.weight_numel), float("nan"), device=DEV)  # see test_uvu_plain_gradients
        del junk
        gx, gw, gx2 = plan.message_backward(x, a, ww, g, edges, want_x2)
        assert_close(gw, rw.numpy(), what="d/dweight")
        # sums of at most E rows: 24-bit products, one rounding per addition
        assert_close(gx, r1.numpy(), atol=1e-5 * max(1.0, float(r1.abs().max())), what="d/dnode_x")
        assert not gx[0].any()
        assert (gx2 is not None) == want_x2
        if want_x2:
            # 64 x 64-channel sums of products of four N(0, 1) factors per path
            assert_close(gx2, r2.numpy(), atol=1e-5 * max(1.0, float(r2.abs().max())), what="d/dedge_attr")
        again = plan.message_backward(x, a, ww, g, edges, want_x2)
        assert torch.equal(again[0], gx) and torch.equal(again[1], gw)


@pytest.mark.parametrize("maker,one_kernel", [(lambda: ks.cfg3(True), True), (lambda: ks.cfg3(False), True), (ks.narrow_message, True), (ks.odd_mul, False),
                                              (ks.message_ragged_groups, True), (ks.message_four_lanes, True),
                                              (lambda: ks.cfg4("A"), False), (ks.ragged_wide_message, False)])  # fmt: skip
@pytest.mark.parametrize("degrees,grouped", [([0, 1, 63, 64, 65, 0, 130, 2], True), ([300, 0, 7], False)])
def test_message_gradients_in_bf16_storage(maker, one_kernel, degrees, grouped):
    # one kernel for every gradient, grouped by source or by destination: against float64 on the same (rounded) inputs, with
    # one rounding to bf16 (8 significant bits: 2^-8 of the value at most) and 1e-5 of the largest entry for the sums in fp32
    tp = maker()
    spec = oracle_spec(tp)
    bf, N, E, n_src = torch.bfloat16, len(degrees), sum(degrees), 9
    dst = torch.repeat_interleave(torch.arange(N), torch.tensor(degrees))
    src = torch.randint(1, n_src, (E,), generator=torch.Generator().manual_seed(3))
    if not grouped:
        dst = dst[torch.randperm(E, generator=torch.Generator().manual_seed(4))]
    node_x, attr, w = seeded(n_src, tp.irreps_in1.dim, seed=1).to(bf), seeded(E, tp.irreps_in2.dim, seed=2).to(bf), seeded(E, tp.weight_numel, seed=3).to(bf)
    cot = seeded(N, tp.irreps_out.dim, seed=4).to(bf)
    ref, grads = _oracle_grads(lambda a, b, c: tp_gather_scatter_torch(spec, a, b, c, src, dst, N), (node_x, attr, w), cot)

    def close(got, want, what):
        assert got.dtype == bf
        err = (got.double().cpu() - want).abs() - 2**-8 * want.abs()
        assert float(err.max()) <= 1e-5 * max(1.0, float(want.abs().max())), what

    edges = DstSortedEdges(src.to(DEV), dst.to(DEV), N, n_src)
    for with_attr in (False, True):
        a, b, c = (t.to(DEV).requires_grad_(r) for t, r in ((node_x, True), (attr, with_attr), (w, True)))
        out = tp.forward_gather_scatter(a, b, c, edges=edges)
        junk = torch.full((E, tp.weight_numel), float("nan"), device=DEV, dtype=bf)  # see test_uvu_plain_gradients
        del junk
        if with_attr and not one_kernel:  # (shares of several kernels would be rounded one by one)
            with pytest.raises(E3xError, match="single-kernel plan"):
                out.backward(cot.to(DEV))
            continue
        out.backward(cot.to(DEV))
        if one_kernel:  # (the matrix-core forward kernel rounds its operands too, and has a test of its own)
            close(out.detach(), ref, "out")
        for got, want, what in zip((a.grad, b.grad, c.grad), grads, ("d/dnode_x", "d/dedge_attr", "d/dweight")):
            if got is not None:
                close(got, want, what)
        assert not a.grad[0].any()  # a source without edges


@pytest.mark.parametrize("maker,Z", [(ks.mfma_full_tiles, 1), (ks.mfma_full_tiles, 31), (ks.mfma_full_tiles, 33), (ks.mfma_full_tiles, 400), (ks.node_block, 65)])
@pytest.mark.parametrize("ramp", [0, 6, -6])
def test_uvw_weight_gradient_on_split_operands(maker, Z, ramp):
    # edges of the chunks of 32 rows; scales that grow along the batch and that fall
    tp = maker()
    spec = oracle_spec(tp)
    scale = torch.logspace(-ramp / 2, ramp / 2, Z)[:, None]
    x1, x2, g = seeded(Z, tp.irreps_in1.dim, seed=1) * scale, seeded(Z, tp.irreps_in2.dim, seed=2), seeded(Z, tp.irreps_out.dim, seed=3) * 1e-20
    w = torch.zeros(tp.weight_numel, dtype=torch.float64, requires_grad=True)
    (ref,) = torch.autograd.grad(tp_forward_torch(spec, x1.double(), x2.double(), w), (w,), g.double())
    plan = tp._plan(torch.float32)
    got = plan.backward_w_uvw(x1.to(DEV), x2.to(DEV), g.to(DEV), True)
    assert "split operands" in plan.arithmetic_weight_gradient
    # sums of at most 400 x 25 products: 6e-7 of the 2-norm from fp32 accumulation, 6e-9 of a term from the pieces
    assert float((got.double().cpu() - ref).norm() / ref.norm()) < 1e-6
    # an infinity spoils the gradients that it enters, and only these
    if tp.irreps_in1.dim == tp.irreps_in1[0].dim + tp.irreps_in1[1].dim and Z > 1:
        x1[0, 0] = float("inf")
        bad = plan.backward_w_uvw(x1.to(DEV), x2.to(DEV), g.to(DEV), True)
        per_u = torch.isfinite(bad).cpu()
        t = tp.instructions[0]
        block = per_u[: t.path_shape[0] * t.path_shape[1] * t.path_shape[2]].view(t.path_shape)
        assert t.i_in1 == 0 and not block[0].any() and block[1:].all()


@pytest.mark.parametrize("Z", [1, 15, 16, 17, 49, 97, 800])
def test_uvw_weight_gradient_of_wide_blocks(Z):
    # stages of 16 rows and their remainders; one batch slice per path (stored) and several (added); every role of the factors
    tp = ks.mfma_wide_blocks()
    spec = oracle_spec(tp)
    x1, x2, g = seeded(Z, tp.irreps_in1.dim, seed=1), seeded(Z, tp.irreps_in2.dim, seed=2), seeded(Z, tp.irreps_out.dim, seed=3)
    w = torch.zeros(tp.weight_numel, dtype=torch.float64, requires_grad=True)
    (ref,) = torch.autograd.grad(tp_forward_torch(spec, x1.double(), x2.double(), w), (w,), g.double())
    got = tp._plan(torch.float32).backward_w_uvw(x1.to(DEV), x2.to(DEV), g.to(DEV), True).double().cpu()
    # sums of at most 800 x 25 products in fp32, as above; block by block, so that no path is lost among the others
    offset = 0
    for t in tp.instructions:
        n = t.path_shape[0] * t.path_shape[1] * t.path_shape[2]
        a, b = got[offset : offset + n], ref[offset : offset + n]
        assert float((a - b).norm() / b.norm()) < 1e-6, t
        offset += n


@pytest.mark.parametrize("maker", [ks.mfma_small, ks.mfma_full_tiles, ks.mfma_wide_blocks, ks.few_outer_indices, ks.unaligned_offsets])
@pytest.mark.parametrize("Z", [1, 17, 33, 400])
def test_uvw_weight_gradient_of_bf16_values(maker, Z):
    # three products in place of six, of the same pieces: the bound of fp32 rows holds, path by path
    tp = maker()
    spec = oracle_spec(tp)
    x1, x2, g = (seeded(Z, d, seed=i).bfloat16().float() for i, d in enumerate((tp.irreps_in1.dim, tp.irreps_in2.dim, tp.irreps_out.dim)))
    w = torch.zeros(tp.weight_numel, dtype=torch.float64, requires_grad=True)
    (ref,) = torch.autograd.grad(tp_forward_torch(spec, x1.double(), x2.double(), w), (w,), g.double())
    got = tp._plan(torch.float32).backward_w_uvw(x1.to(DEV), x2.to(DEV), g.to(DEV), True, True).double().cpu()
    offset = 0
    for t in tp.instructions:
        n = t.path_shape[0] * t.path_shape[1] * t.path_shape[2]
        a, b = got[offset : offset + n], ref[offset : offset + n]
        assert float((a - b).norm() / b.norm()) < 1e-6, t
        offset += n


@pytest.mark.parametrize("Z", [129, 50_003, 400_003])
def test_uvw_weight_gradient_of_few_wide_tiles(Z):
    # 16 tiles for 512 workgroups: how many rows go into one sum decides the error
    tp = ks.dense_one_path().to(DEV)
    x1, x2, g = (seeded(Z, 64, seed=i).to(DEV) for i in (1, 2, 3))
    got = tp._plan(torch.float32).backward_w_uvw(x1, x2, g, True).double()
    ref = torch.zeros(64 * 64, 64, dtype=torch.float64, device=DEV)
    for z in range(0, Z, 8192):
        a, b, c = (x[z : z + 8192].double() for x in (x1, x2, g))
        ref += (a[:, :, None] * b[:, None, :]).flatten(1).T @ c
    ref = tp.instructions[0].path_weight * ref.flatten()
    # at most 3200 rows a sum, six products for every 16 of them: a random walk of 1200 roundings of 2^-24 / sqrt(3), the same
    # share of every slice
    assert float((got - ref).norm() / ref.norm()) < 1200**0.5 * 2.0**-24 / 3**0.5


@pytest.mark.parametrize("maker", [ks.node_block, ks.node_narrow, ks.node_wide_out, ks.node_many_species, ks.radial_layer, ks.node_onto_scalars])
@pytest.mark.parametrize("Z", [1, 16, 17, 63, 65, 2500])
def test_uvw_weight_gradient_of_node_wise_layers(maker, Z):
    # stages of 16 rows and their remainders, one slice and several; tiles of both indices that are not full
    tp = maker()
    spec = oracle_spec(tp)
    x1, x2, g = seeded(Z, tp.irreps_in1.dim, seed=1), seeded(Z, tp.irreps_in2.dim, seed=2), seeded(Z, tp.irreps_out.dim, seed=3)
    w = torch.zeros(tp.weight_numel, dtype=torch.float64, requires_grad=True)
    (ref,) = torch.autograd.grad(tp_forward_torch(spec, x1.double(), x2.double(), w), (w,), g.double())
    got = tp._plan(torch.float32).backward_w_uvw(x1.to(DEV), x2.to(DEV), g.to(DEV), True).double().cpu()
    # sums of at most 2500 x 7 products in fp32: a random walk of some hundred roundings of 6e-8 / sqrt(3)
    assert float((got - ref).norm() / ref.norm()) < 1e-6


@pytest.mark.parametrize("Z", [16_384, 16_385, 50_003])
def test_uvw_weight_gradient_onto_scalars_of_many_rows(Z):
    # beyond 128 rows a workgroup: several trips of 128 rows in each, the last one ragged (50 003 rows: 391 a workgroup)
    tp = ks.node_onto_scalars()
    x1, x2, g = seeded(Z, tp.irreps_in1.dim, seed=1), seeded(Z, tp.irreps_in2.dim, seed=2), seeded(Z, tp.irreps_out.dim, seed=3)
    w = torch.zeros(tp.weight_numel, dtype=torch.float64, requires_grad=True)
    (ref,) = torch.autograd.grad(tp_forward_torch(oracle_spec(tp), x1.double(), x2.double(), w), (w,), g.double())
    got = tp._plan(torch.float32).backward_w_uvw(x1.to(DEV), x2.to(DEV), g.to(DEV), True).double().cpu()
    # a lane adds up at most 16 rows, 32 lanes and 128 workgroups one after the other: a random walk of 176 roundings of
    # 2^-24 / sqrt(3) of sums that are two thirds of the whole on average
    assert float((got - ref).norm() / ref.norm()) < 176**0.5 * 2.0**-24 / 3**0.5


@pytest.mark.parametrize("Z", [1, 31, 65, 129, 16_385])
def test_uvw_weight_gradient_of_long_rows_onto_a_scalar(Z):
    # two rows of 960 numbers in flight a half-wave, trips of 64 rows a workgroup
    tp = ks.node_long_row()
    x1, x2, g = (seeded(Z, n, seed=i) for i, n in ((1, 960), (2, 1), (3, 1)))
    ref = tp.instructions[0].path_weight * ((x2 * g).double().T @ x1.double()).flatten()
    got = tp._plan(torch.float32).backward_w_uvw(x1.to(DEV), x2.to(DEV), g.to(DEV), True).double().cpu()
    # the bound of the sets above (fewer rows a lane here), and two roundings of every product
    assert float((got - ref).norm() / ref.norm()) < (176**0.5 + 2) * 2.0**-24 / 3**0.5


@pytest.mark.parametrize("first", [True, False])
def test_uvw_weight_gradient_of_a_path_with_weight_zero(first):
    # its weights have no part in the output, whatever the path beside it does: zeros exactly, also where rows are not finite
    tp = ks.zero_path(first)
    spec = oracle_spec(tp, [0.0, 1.0] if first else [1.0, 0.0])
    Z = 300
    x1, x2, g = seeded(Z, 64, seed=1), seeded(Z, 4, seed=2), seeded(Z, 2, seed=3)
    w = torch.zeros(tp.weight_numel, dtype=torch.float64, requires_grad=True)
    (ref,) = torch.autograd.grad(tp_forward_torch(spec, x1.double(), x2.double(), w), (w,), g.double())
    dead, alive = (slice(0, 256), slice(256, 512)) if first else (slice(256, 512), slice(0, 256))
    x1[7, 3 if first else 40] = float("inf")
    got = tp._plan(torch.float32).backward_w_uvw(x1.to(DEV), x2.to(DEV), g.to(DEV), True).double().cpu()
    assert not got[dead].any() and ref[alive].all()
    assert float((got - ref)[alive].norm() / ref[alive].norm()) < 1e-6


@pytest.mark.parametrize("maker", [ks.node_ragged, ks.node_narrow, ks.node_partial_tile])
def test_uvw_weight_gradient_of_ragged_node_wise_layers_is_as_exact_as_fp32(maker):
    # multiplicities that are no multiples of 32, which the fp32 vector ALU sums with an error of 1.6e-7 at 1000 rows.  A slice
    # of some 170 rows and components is 11 matrix steps, each cut by 2^-24 / sqrt(3) of a partial sum (two thirds of the
    # whole on average), 0.8e-7; up to 30 slices are added with roundings of 2^-24 / sqrt(12), 0.6e-7; the product of the
    # second input and g is rounded, 0.2e-7, and the operands' pieces end at 2^-25 of them, 0.4e-7: 1.1e-7 in all
    tp = maker()
    spec = oracle_spec(tp)
    Z = 1000
    x1, x2, g = seeded(Z, tp.irreps_in1.dim, seed=1), seeded(Z, tp.irreps_in2.dim, seed=2), seeded(Z, tp.irreps_out.dim, seed=3)
    w = torch.zeros(tp.weight_numel, dtype=torch.float64, requires_grad=True)
    (ref,) = torch.autograd.grad(tp_forward_torch(spec, x1.double(), x2.double(), w), (w,), g.double())
    got = tp._plan(torch.float32).backward_w_uvw(x1.to(DEV), x2.to(DEV), g.to(DEV), True).double().cpu()
    assert float((got - ref).norm() / ref.norm()) < 1.6e-7


@pytest.mark.parametrize("maker", [ks.mfma_full_tiles, ks.node_block])
@pytest.mark.parametrize("sizes", ["x1 against x2", "x1 against g", "x2 against g", "masked row", "largest number", "channels"])
def test_uvw_weight_gradient_of_numbers_of_different_sizes(maker, sizes):
    # the sum runs over the rows: factors of very different sizes whose products are of one size, rows that contribute
    # nothing beside large entries, channels of different sizes.  Powers of two, so that the scales are exact.
    tp = maker()
    spec = oracle_spec(tp)
    Z = 300
    x1, x2, g = seeded(Z, tp.irreps_in1.dim, seed=1), seeded(Z, tp.irreps_in2.dim, seed=2), seeded(Z, tp.irreps_out.dim, seed=3)
    scale = [torch.ones(t.path_shape) for t in tp.instructions]
    if "against" in sizes:
        s = 2.0 ** torch.randint(-40, 41, (Z, 1), generator=torch.Generator().manual_seed(4))
        factors = {"x1": x1, "x2": x2, "g": g}
        up, down = sizes.split(" against ")
        factors[up].mul_(s), factors[down].div_(s)
    if sizes == "masked row":
        x1[7] *= 2.0**33
        g[7] = 0
        x2[150] *= 2.0**40
        x1[150] = 0
    if sizes == "largest number":
        x1[5] *= 2.0**-100
        x2[5, 0] = 2e38
        g[5] *= 0.1
    if sizes == "channels":
        def spread(x, irreps):
            per_mul = [2.0 ** -torch.linspace(0, 27, m.mul).round() for m in irreps]
            x.mul_(torch.cat([v.repeat_interleave(m.ir.dim) for v, m in zip(per_mul, irreps)]))
            return per_mul
        of1, ofo = spread(x1, tp.irreps_in1), spread(g, tp.irreps_out)
        scale = [of1[t.i_in1][:, None, None] * ofo[t.i_out] * torch.ones(t.path_shape) for t in tp.instructions]
    w = torch.zeros(tp.weight_numel, dtype=torch.float64, requires_grad=True)
    (ref,) = torch.autograd.grad(tp_forward_torch(spec, x1.double(), x2.double(), w), (w,), g.double())
    got = tp._plan(torch.float32).backward_w_uvw(x1.to(DEV), x2.to(DEV), g.to(DEV), True)
    scale = torch.cat([s.double().reshape(-1) for s in scale])
    # as above: 1e-6 of the 2-norm, every channel measured in units of its own size
    assert float(((got.double().cpu() - ref) / scale).norm() / (ref / scale).norm()) < 1e-6


@pytest.mark.parametrize("maker,Z", [(lambda: ks.golden_tp("fctp_small_cfg5_like"), 6), (ks.cfg1, 50), (ks.mfma_small, 70),
                                     (lambda: ks.golden_tp("fctp_per_sample_weights"), 5), (ks.node_fctp, 90), (ks.radial_layer, 77), (ks.node_wide_out, 45), (ks.node_narrow, 40)])  # fmt: skip
def test_uvw_input_gradients(maker, Z):
    tp = maker().to(DEV)
    spec = oracle_spec(tp)
    x1, x2 = seeded(Z, tp.irreps_in1.dim, seed=1), seeded(Z, tp.irreps_in2.dim, seed=2)
    w = seeded(*((Z,) if not tp.shared_weights else ()), tp.weight_numel, seed=3) / 4
    cot = seeded(Z, tp.irreps_out.dim, seed=4)
    ref_out, (r1, r2) = _oracle_grads(lambda a, b: tp_forward_torch(spec, a, b, w.double()), (x1, x2), cot)
    a, b = (t.to(DEV).requires_grad_(True) for t in (x1, x2))
    out = tp(a, b, w.to(DEV))
    out.backward(cot.to(DEV))
    assert_close(out, ref_out.numpy())
    assert_close(a.grad, r1.numpy(), what="d/dx1")
    assert_close(b.grad, r2.numpy(), what="d/dx2")


@pytest.mark.parametrize("maker,Z", [(lambda: ks.golden_tp("fctp_small_cfg5_like"), 6), (ks.cfg1, 50), (ks.cfg1, 4099),
                                     (lambda: ks.golden_tp("fctp_per_sample_weights"), 5), (ks.mfma_small, 70),
                                     (ks.mfma_small, 1500), (ks.mfma_full_tiles, 70), (ks.mfma_full_tiles, 1237), (ks.node_fctp, 700), (ks.node_block, 333), (ks.node_block, 20), (ks.outer_split, 410), (ks.radial_layer, 513), (ks.node_wide_out, 300), (ks.node_narrow, 260),
                                     (ks.node_partial_tile, 100), (ks.unaligned_mfma, 300), (ks.unaligned_offsets, 129)])  # fmt: skip
def test_uvw_weight_gradients(maker, Z):
    tp = maker().to(DEV)
    spec = oracle_spec(tp)
    x1, x2 = seeded(Z, tp.irreps_in1.dim, seed=1), seeded(Z, tp.irreps_in2.dim, seed=2)
    w = seeded(*((Z,) if not tp.shared_weights else ()), tp.weight_numel, seed=3) / 4
    cot = seeded(Z, tp.irreps_out.dim, seed=4)
    _, (r1, r2, rw) = _oracle_grads(lambda a, b, c: tp_forward_torch(spec, a, b, c), (x1, x2, w), cot)
    a, b, c = (t.to(DEV).requires_grad_(True) for t in (x1, x2, w))
    tp(a, b, c).backward(cot.to(DEV))
    # shared weights: the gradient is a sum over the batch, held to a tolerance scaled by its size; everything else
    # is a per-sample contraction (1e-4 + 1e-5 |ref|)
    w_atol = 1e-4 * max(1.0, float(rw.abs().max())) if tp.shared_weights else 1e-4
    assert_close(c.grad, rw.numpy(), atol=w_atol, what="d/dw")
    assert_close(a.grad, r1.numpy(), what="d/dx1")
    assert_close(b.grad, r2.numpy(), what="d/dx2")
    # the weights alone
    c2 = w.to(DEV).requires_grad_(True)
    tp(x1.to(DEV), x2.to(DEV), c2).backward(cot.to(DEV))
    assert_close(c2.grad, rw.numpy(), atol=w_atol, what="d/dw alone")


@pytest.mark.parametrize("maker", [ks.few_channels, ks.few_channels_ragged, ks.few_outputs, lambda: ks.few_outputs(True)])
@pytest.mark.parametrize("Z", [1, 3, 66, 1025])
def test_uvw_products_of_few_channels(maker, Z):
    tp = maker().to(DEV)
    spec = oracle_spec(tp)
    x1, x2 = seeded(Z, tp.irreps_in1.dim, seed=1), seeded(Z, tp.irreps_in2.dim, seed=2)
    w = seeded(*((Z,) if not tp.shared_weights else ()), tp.weight_numel, seed=3)
    cot = seeded(Z, tp.irreps_out.dim, seed=4)
    ref_out, ref = _oracle_grads(lambda a, b, c: tp_forward_torch(spec, a, b, c), (x1, x2, w), cot)
    args = [t.to(DEV).requires_grad_(True) for t in (x1, x2, w)]
    out = tp(*args)
    got = [out, *torch.autograd.grad(out, args, cot.to(DEV))]
    for g, r, what in zip(got, [ref_out, *ref], ["out", "d/dx1", "d/dx2", "d/dw"]):
        # sums of up to a few thousand terms in fp32: about 4e-7 of the 2-norm at random
        assert float((g.detach().double().cpu() - r).norm()) <= 1e-6 * float(r.norm()) + 1e-30, what


def test_internal_weights_train():
    tp = ks.cfg1().to(DEV)
    x1, x2 = seeded(40, 64).to(DEV), seeded(40, 9).to(DEV)
    tp(x1, x2).square().sum().backward()
    assert tp.weight.grad is not None and tp.weight.grad.shape == tp.weight.shape and bool(tp.weight.grad.abs().sum() > 0)


def test_shared_uvu_weight_gradient():
    tp = ks.golden_tp("uvu_shared_v2").to(DEV)
    assert tp.shared_weights and tp.weight_numel
    spec = oracle_spec(tp)
    Z = 300
    x1, x2, w = seeded(Z, tp.irreps_in1.dim, seed=1), seeded(Z, tp.irreps_in2.dim, seed=2), seeded(tp.weight_numel, seed=3)
    cot = seeded(Z, tp.irreps_out.dim, seed=4)
    _, (r1, r2, rw) = _oracle_grads(lambda a, b, c: tp_forward_torch(spec, a, b, c), (x1, x2, w), cot)
    a, b, c = (t.to(DEV).requires_grad_(True) for t in (x1, x2, w))
    tp(a, b, c).backward(cot.to(DEV))
    assert_close(c.grad, rw.numpy(), atol=1e-4 * max(1.0, float(rw.abs().max())), what="d/dw (shared, summed over the batch)")
    assert_close(a.grad, r1.numpy(), what="d/dx1")
    assert_close(b.grad, r2.numpy(), what="d/dx2")


@pytest.mark.parametrize("maker", [ks.mixed_modes, lambda: ks.golden_tp("modes_uuu_uvuv_uuw_uvv"), lambda: ks.golden_tp("modes_triangular")])
def test_general_mode_gradients(maker):
    """Connection modes outside pure uvu / pure uvw are differentiated through the equivalent uvw product with structured
    weights.  The map is trilinear, so central differences of the float64 oracle along a direction are exact."""
    from oracle import tensor_product as otp

    tp = maker().to(DEV)
    assert tp._live_mode() == "general"
    spec = oracle_spec(tp)
    Z = 37
    wshape = (tp.weight_numel,) if tp.shared_weights else (Z, tp.weight_numel)
    x1, x2, w = seeded(Z, tp.irreps_in1.dim, seed=1), seeded(Z, tp.irreps_in2.dim, seed=2), seeded(*wshape, seed=3)
    cot = seeded(Z, tp.irreps_out.dim, seed=4)
    a, b, c = (t.to(DEV).requires_grad_(True) for t in (x1, x2, w))
    out = tp(a, b, c)
    f = lambda p, q, r: otp.tp_forward(spec, p, q, r if tp.weight_numel else None)  # noqa: E731
    n1, n2, nw = (t.numpy().astype(np.float64) for t in (x1, x2, w))
    assert_close(out, f(n1, n2, nw), what="forward through the dense equivalent")
    with torch.no_grad():
        assert_close(tp(a, b, c), f(n1, n2, nw), what="forward, mode-specific kernel")
    out.backward(cot.to(DEV))
    rng = np.random.default_rng(5)
    c64 = cot.numpy().astype(np.float64)
    for got, which in ((a.grad, 0), (b.grad, 1), (c.grad, 2)):
        if which == 2 and not tp.weight_numel:
            continue
        for _ in range(3):
            args = [n1, n2, nw]
            v = rng.normal(size=args[which].shape)
            plus, minus = list(args), list(args)
            plus[which], minus[which] = args[which] + v, args[which] - v
            want = ((f(*plus) - f(*minus)) * c64).sum() / 2
            assert float((got.cpu().double().numpy() * v).sum()) == pytest.approx(want, rel=2e-4, abs=1e-3)


@pytest.mark.parametrize("maker", [lambda **kw: ks.golden_tp("fctp_small_cfg5_like", **kw), lambda **kw: ks.golden_tp("uvu_merged_cfg3_like_mul4", **kw), ks.mixed_modes])
def test_right(maker):
    """right(y, w) is the matrix with forward(x, y, w) == x @ right(y, w) (the reference's own test of right(),
    tests/o3/tensor_product_test.py, checks this identity); the forward side is the oracle's."""
    from oracle import tensor_product as otp

    with pytest.raises(AssertionError):  # as in the reference, right() is there only when asked for at construction
        maker().right(seeded(1, maker().irreps_in2.dim).to(DEV))
    tp = maker(compile_right=True).to(DEV)
    spec = oracle_spec(tp)
    Z = 5
    wshape = (tp.weight_numel,) if tp.shared_weights else (Z, tp.weight_numel)
    x1, x2, w = seeded(Z, tp.irreps_in1.dim, seed=1), seeded(Z, tp.irreps_in2.dim, seed=2), seeded(*wshape, seed=3)
    with torch.no_grad():
        r = tp.right(x2.to(DEV), w.to(DEV) if tp.weight_numel else None)
    assert r.shape == (Z, tp.irreps_in1.dim, tp.irreps_out.dim)
    got = torch.einsum("zik,zi->zk", r.cpu().double(), x1.double())
    want = otp.tp_forward(spec, *(t.numpy().astype(np.float64) for t in (x1, x2)), w.numpy().astype(np.float64) if tp.weight_numel else None)
    assert_close(got, want, what="x @ right(y, w)")
    # rows of the operator that belong to an input irrep no instruction reads are zero
    assert torch.isfinite(r).all()


@pytest.mark.parametrize("lmax", [1, 2, 3])
@pytest.mark.parametrize("normalize,normalization", [(True, "component"), (False, "integral"), (True, "norm")])
def test_spherical_harmonics_gradient(lmax, normalize, normalization):
    from e3nn_amd import o3
    from oracle.torch_cpu import spherical_harmonics_torch
    import math

    x = seeded(301, 3, seed=lmax)
    cot = seeded(301, (lmax + 1) ** 2, seed=9)

    def ref_fn(v):
        y = spherical_harmonics_torch(lmax, v, normalize)
        if normalization == "integral":
            y = y / math.sqrt(4 * math.pi)
        elif normalization == "norm":
            y = y / torch.cat([math.sqrt(2 * l + 1) * torch.ones(2 * l + 1, dtype=y.dtype) for l in range(lmax + 1)])
        return y

    _, (rx,) = _oracle_grads(ref_fn, (x,), cot)
    xd = x.to(DEV).requires_grad_(True)
    o3.spherical_harmonics(list(range(lmax + 1)), xd, normalize, normalization).backward(cot.to(DEV))
    assert_close(xd.grad, rx.numpy(), atol=1e-4 * max(1.0, float(rx.abs().max())), what="d/dxyz")
    # float64 finite differences of the oracle agree with its autograd (the reference's gradcheck, test :62-80)
    eps = 1e-6
    xp = x.double().clone()
    xp[0, 1] += eps
    fd = ((ref_fn(xp) - ref_fn(x.double()))[0] * cot[0].double()).sum() / eps
    assert abs(fd - rx[0, 1]) < 1e-4 * max(1.0, abs(float(fd)))


@pytest.mark.parametrize("ls,normalize,normalization", [
    ([0, 1, 2, 3, 4, 5], True, "component"), ([6], False, "integral"), ([2, 2, 0, 7], True, "norm"), ([1, 3], False, "component"),
    (list(range(11)), True, "integral"), (list(range(13)), True, "component"), ([12, 11], False, "norm"),
])  # fmt: skip
def test_spherical_harmonics_gradient_any_l_list(ls, normalize, normalization):
    """l lists beyond 0..3 take the reverse sweep of the recurrence: against central differences of the float64 oracle
    along random directions, point by point."""
    from e3nn_amd import o3
    from oracle import spherical_harmonics as osh

    n = 203
    x = seeded(n, 3, seed=len(ls))
    n_out = sum(2 * l + 1 for l in ls)
    cot = seeded(n, n_out, seed=11)
    xd = x.to(DEV).requires_grad_(True)
    out = o3.spherical_harmonics(ls, xd, normalize, normalization)
    assert out.shape == (n, n_out)
    out.backward(cot.to(DEV))
    got = xd.grad.cpu().double().numpy()
    x64, c64 = x.numpy().astype(np.float64), cot.numpy().astype(np.float64)
    rng = np.random.default_rng(7)
    f = lambda p: osh.spherical_harmonics(ls, p, normalize, normalization)  # noqa: E731
    for _ in range(3):
        v = rng.normal(size=x64.shape)
        eps = 1e-6
        want = ((f(x64 + eps * v) - f(x64 - eps * v)) * c64).sum(axis=1) / (2 * eps)
        have = (got * v).sum(axis=1)
        scale = max(1.0, float(np.abs(want).max()))
        assert np.abs(have - want).max() < 2e-4 * scale, (np.abs(have - want).max(), scale)


@pytest.mark.parametrize("maker,Z,shared", [(ks.mfma_small, 300, True), (lambda: ks.golden_tp("uvu_shared_v2"), 200, True),
                                            (lambda: ks.cfg3(True), 130, False), (ks.wide_k_l3, 150, True)])  # fmt: skip
def test_gradients_in_bf16_storage(maker, Z, shared):
    """bf16 storage, fp32 accumulation: every gradient against float64 autograd of the oracle on the same (bf16-rounded)
    inputs, to the bf16 tolerance rel 1e-2 of the largest entry (inputs, outputs and gradients are rounded to bf16)."""
    tp = maker().to(DEV)
    spec = oracle_spec(tp)
    bf = torch.bfloat16
    wshape = (tp.weight_numel,) if shared else (Z, tp.weight_numel)
    x1, x2 = seeded(Z, tp.irreps_in1.dim, seed=1).to(bf), seeded(Z, tp.irreps_in2.dim, seed=2).to(bf)
    w, cot = seeded(*wshape, seed=3).to(bf), seeded(Z, tp.irreps_out.dim, seed=4).to(bf)
    _, (r1, r2, rw) = _oracle_grads(lambda a, b, c: tp_forward_torch(spec, a, b, c), (x1.float(), x2.float(), w.float()), cot.float())
    a, b, c = (t.to(DEV).requires_grad_(True) for t in (x1, x2, w))
    tp(a, b, c).backward(cot.to(DEV))
    for got, ref, what in ((a.grad, r1, "d/dx1"), (b.grad, r2, "d/dx2"), (c.grad, rw, "d/dw")):
        assert got.dtype == bf
        err = (got.float().cpu().double() - ref).abs().max().item()
        assert err <= 2e-2 * max(1.0, ref.abs().max().item()), f"{what}: {err} vs {ref.abs().max().item()}"
