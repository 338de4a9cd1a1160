"""The package's instruction-set list (e3nn_amd.kernel_sets) plus the cases of tests/golden: instruction tables and
constructor arguments written from the reference (tp_cases.json, nn_cases.json and their .npz arrays)."""
import json
import os

import torch

from e3nn_amd import kernel_sets as _ks
from e3nn_amd import nn, o3
from e3nn_amd.kernel_sets import *  # noqa: F401,F403
from e3nn_amd.kernel_sets import FUSED_FC_CASES, SH2, SH3  # noqa: F401

GOLDEN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden")

GOLDEN_GPU_CASES = [
    "fctp_cfg1", "fctp_small_cfg5_like", "fctp_per_sample_weights", "fctp_norm_path",
    "uvu_merged_cfg3_like_mul4", "uvu_builder_cfg3_like_mul4", "uvu_builderA_cfg4_like_mul2",
    "uvu_builderB_cfg4_like_mul2", "uvu_shared_v2", "uvu_mixed_weightless", "empty_path_and_missing_output",
    "modes_uuu_uvuv_uuw_uvv", "modes_triangular", "conv_small",
]  # fmt: skip

# instruction sets whose backward pass the GPU tests run (transposed plans are separate kernels)
BACKWARD_CASES = _ks.BACKWARD_CASES + ["uvu_merged_cfg3_like_mul4", "uvu_builderA_cfg4_like_mul2", "uvu_shared_v2", "fctp_small_cfg5_like",
                                       "fctp_per_sample_weights", "modes_uuu_uvuv_uuw_uvv", "modes_triangular", "zero_path_first", "zero_path_last",
                                       "dense_one_path", "node_ragged", "node_long_row", "few_channels", "few_channels_ragged",
                                       "few_outputs", "few_outputs_per_sample", "message_ragged_groups", "message_four_lanes"]  # fmt: skip
BACKWARD_BF16_CASES = _ks.BACKWARD_BF16_CASES + ["uvu_shared_v2", "cfg3_builder", "cfg4_A", "odd_mul", "narrow_message", "ragged_wide_message",
                                                 "mfma_full_tiles", "mfma_wide_blocks", "few_outer_indices", "unaligned_offsets", "cfg5"]  # fmt: skip


def golden_meta():
    with open(os.path.join(GOLDEN, "tp_cases.json")) as f:
        return json.load(f)


def tp_from_meta(m, **extra):
    upw = m.get("user_path_weights", [1.0] * len(m["instructions"]))
    ins = [tuple(t[:5]) + (pw,) for t, pw in zip(m["instructions"], upw)]
    kw = {}
    if m.get("irrep_normalization"):
        kw = dict(irrep_normalization=m["irrep_normalization"], path_normalization=m["path_normalization"])
    return o3.TensorProduct(
        m["irreps_in1"], m["irreps_in2"], m["irreps_out"], ins,
        internal_weights=m["internal_weights"], shared_weights=m["shared_weights"], **kw, **extra,
    )  # fmt: skip


def golden_tp(name, meta=None, **extra):
    m = dict((meta or golden_meta())[name])
    if name == "fctp_norm_path":
        m.update(irrep_normalization="norm", path_normalization="path")
    return tp_from_meta(m, **extra)


def nn_golden():
    import numpy as np

    with open(os.path.join(GOLDEN, "nn_cases.json")) as f:
        meta = json.load(f)
    return np.load(os.path.join(GOLDEN, "nn_cases.npz")), meta


# (features, node attributes) of blocks whose mixing coefficient is read from messages of 4224 numbers, too long for the
# vector-ALU kernel to stage; of an ordinary width; with a handful of weights; and that are not whole 16-byte pieces, with
# scalars that are and scalars that are not
ALPHA_CASES = [("384x0e+384x1o", "1x0e"), ("16x0e+16x1o", "4x0e"), ("8x0e+8x1o", "1x0e"), ("16x0e+16x1o+1x1e", "4x0e"), ("8x0e+7x1o", "9x0e")]


def alpha_block(features, attr):
    torch.manual_seed(1)
    return nn.Convolution(features, attr, SH2, features, [8, 16], 4.0)


def alpha_modules():
    out = []
    for i, case in enumerate(ALPHA_CASES):
        conv = alpha_block(*case)
        # (lin2 and alpha on the long messages have no kernel for the gradient of the node attributes, which a block does not
        # ask for; those of a training step are built as they are used)
        parts = [conv.sc, conv.lin1, conv.tp, conv.fc, conv.__dict__["_alpha_head"]] if i == 0 else [conv]
        out.append((f"alpha_block{i}", torch.nn.ModuleList(p for p in parts if p is not None)))
    return out


def zero_path(first):
    # scalars onto scalars, few weights, one of the two paths with a path weight of zero
    return o3.TensorProduct("32x0e+32x0e", "4x0e", "2x0e", [(0, 0, 0, "uvw", True, 0.0 if first else 1.0), (1, 0, 0, "uvw", True, 1.0 if first else 0.0)])


def scalar_outputs():
    # scalar outputs of l x l, l = 0, 1, 2, whose path coefficients are about 1, larger, and a hundred
    weights = (1.0, 2.0, 1e4)
    return o3.TensorProduct("64x0e+64x1o+64x2e", "64x0e+64x1o+64x2e", "64x0e+64x0e+64x0e",
                            [(l, l, o, "uvw", True, pw) for o, pw in enumerate(weights) for l in range(3)], path_normalization="none")  # fmt: skip


def wide_scalar_output():
    return o3.FullyConnectedTensorProduct("64x0e+64x1o+64x2e", "64x0e+64x1o+64x2e", "128x0e")


def dense_one_path():
    return o3.FullyConnectedTensorProduct("64x0e", "64x0e", "64x0e")


def node_ragged():
    return o3.FullyConnectedTensorProduct("16x0e+16x1o+16x2e", "4x0e", "16x0e+16x1o+16x2e")


def node_long_row():
    # scalars onto one scalar, the longest row whose gradient the kernel for few scalars takes
    return o3.FullyConnectedTensorProduct("960x0e", "1x0e", "1x0e")


def few_channels():
    return o3.FullyConnectedTensorProduct("16x0e+16x1o", "0e+1o+2e", "16x0e+16x1o+16x2e")


def few_channels_ragged():
    # either input the one of more indices; more columns (v, w) than a workgroup has threads, and 9 u to blocks of 8
    return o3.FullyConnectedTensorProduct("9x0e+5x1o", "3x0e+30x1o", "6x0e+11x1o")


def few_outer_indices():
    # tiles of 32 channels, whose second wave column takes every other outer index, an odd number of which is left
    return o3.FullyConnectedTensorProduct("128x0e+64x1o", "33x0e+3x1o", "32x1o+32x1e+32x2e")


def few_outputs(per_sample=False):
    # outputs summed over the lanes, with indices that are no multiple of them and more of them than lanes
    kw = dict(internal_weights=False, shared_weights=False) if per_sample else {}
    return o3.FullyConnectedTensorProduct("12x0e+7x1o", "20x0e+70x1o", "1x0e+2x1o+1x2e", **kw)


def message_ragged_groups():
    # 5 of the 8 lanes of a group have indices; rows summed over the groups through LDS
    return _ks.message_tensor_product("20x0e+20x1o+20x2e", SH2, irreps_out="20x0e+20x1o+20x2e")


def message_four_lanes():
    # groups of four lanes whose rows are too wide to be summed through LDS
    return _ks.message_tensor_product("16x0e+16x1o+16x2e", SH2, keep="0e+1o+2e")


def golden_tensor_products():
    meta = golden_meta()
    return [(n, golden_tp(n, meta), (torch.float32,)) for n in GOLDEN_GPU_CASES]


def edge_case_tensor_products():
    return [
        ("zero_path_first", zero_path(True), (torch.float32,)), ("zero_path_last", zero_path(False), (torch.float32,)),
        ("scalar_outputs", scalar_outputs(), (torch.bfloat16,)), ("wide_scalar_output", wide_scalar_output(), (torch.float32, torch.bfloat16)),
        ("dense_one_path", dense_one_path(), (torch.float32,)), ("node_ragged", node_ragged(), (torch.float32,)),
        ("node_long_row", node_long_row(), (torch.float32,)), ("few_channels", few_channels(), (torch.float32,)),
        ("few_channels_ragged", few_channels_ragged(), (torch.float32,)), ("few_outputs", few_outputs(), (torch.float32, torch.bfloat16)),
        ("few_outer_indices", few_outer_indices(), (torch.float32,)), ("few_outputs_per_sample", few_outputs(True), (torch.float32,)),
        ("message_ragged_groups", message_ragged_groups(), (torch.float32, torch.bfloat16)),
        ("message_four_lanes", message_four_lanes(), (torch.float32, torch.bfloat16)),
    ]  # fmt: skip


def golden_modules():
    _, meta = nn_golden()
    out = []
    for name in ("linear_mixed", "linear_path_norm", "linear_bias"):
        m = meta[name]
        out.append((name, o3.Linear(m["irreps_in"], m["irreps_out"], **m["kwargs"])))
    out.append(("fc_golden", nn.FullyConnectedNet(meta["fc"]["hs"], torch.nn.functional.silu)))
    a = meta["conv"]["args"]
    out.append(("conv_golden", nn.Convolution(a[0], a[1], a[2], a[3], a[4], a[5])))
    return out


def prebuild(verbose=True):
    """Every kernel the tests and the benchmark use: the package's list plus the fixtures' instruction sets."""
    _ks.prebuild(verbose=verbose, extra_tensor_products=golden_tensor_products() + edge_case_tensor_products(), extra_modules=golden_modules() + alpha_modules(),
                 backward_cases=BACKWARD_CASES, backward_bf16_cases=BACKWARD_BF16_CASES)  # fmt: skip
