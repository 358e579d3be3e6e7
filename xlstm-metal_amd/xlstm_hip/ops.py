"""``torch.library`` operators ``xlstm_hip::*`` backed by libxlstm_hip.so.

Schemas and fake (meta) kernels are declared here, so the ops are traceable; the GPU kernels are native
(csrc/torch_ops.cpp, lib/libxlstm_torch.so): they validate shapes and dtypes, allocate the outputs with
torch's caching allocator (the library itself never allocates), pass raw pointers and the current HIP
stream through the C-ABI and return without synchronising.  There is no CPU path: CPU tensors raise.
``mlstm_chunkwise`` differentiates through the reference's custom backward; a backward through any other
op raises.
"""

from __future__ import annotations

import ctypes
import warnings

import torch
from torch import Tensor

from . import _lib

__all__ = [
    "soft_cap_op", "mlstm_step_op", "mlstm_step_inplace_op", "mlstm_chunkwise_op", "mlstm_chunkwise_bwd_op", "mlstm_sequence_op",
    "slstm_step_op", "slstm_sequence_op", "causal_conv1d_op", "group_norm_op", "mh_rmsnorm_gate_op",
    "gate_proj_softcap_op", "gate_proj2_softcap_op", "lm_head_softcap_op", "rms_norm_op", "add_rmsnorm_op", "silu_mul_op",
    "chunkwise_workspace_bytes", "chunkwise_algorithm",
]

_EMPTY_SHAPE = (0,)

_SCHEMAS = {
    "soft_cap": ("(Tensor x, float cap) -> Tensor"),
    "mlstm_step": ("(Tensor q, Tensor k, Tensor v, Tensor i, Tensor f, Tensor c, Tensor n, Tensor m, float "
                  "eps, float qk_scale) -> (Tensor, Tensor, Tensor, Tensor)"),
    # decode step updating the float32 C state in place; returns (h, n', m')
    "mlstm_step_": ("(Tensor q, Tensor k, Tensor v, Tensor i, Tensor f, Tensor(a!) c, Tensor n, Tensor m, "
                   "float eps, float qk_scale) -> (Tensor, Tensor, Tensor)"),
    "mlstm_chunkwise": ("(Tensor q, Tensor k, Tensor v, Tensor i, Tensor f, Tensor? c0, Tensor? n0, Tensor? m0, "
                       "float qk_scale, SymInt chunk_size, float eps, bool return_last_states, SymInt algo) -> "
                       "(Tensor, Tensor, Tensor, Tensor)"),
    # the reference's custom backward (mlstm_chunkwise_bw, bw.py:198-352): dq, dk, dv (q's dtype), di, df
    # (the gates' dtype) and dc0 (float32; an empty placeholder without initial states)
    "mlstm_chunkwise_bwd": ("(Tensor q, Tensor k, Tensor v, Tensor i, Tensor f, Tensor? c0, Tensor? n0, Tensor? m0, "
                           "Tensor dh, Tensor? dc_last, float qk_scale, SymInt chunk_size, float eps) -> (Tensor, "
                           "Tensor, Tensor, Tensor, Tensor, Tensor)"),
    "mlstm_sequence": ("(Tensor q, Tensor k, Tensor v, Tensor i, Tensor f, Tensor? c0, Tensor? n0, Tensor? m0, "
                      "float qk_scale, float eps, bool return_last_states) -> (Tensor, Tensor, Tensor, Tensor)"),
    # h and the new states packed as one flat tensor [c | n | m] (state_views splits it): one
    # allocation and, for 16-bit outputs, one conversion kernel
    "slstm_step": ("(Tensor z, Tensor i, Tensor f, Tensor o, Tensor c, Tensor n, Tensor m, float eps) -> "
                  "(Tensor, Tensor)"),
    # h and the last states packed as one flat tensor [c | n | m] (state_views)
    "slstm_sequence": ("(Tensor z, Tensor i, Tensor f, Tensor o, Tensor? c0, Tensor? n0, Tensor? m0, float eps) "
                      "-> (Tensor, Tensor)"),
    "causal_conv1d": ("(Tensor x, Tensor weight, Tensor? bias, SymInt act) -> Tensor"),
    "group_norm": ("(Tensor x, SymInt num_groups, Tensor? weight, Tensor? bias, float eps) -> Tensor"),
    "mh_rmsnorm_gate": ("(Tensor h, Tensor? weight, Tensor? o_preact, bool heads_first, float eps) -> Tensor"),
    "gate_proj_softcap": ("(Tensor x, Tensor weight, Tensor? bias, float cap, SymInt cap_rounding=0) -> Tensor"),
    # gate_proj_softcap for two projections of one input [B, S, D], their weights not stacked; the
    # outputs [B, S, G], or [B, G, S] with heads_first
    "gate_proj2_softcap": ("(Tensor x, Tensor w1, Tensor? b1, Tensor w2, Tensor? b2, float cap, SymInt cap_rounding, "
                          "bool heads_first) -> (Tensor, Tensor)"),
    # soft_cap(x weight^T, cap) for at most LM_HEAD_MAX_ROWS rows
    "lm_head_softcap": ("(Tensor x, Tensor weight, float cap) -> Tensor"),
    # x / rms(x) * weight over the last axis, float32, rounded once (bf16 / f16)
    "rms_norm": ("(Tensor x, Tensor weight, float eps) -> Tensor"),
    # (x + residual, rms_norm of it); up to two float32 states copied along
    "add_rmsnorm": ("(Tensor x, Tensor residual, Tensor weight, float eps, Tensor[] copy_src, Tensor(a!)[] "
                   "copy_dst) -> (Tensor, Tensor)"),
    # silu(gate) * up, the SiLU rounded to the dtype first (bf16 / f16)
    "silu_mul": ("(Tensor gate, Tensor up) -> Tensor"),
}

_library = torch.library.Library("xlstm_hip", "DEF")
for _name, _schema in _SCHEMAS.items():
    _library.define(_name + _schema, tags=(torch.Tag.pt2_compliant_tag,))


def _no_path(name: str, reason):
    def raises(*args, **kwargs):
        raise RuntimeError(f"{name}: {reason()}")
    return raises


for _name in _SCHEMAS:
    _library.impl(_name, _no_path(_name, lambda: "tensors must be on the GPU (got cpu); there is no CPU path"), "CPU")
unavailable = _lib.load_ops()  # "" or why the GPU kernels cannot run
if unavailable:
    for _name in _SCHEMAS:
        _library.impl(_name, _no_path(_name, lambda: unavailable), "CUDA")


def _fake(name: str):
    return torch.library.register_fake(f"xlstm_hip::{name}", lib=_library)


@_fake("soft_cap")
def _(x, cap):
    return torch.empty_like(x, memory_format=torch.contiguous_format)


@_fake("mlstm_step")
def _(q, k, v, i, f, c, n, m, eps, qk_scale):
    B, NH, DQK = q.shape
    DV = v.shape[-1]
    return (q.new_empty((B, NH, DV)), q.new_empty((B, NH, DQK, DV), dtype=torch.float32),
            q.new_empty((B, NH, DQK), dtype=torch.float32), q.new_empty((B, NH, 1), dtype=torch.float32))


@_fake("mlstm_step_")
def _(q, k, v, i, f, c, n, m, eps, qk_scale):
    B, NH, DQK = q.shape
    DV = v.shape[-1]
    return (q.new_empty((B, NH, DV)), q.new_empty((B, NH, DQK), dtype=torch.float32),
            q.new_empty((B, NH, 1), dtype=torch.float32))


@_fake("mlstm_chunkwise")
def _(q, k, v, i, f, c0, n0, m0, qk_scale, chunk_size, eps, return_last_states, algo):
    B, NH, S, DQK = q.shape
    DV = v.shape[-1]
    h = q.new_empty((B, NH, S, DV))
    if not return_last_states:
        return (h,) + tuple(q.new_empty(_EMPTY_SHAPE, dtype=torch.float32) for _ in range(3))
    return (h, q.new_empty((B, NH, DQK, DV), dtype=torch.float32), q.new_empty((B, NH, DQK), dtype=torch.float32),
            q.new_empty((B, NH, 1), dtype=torch.float32))


@_fake("mlstm_chunkwise_bwd")
def _(q, k, v, i, f, c0, n0, m0, dh, dc_last, qk_scale, chunk_size, eps):
    dc0 = (q.new_empty(tuple(c0.shape), dtype=torch.float32) if c0 is not None
           else q.new_empty(_EMPTY_SHAPE, dtype=torch.float32))
    return q.new_empty(q.shape), k.new_empty(k.shape), v.new_empty(v.shape), i.new_empty(i.shape), \
        f.new_empty(f.shape), dc0


@_fake("mlstm_sequence")
def _(q, k, v, i, f, c0, n0, m0, qk_scale, eps, return_last_states):
    B, NH, S, DQK = q.shape
    DV = v.shape[-1]
    h = q.new_empty((B, NH, S, DV))
    if not return_last_states:
        return (h,) + tuple(q.new_empty(_EMPTY_SHAPE, dtype=torch.float32) for _ in range(3))
    return (h, q.new_empty((B, NH, DQK, DV), dtype=torch.float32), q.new_empty((B, NH, DQK), dtype=torch.float32),
            q.new_empty((B, NH, 1), dtype=torch.float32))


def _slstm_out_dtype(z, i, c):
    return torch.promote_types(torch.promote_types(z.dtype, i.dtype), c.dtype)


@_fake("slstm_step")
def _(z, i, f, o, c, n, m, eps):
    out_dt = _slstm_out_dtype(z, i, c)
    B, NH, H = z.shape
    return z.new_empty((B, NH, H), dtype=out_dt), z.new_empty((2 * B * NH * H + B * NH,), dtype=out_dt)


@_fake("slstm_sequence")
def _(z, i, f, o, c0, n0, m0, eps):
    B, S, NH, H = z.shape
    out_dt = torch.promote_types(z.dtype, i.dtype) if c0 is None else _slstm_out_dtype(z, i, c0)
    return z.new_empty((B, S, NH, H), dtype=out_dt), z.new_empty((2 * B * NH * H + B * NH,), dtype=out_dt)


@_fake("causal_conv1d")
def _(x, weight, bias, act):
    return torch.empty_like(x, memory_format=torch.contiguous_format)


@_fake("group_norm")
def _(x, num_groups, weight, bias, eps):
    return torch.empty_like(x, memory_format=torch.contiguous_format)


@_fake("mh_rmsnorm_gate")
def _(h, weight, o_preact, heads_first, eps):
    if heads_first:
        B, NH, S, DH = h.shape
    else:
        B, S, NH, DH = h.shape
    return h.new_empty((B, S, NH * DH))


@_fake("gate_proj_softcap")
def _(x, weight, bias, cap, cap_rounding=0):
    return x.new_empty(tuple(x.shape[:-1]) + (weight.shape[0],))


@_fake("gate_proj2_softcap")
def _(x, w1, b1, w2, b2, cap, cap_rounding, heads_first):
    B, S, _ = x.shape
    return tuple(x.new_empty((B, w.shape[0], S) if heads_first else (B, S, w.shape[0])) for w in (w1, w2))


@_fake("lm_head_softcap")
def _(x, weight, cap):
    return x.new_empty(tuple(x.shape[:-1]) + (weight.shape[0],))


@_fake("rms_norm")
def _(x, weight, eps):
    return torch.empty_like(x, memory_format=torch.contiguous_format)


@_fake("add_rmsnorm")
def _(x, residual, weight, eps, copy_src, copy_dst):
    return tuple(torch.empty_like(x, memory_format=torch.contiguous_format) for _ in range(2))


@_fake("silu_mul")
def _(gate, up):
    return torch.empty_like(gate, memory_format=torch.contiguous_format)


soft_cap_op = torch.ops.xlstm_hip.soft_cap.default
mlstm_step_op = torch.ops.xlstm_hip.mlstm_step.default
mlstm_step_inplace_op = torch.ops.xlstm_hip.mlstm_step_.default
mlstm_sequence_op = torch.ops.xlstm_hip.mlstm_sequence.default
slstm_step_op = torch.ops.xlstm_hip.slstm_step.default
slstm_sequence_op = torch.ops.xlstm_hip.slstm_sequence.default
causal_conv1d_op = torch.ops.xlstm_hip.causal_conv1d.default
group_norm_op = torch.ops.xlstm_hip.group_norm.default
mh_rmsnorm_gate_op = torch.ops.xlstm_hip.mh_rmsnorm_gate.default
gate_proj_softcap_op = torch.ops.xlstm_hip.gate_proj_softcap.default
gate_proj2_softcap_op = torch.ops.xlstm_hip.gate_proj2_softcap.default
lm_head_softcap_op = torch.ops.xlstm_hip.lm_head_softcap.default
rms_norm_op = torch.ops.xlstm_hip.rms_norm.default
add_rmsnorm_op = torch.ops.xlstm_hip.add_rmsnorm.default
silu_mul_op = torch.ops.xlstm_hip.silu_mul.default

CONV_ACTS = {None: 0, "silu": 1}
# csrc/torch_ops.cpp's own (0 where no kernel can run): the most rows of lm_head_softcap and the LDS of its
# staging, and the input and forget gate of the tokens that the backward pads a ragged sequence with
LM_HEAD_MAX_ROWS, LM_HEAD_MAX_LDS, _PAD_I, _PAD_F = (
    ctype().value if unavailable else _lib.ops_constant(_name, ctype)
    for _name, ctype in (("xl_lm_head_max_rows", ctypes.c_int64), ("xl_lm_head_max_lds", ctypes.c_int64),
                         ("xl_pad_i", ctypes.c_double), ("xl_pad_f", ctypes.c_double)))


def state_views(st: Tensor, B: int, NH: int, H: int) -> tuple[Tensor, Tensor, Tensor]:
    """c [B,NH,H], n [B,NH,H], m [B,NH]: the consecutive pieces of a flat sLSTM state tensor."""
    k = B * NH * H
    return st[:k].view(B, NH, H), st[k:2 * k].view(B, NH, H), st[2 * k:].view(B, NH)


_ALGO_NAMES = {1: "two_pass", 2: "fused", 3: "pipelined"}
_fallback_warned: set = set()


def chunkwise_algorithm(B, NH, S, DQK, DV, L, dtype, algo="auto") -> str:
    """The algorithm ("fused", "pipelined" or "two_pass") xl_mlstm_chunkwise_fwd takes for these arguments."""
    lib = _lib.load()
    rc = int(lib.xl_mlstm_chunkwise_algo(B, NH, S, DQK, DV, L, _lib.XL_DTYPE[dtype], _lib.ALGO[algo]))
    if rc < 0:
        _lib.check(rc, "mlstm_chunkwise")
    return _ALGO_NAMES[rc]


def _warn_slow_fallback(B, NH, S, DQK, DV, L, dtype) -> None:
    """One warning per reason when algo="auto" leaves 16-bit inputs on the two-pass kernels (several
    times slower than the single-pass kernels, and holding every chunk's state in a workspace)."""
    lib = _lib.load()
    if int(lib.xl_mlstm_chunkwise_algo(B, NH, S, DQK, DV, L, _lib.XL_DTYPE[dtype], 0)) != 1:
        return
    why = lib.xl_last_error().decode(errors="replace")
    if why not in _fallback_warned:
        _fallback_warned.add(why)
        warnings.warn(f"xlstm_hip.mlstm_chunkwise: {dtype} inputs run the two-pass kernels ({why}); "
                      "bf16 or f16 q/k/v with DQK 32, 64, 96, 128, 192 or 256 and DV a multiple of 64 take "
                      "the single-pass kernels",
                      RuntimeWarning, stacklevel=3)


def chunkwise_workspace_bytes(B, NH, S, DQK, DV, L, dtype, algo="auto") -> int:
    return int(_lib.load().xl_mlstm_chunkwise_workspace_size(B, NH, S, DQK, DV, L, _lib.XL_DTYPE[dtype],
                                                             _lib.ALGO[algo]))


_SINGLE_PASS_DQK = (32, 64, 96, 128, 192, 256)


def _whole_chunks(q: Tensor, chunk_size: int) -> None:
    """The reference's own error for a ragged sequence (fw.py:303-305)."""
    if q.dim() == 4 and q.shape[2] % chunk_size != 0:
        raise AssertionError(f"Sequence length {q.shape[2]} is not divisible by chunk size {chunk_size}.")


def mlstm_chunkwise_op(q, k, v, i, f, c0, n0, m0, qk_scale: float, chunk_size: int, eps: float, return_last_states: bool,
                       algo: int):
    if q.is_cuda and q.dim() == 4:
        if algo < _lib.ALGO["fused"]:  # the single-pass algorithms, asked for, take a ragged last chunk
            _whole_chunks(q, chunk_size)
        if algo == _lib.ALGO["auto"] and q.dtype != torch.float32 and v.dim() == 4 and (
                v.shape[-1] % 64 or q.shape[-1] not in _SINGLE_PASS_DQK) and not torch.compiler.is_compiling() \
                and q.dtype in _lib.XL_DTYPE:
            _warn_slow_fallback(*q.shape, v.shape[-1], chunk_size, q.dtype)
    return torch.ops.xlstm_hip.mlstm_chunkwise.default(q, k, v, i, f, c0, n0, m0, qk_scale, chunk_size, eps,
                                                       return_last_states, algo)


def mlstm_chunkwise_bwd_op(q, k, v, i, f, c0, n0, m0, dh, dc_last, qk_scale: float, chunk_size: int, eps: float):
    if q.is_cuda:
        _whole_chunks(q, chunk_size)
    return torch.ops.xlstm_hip.mlstm_chunkwise_bwd.default(q, k, v, i, f, c0, n0, m0, dh, dc_last, qk_scale, chunk_size, eps)
