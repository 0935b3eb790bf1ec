"""``cdist_grad``: fused kernel-gradient contraction (AGOP / RFM gradient).

Same signature as the reference's ``kermac.cdist_grad``
(src/kermac/cdist_grad.py:10-18).
"""
from __future__ import annotations

import os
from typing import Union

import numpy as np
import torch

from . import _backend
from . import _scratch
from .build_a_kernel import _current_stream_for
from .common import launch_cuts_enabled, matrix_layout, merge_batch_size

_NORM_L1, _NORM_L2, _NORM_P = 0, 1, 2


class _GradPlan:
    __slots__ = ("params", "out", "keepalive", "L", "M", "N", "O", "K")


def _plan_cdist_grad(a, b, c, d, out, p, require_device=True) -> _GradPlan:
    """Validation and parameter marshalling of ``cdist_grad``
    (reference: cdist_grad.py:62-235), without the launch."""
    inputs = (a, b, c, d)
    for x in inputs:
        if not isinstance(x, torch.Tensor):
            raise TypeError("All inputs must be PyTorch tensors")
    if out is not None and not isinstance(out, torch.Tensor):
        raise TypeError("out must be a PyTorch tensor if provided")
    for x in inputs:
        if x.dtype is not torch.float32:
            raise TypeError("All inputs must have dtype torch.float32")
    if out is not None and out.dtype != torch.float32:
        raise TypeError("out must have dtype torch.float32")
    for x in inputs:
        if x.dim() not in (2, 3):
            raise ValueError("All inputs must be 2-dimensional or 3-dimensional with a batch mode")
    if out is not None and out.dim() not in (3, 4):
        raise ValueError("out must be 3-dimensional or 4-dimensional with a batch mode")
    if require_device:
        for x in inputs:
            if not x.is_cuda:
                raise ValueError("All inputs must be on a CUDA device")
        if out is not None and not out.is_cuda:
            raise ValueError("out must be on a CUDA device")
    device = a.device
    for x in inputs[1:]:
        if x.device != device:
            raise ValueError(f"All inputs must be on the same CUDA device: got {[x.device for x in inputs]}")
    if out is not None and out.device != device:
        raise ValueError(f"out must be on the same CUDA device as inputs: got {out.device}, expected {device}")

    if isinstance(p, int) and not isinstance(p, bool):
        p = float(p)

    _, K, M, _, a_ld, a_bs = matrix_layout(a)
    _, N, K_b, _, b_ld, b_bs = matrix_layout(b)
    _, O, K_c, _, c_ld, c_bs = matrix_layout(c)
    _, N_d, M_d, _, d_ld, d_bs = matrix_layout(d)

    L = 1
    L = merge_batch_size("p", L, p, expected_dims=0, can_be_none=False)
    for name, x in zip("abcd", inputs):
        if x.dim() != 2:            # (a matrix without a batch leaves L as it is)
            L = merge_batch_size(name, L, x, expected_dims=2, can_be_none=False)
    L = merge_batch_size("out", L, out, expected_dims=3, can_be_none=True)

    if (N, K_b) != (N, K):
        raise ValueError(f"Expected shape {(N, K)} for b, got {(N, K_b)}")
    if (O, K_c) != (O, K):
        raise ValueError(f"Expected shape {(O, K)} for c, got {(O, K_c)}")
    if (N_d, M_d) != (N, M):
        raise ValueError(f"Expected shape {(N, M)} for d, got {(N_d, M_d)}")
    if out is not None:
        if L == 1:
            if tuple(out.shape) not in ((O, N, M), (1, O, N, M)):
                raise ValueError(f"Expected shape {(O, N, M)} or {(L, O, N, M)} for out, got {tuple(out.shape)}")
        elif tuple(out.shape) != (L, O, N, M):
            raise ValueError(f"Expected shape {(L, O, N, M)} for out, got {tuple(out.shape)}")

    for name, x in zip("abcd", inputs):
        if x.stride(-1) != 1:
            raise ValueError(f"{name} must have stride 1 in last dimension")
    if out is not None and out.stride(-1) != 1:
        raise ValueError("out must have stride 1 in last dimension")

    if isinstance(p, float):
        p_ptr, p_bs, p_value, p_keep = 0, 0, float(np.float32(p)), None
        scalar_p = p_value
    else:
        if not isinstance(p, torch.Tensor):
            raise TypeError("`p` must be a float or a torch.Tensor")
        if p.dtype != torch.float32:
            raise TypeError("`p` tensor must have dtype torch.float32")
        if require_device and (not p.is_cuda or p.device != device):
            raise ValueError("`p` tensor must be on the same CUDA device as inputs")
        if p.numel() != 1 and p.numel() != L:
            raise ValueError(f"`p` tensor has {p.numel()} elements but the batch size is {L}")
        p_ptr, p_value, p_keep = p.data_ptr(), 0.0, p
        p_bs = 0 if p.numel() == 1 else p.stride(0)
        # One device-to-host read, as in the reference (cdist_grad.py:181-190), to
        # pick the transcendental-free kernels for p = 1 and p = 2.
        scalar_p = p.item() if p.numel() == 1 else None

    if scalar_p == 1.0:
        norm_type = _NORM_L1
    elif scalar_p == 2.0:
        norm_type = _NORM_L2
    else:
        norm_type = _NORM_P

    if out is None:
        # every element is written by the kernel, so no fill is needed
        out = torch.empty((L, O, N, M), dtype=torch.float32, device=device)

    params = _backend.NormGradientParams(norm_type, 0, M, N, O, K, L, a.data_ptr(), a_ld, a_bs, b.data_ptr(), b_ld, b_bs,
                                         c.data_ptr(), c_ld, c_bs, d.data_ptr(), d_ld, d_bs)
    params.e = out.data_ptr()
    params.e_ld_n = out.stride(-2)
    params.e_ld_o = out.stride(-3)
    params.e_bs = 0 if (L == 1 or out.dim() == 3) else out.stride(-4)
    params.p, params.p_bs, params.p_value = p_ptr, p_bs, p_value

    plan = _GradPlan()
    plan.params, plan.out, plan.keepalive = params, out, [a, b, c, d, out, p_keep]
    plan.L, plan.M, plan.N, plan.O, plan.K = L, M, N, O, K
    return plan


@_scratch.operator
def cdist_grad(
    a: torch.Tensor,           # [K,M]   m contiguous   kernel_matrix
    b: torch.Tensor,           # [N,K]   k contiguous   x
    c: torch.Tensor,           # [O,K]   k contiguous   coefs
    d: torch.Tensor,           # [N,M]   m contiguous   z
    out: torch.Tensor = None,  # [O,N,M] m contiguous   grad
    p: Union[float, torch.Tensor] = 2.0,
    debug=False,
    _may_split=True,
):
    """Gradient of the p-norm kernel contracted with coefficients::

        out[o, n, m] = sum_k c[o, k] * a[k, m] * sign(d[n, m] - b[n, k]) * |d[n, m] - b[n, k]| ** (p - 1)

    ``sign`` is ``copysign(1, x)`` (so ``sign(0) = 1``); for ``p = 2`` the weight is
    simply the difference.  Every tensor may carry a leading batch dimension of 1
    or L.  Returns ``out`` (allocated ``[L, O, N, M]`` when None; every element is written).

    Raises:
        TypeError: non-tensor inputs or a dtype other than fp32.
        ValueError: bad shapes, strides, batch sizes or devices.
    """
    plan = _plan_cdist_grad(a, b, c, d, out, p)
    route = _route_of_any_size(plan) if _may_split else None
    if route is not None and _run_cut((*route, True), plan, a, b, c, d, p, debug, any_size=True):
        return plan.out
    if _may_split:
        for cut in _cuts_over_contraction(plan):
            if _run_cut(cut, plan, a, b, c, d, p, debug):
                return plan.out
    _launch(plan, a.device, debug)
    return plan.out


def _launch(plan, device, debug, needs_workspace=False, any_size=False):
    """Launches the call as it is; with `needs_workspace` only if it gets the workspace that the library wants for it, which
    with `any_size` does not ask whether the route pays."""
    plan.params.flags = _backend.FLAG_GRAM_WORKSPACE_ANY_SIZE if any_size else 0
    workspace = _attach_workspace(plan.params, device)
    if needs_workspace and workspace is None:
        plan.params.flags = 0
        return False
    if debug:
        print(f"(Kermac Debug) Launching kernel: norm_kernel_gradient<{('L1', 'L2', 'P')[plan.params.norm_type]}>")
    _backend.norm_kernel_gradient(plan.params, _current_stream_for(device))
    del workspace           # the launches are queued: the allocator hands the memory on in stream order
    return True


def _workspace_enabled():
    return os.environ.get("KERMAC_AMD_GRADIENT_WORKSPACE", "1") not in ("", "0")


def _attach_workspace(params, device):
    """Large L1 and L2 gradients run on the fp16 matrix instruction through a workspace (include/kermac_amd.h,
    kmc_norm_gradient_params::workspace.  L1: rows of b and d ranked, d >= b as an exact 0 or 1 times a c in two fp16 pieces.
    L2: the sum factors into (d - s) (c a) - (c (b - s)) a, one product of pieces); the library says how much it wants for
    this call, 0 when it would not use one.  KERMAC_AMD_GRADIENT_WORKSPACE=0 keeps every call on
    the fp32 kernels."""
    if not _workspace_enabled():
        return None
    needed = _backend.norm_gradient_workspace_bytes(params)
    if needed == 0:
        return None
    workspace = _scratch.allocate(needed, device)
    if workspace is None:
        return None             # no room for it, or the caller's limit: the fp32 kernels need none
    params.workspace, params.workspace_bytes = workspace.data_ptr(), needed
    return workspace


# A workgroup owns 64 (m) x 32 or 16 (n) results and walks the whole contraction index k,
# so few samples and features against many centres (M = 2000, N = 100, K = 10000) launch a
# hundred workgroups on 256 CUs, and a few hundred workgroups, all started together, leave
# the CUs unevenly loaded (256 workgroups at O = 16: 65 TFLOP/s where 4096 reach 120).  Such
# an unbatched call is cut over k: slices of a, b and c become the batch of one launch
# through strided views (d broadcasts), every slice writes a partial result, and the
# partial results are summed in a fixed order.  Measured at N = 128, K = 4096, cut in 8:
# O = 16, M = 2048: 65 -> 96 TFLOP/s; O = 1, M = 4096: 24 -> 60; nothing from 1536
# workgroups on.
_SPLIT_BELOW_WORKGROUPS = 1536
_SPLIT_TARGET_WORKGROUPS = 3072
_SPLIT_MIN_DEPTH = 512                      # from 512 workgroups on: 1024, and 2048 for the matrix-core kernels
_SPLIT_MAX_SLICES = 24
_SPLIT_MAX_PARTIAL_BYTES = 512 << 20
# Calls that go to the fp16 matrix instruction (p = 1, the workspace granted): its workgroups own 16 (m) x 128 (n) x 16 (o)
# results or more, one per CU at a time, and every slice ranks its rows again, so fewer slices are wanted: 2000 x 24 x 16 x 9000 in
# 17 slices 166 us, in 5 147; 200 x 1000 x 16 x 12000 in 12 472, in 5 401.
_SPLIT_F16_TARGET_WORKGROUPS = 512


def _shape_of_cuts(plan):
    """(workgroups of the fp32 kernels, the most slices over k), or None for a call that is not cut."""
    if plan.L != 1 or plan.M == 0 or plan.N == 0 or plan.O == 0 or not launch_cuts_enabled():
        return None
    M, N, O, K = plan.M, plan.N, plan.O, plan.K
    n_tile = 32 if O <= 8 else 16
    workgroups = -(-M // 64) * -(-N // n_tile) * max(1, -(-O // 32))
    min_depth = _SPLIT_MIN_DEPTH * (1 if workgroups < 512 else 2 if O <= 8 else 4)
    if workgroups >= _SPLIT_BELOW_WORKGROUPS or K < 2 * min_depth:
        return None
    return workgroups, min(K // min_depth, _SPLIT_MAX_SLICES, _SPLIT_MAX_PARTIAL_BYTES // (4 * O * N * M) - 1)


def _cut_into(K, wanted, most):
    depth = K // min(wanted, most) // 64 * 64           # whole K slices of the kernels; 16-byte alignment survives
    slices = K // depth
    return slices, depth, K - slices * depth


def _f16_slices(M, N, O):
    """Slices over k that the L1 route wants: the number that fills the CUs, and the fewer that reach its number of workgroups."""
    f16_workgroups = -(-M // 16) * -(-N // 128) * -(-O // 16)
    wanted = -(-_SPLIT_F16_TARGET_WORKGROUPS // f16_workgroups)
    filled = wanted
    # a workgroup has its CU to itself: up to twice as many slices where their last round of 256 would be nearly empty
    # (1408 x 128 x 32 x 9522, 176 workgroups: 3 slices 424 us, 4 slices 354)
    if wanted > 1:
        parts = [n * f16_workgroups / (256 * -(-n * f16_workgroups // 256)) for n in range(wanted, 2 * wanted + 1)]
        filled += next((extra for extra, part in enumerate(parts) if part >= 0.85), parts.index(max(parts)))
    return filled, wanted


# The library's own rule for the L1 gradient's fp16 route (kmc_norm_gradient_workspace_bytes) takes the calls that are large enough for the route to win
# everywhere; below it stand calls that the fp32 kernels, a workgroup walking the whole of k, take far longer for.  Which is
# the faster one there follows from launch times in microseconds, fitted to sweeps of M 64 .. 12000, N 8 .. 1024, K 64 .. 12000, O 1 .. 64, one
# problem or a batch of two (the fits are off by 13 .. 19 %).  An uncut route that they favour by 25 % is taken, one cut
# over k by 15 %.  Of 260 other calls that they favour at all, the 171 uncut ones beyond 25 % are 0.97 .. 8.1 times as fast and the 41 cut ones beyond 15 % 0.94 .. 2.1 (two
# slower, 68 x 13 x 2 x 3117 77 -> 82 us); the 16 uncut ones favoured by 15 to 25 % were 0.82 .. 1.6 (8808 x 37 x 16 x 174 44 -> 53 us).
# fp32 / route, us: 768 x 28 x 1 x 1651 twice 191 / 56; 192 x 22 x 32 x 1088 118 / 39; 428 x 18 x 4 x 256 40 / 23; 10304 x 675 x 1 x 175 117 / 227.
# Not the L2 gradient, below its own rule: the pieces of a and of c (b - s) are scaled by the largest magnitude of a row and hold what lies far below it to
# fewer bits, and nothing in the sum of their products tells the call that its result is off.  Error (2-norm) of fp32 / route with the rows of a scaled over 8 decades and those of
# c by the inverse: 717 x 52 x 16 x 390 twice 3.7e-7 / 1.6e-5, 2432 x 256 x 4 x 1984 4.9e-7 / 4.0e-5 (on normal values 0.4 to 0.6 of the fp32 kernels',
# at 732 x 22 x 10 x 11840 twice 1650 / 468 us).  In the L1 gradient the pieces of a c meet 0 or 1: the route's error is 0.2 to 0.8 of theirs on such values too.
_ROUTE_ADVANTAGE = 1.25
_ROUTE_ADVANTAGE_CUT = 1.15
# The sums of the fp32 kernels hold their rounding, which short slices keep small: the route's error (in the 2-norm, against 64 bits,
# normal, uniform, heavy-tailed and scaled values) is 0.2 .. 0.8 of theirs on slices of the same depth, 0.9 at four times the depth, above theirs
# from seven times on (1602 x 178 x 10 x 4485 uncut against 8 slices 5.8e-7 / 4.2e-7).
_ROUTE_MAX_DEPTH_RATIO = 4
_ROUTE_MIN_FP32_US = 24.0


def _fp32_us(plan, slices, depth):
    L, M, N, O = plan.L, plan.M, plan.N, plan.O
    rounds = max(1.0, -(-M // 64) * -(-N // (32 if O <= 8 else 16)) * -(-O // 32) * L * slices / 256)
    outputs = O if O <= 2 else 4 if O <= 4 else 8 if O <= 8 else 16 if O <= 16 else 32
    us = 4.5 + depth * (0.081 + rounds * (0.0356 + 0.0035 * outputs)) + 1.84e-6 * L * M * N * O
    return us + 30.0 + 1.84e-6 * slices * M * N * O if slices > 1 else us


def _route_us(plan, slices, depth):
    L, M, N, O, K = plan.L, plan.M, plan.N, plan.O, plan.K
    parts = L if slices == 1 else slices
    workgroups = -(-M // 16) * -(-N // 128) * -(-O // 16) * parts
    us = (18.5 + 0.0194 * depth * max(1.0, workgroups / 256) + (11e-6 * N + 2.6e-6 * M) * K * L + 23e-6 * N * (M + 256) * parts
          + 1.7e-6 * L * M * N * O)
    return us + 36.0 + 1.7e-6 * slices * M * N * O if slices > 1 else us


def _route_of_any_size(plan):
    """(slices, k per slice, leftover k) with which an L1 gradient that the library's rule leaves to the fp32 kernels is faster on the fp16
    matrix instruction, or None."""
    if plan.params.norm_type != _NORM_L1 or min(plan.L, plan.M, plan.N, plan.O, plan.K) < 1 or not _workspace_enabled():
        return None
    shape = _shape_of_cuts(plan)
    fp32 = (1, plan.K, 0)
    forms = [fp32]
    if shape is not None and shape[1] >= 2:
        workgroups, most = shape
        fp32 = _cut_into(plan.K, max(2, round(_SPLIT_TARGET_WORKGROUPS / workgroups)), most)
        wanted = _f16_slices(plan.M, plan.N, plan.O)[0]
        if min(wanted, most) >= 2:
            forms.append(_cut_into(plan.K, wanted, most))
    fp32_us = _fp32_us(plan, *fp32[:2])
    if fp32_us < _ROUTE_MIN_FP32_US:
        return None
    forms = [form for form in forms if form[1] <= _ROUTE_MAX_DEPTH_RATIO * fp32[1]]
    if not forms:
        return None
    route_us, route = min((_route_us(plan, *form[:2]), form) for form in forms)
    if (_ROUTE_ADVANTAGE if route[0] == 1 else _ROUTE_ADVANTAGE_CUT) * route_us >= fp32_us or _backend.norm_gradient_workspace_bytes(plan.params) > 0:
        return None
    return route


def _takes_f16_route(params, slices=1, depth=None):
    """Whether the library wants a workspace for this L1 gradient, or for `slices` of `depth` k each as a batch of one launch."""
    if params.norm_type != _NORM_L1 or not _workspace_enabled():
        return False
    if slices > 1:
        params = type(params).from_buffer_copy(params)
        params.k, params.l = depth, slices
        params.a_bs, params.b_bs, params.c_bs, params.d_bs = depth * params.a_ld, depth, depth, 0
    return _backend.norm_gradient_workspace_bytes(params) > 0


def _cuts_over_contraction(plan):
    """How the call is cut over k: (slices, k per slice, leftover k, whether only with a workspace), the best first.  Behind the cuts for the fp16
    matrix instruction stands the one for the fp32 kernels, which run where the workspace is refused; the last resort is the call as it is."""
    shape = _shape_of_cuts(plan)
    if shape is None:
        return
    workgroups, most = shape
    M, N, O, K = plan.M, plan.N, plan.O, plan.K

    def cut(wanted):
        return _cut_into(K, wanted, most)

    if _takes_f16_route(plan.params):
        filled, wanted = _f16_slices(M, N, O)
        # more slices take more memory: where that is refused, the fewer ones
        for slices in dict.fromkeys((filled, wanted)):
            if min(slices, most) < 2:
                yield 1, K, 0, True
            elif _takes_f16_route(plan.params, *cut(slices)[:2]):
                yield (*cut(slices), True)
    if most >= 2:
        yield (*cut(max(2, round(_SPLIT_TARGET_WORKGROUPS / workgroups))), False)


def _split_over_contraction(plan):
    """(slices, k per slice, leftover k), or None when the call is launched as it is, if all the memory it asks for is granted."""
    best = next(_cuts_over_contraction(plan), None)
    return best[:3] if best is not None and best[0] > 1 else None


def _run_cut(cut, plan, a, b, c, d, p, debug, any_size=False):
    """Launches the call in slices, or returns False with nothing launched: no memory for the partial results, or for the workspace of a
    cut that is none without."""
    slices, depth, leftover, needs_workspace = cut
    if slices == 1:
        return _launch(plan, a.device, debug, needs_workspace, any_size)
    taken = _scratch.mark()
    if _run_slices(slices, depth, leftover, needs_workspace, plan, a, b, c, d, p, debug, any_size):
        return True
    _scratch.give_back_to(taken)
    return False


def _run_slices(slices, depth, leftover, needs_workspace, plan, a, b, c, d, p, debug, any_size=False):
    a2, b2, c2, d2 = (t[0] if t.dim() == 3 else t for t in (a, b, c, d))
    M, N, O = plan.M, plan.N, plan.O
    partial = _scratch.allocate_floats((slices + (1 if leftover else 0), O, N, M), a.device)
    target = plan.out[0] if plan.out.dim() == 4 else plan.out
    # the order in which torch adds the slices depends on the layout of the result: a strided `out` gets the
    # bits of a contiguous one, through a buffer of its own
    staged = None if target.is_contiguous() or partial is None else _scratch.allocate_floats((O, N, M), a.device)
    if partial is None or (staged is None and not target.is_contiguous()):
        return False
    a_slices = a2.as_strided((slices, depth, M), (depth * a2.stride(0), a2.stride(0), a2.stride(1)), a2.storage_offset())
    b_slices = b2.as_strided((slices, N, depth), (depth * b2.stride(1), b2.stride(0), b2.stride(1)), b2.storage_offset())
    c_slices = c2.as_strided((slices, O, depth), (depth * c2.stride(1), c2.stride(0), c2.stride(1)), c2.storage_offset())
    if not _launch(_plan_cdist_grad(a_slices, b_slices, c_slices, d2, partial[:slices], p), a.device, debug, needs_workspace, any_size):
        return False
    if leftover:
        done = slices * depth
        _launch(_plan_cdist_grad(a2[done:], b2[:, done:], c2[:, done:], d2, partial[slices:], p), a.device, debug)
    if staged is None:
        torch.sum(partial, dim=0, out=target)
    else:
        torch.sum(partial, dim=0, out=staged)
        target.copy_(staged)
    return True
