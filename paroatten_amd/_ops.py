"""The `_ops` submodule of the compiled extension (csrc/torch_binding.cpp) through ctypes, for a tree that has the library
alone (`python paroatten_amd/build.py --no-ext`): the same functions, arguments, checks, kernels and results; a call costs
some tens of microseconds more on the host."""
from __future__ import annotations

import torch
from torch.autograd import forward_ad

from . import _lib
from ._lib import load, ptr, require_gpu, stream_of


def _need(cond, msg):
    if not cond:
        raise RuntimeError(msg)


def _check_mask(sparse, B, H, nbq, nbk):
    _need(sparse.is_cuda, "Tensor sparse must be on CUDA")
    _need(sparse.dtype in (torch.bool, torch.uint8), "Tensor sparse must have dtype (torch::kBool)")
    _need(sparse.is_contiguous(), "Tensor sparse must be contiguous")
    if sparse.dim() == 4:
        _need(tuple(sparse.shape) == (B, H, nbq, nbk),
              f"Tensor sparse must have shape (batch_size, num_qo_heads, {nbq}, {nbk}), got {tuple(sparse.shape)}")
        return sparse.stride(0)
    _need(tuple(sparse.shape) == (H, nbq, nbk),
          f"Tensor sparse must have shape ([batch_size,] num_qo_heads, {nbq}, {nbk}), got {tuple(sparse.shape)}")
    return 0


def _check_heads(H, Hkv, D):
    if D not in (64, 128):
        raise ValueError(f"Unsupported head dim: {D}")
    if Hkv == 0 or H % Hkv != 0:
        raise ValueError(f"num_qo_heads ({H}) must be divisible by num_kv_heads ({Hkv})")


def attn_operator(q, k, v, sparse, tensor_layout, is_causal, qk_quant_gran, sm_scale, return_lse, smooth_k, smooth_v, flags):
    for t, n in ((q, "query"), (k, "key"), (v, "value")):
        _need(t.dim() == 4, f"Tensor {n} must have dimension number (4)")
    sn, sh = (1, 2) if tensor_layout == 0 else (2, 1)
    B, D, H, Hkv, Nq, Nk = q.size(0), q.size(3), q.size(sh), k.size(sh), q.size(sn), k.size(sn)
    _check_heads(H, Hkv, D)
    _need(k.size(0) == B and k.size(3) == D, "Tensor key must have the batch size and head dim of query")
    _need(v.shape == k.shape, "Tensor value must have the shape of key")
    sparse_bs = _check_mask(sparse, B, H, (Nq + 63) // 64, (Nk + 63) // 64)
    out = torch.empty(q.shape, dtype=q.dtype, device=q.device)
    lse = torch.empty((B, H, Nq), dtype=torch.float32, device=q.device) if return_lse else None
    ws = torch.empty(int(load().paro_attn_operator_workspace_bytes(B, H, Hkv, Nq, Nk, D, smooth_k, return_lse, qk_quant_gran,
                                                                   flags)), dtype=torch.uint8, device=q.device)
    strides = [t.stride(d) for t in (q, k, v, out) for d in (0, sh, sn)]
    _lib.on(q).paro_attn_operator(
        ptr(q), ptr(k), ptr(v), _lib.DTYPE_CODE[q.dtype], ptr(out), ptr(sparse), sparse_bs, ptr(lse), ptr(ws), ws.numel(),
        B, H, Hkv, Nq, Nk, D, *strides, int(is_causal), qk_quant_gran, float(sm_scale), int(smooth_k), int(smooth_v), flags,
        stream_of(q))
    return (out, lse) if return_lse else out


def attn_sparse_prepacked(q8, k8, v8, v_scale, v_mean, output, q_scale, k_scale, sm_scale, sparse, is_causal, return_lse, flags,
                          orders, F, Hh, W, n_text):
    pv16 = flags & _lib.PARO_ATTN_PV_F16 != 0
    for t, n in ((q8, "query"), (k8, "key"), (v8, "value"), (output, "output"), (q_scale, "query_scale"),
                 (k_scale, "key_scale"), (v_scale, "v_scale"), (sparse, "sparse")):
        if t is None and n == "v_scale":
            _need(pv16, "Tensor v_scale must be given")
            continue
        _need(t.is_cuda, f"Tensor {n} must be on CUDA")
        _need(t.is_contiguous() or n == "output", f"Tensor {n} must be contiguous")
    _need(q8.dtype == torch.int8 and k8.dtype == torch.int8, "Tensor query/key must have dtype (torch::kInt8)")
    _need(q8.dim() == 4 and k8.dim() == 4, "Tensor query/key must have dimension number (4)")
    B, H, Nq, D = q8.shape
    Hkv, Nk = k8.size(1), k8.size(2)
    _check_heads(H, Hkv, D)
    _need(k8.size(0) == B and k8.size(3) == D, "Tensor key must have the batch size and head dim of query")
    nbq, nbk = (Nq + 63) // 64, (Nk + 63) // 64
    tiles = load().paro_v_f16_bytes if pv16 else load().paro_v_fp8_bytes
    _need(v8.numel() * v8.element_size() == tiles(B, Hkv, Nk, D),
          f"Tensor value has the wrong size for {'float16' if pv16 else 'FP8'} tiles")
    _need(q_scale.dtype == torch.float32 and k_scale.dtype == torch.float32 and tuple(q_scale.shape) == (B, H, nbq * 2)
          and tuple(k_scale.shape) == (B, Hkv, nbk), "Tensor query_scale / key_scale must have shapes (B, H, 2*nbq) / (B, Hkv, nbk)")
    for t in (v_scale, v_mean):
        _need(t is None or (t.is_cuda and t.dtype == torch.float32 and tuple(t.shape) == (B, Hkv, D)),
              "Tensor v_scale / v_mean must have shape (B, Hkv, head_dim)")
    _need(tuple(output.shape) == (B, H, Nq, D) and output.stride(-1) == 1 and output.dtype in _lib.DTYPE_CODE,
          "Tensor output must be float16/bfloat16 [B,H,N,D] with a contiguous last dimension")
    sparse_bs = _check_mask(sparse, B, H, nbq, nbk)
    lse = torch.empty((B, H, Nq), dtype=torch.float32, device=q8.device) if return_lse else torch.empty(0)
    head = (ptr(q8), ptr(k8), ptr(v8), ptr(q_scale), ptr(k_scale), ptr(v_scale), ptr(v_mean), ptr(sparse), sparse_bs, ptr(output),
            _lib.DTYPE_CODE[output.dtype], ptr(lse) if return_lse else None)
    tail = (B, H, Hkv, Nq, Nk, D, *q8.stride()[:3], *k8.stride()[:3], *output.stride()[:3], float(sm_scale), int(is_causal), flags)
    n_scratch = load().paro_attn_scratch_bytes(B, H, Nq, Nk, D, int(is_causal), int(return_lse), flags)
    scratch = torch.empty(n_scratch, dtype=torch.uint8, device=q8.device) if n_scratch else None
    if orders is not None:
        _need(orders.is_cuda and orders.dtype == torch.int32 and orders.dim() == 1 and orders.numel() == H
              and orders.is_contiguous(), f"orders must be a contiguous int32 GPU tensor of {H} entries")
    _lib.on(q8).paro_attn_sparse_scratch_fwd(*head, *tail, ptr(orders), n_text, F, Hh, W, ptr(scratch), stream_of(q8))
    return lse


def _hnd(t, name):
    require_gpu(t, name)
    _need(t.dim() == 4, f"Tensor {name} must have dimension number (4)")
    _need(t.dtype in _lib.DTYPE_CODE, f"Tensor {name} must be float16 or bfloat16")
    _need(t.stride(-1) == 1, f"Tensor {name} must be contiguous at the last dimension")


def _check_orders(orders, H):
    require_gpu(orders, "orders")
    _need(orders.dtype == torch.int32 and orders.dim() == 1 and orders.numel() == H and orders.is_contiguous(),
          f"orders must be a contiguous int32 tensor of {H} entries (one per head)")


def _check_tables(cos, sin, n_img, D):
    if cos is None:
        return
    _need(sin is not None, "cos and sin must be given together")
    for t, n in ((cos, "cos"), (sin, "sin")):
        require_gpu(t, n)
        _need(t.dtype == torch.float32 and tuple(t.shape) == (n_img, D) and t.is_contiguous(),
              f"Tensor {n} must be contiguous float32 of shape ({n_img}, {D})")


def rope_permute(q, k, v, orders, F, Hh, W, n_text, cos, sin):
    given = [t for t in (q, k, v) if t is not None]
    _need(given, "one of q, k, v must be given")
    ref = given[0]
    for t in given:
        _hnd(t, "input")
        _need(t.shape == ref.shape and t.stride() == ref.stride() and t.dtype == ref.dtype,
              "q, k, v must share shape, strides and dtype")
    B, H, N, D = ref.shape
    _check_orders(orders, H)
    _check_tables(cos, sin, F * Hh * W, D)
    outs = [None if t is None else torch.empty((B, H, N, D), dtype=t.dtype, device=t.device) for t in (q, k, v)]
    _lib.on(ref).paro_rope_permute_fwd(
        ptr(q), ptr(k), ptr(v), *map(ptr, outs), _lib.DTYPE_CODE[ref.dtype], ptr(cos), ptr(None if cos is None else sin),
        ptr(orders), B, H, N, D, n_text, F, Hh, W, *ref.stride()[:3], H * N * D, N * D, D, stream_of(ref))
    return outs


def rope_permute_quant(q, k, v, orders, F, Hh, W, n_text, cos, sin, km, compute_km, smooth_v):
    for t, n in ((q, "query"), (k, "key"), (v, "value")):
        _hnd(t, n)
    _need(k.shape == q.shape and v.shape == q.shape and k.dtype == q.dtype and v.dtype == q.dtype,
          "q, k, v must share shape and dtype")
    B, H, N, D = q.shape
    _check_orders(orders, H)
    _check_tables(cos, sin, F * Hh * W, D)
    lib, dev, nb = load(), q.device, (N + 63) // 64
    if compute_km:
        km = torch.empty((B, H, 1, D), dtype=q.dtype, device=dev)
    if km is not None:
        require_gpu(km, "km")
        _need(km.dtype == q.dtype and tuple(km.shape) == (B, H, 1, D) and km.stride(-1) == 1,
              f"Tensor km must have shape ({B}, {H}, 1, {D}) and the dtype of key")
    q8, k8 = (torch.empty((B, H, N, D), dtype=torch.int8, device=dev) for _ in range(2))
    q_scale, k_scale, v_scale, v_mean = (torch.empty(s, dtype=torch.float32, device=dev)
                                         for s in ((B, H, nb * 2), (B, H, nb), (B, H, D), (B, H, D)))
    v8 = torch.empty(int(lib.paro_v_fp8_bytes(B, H, N, D)), dtype=torch.uint8, device=dev)
    need = lib.paro_prep_smooth_workspace_bytes if compute_km else lib.paro_prep_workspace_bytes
    ws = torch.empty(int(need(B, H, N, D)), dtype=torch.uint8, device=dev)
    entry = _lib.on(q).paro_rope_k_mean_permute_quant_fwd if compute_km else _lib.on(q).paro_rope_permute_quant_fwd
    ms = (0, 0) if km is None else (km.stride(0), km.stride(1))
    entry(ptr(q), ptr(k), ptr(v), _lib.DTYPE_CODE[q.dtype], ptr(cos), ptr(None if cos is None else sin), ptr(orders), ptr(km),
          ptr(q8), ptr(q_scale), ptr(k8), ptr(k_scale), ptr(v8), ptr(v_scale), ptr(v_mean), ptr(ws), ws.numel(),
          B, H, N, D, n_text, F, Hh, W, *q.stride()[:3], *k.stride()[:3], *v.stride()[:3], *ms, int(smooth_v), stream_of(q))
    return q8, q_scale, k8, k_scale, v8, v_scale, v_mean if smooth_v else None, km if compute_km else None


def permute_inverse(o, orders, F, Hh, W, n_text, out):
    _hnd(o, "attn_out")
    B, H, N, D = o.shape
    _check_orders(orders, H)
    if out is None:
        out = torch.empty((B, H, N, D), dtype=o.dtype, device=o.device)
    else:
        _hnd(out, "out")
        _need(out.shape == o.shape and out.dtype == o.dtype and out.device == o.device,
              "out must have attn_out's shape, dtype and device")
    _lib.on(o).paro_permute_inv(ptr(o), ptr(out), _lib.DTYPE_CODE[o.dtype], ptr(orders), B, H, N, D, n_text, F, Hh, W,
                                *o.stride()[:3], *out.stride()[:3], stream_of(o))
    return out


def _has_tangent(t):
    return forward_ad._current_level >= 0 and forward_ad.unpack_dual(t).tangent is not None


def head_norm(q, k, q_weight, q_bias, q_eps, k_weight, k_bias, k_eps):
    params = [w for w in (q_weight, q_bias, k_weight, k_bias) if w is not None]
    if (any(type(t) not in (torch.Tensor, torch.nn.Parameter) or not t.is_cuda or t.device != q.device or t.dtype != q.dtype
            or torch._C._functorch.is_functorch_wrapped_tensor(t) or t.is_neg() or t._is_zerotensor()
            or torch.is_grad_enabled() and t.requires_grad or _has_tangent(t) or t.data_ptr() % 16 for t in (q, k, *params))
            or q.dtype not in _lib.DTYPE_CODE or q.dim() != 4 or q.size(-1) not in (64, 128) or q.numel() == 0 or k.shape != q.shape
            or any(w.dim() != 1 or w.numel() != q.size(-1) or not w.is_contiguous() for w in params)
            or not q.transpose(1, 2).is_contiguous() or not k.transpose(1, 2).is_contiguous()
            or torch.is_autocast_enabled() or torch.jit.is_tracing()
            or torch._C._len_torch_dispatch_stack() or torch._C._len_torch_function_stack()):
        return []
    B, H, N, D = q.shape
    qo, ko = (torch.empty((B, N, H, D), dtype=q.dtype, device=q.device) for _ in range(2))
    _lib.on(q).paro_head_norm(ptr(q), ptr(k), ptr(qo), ptr(ko), _lib.DTYPE_CODE[q.dtype], ptr(q_weight), ptr(q_bias),
                              ptr(k_weight), ptr(k_bias), q_eps, k_eps, B * N * H, D, stream_of(q))
    return [qo.transpose(1, 2), ko.transpose(1, 2)]
