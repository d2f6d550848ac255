"""The work a user of this package has it do, as cases that can be timed and compared.

Four kinds of call, all through the public entry points:

  operator   paroattn_qk_int8_pv_fp16_cuda on 16-bit q, k, v and a block mask (INT8 quantisation of q and k, V
             conversion, block-sparse attention)
  layer      what a diffusion transformer's layer runs on its projections: rope_permute_quant, then
             attn_sparse_prepacked storing through the inverse permutation into a token-major buffer
  processor  a CogVideoX attention processor called on hidden states, projections included
  permute    rope_permute of q and k and permute_inverse of an attention output, the stand-alone kernels

Sizes: the benchmark configurations of paroatten_amd.synth, the sequence lengths and ratios of the operator
benchmark the package follows (N = 8192 / 17776, 48 heads, ratio 0.2 to 0.5), the shapes of the tests, and generic
ragged ones.  A case is a dict of plain values; run() is one pass and returns its outputs whole.
"""
import math

import torch

import paroatten_amd as P
from paroatten_amd import _qattn_sm80 as qattn
from paroatten_amd import permute as PM
from paroatten_amd import rope, synth

DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16}
DEVICE = "cuda"


def _operator(name, B, H, N, D, dtype, density, mask="band", Hkv=None, layout="HND", smooth_k=False, causal=False,
              lse=False, pv_f16=False, exact_exp=False, gran="per_warp"):
    c = {"kind": "operator", "B": B, "H": H, "Hkv": Hkv or H, "N": N, "D": D, "dtype": dtype, "density": density,
         "mask": mask, "layout": layout, "smooth_k": smooth_k, "causal": causal, "lse": lse, "pv_f16": pv_f16,
         "exact_exp": exact_exp, "gran": gran}
    return dict(c, name=name) if name else c


def _gridded(kind, name, B, H, D, grid, n_text, dtype, density=0.3, mask="band", smooth_k=False, pv_f16=False):
    c = {"kind": kind, "B": B, "H": H, "D": D, "F": grid[0], "Hh": grid[1], "W": grid[2], "n_text": n_text,
         "N": n_text + grid[0] * grid[1] * grid[2], "dtype": dtype, "density": density, "mask": mask,
         "smooth_k": smooth_k, "pv_f16": pv_f16}
    return dict(c, name=name) if name else c


def listed():
    return [
        # the smallest call: a few hundred tokens, launches and latency
        _operator("op_416_tokens", 1, 2, 416, 64, "fp16", 0.5, smooth_k=True),
        # one short clip on two heads (the 16 x 16 x 16 configuration): fewer q-blocks than compute units
        _operator("op_4096_two_heads", 1, 2, 4096, 64, "fp16", 0.5, smooth_k=True),
        # the operator benchmark's middle length, its mask generator and ratio
        _operator("op_8192", 1, 48, 8192, 64, "fp16", 0.3, mask="bernoulli"),
        # the CogVideoX-5b self-attention through the operator, with the K mean taken off
        _operator("op_cogvideox", 2, 48, 17776, 64, "fp16", 0.3, smooth_k=True),
        # the same attention with the float16 P.V product, for users who cannot take FP8 rounding
        _operator("op_cogvideox_pv_f16", 2, 48, 17776, 64, "fp16", 0.3, smooth_k=True, pv_f16=True),
        # partial attention whose log-sum-exp is merged elsewhere: token-major, ragged, smoothed
        _operator("op_lse_ragged", 1, 48, 9001, 64, "bf16", 0.5, layout="NHD", smooth_k=True, lse=True),
        # causal, grouped heads, head size 128, every block below the diagonal
        _operator("op_causal_gqa", 2, 32, 8192, 128, "bf16", 1.0, mask="bernoulli", Hkv=8, causal=True),
        # one CogVideoX layer on small latents, called as the pipeline calls it
        _gridded("processor", "processor_small", 2, 4, 64, (4, 16, 24), 226, "bf16", density=0.5),
        # one CogVideoX-5b layer
        _gridded("layer", "layer_cogvideox", 2, 48, 64, (13, 30, 45), 226, "bf16", density=0.2, smooth_k=True),
        # one Wan 2.1 14B layer at 480p, and at 720p with masks of contiguous runs
        _gridded("layer", "layer_wan_480p", 1, 40, 128, (21, 30, 52), 0, "bf16", density=0.3),
        _gridded("layer", "layer_wan_720p", 1, 40, 128, (21, 45, 80), 0, "bf16", density=0.2, mask="window"),
        # RoPE + permutation of q and k and the inverse permutation as passes of their own
        _gridded("permute", "permute_cogvideox", 2, 48, 64, (13, 30, 45), 226, "bf16"),
    ]


MOST_FLOPS = 2.4e13   # about layer_wan_720p, the largest listed case
MOST_ELEMENTS = 4e8   # of one of q, k, v: the same case's


def draw(rng):
    """One more case of the ranges above."""
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    while True:
        kind = rng.choices(("operator", "layer", "processor", "permute"), (5, 3, 1, 1))[0]
        D = rng.choice((64, 64, 128))
        dtype = rng.choice(("fp16", "bf16"))
        B = rng.choice((1, 2))
        density = round(rng.uniform(0.1, 1.0) if rng.random() < 0.3 else rng.uniform(0.15, 0.5), 3)
        mask = rng.choice(("band", "bernoulli", "window"))
        if kind == "operator":
            Hkv = log_int(1, 48)
            H = Hkv
            if rng.random() < 0.2:
                Hkv = max(1, H // 4)
                H = 4 * Hkv
            # what the pv_f16 mode and per-thread scales cannot be combined with is left out
            pv_f16 = rng.random() < 0.2
            c = _operator("", B, H, log_int(100, 33000), D, dtype, density, mask, Hkv, rng.choice(("HND", "HND", "NHD")),
                          smooth_k=rng.random() < 0.5, causal=rng.random() < 0.15, lse=rng.random() < 0.2,
                          pv_f16=pv_f16, exact_exp=not pv_f16 and rng.random() < 0.1,
                          gran="per_thread" if not pv_f16 and rng.random() < 0.1 else "per_warp")
        else:
            D = 64 if kind == "processor" else D
            grid = (rng.randint(2, 21), log_int(6, 45), log_int(8, 80))
            n_text = 0 if D == 128 else rng.choice((0, 32, 226))
            heads = log_int(1, 16 if kind == "processor" else 48)
            c = _gridded(kind, "", B, heads, D, grid, max(n_text, 32) if kind == "processor" else n_text, dtype, density,
                         mask, smooth_k=rng.random() < 0.5, pv_f16=kind != "permute" and rng.random() < 0.15)
        if work(c)["flops"] <= MOST_FLOPS and c["B"] * c["H"] * c["N"] * c["D"] <= MOST_ELEMENTS:
            return c


# ---- inputs --------------------------------------------------------------------------------------------------
def _block_mask(H, nb, kind, density, seed, batch=None):
    """bool [H,nb,nb] (or [batch,H,nb,nb]): a band plus scattered blocks, one contiguous run per row, or independent
    blocks with the last column kept."""
    if kind == "window":
        m = synth.make_window_mask(H, nb, density, device=DEVICE)
    elif kind == "band":
        m = synth.make_block_mask(H, nb, density, seed=seed, device=DEVICE)
    else:
        g = torch.Generator(device=DEVICE).manual_seed(seed)
        m = torch.rand(H, nb, nb, generator=g, device=DEVICE) < density
        m[:, :, -1] = True
    return m if batch is None else m[None].expand(batch, H, nb, nb).contiguous()


def _qkv(B, H, Hkv, N, D, dtype, seed, token_major):
    """q, k, v ~ N(0, 1), a bias per head and channel on k, as [B,N,H,D] memory or [B,H,N,D] memory."""
    g = torch.Generator(device=DEVICE).manual_seed(seed)

    def make(h):
        shape = (B, N, h, D) if token_major else (B, h, N, D)
        return torch.randn(shape, generator=g, device=DEVICE, dtype=torch.float32)
    q, k, v = make(H).to(dtype), make(Hkv), make(Hkv).to(dtype)
    bias = torch.randn(Hkv, D, generator=g, device=DEVICE) * 3.0
    k = (k + (bias if token_major else bias[:, None])).to(dtype)
    return q, k, v


def _grid_of(c):
    return (c["F"], c["Hh"], c["W"])


def _tables(c):
    make = rope.rope_table_cog if c["D"] == 64 else rope.rope_table_wan_real
    return make(c["D"], _grid_of(c), device=DEVICE)


class _Attention(torch.nn.Module):
    """The part of a CogVideoX attention block that a processor uses."""

    def __init__(self, heads, head_dim):
        super().__init__()
        dim = heads * head_dim
        self.heads, self.is_cross_attention = heads, False
        self.to_q, self.to_k, self.to_v = (torch.nn.Linear(dim, dim) for _ in range(3))
        self.norm_q, self.norm_k = torch.nn.LayerNorm(head_dim), torch.nn.LayerNorm(head_dim)
        self.to_out = torch.nn.ModuleList([torch.nn.Linear(dim, dim), torch.nn.Dropout(0.0)])


def prepare(case, seed):
    c = case
    dtype = DTYPES[c["dtype"]]
    nb = (c["N"] + 63) // 64
    s = {"case": c}
    if c["kind"] == "operator":
        s["qkv"] = _qkv(c["B"], c["H"], c["Hkv"], c["N"], c["D"], dtype, seed, c["layout"] == "NHD")
        s["mask"] = _block_mask(c["H"], nb, c["mask"], c["density"], seed + 1)
        return s
    plan = synth.make_permute_plan(1, c["H"], seed=seed + 2)
    s["tables"] = _tables(c)
    if c["kind"] == "processor":
        with torch.random.fork_rng(devices=[torch.device(DEVICE)] if torch.cuda.is_available() else []):
            torch.manual_seed(seed)
            s["attn"] = _Attention(c["H"], c["D"]).to(DEVICE, dtype).eval().requires_grad_(False)
        g = torch.Generator(device=DEVICE).manual_seed(seed + 3)
        dim = c["H"] * c["D"]
        s["hidden"] = torch.randn(c["B"], c["N"] - c["n_text"], dim, generator=g, device=DEVICE).to(dtype)
        s["text"] = torch.randn(c["B"], c["n_text"], dim, generator=g, device=DEVICE).to(dtype)
        proc = P.PARO_CogVideoXAttnProcessor2_0(grid=_grid_of(c), smooth_k=c["smooth_k"], pv_f16=c["pv_f16"])
        proc.permute_plan, proc.i_block, proc.i_timestep = plan, 0, 0
        proc.sparse_mask = _block_mask(c["H"], nb, c["mask"], c["density"], seed + 1)[None, None]
        s["processor"] = proc
        return s
    q, k, v = _qkv(c["B"], c["H"], c["H"], c["N"], c["D"], dtype, seed, True)
    s["qkv"] = tuple(t.transpose(1, 2) for t in (q, k, v))   # the [B,H,N,D] views of token-major projections
    s["orders"] = PM.head_orders(plan, 0, DEVICE)
    if c["kind"] == "layer":
        s["mask"] = _block_mask(c["H"], nb, c["mask"], c["density"], seed + 1)
    else:
        s["attn_out"] = v.transpose(1, 2).contiguous()
    return s


# ---- one pass ------------------------------------------------------------------------------------------------
def _run_layer(s, c):
    q, k, v = s["qkv"]
    cos, sin = s["tables"]
    grid, n_text = _grid_of(c), c["n_text"]
    ops = PM.rope_permute_quant(q, k, v, s["orders"], grid, n_text, cos, sin, km="mean" if c["smooth_k"] else None)
    v8, v_scale, v_mean = ops.v8, ops.v_scale, ops.v_mean
    if c["pv_f16"]:
        _, _, vp = PM.rope_permute(None, None, v, s["orders"], grid, n_text)
        v8, v_scale, v_mean = qattn.v_f16_tiles(vp), None, None
    out = torch.empty((c["B"], c["N"], c["H"], c["D"]), dtype=q.dtype, device=q.device)
    qattn.attn_sparse_prepacked(ops.q8, ops.k8, v8, v_scale, v_mean, out.transpose(1, 2), ops.q_scale, ops.k_scale,
                                c["D"] ** -0.5, s["mask"], unpermute=(s["orders"], grid, n_text), pv_f16=c["pv_f16"])
    return out


def run(state):
    s, c = state, state["case"]
    if c["kind"] == "operator":
        q, k, v = s["qkv"]
        return P.paroattn_qk_int8_pv_fp16_cuda(q, k, v, s["mask"], tensor_layout=c["layout"], is_causal=c["causal"],
                                               qk_quant_gran=c["gran"], return_lse=c["lse"], smooth_k=c["smooth_k"],
                                               exact_exp=c["exact_exp"], pv_f16=c["pv_f16"])
    if c["kind"] == "layer":
        return _run_layer(s, c)
    if c["kind"] == "processor":
        return s["processor"](s["attn"], s["hidden"], s["text"], image_rotary_emb=s["tables"])
    q, k, _ = s["qkv"]
    cos, sin = s["tables"]
    qp, kp, _ = PM.rope_permute(q, k, None, s["orders"], _grid_of(c), c["n_text"], cos, sin)
    return qp, kp, PM.permute_inverse(s["attn_out"], s["orders"], _grid_of(c), c["n_text"])


# ---- what a pass cannot do without ---------------------------------------------------------------------------
def work(case):
    """16-bit q, k, v and the mask read once, the 16-bit output written once; the two products of every kept block
    (half of them when causal), each 2 * 64 * 64 * D operations."""
    c = case
    B, H, N, D = c["B"], c["H"], c["N"], c["D"]
    Hkv = c.get("Hkv", H)
    nb = (N + 63) // 64
    el = B * N * D
    if c["kind"] == "permute":
        tables = 2 * (N - c["n_text"]) * D * 4
        return {"bytes": 2 * 3 * el * H * 2 + tables, "flops": 2 * 3 * el * H}
    blocks = B * H * max(nb, c["density"] * nb * nb) * (0.5 if c.get("causal") else 1.0)
    w = {"bytes": 2 * el * (2 * H + 2 * Hkv) + H * nb * nb, "flops": 4.0 * 64 * 64 * D * blocks}
    if c.get("lse"):
        w["bytes"] += 4 * B * H * N
    if c["kind"] != "operator":
        w["bytes"] += 2 * (N - c["n_text"]) * D * 4
    if c["kind"] == "processor":   # hidden states in and out and the weights instead of q, k, v and o
        dim = H * D
        w = {"bytes": 2 * 2 * B * N * dim + 4 * 2 * dim * dim + H * nb * nb, "flops": w["flops"] + 8.0 * B * N * dim * dim}
    return w


def tolerance(case):
    """Measured on the path itself.
    permute: rotated in fp32 against rotated in fp64, both rounded to 16 bits: relative 1.5e-5 (bf16), 4e-6 (fp16), one
    unit in the last place at most (7e-3, 1e-3).
    Float16 P.V product: the same attention with its key blocks in reverse order differs by 3.9e-4 / 1.0e-3 (fp16 / bf16
    outputs) and 1.8e-3 / 7.8e-3 at most, which is the rounding of weights and outputs to 16 bits.
    FP8 P.V product: in reverse order the weights are rounded to e4m3 against other running maxima and the outputs
    differ by 4.4e-2, 0.3 at most.  Half of that is allowed: who keeps the order of the blocks keeps most codes."""
    f16 = case["dtype"] == "fp16"
    if case["kind"] == "permute":
        return {"rel": 2e-5, "max": 4e-3} if f16 else {"rel": 6e-5, "max": 1.5e-2}
    if case["pv_f16"]:
        return {"rel": 1.6e-3, "max": 8e-3} if f16 else {"rel": 4e-3, "max": 3.2e-2}
    return {"rel": 2e-2, "max": 0.3}
