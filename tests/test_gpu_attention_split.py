"""The attention kernel for few q-blocks (several kept key blocks of a q-block at a time) against the two-wave kernel, which
is held to the oracle elsewhere: the same weights, code for code, so that outputs differ by the order of fp32 sums and the
rounding to 16 bits only."""
import pytest
import torch

from paroatten_amd import synth

pytestmark = pytest.mark.gpu


def _close(a, b, v):
    """One unit in the last place of the 16-bit output, and 2^-18 of max|v| for the fp32 sums (a few dozen partial sums,
    each off by 2^-24 of sums of |p v| <= max|v|)."""
    ulp = 2.0 ** -10 if a.dtype == torch.float16 else 2.0 ** -7
    a, b = a.double(), b.double()
    assert torch.isfinite(a).all()
    assert ((a - b).abs() <= ulp * b.abs() + 2.0 ** -18 * float(v.abs().max())).all()


# (B, H, blocks of 64 tokens): four blocks at a time up to 128 q-blocks, two up to 256; 20 blocks is the shortest list
@pytest.mark.parametrize("B,H,nb", [(1, 1, 20), (1, 6, 21), (2, 4, 32), (1, 1, 129), (1, 4, 64)])
@pytest.mark.parametrize("D,dtype", [(64, torch.float16), (128, torch.bfloat16)])
@pytest.mark.parametrize("causal,mode", [(False, "fast"), (True, "fast"), (False, "exact"), (True, "lse")])
def test_same_result_as_two_waves(dev, B, H, nb, D, dtype, causal, mode):
    """Rows of 0, 1, 2 ... kept blocks (so that a round is full, ragged or empty), a last block of 45 tokens."""
    import paroatten_amd as P
    N = nb * 64 - 19
    q, k, v = (t.to(dev) for t in synth.make_qkv(B, H, N, D, dtype, seed=nb))
    mask = synth.make_block_mask(H, nb, 0.4, seed=nb, device=dev)
    for i in range(min(nb, 12)):   # the first rows of head 0 keep i blocks from the diagonal down
        mask[0, i] = False
        for j in range(i):
            mask[0, i, (i - j) % nb] = True
    kw = dict(is_causal=causal, smooth_k=True, exact_exp=mode == "exact", return_lse=mode == "lse")
    a = P.paroattn_qk_int8_pv_fp16_cuda(q, k, v, mask, **kw)
    b = P.paroattn_qk_int8_pv_fp16_cuda(q, k, v, mask, two_waves=True, **kw)
    if mode == "lse":
        finite = torch.isfinite(b[1])
        assert torch.equal(torch.isfinite(a[1]), finite)
        assert ((a[1] - b[1])[finite].abs() <= 1e-5).all()   # log of a sum whose terms are added in another order
        a, b = a[0], b[0]
    _close(a, b, v)
    assert torch.count_nonzero(a[:, 0, :64]) == 0   # the q-block without a kept block


# around the lines of split_width: more than 256 q-blocks, and few key blocks
@pytest.mark.parametrize("B,H,nb,D", [(1, 9, 32, 64), (1, 16, 32, 64), (2, 5, 20, 64), (1, 2, 12, 64), (1, 3, 7, 64), (1, 6, 31, 64),
                                      (1, 3, 2, 128), (1, 8, 16, 128), (1, 9, 15, 128), (2, 2, 64, 128), (1, 5, 1, 128)])
@pytest.mark.parametrize("causal,mode", [(False, "fast"), (True, "exact"), (True, "lse")])
def test_same_result_as_two_waves_around_the_lines(dev, B, H, nb, D, causal, mode):
    from paroatten_amd import _lib as L
    N, lse = nb * 64 - 19, mode == "lse"
    form = L.load().paro_attn_kernel_form(B, H, N, N, D, int(causal), int(lse), L.PARO_ATTN_EXACT_EXP if mode == "exact" else 0)
    assert (form == L.PARO_ATTN_FORM_SPLIT) == (not lse or (nb >= 20 and B * H * nb <= 448))
    test_same_result_as_two_waves(dev, B, H, nb, D, torch.bfloat16, causal, mode)


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("H", [4, 8])
@pytest.mark.parametrize("pattern,causal,density", [("ramp", False, 1.0), ("ramp", True, 1.0), ("ramp", False, 0.5), ("spike", False, 0.5)])
def test_maximum_settled_in_list_order(dev, D, H, pattern, causal, density):
    """Scores that climb by 4.3 octaves a block move the maximum in every block of a round (each wave in turn, the later
    ones after computing their weights again), spikes in single ones; four and two blocks a round."""
    import paroatten_amd as P
    from test_gpu_attention import _ramp_case
    B, nb = 1, 24
    q, k, v = (t.to(dev) for t in _ramp_case(B, H, 64 * nb - 19, D, torch.float16, 7 + D, pattern))
    mask = synth.make_block_mask(H, nb, density, seed=5, device=dev)
    if density == 1.0:
        mask[:] = True
    for exact in (False, True):
        a = P.paroattn_qk_int8_pv_fp16_cuda(q, k, v, mask, is_causal=causal, exact_exp=exact)
        b = P.paroattn_qk_int8_pv_fp16_cuda(q, k, v, mask, is_causal=causal, exact_exp=exact, two_waves=True)
        _close(a, b, v)


def test_grouped_heads_and_unpermuting_store(dev):
    """Grouped heads, keys of another length than the queries, token-major output through the inverse permutation."""
    from paroatten_amd import _qattn_sm80 as qattn, quant as Q
    H, Hkv, D, grid, n_text = 4, 2, 64, (4, 12, 27), 32
    N, Nk = n_text + grid[0] * grid[1] * grid[2], 1500
    q, _, _ = (t.to(dev) for t in synth.make_qkv(1, H, N, D, torch.float16, seed=1))
    _, k, v = (t.to(dev) for t in synth.make_qkv(1, Hkv, Nk, D, torch.float16, seed=2))
    mask = torch.rand(H, (N + 63) // 64, (Nk + 63) // 64, device=dev) < 0.4
    q8, qs, _, _ = Q.per_warp_int8(q, q, None, BLKQ=64, WARPQ=32, BLKK=64)
    _, _, k8, ks = Q.per_warp_int8(k, k, None, BLKQ=64, WARPQ=32, BLKK=64)
    v8, vsc, vm = Q.per_channel_fp8(v)
    orders = torch.tensor([0, 2, 3, 5], dtype=torch.int32, device=dev)
    outs = []
    for two in (False, True):
        o = torch.zeros(1, N, H, D, dtype=torch.float16, device=dev).transpose(1, 2)
        qattn.attn_sparse_prepacked(q8, k8, v8, vsc, vm, o, qs, ks, D ** -0.5, mask, unpermute=(orders, grid, n_text),
                                    two_waves=two)
        outs.append(o)
    _close(outs[0], outs[1], v)


@pytest.mark.parametrize("H,grid,n_text", [(9, (8, 16, 16), 0), (16, (8, 16, 15), 100), (3, (7, 8, 7), 40), (12, (9, 8, 8), 0),
                                           (5, (16, 15, 17), 7)])
def test_layers_stay_with_two_waves_where_those_are_faster(dev, H, grid, n_text):
    """Stores through the inverse permutation: with more than 256 q-blocks below 76 key blocks, and with fewer than 12 key blocks,
    the bits of two waves, which the other order of sums does not give."""
    from paroatten_amd import _qattn_sm80 as qattn
    from paroatten_amd import permute as PM
    N, D = n_text + grid[0] * grid[1] * grid[2], 64
    q, k, v = (t.to(dev) for t in synth.make_qkv(1, H, N, D, torch.float16, seed=N))
    mask = synth.make_block_mask(H, (N + 63) // 64, 0.7, seed=N, device=dev)
    orders = PM.head_orders(synth.make_permute_plan(1, H, seed=3), 0, dev)
    ops = PM.rope_permute_quant(q, k, v, orders, grid, n_text)
    outs = [torch.empty_like(q) for _ in range(2)]
    for two, o in enumerate(outs):
        qattn.attn_sparse_prepacked(ops.q8, ops.k8, ops.v8, ops.v_scale, ops.v_mean, o, ops.q_scale, ops.k_scale, D ** -0.5, mask,
                                    unpermute=(orders, grid, n_text), two_waves=bool(two))
    assert torch.equal(*outs)
