"""GPU test of the operator in one native call (paro_attn_operator) against the chain of its parts: the quantisers and the
extension entry point, each of which has its own parity tests against the oracle."""
import pytest
import torch

from paroatten_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,D,layout,groups,mode", [
    (1, 64, "HND", 1, "fp8"), (63, 64, "NHD", 2, "fp8"), (64, 128, "HND", 1, "fp8"), (65, 64, "HND", 1, "f16"),
    (129, 128, "NHD", 1, "f16"), (257, 64, "HND", 2, "thread"), (300, 128, "NHD", 1, "thread"), (1000, 64, "HND", 1, "fp8"),
])
@pytest.mark.parametrize("smooth_k", [False, True])
def test_operator_equals_the_chain_of_its_parts(dev, N, D, layout, groups, mode, smooth_k):
    """Edges of the groups of 32 and 64 tokens, of four groups per workgroup and of the statistics chunks; both layouts,
    grouped heads, every product and granularity, with and without the mean and the log-sum-exp."""
    import paroatten_amd as P
    from paroatten_amd import _qattn_sm80 as qattn
    from paroatten_amd import quant as Q
    B, Hkv, dtype = 2, 2, torch.float16 if D == 64 else torch.bfloat16
    H, nb, sd = Hkv * groups, (N + 63) // 64, 2 if layout == "HND" else 1
    g = torch.Generator().manual_seed(N + D)

    def make(h):   # multiples of 1/8 below 8: sums of up to 1000 of them are exact in fp32, whatever their order
        shape = (B, h, N, D) if layout == "HND" else (B, N, h, D)
        return (torch.randint(-63, 64, shape, generator=g) / 8).to(dtype).to(dev)
    q, k, v = make(H), make(Hkv), make(Hkv)
    mask = synth.make_block_mask(H, nb, 0.6, seed=N, device=dev)
    km = k.double().mean(dim=sd, keepdim=True).float().to(dtype) if smooth_k else None
    if mode == "thread":
        q8, qs, k8, ks = Q.per_thread_int8(q, k, km, tensor_layout=layout)
    else:
        q8, qs, k8, ks = Q.per_warp_int8(q, k, km, BLKQ=64, WARPQ=32, BLKK=64, tensor_layout=layout)
    kw = dict(pv_f16=mode == "f16")
    args = (0 if layout == "NHD" else 1, 0, 3 if mode == "thread" else 2, D ** -0.5)
    o_ref = torch.empty_like(q)
    qattn.qk_int8_sv_f16_accum_f16_attn(q8, k8, v, o_ref, qs, ks, *args, 0, mask, **kw)
    o_lse_ref = torch.empty_like(q)
    lse2 = qattn.qk_int8_sv_f16_accum_f16_attn(q8, k8, v, o_lse_ref, qs, ks, *args, 1, mask, **kw)
    call = dict(tensor_layout=layout, smooth_k=smooth_k, qk_quant_gran="per_thread" if mode == "thread" else "per_warp", **kw)
    assert torch.equal(P.paroattn_qk_int8_pv_fp16_cuda(q, k, v, mask, **call), o_ref)
    o, lse = P.paroattn_qk_int8_pv_fp16_cuda(q, k, v, mask, return_lse=True, **call)
    assert torch.equal(o, o_lse_ref)
    want = lse2.double() * 0.6931471805599453
    scale = want.abs()
    if smooth_k:
        qh = q if layout == "HND" else q.transpose(1, 2)
        kh = (km if layout == "HND" else km.transpose(1, 2)).repeat_interleave(groups, dim=1).double()
        corr = (qh.double() * kh).sum(-1) * D ** -0.5
        want = want + corr
        scale = scale + (qh.double() * kh).abs().sum(-1) * D ** -0.5
    # one product and one sum in fp32, and an fp32 dot product of D terms
    assert ((lse.double() - want).abs() <= (D + 4) * 2.0 ** -24 * scale + 1e-30).all()


@pytest.mark.parametrize("N,D,H,mode", [
    (1, 64, 3, "fp8"), (64, 128, 3, "f16"), (255, 64, 3, "fp8"), (256, 128, 3, "fp8"), (257, 64, 3, "f16"), (513, 128, 3, "fp8"),
    (1023, 64, 3, "fp8"), (1024, 64, 3, "fp8"), (1024, 128, 3, "fp8"),
    (1025, 64, 3, "fp8"), (2000, 64, 3, "f16"), (4096, 128, 3, "fp8"), (4097, 64, 3, "fp8"), (8192, 64, 9, "fp8"),
    (1000, 64, 60, "fp8"), (1024, 128, 60, "f16"), (700, 128, 60, "fp8"), (300, 128, 110, "fp8"), (300, 64, 180, "fp8"),
    (1024, 64, 42, "fp8"), (1024, 64, 43, "fp8"), (1024, 64, 86, "fp8"), (1024, 64, 150, "fp8"), (769, 128, 51, "fp8"),
    (512, 128, 102, "fp8"), (513, 128, 52, "fp8"), (768, 64, 64, "f16"), (769, 64, 51, "f16"), (512, 128, 170, "f16"), (1, 64, 180, "fp8"),
])
@pytest.mark.parametrize("smooth_k,smooth_v", [(False, True), (True, True), (True, False)])
def test_one_launch_preparation_equals_the_separate_ones(dev, N, D, H, mode, smooth_k, smooth_v):
    """Edges of the 64-token tiles, the 256-token chunks and the 1024 tokens of the one-launch preparation; K by 256 tokens
    (3 heads, 42 at N = 1024), by heads (43, 60; in two rounds 102, 150), and more heads than it takes; there and beyond, the
    preparation that adds up the chunks itself, at its edges of 4096 and (512 channels) 8192 tokens.  K's sums are exact, V is
    arbitrary: the same bits."""
    import paroatten_amd as P
    from paroatten_amd import _qattn_sm80 as qattn
    from paroatten_amd import quant as Q
    dtype = torch.bfloat16 if N % 2 else torch.float16
    g = torch.Generator(device=dev).manual_seed(N + D + H)
    q, v = (torch.randn(1, H, N, D, generator=g, device=dev).to(dtype) for _ in range(2))
    v = v + torch.randn(1, H, 1, D, generator=g, device=dev).to(dtype)
    k = (torch.randint(-63, 64, (1, H, N, D), generator=g, device=dev) / 8).to(dtype)
    mask = synth.make_block_mask(H, (N + 63) // 64, 0.6, seed=N, device=dev)
    km = k.double().mean(dim=2, keepdim=True).float().to(dtype) if smooth_k else None
    q8, qs, k8, ks = Q.per_warp_int8(q, k, km, BLKQ=64, WARPQ=32, BLKK=64, tensor_layout="HND")
    o_ref = torch.empty_like(q)
    qattn.qk_int8_sv_f16_accum_f16_attn(q8, k8, v, o_ref, qs, ks, 1, 0, 2, D ** -0.5, 0, mask, pv_f16=mode == "f16",
                                        smooth_v=smooth_v)
    got = P.paroattn_qk_int8_pv_fp16_cuda(q, k, v, mask, smooth_k=smooth_k, smooth_v=smooth_v, pv_f16=mode == "f16")
    assert torch.equal(got, o_ref)


@pytest.mark.parametrize("N,D,dtype", [(416, 64, torch.float16), (2000, 128, torch.bfloat16), (32760, 128, torch.float16)])
def test_k_mean_is_the_rounded_mean(dev, N, D, dtype):
    """The K mean that the operator takes is the one that 64-bit sums round to, on inputs of which sums in one fp32
    accumulator per thread give a few channels the neighbouring value."""
    import paroatten_amd as P
    from paroatten_amd import _qattn_sm80 as qattn
    from paroatten_amd import quant as Q
    H, nb = 64, (N + 63) // 64
    g = torch.Generator(device=dev).manual_seed(N)
    k = (torch.randn(H, N, D, generator=g, device=dev) + 3 * torch.randn(H, 1, D, generator=g, device=dev)).to(dtype)[None]
    q, v = k[..., :64, :].contiguous(), k.flip(2).contiguous()
    mask = torch.ones(H, 1, nb, dtype=torch.bool, device=dev)
    km = k.double().mean(dim=2, keepdim=True).to(dtype)
    q8, qs, k8, ks = Q.per_warp_int8(q, k, km, BLKQ=64, WARPQ=32, BLKK=64)
    o_ref = torch.empty_like(q)
    qattn.qk_int8_sv_f16_accum_f16_attn(q8, k8, v, o_ref, qs, ks, 1, 0, 2, D ** -0.5, 0, mask, two_waves=True)
    assert torch.equal(P.paroattn_qk_int8_pv_fp16_cuda(q, k, v, mask, smooth_k=True, two_waves=True), o_ref)


@pytest.mark.parametrize("B,H,smooth_k", [(32769, 1, True), (1, 32769, False)])
def test_operator_batch_and_head_counts_of_16_bits(dev, B, H, smooth_k):
    """Batch and head counts above half a grid dimension, as the quantisers and the V conversion take them: the same as the
    last 1100 batch entries or heads by themselves (both calls have more than the 1024 q-blocks of the split kernels)."""
    import paroatten_amd as P
    g = torch.Generator(device=dev).manual_seed(3)
    q, k, v = (torch.randn(B, H, 17, 64, generator=g, device=dev).half() for _ in range(3))
    mask = torch.ones(H, 1, 1, dtype=torch.bool, device=dev)
    kw = dict(tensor_layout="HND", smooth_k=smooth_k)
    o = P.paroattn_qk_int8_pv_fp16_cuda(q, k, v, mask, **kw)
    tail = (slice(-1100, None),) if B > 1 else (slice(None), slice(-1100, None))
    part = P.paroattn_qk_int8_pv_fp16_cuda(q[tail].contiguous(), k[tail].contiguous(), v[tail].contiguous(),
                                           mask if B > 1 else mask[-1100:], **kw)
    assert torch.equal(o[tail], part)


@pytest.mark.parametrize("H,N,D,form,causal", [
    (2, 1345, 64, "SPLIT", False), (2, 1345, 128, "SPLIT", True), (6, 1345, 128, "SPLIT", False),
    (75, 1345, 64, "ONE_WAVE", False), (200, 1345, 64, "ONE_WAVE", True), (30, 700, 64, "TWO_WAVES", True),
    (90, 1345, 64, "PACED", False), (60, 1345, 128, "PACED", True),
])
@pytest.mark.parametrize("lse", [False, True])
def test_queries_quantised_by_every_kernel_form(dev, monkeypatch, H, N, D, form, causal, lse):
    """The operator's attention kernels read 16-bit queries and quantise them themselves: the same bits as on queries that
    the quantiser has made, in every form, with a last q-block of one row, an empty row of the mask and queries of zero."""
    import paroatten_amd as P
    from paroatten_amd import _lib
    from paroatten_amd import _qattn_sm80 as qattn
    from paroatten_amd import quant as Q
    if form == "PACED":
        monkeypatch.setenv("PARO_ATTN_PACING", "1")
    assert _lib.load().paro_attn_kernel_form(1, H, N, N, D, int(causal), int(lse), 0) == getattr(_lib, "PARO_ATTN_FORM_" + form)
    g = torch.Generator(device=dev).manual_seed(N + D + H)
    q, k, v = (torch.randn(1, H, N, D, generator=g, device=dev).to(torch.bfloat16) for _ in range(3))
    q[:, 0, 64:96] = 0
    mask = synth.make_block_mask(H, (N + 63) // 64, 0.4, seed=N, device=dev)
    mask[1, 2] = False
    q8, qs, k8, ks = Q.per_warp_int8(q, k, None, BLKQ=64, WARPQ=32, BLKK=64, tensor_layout="HND")
    o_ref = torch.empty_like(q)
    lse2 = qattn.qk_int8_sv_f16_accum_f16_attn(q8, k8, v, o_ref, qs, ks, 1, int(causal), 2, D ** -0.5, int(lse), mask)
    got = P.paroattn_qk_int8_pv_fp16_cuda(q, k, v, mask, is_causal=causal, smooth_k=False, return_lse=lse)
    assert torch.equal(got[0] if lse else got, o_ref)
    if lse:
        assert torch.equal(got[1], lse2 * 0.6931471805599453)


@pytest.mark.parametrize("B,H,Hkv,N,D,form,causal", [
    (1, 4, 2, 1345, 64, "SPLIT", False), (2, 3, 1, 1345, 128, "SPLIT", True), (2, 15, 5, 700, 64, "TWO_WAVES", False),
    (3, 20, 10, 700, 128, "TWO_WAVES", True), (3, 25, 5, 1345, 64, "ONE_WAVE", False), (2, 100, 25, 1345, 64, "ONE_WAVE", True),
    (3, 30, 6, 1345, 64, "PACED", False), (3, 32, 8, 1345, 64, "PACED", True), (2, 30, 10, 1345, 128, "PACED", False),
    (2, 6, 2, 700, 64, "PV_F16", False), (2, 6, 3, 700, 128, "PV_F16", True),
])
def test_log_sum_exp_with_the_k_mean_in_every_kernel_form(dev, monkeypatch, B, H, Hkv, N, D, form, causal):
    """sm_scale * q . k_mean, which the attention kernels put into the row of the log-sum-exp before their loop and add to at
    its end: every form, grouped heads in a batch (the mean is that of the row's key head), token-major, a last q-block of
    one row (N = 1345) and an empty row of the mask.  K's sums are exact, so that its mean, and the outputs, are the same bits."""
    import paroatten_amd as P
    from paroatten_amd import _lib
    from paroatten_amd import _qattn_sm80 as qattn
    from paroatten_amd import quant as Q
    pv_f16 = form == "PV_F16"
    if form == "PACED":
        monkeypatch.setenv("PARO_ATTN_PACING", "1")
    flags = qattn._flags(False, None, False, pv_f16)
    assert _lib.load().paro_attn_kernel_form(B, H, N, N, D, int(causal), 1, flags) == getattr(_lib, "PARO_ATTN_FORM_" + form)
    dtype = torch.float16 if D == 64 else torch.bfloat16
    g = torch.Generator(device=dev).manual_seed(N + D + H)
    q, v = (torch.randn(B, N, h, D, generator=g, device=dev).to(dtype) for h in (H, Hkv))
    k = ((torch.randint(-40, 41, (B, N, Hkv, D), generator=g, device=dev)
          + torch.randint(-20, 21, (B, 1, Hkv, D), generator=g, device=dev)) / 8).to(dtype)
    mask = synth.make_block_mask(H, (N + 63) // 64, 0.4, seed=N, device=dev)
    mask[1, 2] = False
    km = k.double().mean(dim=1, keepdim=True).float().to(dtype)
    q8, qs, k8, ks = Q.per_warp_int8(q, k, km, BLKQ=64, WARPQ=32, BLKK=64, tensor_layout="NHD")
    o_ref = torch.empty_like(q)
    lse2 = qattn.qk_int8_sv_f16_accum_f16_attn(q8, k8, v, o_ref, qs, ks, 0, int(causal), 2, D ** -0.5, 1, mask, pv_f16=pv_f16)
    o, lse = P.paroattn_qk_int8_pv_fp16_cuda(q, k, v, mask, tensor_layout="NHD", is_causal=causal, smooth_k=True,
                                             return_lse=True, pv_f16=pv_f16)
    assert torch.equal(o, o_ref)
    terms = q.transpose(1, 2).double() * km.transpose(1, 2).repeat_interleave(H // Hkv, dim=1).double()
    want = lse2.double() * 0.6931471805599453 + terms.sum(-1) * D ** -0.5
    empty = lse2 == -float("inf")
    assert empty[:, 1, 128:192].all() and torch.equal(lse == -float("inf"), empty)
    # one product and one sum in fp32, and an fp32 dot product of D terms
    bound = (D + 4) * 2.0 ** -24 * (lse2.double().abs() + terms.abs().sum(-1) * D ** -0.5)
    assert ((lse.double() - want).abs() <= bound)[~empty].all()


@pytest.mark.parametrize("H,Hkv,Nq,Nk,D,mode", [
    (4, 2, 1, 1, 64, "f16"), (3, 1, 33, 33, 128, "f16"), (2, 2, 4096, 4096, 64, "f16"), (3, 3, 2752, 2752, 64, "f16"),
    (4, 4, 4096, 4096, 128, "f16"), (4, 2, 65, 4200, 64, "fp8"), (6, 3, 1, 4097, 128, "fp8"), (9, 3, 129, 8200, 128, "exact"),
    (2, 1, 4097, 4097, 64, "fp8"), (1, 1, 8200, 8200, 64, "fp8"), (3, 1, 95, 5000, 64, "f16"),
])
@pytest.mark.parametrize("smooth_k", [False, True])
def test_queries_in_a_pass_of_their_own(dev, H, Hkv, Nq, Nk, D, mode, smooth_k):
    """With few q-blocks and a preparation launch that takes K and V tile by tile, Q is quantised in that launch: token-major,
    grouped heads, last groups of one row, both sides of the lines (128 q-blocks at D = 64, 256 at 128; 4096 keys where there is
    something to sum up).  K's sums are exact: the same bits as the chain of its parts, and the log-sum-exp within its bound."""
    import paroatten_amd as P
    from paroatten_amd import _qattn_sm80 as qattn
    from paroatten_amd import quant as Q
    dtype = torch.bfloat16 if Nk % 2 else torch.float16
    g = torch.Generator(device=dev).manual_seed(Nq + Nk + D + H)
    q = torch.randn(2 if Nq < 4000 else 1, Nq, H, D, generator=g, device=dev).to(dtype)
    B = q.size(0)
    v = torch.randn(B, Nk, Hkv, D, generator=g, device=dev).to(dtype)
    k = (torch.randint(-63, 64, (B, Nk, Hkv, D), generator=g, device=dev) / 8).to(dtype)
    mask = torch.rand(H, (Nq + 63) // 64, (Nk + 63) // 64, generator=g, device=dev) < 0.4
    mask[:, :, 0] = True
    km = k.double().mean(dim=1, keepdim=True).float().to(dtype) if smooth_k else None
    q8, qs, k8, ks = Q.per_warp_int8(q, k, km, BLKQ=64, WARPQ=32, BLKK=64, tensor_layout="NHD")
    kw = dict(pv_f16=mode == "f16", exact_exp=mode == "exact")
    o_ref, o_lse_ref = torch.empty_like(q), torch.empty_like(q)
    args = (0, 0, 2, D ** -0.5)
    qattn.qk_int8_sv_f16_accum_f16_attn(q8, k8, v, o_ref, qs, ks, *args, 0, mask, **kw)
    lse2 = qattn.qk_int8_sv_f16_accum_f16_attn(q8, k8, v, o_lse_ref, qs, ks, *args, 1, mask, **kw)
    call = dict(tensor_layout="NHD", smooth_k=smooth_k, **kw)
    assert torch.equal(P.paroattn_qk_int8_pv_fp16_cuda(q, k, v, mask, **call), o_ref)
    o, lse = P.paroattn_qk_int8_pv_fp16_cuda(q, k, v, mask, return_lse=True, **call)
    assert torch.equal(o, o_lse_ref)
    want, scale = lse2.double() * 0.6931471805599453, lse2.double().abs()
    if smooth_k:
        terms = q.transpose(1, 2).double() * km.transpose(1, 2).repeat_interleave(H // Hkv, dim=1).double()
        want = want + terms.sum(-1) * D ** -0.5
        scale = scale + terms.abs().sum(-1) * D ** -0.5
    # one product and one sum in fp32, and an fp32 dot product of D terms
    assert ((lse.double() - want).abs() <= (D + 4) * 2.0 ** -24 * scale + 1e-30).all()


@pytest.mark.parametrize("N,D,H,dtype", [
    (1025, 64, 1, torch.float16), (1473, 64, 2, torch.bfloat16), (2049, 64, 12, torch.float16), (4033, 64, 8, torch.float16),
    (4096, 64, 2, torch.bfloat16), (4097, 64, 2, torch.float16),
    (1025, 128, 1, torch.float16), (2047, 128, 4, torch.bfloat16), (4096, 128, 2, torch.bfloat16), (4096, 128, 3, torch.float16),
])
@pytest.mark.parametrize("with_lse", [False, True])
def test_residual_sums_in_the_attention_launch(dev, N, D, H, dtype, with_lse):
    """Both sides of the rule by which the kernel of few q-blocks adds up what v_mean lacks: a V with a mean beside a wide channel, so
    that the sums matter, against the extension entry point, which has a launch of their own for them.  The same bits."""
    import paroatten_amd as P
    from paroatten_amd import _qattn_sm80 as qattn
    from paroatten_amd import quant as Q
    g = torch.Generator().manual_seed(N + D)
    q, k, v = ((torch.randint(-63, 64, (1, H, N, D), generator=g) / 8).to(dtype).to(dev) for _ in range(3))
    v[..., ::3] += 5
    nb = (N + 63) // 64
    mask = synth.make_block_mask(H, nb, 0.6, seed=N, device=dev)
    mask[0, 1] = False
    q8, qs, k8, ks = Q.per_warp_int8(q, k, None, BLKQ=64, WARPQ=32, BLKK=64, tensor_layout="HND")
    ref = torch.empty_like(q)
    qattn.qk_int8_sv_f16_accum_f16_attn(q8, k8, v, ref, qs, ks, 1, 0, 2, D ** -0.5, int(with_lse), mask)
    got = P.paroattn_qk_int8_pv_fp16_cuda(q, k, v, mask, return_lse=with_lse)
    assert torch.equal(got[0] if with_lse else got, ref)
