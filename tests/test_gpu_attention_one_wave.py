"""The one-wave kernel (head size 64, where there are enough q-blocks) against the two-wave kernel, bit for bit: rows with no, one,
two, odd and even numbers of kept blocks, a ragged tail, scores that keep moving the running maximum, both exponentials, the
log-sum-exp, causal diagonals, and a number of heads that does not divide among the eight XCDs (whose q-blocks the causal
order deals out one by one)."""
import pytest
import torch

from oracle import paro_oracle as O
from paroatten_amd import _lib as L
from paroatten_amd import _qattn_sm80 as qattn
from paroatten_amd import permute as PM

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["fast", "exact", "lse"])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("B,H", [(1, 448), (1, 451)])
def test_one_wave_equals_two_waves(dev, mode, causal, B, H):
    N, D, nb = 64 * 11 - 21, 64, 11
    assert L.load().paro_attn_kernel_form(B, H, N, N, D, int(causal), int(mode == "lse"),
                                          L.PARO_ATTN_EXACT_EXP if mode == "exact" else 0) == L.PARO_ATTN_FORM_ONE_WAVE
    g = torch.Generator().manual_seed(17)
    q, k, v = (torch.randn(B, H, N, D, generator=g) for _ in range(3))
    k[:, 1::2] *= torch.linspace(0.1, 4.0, N)[:, None]       # the maxima of these heads grow along the row
    mask = torch.rand(H, nb, nb, generator=g) < 0.5
    mask[::4] = True
    for i in range(nb):                                      # row i keeps min(i, kept by causal) blocks
        mask[1::4, i] = (torch.arange(nb) < i)
    k_dev = k.half().to(dev)
    ops = PM.rope_permute_quant(q.half().to(dev), k_dev, v.half().to(dev), torch.zeros(H, dtype=torch.int32, device=dev),
                                (1, 1, N), 0, None, None)
    outs = []
    for two in (False, True):
        o = torch.full((B, H, N, D), float("nan"), dtype=torch.float16, device=dev)
        lse = qattn.attn_sparse_prepacked(ops.q8, ops.k8, ops.v8, ops.v_scale, ops.v_mean, o, ops.q_scale, ops.k_scale,
                                          D ** -0.5, mask.to(dev), is_causal=int(causal), return_lse=int(mode == "lse"),
                                          exact_exp=mode == "exact", two_waves=two)
        outs.append((o.cpu(), lse.cpu() if mode == "lse" else torch.zeros(0)))
    assert torch.isfinite(outs[0][0].float()).all()
    assert torch.equal(outs[0][0], outs[1][0])
    assert torch.equal(outs[0][1], outs[1][1])
    assert torch.count_nonzero(outs[0][0][:, 1, :64]) == 0
    if mode == "lse":
        assert torch.isneginf(outs[0][1][:, 1, :64]).all()
        # two heads against the oracle: exact fp32 sums of the same integer scores
        _, ref = O.sparse_attention(ops.q8[:, :2].cpu(), ops.k8[:, :2].cpu(), v[:, :2].half(), ops.q_scale[:, :2].cpu(),
                                    ops.k_scale[:, :2].cpu(), mask[None, :2].expand(B, 2, nb, nb), D ** -0.5,
                                    is_causal=causal, out_dtype=torch.float32)
        a, r = outs[0][1][:, :2], ref.float()
        fin = torch.isfinite(r) & (r > -1e5)
        # a score enters the exponent as fma(S + 1.5 * 2^23, c, bias) with bias = fp32(m_off - 1.5 * 2^23 * c): half an
        # ulp of the bias, 2^-24 * 1.5 * 2^23 * c, once in the weights and once in the maximum, and 704 fp32 terms
        c = ops.q_scale[:, :2].max() * ops.k_scale[:, :2].max() * D ** -0.5 * O.LOG2E
        assert (a[fin] - r[fin]).abs().max() <= 1.5 * c.item() + 1e-4
