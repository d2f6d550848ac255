"""True exponentials (exact_exp, and with the log-sum-exp): when the running maximum moves.  A key block whose maximum is up to
3.75 octaves above the running one keeps it, and its largest weight is rounded where it is, between 2^5 and 2^8.75; above
that the maximum moves, and the weight is exactly 2^5.  Rows of two keys that count, the second a chosen distance above the
first, show which of the two happened."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu

C = 0.0005                     # octaves per unit of an integer score
UNITS = [90, 124, 126, 127, 128, 130, 200]   # the second key above the first, in steps of 60 * C = 0.03 octaves


@pytest.mark.parametrize("mode", ["exact", "lse"])
@pytest.mark.parametrize("D,H,nb,kept,two_waves", [
    (64, 1600, 2, (0, 1), False),                       # one wave per q-block
    (64, 7, 24, (3, 17), False),                        # two blocks of a list at a time
    (64, 5, 24, (3, 4, 5, 6, 7, 17), False),            # four at a time, the second key in a later round
    (64, 7, 24, (3, 17), True), (128, 14, 24, (3, 9, 17), True), (128, 7, 24, (3, 17), False), (128, 5, 24, (3, 9, 17), False),
])
def test_maximum_moves_beyond_the_headroom(dev, mode, D, H, nb, kept, two_waves):
    import paroatten_amd as P
    N = nb * 64
    q, k, v = torch.zeros(1, H, N, D), torch.zeros(1, H, N, D), torch.zeros(1, H, N, D)
    q[..., 0], q[..., 1] = 60, 127          # (channels 1 of q and 2 of k make both scales exactly 1)
    q[..., 3:9] = 127
    k[..., 2], k[..., 3:9] = 127, -127      # every key is 48 octaves below ...
    step = torch.tensor([UNITS[h % len(UNITS)] for h in range(H)], dtype=torch.float32)
    first, second = 64 * kept[0] + 21, 64 * kept[-1] + 42
    k[..., first, 3:9], k[..., second, 3:9] = 0, 0     # ... but one of the first and one of the last kept block
    k[..., first, 0], k[..., second, 0] = -80, -80 + step
    v[..., first, :] = 1
    mask = torch.zeros(H, nb, nb, dtype=torch.bool)
    mask[..., list(kept)] = True
    out = P.paroattn_qk_int8_pv_fp16_cuda(q.half().to(dev), k.half().to(dev), v.half().to(dev), mask.to(dev), sm_scale=C * math.log(2.0),
                                          smooth_v=False, exact_exp=True, return_lse=mode == "lse", two_waves=two_waves)
    delta = step.double() * 60 * C
    stays = torch.exp2(5 + delta).float().to(torch.float8_e4m3fn).double()
    want = torch.where(delta > 3.75, 1 / (1 + torch.exp2(delta)), 32 / (32 + stays))
    o = (out[0] if mode == "lse" else out).cpu().double()[0]
    # a score enters an exponent with half an ulp of 1.5 * 2^23 * C, once in the weight and once in the maximum; one rounding
    # to the output's 11 bits
    rel = 2 * 0.75 * C * math.log(2.0) + 2.0 ** -11 + 1e-5
    assert ((o - want[:, None, None]).abs() <= rel * want[:, None, None]).all()
    if mode == "lse":
        lse = math.log(2.0) * ((60 * -80) * C + torch.log2(1 + torch.exp2(delta)))
        assert ((out[1].cpu().double()[0] - lse[:, None]).abs() <= 2 * 0.75 * C + 1e-5).all()
