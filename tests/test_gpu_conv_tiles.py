"""The front end's token tile depends on the packed length (shorter tiles on
short inputs): the tile must not show in the results."""

import pytest
import torch

from oracle import gdn as ref
from tests.gpu_util import DEV, assert_bf16_close, gen, randn

pytestmark = pytest.mark.gpu


# one 2048-channel slab: tiles 2 | 4 | 8 | 12 | ... | 28 | 32 from 1, 2049, 4097, 8193, ..., 24577 and 28673 tokens on
@pytest.mark.parametrize("total", [2048, 2049, 2812, 2813, 4097, 5631, 8193, 11250, 22503, 28672, 28673])
def test_packed_front_end_equals_its_sequences_alone(total):
    from logssms_amd.kernel.linear_attention.fused_backend import prefill_frontend
    from logssms_amd.layers import GatedDeltaConfig
    g = gen(total)
    H, HV, d = 2, 2, 32
    cfg = GatedDeltaConfig(H, HV, d, d, (2 * H + HV) * d, 3, 0)
    lengths = [1, 2, 3, 33, 517, 1030]
    lengths.append(total - sum(lengths))
    mixed = randn(total, cfg.conv_dim, g=g, dtype=torch.bfloat16)
    gate, beta = (randn(total, HV, g=g, dtype=torch.bfloat16) for _ in range(2))
    weight = randn(cfg.conv_dim, 1, 4, g=g, dtype=torch.bfloat16, std=0.3)
    A_log, dt_bias = randn(HV, g=g), randn(HV, g=g)
    pool = randn(len(lengths), 1, cfg.conv_dim, 3, g=g, dtype=torch.bfloat16)
    base = torch.tensor([0, -1, 2, 3, 4, -1, 6])
    cu = torch.tensor([0] + lengths).cumsum(0)

    def front(a, b, cu, base):
        out = prefill_frontend(mixed[a:b].to(DEV), gate[a:b].to(DEV), beta[a:b].to(DEV), weight.to(DEV),
                               A_log.to(DEV), dt_bias.to(DEV), cfg, pool.to(DEV), cu.to(DEV), base.to(DEV))
        return [x[0].cpu() for x in out]

    got = front(0, total, cu, base)
    for i in range(len(lengths) - 1):  # short inputs: the smallest tile
        a, b = int(cu[i]), int(cu[i + 1])
        alone = front(a, b, torch.tensor([0, b - a]), base[i:i + 1])
        for x, y in zip(got, alone):
            assert torch.equal(x[a:b], y)
    hist = torch.where(base[:, None, None] >= 0, pool[base.clamp_min(0), 0], torch.zeros((), dtype=pool.dtype))
    y, _ = ref.packed_causal_conv1d(mixed, weight, hist, cu, window_rows=[])
    want = ref.prepare_gdn(*ref.split_qkv(y[None], H, d, HV, d), gate[None], beta[None], A_log, dt_bias)
    for x, e in zip(got, want):
        assert_bf16_close(x, e[0], rel=1e-2, atol=1e-2)  # the bars of the front end's own tests


# 512 channels a wave: v alone in its wave (2 key heads), v behind q and k in the same wave (1 key head)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("total", [1, 5, 67])
def test_v_does_not_depend_on_the_wave_it_is_in(total, dtype):
    from logssms_amd.kernel.linear_attention.fused_backend import prefill_frontend
    from logssms_amd.layers import GatedDeltaConfig
    g = gen(total)
    HV, d = 2, 128
    v_in = randn(total, HV * d, g=g, dtype=dtype, std=3.0)
    v_in[0, 3], v_in[0, 7], v_in[-1, 11] = float("inf"), float("nan"), torch.finfo(dtype).max
    v_weight = randn(HV * d, 1, 4, g=g, dtype=dtype, std=0.5)
    gate, beta = (randn(total, HV, g=g, dtype=dtype) for _ in range(2))
    A_log, dt_bias = randn(HV, g=g), randn(HV, g=g)
    cu, base = torch.tensor([0, total]), torch.tensor([-1])
    got = []
    for H in (1, 2):
        cfg = GatedDeltaConfig(H, HV, d, d, (2 * H + HV) * d, 3, 0)
        mixed = torch.cat([randn(total, 2 * H * d, g=g, dtype=dtype), v_in], 1)
        weight = torch.cat([randn(2 * H * d, 1, 4, g=g, dtype=dtype, std=0.5), v_weight])
        pool = torch.zeros(1, 1, cfg.conv_dim, 3, dtype=dtype)
        out = prefill_frontend(mixed.to(DEV), gate.to(DEV), beta.to(DEV), weight.to(DEV), A_log.to(DEV),
                               dt_bias.to(DEV), cfg, pool.to(DEV), cu.to(DEV), base.to(DEV))
        got.append(out[2].cpu().view(torch.int16))
    nan = got[0].view(dtype).isnan()
    assert torch.equal(nan, got[1].view(dtype).isnan())
    assert torch.equal(got[0][~nan], got[1][~nan])
