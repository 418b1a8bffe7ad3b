"""LogState conv windows of a packed prefill (``conv_windows_logstate``), the
16-byte and the per-element form, bit for bit against the oracle's windows."""

import numpy as np
import pytest
import torch

from oracle import frames as ofr
from oracle import gdn as ref
from tests.gpu_util import DEV, gen, randn

pytestmark = pytest.mark.gpu


# 2056 channels: two channel blocks of the 16-byte form, nine of the other
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("scaled", [False, True])
@pytest.mark.parametrize("case", ["vector", "odd_column", "two_frames", "width_3"])
def test_conv_windows_match_oracle(case, scaled, dtype):
    from logssms_amd.kernel.linear_attention.packed_conv import PackedConvStateIO, conv_windows_logstate
    g = gen(7)
    C, width = 2056, 3 if case == "width_3" else 4
    S = width - 1
    lengths = [1, 2, 3, 31, 65]
    T, N = sum(lengths), len(lengths)
    cu = torch.tensor([0] + lengths).cumsum(0)
    granules, slots = 2, T + N
    layers, layer = 2, 1
    frame = 2 * C * S if case == "two_frames" else 2 * layers * C * S + 16
    cf = 2 if case == "two_frames" else 1
    order = torch.randperm(slots * granules * cf, generator=g).to(torch.int32)
    table = order.view(slots, granules, cf).clone()
    table[3, 1] = -1  # an unmapped snapshot takes no write
    storage = randn(slots * granules * cf, frame // 2, g=g, dtype=dtype)
    wide = randn(T, C + 8, g=g, dtype=dtype)
    first = 1 if case == "odd_column" else 0
    x = wide[:, first:first + C]
    hist = randn(N, C, S, g=g, dtype=dtype)
    token_slots = torch.where(torch.rand(T, generator=g) < 0.4, torch.arange(T), -1).to(torch.int32)
    token_slots[:3] = torch.arange(3)  # the first rows of sequences 0 and 1 (windows reach into the history)
    token_granules = torch.randint(0, granules, (T,), generator=g, dtype=torch.int32)
    token_granules[3] = 1
    finals = torch.arange(T, T + N, dtype=torch.int32)
    finals[2] = -1
    scale, xs = {}, x
    if scaled:
        scale = dict(input_boundaries=(100, 1111), input_scales=(0.7, 1.0, 0.45))
        factor = torch.tensor([0.7] * 100 + [1.0] * 1011 + [0.45] * (C - 1111))
        if dtype == torch.float16:  # a mixed-precision multiply: the exact product rounded once
            xs = torch.from_numpy((x.double() * factor.double()).numpy().astype(np.float16))
        else:  # the fp32 product, rounded
            xs = (x.float() * factor).to(dtype)
    weight = randn(C, 1, width, g=g, dtype=dtype)
    _, windows = ref.packed_causal_conv1d(xs, weight, hist, cu)
    want = storage.clone()
    last = {int(cu[i + 1]) - 1: int(finals[i]) for i in range(N)}
    for t in range(T):
        for slot, gr in ((int(token_slots[t]), int(token_granules[t])), (last.get(t, -1), 0)):
            if slot < 0 or int(table[slot, gr, 0]) < 0:
                continue
            idx = ofr.conv_element_index(table, [slot], [gr], layer, C, S, frame // 2)
            want.view(-1)[idx[0]] = windows[t].reshape(-1)
    dev = storage.to(DEV)
    conv_windows_logstate(wide.to(DEV)[:, first:first + C], hist.to(DEV), cu.to(DEV),
                          PackedConvStateIO(storage=dev, slots=token_slots.to(DEV),
                                            granules=token_granules.to(DEV), final_slots=finals.to(DEV),
                                            frame_table=table.to(DEV), frame_bytes=frame, layer=layer),
                          width, **scale)
    assert torch.equal(dev.cpu(), want)
