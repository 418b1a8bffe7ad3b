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


def _dense(T, C, g, share=1.0):
    """Inputs of one sequence of T rows of which a share writes a window to a slot of its own."""
    from logssms_amd.kernel.linear_attention.packed_conv import PackedConvStateIO
    x, hist = (randn(*s, g=g, dtype=torch.bfloat16) for s in ((T, C), (1, C, 3)))
    slots = torch.where(torch.rand(T, generator=g) < share, torch.randperm(T, generator=g), -1).to(torch.int32)
    storage = torch.zeros(T, C * 3, dtype=torch.bfloat16, device=DEV)
    table = torch.arange(T, dtype=torch.int32).view(T, 1, 1)
    io = PackedConvStateIO(storage=storage, slots=slots.to(DEV), granules=torch.zeros(T, dtype=torch.int32, device=DEV),
                           final_slots=None, frame_table=table.to(DEV), frame_bytes=C * 6, layer=0)
    return x, hist, slots, io


# the rows of a tile over 32, 8 and 7 blocks and over one (8 channels per thread: 1024 / (tiles x column blocks))
@pytest.mark.parametrize("T,C,share", [(33, 2056, 1.0), (2048, 2056, 0.5), (1153, 8200, 1.0), (16385, 2056, 0.2)])
def test_rows_of_a_tile_spread_over_blocks(T, C, share):
    from logssms_amd.kernel.linear_attention.packed_conv import conv_windows_logstate
    x, hist, slots, io = _dense(T, C, gen(T), share)
    conv_windows_logstate(x.to(DEV), hist.to(DEV), torch.tensor([0, T], device=DEV), io, 4)
    rows = torch.cat([hist[0].t(), x])  # window of row t: the 3 rows ending at t
    want = torch.zeros(T, C, 3, dtype=torch.bfloat16)
    on = slots >= 0
    want[slots[on].long()] = torch.stack([rows[1:T + 1], rows[2:T + 2], rows[3:T + 3]], 2)[on]
    assert torch.equal(io.storage.cpu().view(T, C, 3), want)


def test_every_row_of_a_tile_takes_little_more_than_one():
    """32 windows in one tile: walked by one block they took 12 times as long as one (45 us against 3.6)."""
    from logssms_amd.kernel.linear_attention.packed_conv import conv_windows_logstate

    def us(only_last):
        x, hist, slots, io = _dense(32, 8192, gen(5))
        x, hist, cu = x.to(DEV), hist.to(DEV), torch.tensor([0, 32], device=DEV)
        if only_last:
            io.slots[:-1] = -1
        conv_windows_logstate(x, hist, cu, io, 4)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            for _ in range(20):
                conv_windows_logstate(x, hist, cu, io, 4)
        times = []
        for _ in range(9):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            graph.replay()
            b.record()
            torch.cuda.synchronize()
            times.append(a.elapsed_time(b))
        return sorted(times)[4] * 1e3 / 20

    one, every = us(True), us(False)
    assert every < 4 * one, f"{every:.1f} us for 32 rows, {one:.1f} us for one"
