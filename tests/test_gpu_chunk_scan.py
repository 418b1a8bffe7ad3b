"""The two-launch chunked rule (records, then the recurrence) against the
one-launch kernel: outputs, v', states and, on LogState frames, the whole
storage, bit for bit; and each of the two forms, chosen by force, against the
oracle and the committed fixture (the tests of test_gpu_chunk.py alone take
whichever form the sizes select)."""

import pytest
import torch

from tests import test_gpu_backend, test_gpu_chunk, test_gpu_fused_prefill
from tests.gpu_util import DEV, gen, rand, randn
from tests.test_gpu_fused_prefill import _cfg, _fused, _setup, _two_step
from tests.test_gpu_logstate_backend import _logstate_world

pytestmark = pytest.mark.gpu

RULE, PREFILL = "gdn_chunk_workspace_bytes", "gdn_prefill_workspace_bytes"


@pytest.fixture
def force(monkeypatch):
    """force(RULE), force(PREFILL): a workspace at every size for that entry
    and none for the other; force(None): none at all."""
    from logssms_amd import _lib

    def set_form(which):
        def workspace(name, device, N, T, H, HV, dk, dv, *log):
            if name != which:
                return None, 0
            n = (T // 64 + N) * HV * (13312 + 512 * -(-dv // 64))
            if name == PREFILL:  # and the front end's outputs, 256-byte aligned
                n += sum(-(-b // 256) * 256 for b in (T * H * dk * 2,) * 2 + (T * HV * dv * 2,) + (T * HV * 4,) * 2)
            return torch.full((n,), 255, dtype=torch.uint8, device=device), n
        monkeypatch.setattr(_lib, "workspace", workspace)

    return set_form


ORACLE_TESTS = [
    (test_gpu_chunk.test_config1_against_token_recurrence,),
    (test_gpu_chunk.test_config1_against_committed_fixture,),
    (test_gpu_chunk.test_varlen_gqa_pool_semantics, (128, 128)),
    (test_gpu_chunk.test_varlen_gqa_pool_semantics, (128, 64)),
    (test_gpu_chunk.test_varlen_gqa_pool_semantics, (64, 64)),
    (test_gpu_chunk.test_varlen_gqa_pool_semantics, (32, 32)),
    (test_gpu_chunk.test_dispatch_style_recurrence_checkpoints_and_graph, [17, 31, 33, 65], torch.float16),
    (test_gpu_chunk.test_dispatch_style_recurrence_checkpoints_and_graph, [17, 31, 33, 65], torch.bfloat16),
    (test_gpu_chunk.test_bf16_pool_and_chunk_aligned_resume,),
    (test_gpu_chunk.test_large_magnitude_values, 1e3),
    (test_gpu_chunk.test_large_magnitude_values, 1e5),
]


@pytest.mark.parametrize("which", [None, RULE], ids=["one_launch", "two_launches"])
@pytest.mark.parametrize("test", ORACLE_TESTS, ids=["-".join([t[0].__name__[5:]] + [str(a) for a in t[1:]])
                                                    for t in ORACLE_TESTS])
def test_each_form_meets_the_oracle(test, which, force):
    print(f"{test[0].__name__}{test[1:]} workspace={which}", flush=True)
    force(which)
    test[0](*test[1:])


CASES = [
    # H, HV, dk, dv, lengths, io, state dtype: ragged chunks, an empty sequence, every width of the kernel
    (2, 4, 128, 128, [1, 63, 64, 65, 0, 200, 128], torch.bfloat16, torch.float32),
    (1, 2, 128, 192, [130, 17], torch.bfloat16, torch.bfloat16),
    (3, 3, 128, 128, [16, 48, 321], torch.float16, torch.float32),
    (4, 4, 64, 64, [191, 2, 64], torch.float16, torch.float16),
    (2, 4, 32, 32, [100, 33, 129], torch.bfloat16, torch.float32),
    (1, 4, 64, 128, [1], torch.bfloat16, torch.float32),
] + [(1, 2, 128, 128, [n % 7 + 1 for n in range(70)], torch.bfloat16, torch.float32)]  # more sequences than lanes


@pytest.mark.parametrize("case", CASES, ids=[f"H{c[0]}_HV{c[1]}_dk{c[2]}_dv{c[3]}_n{len(c[4])}" for c in CASES])
def test_scan_equals_one_launch(case, force):
    from logssms_amd.kernel.linear_attention import ChunkStateIO, chunk_gated_delta_rule_to_cache
    H, HV, dk, dv, lengths, io, sdt = case
    print(f"scan case {case[:4]} lengths={lengths[:8]} io={io} state={sdt}", flush=True)
    g = gen(sum(lengths) + dv)
    T, N = sum(lengths), len(lengths)
    norm = torch.nn.functional.normalize
    q, k = (norm(randn(1, T, H, dk, g=g), dim=-1).to(io).to(DEV) for _ in range(2))
    v = randn(1, T, HV, dv, g=g, dtype=io).to(DEV)
    gate, beta = (-rand(1, T, HV, g=g)).to(DEV), rand(1, T, HV, g=g).to(DEV)
    cu = torch.tensor([0] + lengths).cumsum(0).to(DEV)
    nch = sum(-(-n // 64) for n in lengths)
    pool0 = randn(N + nch + N, 2, HV, dk, dv, g=g, std=0.1).to(sdt).to(DEV)
    reads = torch.tensor([i if i % 3 != 1 else -1 for i in range(N)], dtype=torch.int32, device=DEV)
    writes = torch.tensor([N + c if c % 2 == 0 else -1 for c in range(nch)], device=DEV)
    finals = torch.arange(N + nch, N + nch + N, device=DEV)

    def run(scan):
        force(RULE if scan else None)
        pool = pool0.clone()
        o, vn = chunk_gated_delta_rule_to_cache(q, k, v, gate, beta,
                                                ChunkStateIO(pool, reads, writes, final_write_slots=finals, layer=1), cu)
        return o, vn, pool

    want, got = run(False), run(True)
    torch.cuda.synchronize()
    for name, a, b in zip(("output", "v_new", "states"), got, want):
        assert torch.equal(a, b), name
    assert not torch.equal(got[2], pool0)


@pytest.mark.parametrize("gran,d", [(16, 64), (32, 128), (64, 64), (16, 32)])
def test_scan_equals_one_launch_on_logstate_frames(gran, d, force):
    from logssms_amd.core import Batch, LogStateCacheMetadata, Request
    from logssms_amd.layers import GatedDeltaConfig, GatedDeltaLogStateBackend
    g = gen(500 + gran + d)
    H, HV = 2, 4
    ctx, C = _logstate_world(g, rows=3, page=128, gran=gran, d=d, H=H, HV=HV)
    pool, cfg = ctx.linear_state, GatedDeltaConfig(H, HV, d, d, C, 3, 0)
    lens, cached = [70, 45, 129], [0, 20, 64]
    T = sum(lens)
    mixed = randn(T, C, g=g, dtype=torch.bfloat16, std=0.5).to(DEV)
    gate, beta = (randn(T, HV, g=g, dtype=torch.bfloat16).to(DEV) for _ in range(2))
    weight = randn(C, 1, 4, g=g, dtype=torch.bfloat16, std=0.3).to(DEV)
    A_log, dt_bias = -rand(HV, g=g).to(DEV), randn(HV, g=g).to(DEV)
    start = pool.storage.clone()

    def run(scan):
        force(RULE if scan else None)
        pool.storage.copy_(start)
        # (checkpoints into log slots no token of the batch is logged to)
        pos = torch.cat([torch.arange(k, k + n, dtype=torch.int32) for n, k in zip(lens, cached)]).to(DEV)
        batch = Batch([Request(i, k, k + n) for i, (n, k) in enumerate(zip(lens, cached))], "prefill", positions=pos,
                      out_loc=pos, cache_metadata=LogStateCacheMetadata(checkpoint_writes=[(31, 1), (63, 3)]))
        backend = GatedDeltaLogStateBackend(ctx)
        backend.prepare_metadata(batch)
        out = backend.forward(mixed, gate, beta, weight, A_log, dt_bias, cfg, batch)
        torch.cuda.synchronize()
        return out, pool.storage.clone()

    print(f"scan on LogState frames gran={gran} d={d}", flush=True)
    want, got = run(False), run(True)
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
    assert not torch.equal(got[1], start)


@pytest.mark.parametrize("case", test_gpu_fused_prefill.CASES,
                         ids=[f"H{c[0]}_HV{c[1]}_dk{c[2]}_dv{c[3]}_{str(c[5])[6:]}_{str(c[6])[6:]}"
                              for c in test_gpu_fused_prefill.CASES])
def test_split_prefill_equals_two_step_path(case, force):
    force(PREFILL)
    test_gpu_fused_prefill.test_fused_prefill_equals_two_step_path(case)


def test_split_prefill_pool_offsets_beyond_2gib(force):
    force(PREFILL)
    test_gpu_fused_prefill.test_prefill_pool_offsets_beyond_2gib()


def test_split_prefill_writes_windows_after_reading_history(force):
    force(PREFILL)
    test_gpu_backend.test_prefill_resuming_mid_page_writes_windows_after_reading_history((128, 128))


def _strided(w, cfg, head_stride):
    """The projections as column slices of one wider buffer, as the layer passes them."""
    T, C = w["mixed"].shape
    HV = cfg.num_v_heads
    wide = torch.empty(T, C + 8 + 2 * HV * head_stride, dtype=w["mixed"].dtype, device=DEV)
    parts = dict(mixed=wide[:, 8:8 + C], gate=wide[:, 8 + C:8 + C + HV * head_stride:head_stride],
                 beta=wide[:, 8 + C + HV * head_stride::head_stride])
    for name, part in parts.items():
        part.copy_(w[name])
    return {**w, **parts}


@pytest.mark.parametrize("head_stride", [1, 2])
def test_split_prefill_takes_row_strided_projections(head_stride, monkeypatch):
    from logssms_amd import _lib
    cfg = _cfg(2, 4, 128, 128)
    calls = []
    real = _lib.call
    monkeypatch.setattr(_lib, "call", lambda name, *a: (calls.append(name), real(name, *a))[1])
    results = []
    for strided in (False, True):
        pool, w, meta = _setup(cfg, [1, 900, 130], gen(62))
        if strided:
            w = _strided(w, cfg, head_stride)
            assert not w["mixed"].is_contiguous() and not w["gate"].is_contiguous()
        calls.clear()
        o = _fused(cfg, pool, w, meta) if strided else _two_step(cfg, pool, w, meta)
        torch.cuda.synchronize()
        if strided:
            assert calls == ["gdn_prefill_split"]
        results.append((o, pool.conv_state, pool.recurrent_state))
    for a, b in zip(*results):
        assert torch.equal(a, b)


@pytest.mark.parametrize("shape", [(1, 2, 128, [700]), (2, 2, 64, [300, 129])])
def test_split_prefill_is_chosen_and_equals_two_step(shape, monkeypatch):
    """Shapes the rule gives to ``gdn_prefill_split``: equal to the front end
    followed by the one-launch kernel, also from a captured graph whose inputs
    change between replays."""
    from logssms_amd import _lib
    H, HV, d, lengths = shape
    cfg = _cfg(H, HV, d, d)
    calls = []
    real = _lib.call
    monkeypatch.setattr(_lib, "call", lambda name, *a: (calls.append(name), real(name, *a))[1])
    pool, w, meta = _setup(cfg, lengths, gen(61))
    conv0, state0 = pool.conv_state.clone(), pool.recurrent_state.clone()

    def reset():
        pool.conv_state.copy_(conv0)
        pool.recurrent_state.copy_(state0)

    def two_step():
        reset()
        with monkeypatch.context() as mp:
            mp.setattr(_lib, "workspace", lambda *a: (None, 0))
            o = _two_step(cfg, pool, w, meta).clone()
        return o, pool.conv_state.clone(), pool.recurrent_state.clone()

    want = two_step()
    reset()
    calls.clear()
    got = _fused(cfg, pool, w, meta)
    assert calls == ["gdn_prefill_split"]
    torch.cuda.synchronize()
    assert all(torch.equal(a, b) for a, b in zip((got, pool.conv_state, pool.recurrent_state), want))
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = _fused(cfg, pool, w, meta)
    for i in range(3):
        w["mixed"].mul_(0.5 + i)
        want = two_step()
        reset()
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip((out, pool.conv_state, pool.recurrent_state), want)), i
    graph.reset()
