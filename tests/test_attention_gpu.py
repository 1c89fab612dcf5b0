"""Segmented-KV GQA attention vs the FP32 SDPA-math oracle (MI355X only).

Cases follow tests/e2e/test_compact_attention.py of the reference (history
(2049, 0, 575): empty middle segment and a ragged tail; current-segment V
token stride 6144; graph replay after in-place updates; non-default stream)
and BASELINE config 5 (history 1024/512/256, T in {32, 96, 256}).
"""
import ctypes

import pytest
import torch

from llm_gpu_kernels_amd import _native as N, prepare_segmented_gqa, prepare_cuda_gqa_compact
from oracle import moe_oracle as O

pytestmark = pytest.mark.gpu
LIMITS = {"relative_rms": 5e-3, "normalized_max": 1e-2}


def _values(seed, tokens, history, device, v_stride=None, hq=32, hkv=8):
    g = torch.Generator().manual_seed(seed)

    def rnd(shape):
        return torch.randn(shape, generator=g).to(torch.bfloat16).to(device)

    q = rnd((tokens, hq, 128))
    segs = [(rnd((L, hkv, 128)), rnd((L, hkv, 128))) for L in (*history, tokens)]
    if v_stride:
        k, v = segs[-1]
        pv = torch.empty_strided(tuple(v.shape), (v_stride, 128, 1), dtype=v.dtype, device=device)
        pv.copy_(v)
        segs[-1] = (k, pv)
    return q, segs


def _long_chunk(plan, device):
    """{1 long-chunk kernel, 0 short-chunk kernel; key splits} of a plan."""
    out = (ctypes.c_int32 * 2)()
    N.check(N.lib().gqa_seg_choice(ctypes.byref(plan._desc),
                                   torch.cuda.get_device_properties(device).multi_processor_count, out), "choice")
    return tuple(out)


def _check(out, q, segs):
    ref = O.gqa_segmented_reference(q.cpu(), [(k.cpu(), v.cpu()) for k, v in segs])
    m = O.error(out.cpu(), ref, LIMITS)
    assert m["passed"], m


@pytest.mark.parametrize("tokens", [32, 96, 256])
def test_baseline_config5(tokens, gpu_device):
    q, segs = _values(tokens, tokens, (1024, 512, 256), gpu_device)
    plan = prepare_segmented_gqa(q, segs)
    torch.cuda.synchronize()
    _check(plan.output, q, segs)


@pytest.mark.parametrize("tokens,hq,hkv", [(40, 32, 8), (100, 32, 8), (200, 32, 8), (512, 32, 8),
                                           (600, 8, 8)])
def test_launch_shapes(tokens, hq, hkv, gpu_device):
    """Every launch shape on 256 CUs (gqa_shape).  One 16-row block per wave:
    T = 40 four-wave workgroups with the keys split in two (merge launch),
    T = 100 eight-wave workgroups without a split.  Two row blocks per wave:
    T = 200 eight-wave workgroups without a split, T = 512 four-wave
    workgroups, two per CU; T = 600 with one query head per KV head (two
    token blocks per workgroup)."""
    q, segs = _values(tokens + 1, tokens, (300, 0, 129), gpu_device, hq=hq, hkv=hkv)
    plan = prepare_segmented_gqa(q, segs)
    torch.cuda.synchronize()
    _check(plan.output, q, segs)


@pytest.mark.parametrize("tokens,history", [(96, (2049, 0, 575)), (17, (0, 0, 0)), (1, (5, 0, 3)),
                                            (33, (64, 63, 1))])
def test_reference_shapes_and_tails(tokens, history, gpu_device):
    q, segs = _values(7, tokens, history, gpu_device, v_stride=6144 if tokens == 96 else None)
    plan = prepare_cuda_gqa_compact(q, segs, stages=2)
    torch.cuda.synchronize()
    _check(plan.output, q, segs)


@pytest.mark.parametrize("hq,hkv", [(8, 8), (16, 8), (64, 8)])
def test_group_sizes(hq, hkv, gpu_device):
    q, segs = _values(3, 40, (100, 30, 7), gpu_device, hq=hq, hkv=hkv)
    plan = prepare_segmented_gqa(q, segs)
    torch.cuda.synchronize()
    _check(plan.output, q, segs)


@pytest.mark.parametrize("tokens,hq,hkv,history", [
    (2048, 32, 8, (16, 0, 1)),         # mostly causal, one round of workgroups, no split
    (500, 32, 8, (8192, 2049, 575)),   # key splits and the merge, ragged last query block
    (1020, 16, 8, (8000, 100, 3)),     # two heads per KV head
    (2000, 8, 8, (9000, 0, 65)),       # one head per KV head
    (700, 64, 8, (6000, 63, 0)),       # eight heads per KV head, an empty segment
])
def test_long_chunks(tokens, hq, hkv, history, gpu_device):
    """The long-chunk kernel (256 query rows per workgroup over shared 64-key
    stages): every group size, short last tiles of each segment, query blocks
    that end inside a workgroup, with and without key splits; repeated runs are
    bitwise equal."""
    q, segs = _values(tokens, tokens, history, gpu_device, hq=hq, hkv=hkv, v_stride=6144 if tokens == 500 else None)
    plan = prepare_segmented_gqa(q, segs)
    chosen, splits = _long_chunk(plan, gpu_device)
    assert chosen and (splits > 1) == (tokens in (500, 1020, 2000))
    first = plan.run().clone()
    again = plan.run().clone()
    torch.cuda.synchronize()
    assert torch.equal(first.view(torch.int16), again.view(torch.int16))
    _check(first, q, segs)


@pytest.mark.parametrize("hq,hkv", [(32, 8), (8, 1), (4, 4), (1, 1)])
def test_workspace_serves_every_history(hq, hkv, gpu_device):
    """A workspace sized with one history is accepted with every other history of
    the same chunk length and heads, whichever kernels the two choose."""
    base = 1 << 20  # addresses that are only looked at by the validation
    for tokens in (32, 256, 512, 1024, 2048):
        descs, sizes = [], []
        for history in (0, 300, 2000, 9000, 40000):
            d = N.GqaDesc()
            d.T, d.Hq, d.Hkv, d.D, d.num_segments = tokens, hq, hkv, 128, 2
            for i, length in enumerate((history, tokens)):
                d.len[i], d.k[i], d.v[i] = length, base, base
                d.k_stride[i] = d.v_stride[i] = hkv * 128
            d.q = d.out = d.workspace = base
            size = ctypes.c_size_t()
            N.check(N.lib().gqa_seg_workspace_bytes(ctypes.byref(d), ctypes.byref(size)), "size")
            descs.append(d)
            sizes.append(size.value)
        for d in descs:
            for d.workspace_bytes in sizes:
                handle = ctypes.c_void_p()
                N.check(N.lib().gqa_seg_plan_create(ctypes.byref(handle), ctypes.byref(d)), "create")
                N.lib().gqa_seg_plan_destroy(handle)


def test_long_chunk_without_split_workspace(gpu_device):
    """A plan whose workspace does not hold the long-chunk kernel's split states
    is accepted and runs the kernel that needs none."""
    q, segs = _values(9, 500, (8192, 2049, 575), gpu_device)
    plan = prepare_segmented_gqa(q, segs)
    assert plan.splits_workspace_bytes > 0
    plan._desc.workspace, plan._desc.workspace_bytes = None, 0
    handle = ctypes.c_void_p()
    N.check(N.lib().gqa_seg_plan_create(ctypes.byref(handle), ctypes.byref(plan._desc)), "create")
    plan.output.zero_()
    stream = torch.cuda.current_stream(gpu_device).cuda_stream
    N.check(N.lib().gqa_seg_plan_run(handle, ctypes.c_void_p(stream)), "run")
    torch.cuda.synchronize()
    N.lib().gqa_seg_plan_destroy(handle)
    _check(plan.output, q, segs)


@pytest.mark.parametrize("tokens,history", [
    (32, (1024, 512, 256)),    # short chunk, keys split, merge launch
    (256, (1024, 512, 256)),   # short chunk, no split
    (500, (8192, 2049, 575)),  # long chunk, keys split, merge launch
    (2048, (16, 0, 1)),        # long chunk, no split
])
def test_non_finite_scores(tokens, history, gpu_device):
    """NaN in q or K and scores of +inf give NaN rows exactly where the FP32
    oracle has them, split or not; scores of -inf drop their key."""
    q, segs = _values(tokens + 5, tokens, history, gpu_device)
    q[tokens // 2, 3, 7] = float("nan")          # one row
    segs[0][0][9, 2, 100] = float("nan")         # every row of KV head 2
    segs[2][0][0, 7, 31] = float("inf")          # +inf or -inf by the sign of q's element
    ref = O.gqa_segmented_reference(q.cpu(), [(k.cpu(), v.cpu()) for k, v in segs]).float()
    segs[-1][0][tokens - 3, 5, 64] = float("nan")  # the last three tokens of KV head 5
    ref[tokens - 3:, 20:24] = float("nan")         # (the oracle adds its mask: NaN for the tokens before too)
    out = prepare_segmented_gqa(q, segs).output.cpu().float()
    nan = ref.isnan()
    assert 0 < int(nan.sum()) < nan.numel()
    assert torch.equal(out.isnan(), nan)
    m = O.error(out.masked_fill(nan, 0.0), ref.masked_fill(nan, 0.0), LIMITS)
    assert m["passed"], m


@pytest.mark.parametrize("tokens,hq,hkv,history", [
    (256, 32, 8, (1024, 512, 256)),    # short chunk
    (500, 32, 8, (8192, 2049, 575)),   # long chunk, keys split
    (2047, 32, 8, (16, 0, 1)),         # long chunk, no split, 64 tokens per workgroup
    (2000, 8, 8, (9000, 0, 65)),       # 256 tokens per workgroup
    (1020, 16, 8, (8000, 100, 3)),     # 128
    (700, 64, 8, (6000, 63, 0)),       # 32
])
def test_non_finite_values_of_later_tokens(tokens, hq, hkv, history, gpu_device):
    """A row of V that is not finite reaches its own token and the later ones;
    tokens of earlier 16-token blocks keep their values, those of earlier
    32-token blocks their bits.  (The long-chunk kernel adds up the 32 tokens
    around such a row in another order.)"""
    q, segs = _values(tokens + 6, tokens, history, gpu_device, hq=hq, hkv=hkv)
    plan = prepare_segmented_gqa(q, segs)
    clean = plan.output.clone()
    for row in (tokens - 3, tokens // 2 + 21, tokens // 2 + 5, 40, 17, 0):
        segs[-1][1][row] = float("inf") if row % 2 else float("nan")
        out = plan.run()
        same = row // 32 * 32
        assert torch.equal(out[:same].view(torch.int16), clean[:same].view(torch.int16)), row
        if row // 16 * 16 > same:
            m = O.error(out[same:row // 16 * 16].cpu(), clean[same:row // 16 * 16].cpu().float(), LIMITS)
            assert m["passed"], (row, m)
        assert not out[row:].isfinite().any(), row


def test_split_merge_partial_workgroup(gpu_device):
    """T * Hq = 66 (query) rows with the keys split: the merge launch's last
    workgroup holds fewer rows than the others."""
    q, segs = _values(5, 33, (200, 17, 0), gpu_device, hq=2, hkv=1)
    plan = prepare_segmented_gqa(q, segs)
    torch.cuda.synchronize()
    assert plan.splits_workspace_bytes > 0
    _check(plan.output, q, segs)


def test_empty_query(gpu_device):
    q, segs = _values(1, 0, (10, 0, 4), gpu_device)
    plan = prepare_segmented_gqa(q, segs)
    assert plan.run().shape == (0, 32, 128)


@pytest.mark.parametrize("tokens", [96, 32])
def test_graph_replay_and_stream(tokens, gpu_device):
    """T = 96 runs unsplit, T = 32 with a key split and the merge launch."""
    q, segs = _values(11, tokens, (1024, 512, 256), gpu_device)
    plan = prepare_segmented_gqa(q, segs)
    torch.cuda.synchronize()
    stream = torch.cuda.Stream(device=gpu_device)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        gout = plan.run()
    for step in range(2):
        q2, segs2 = _values(100 + step, tokens, (1024, 512, 256), gpu_device)
        q.copy_(q2)
        for (k, v), (k2, v2) in zip(segs, segs2):
            k.copy_(k2)
            v.copy_(v2)
        graph.replay()
        torch.cuda.synchronize()
        replay = gout.clone()
        side = torch.cuda.Stream(device=gpu_device)
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            eager = plan.run().clone()
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        assert torch.equal(replay.view(torch.int16), eager.view(torch.int16))
        _check(replay, q, segs)


@pytest.mark.parametrize("tokens", [32, 64])
def test_split_runs_repeat_bitwise(tokens, gpu_device):
    """Key-split shapes (T = 32: four splits, T = 64: two on 256 CUs):
    repeated runs of one plan merge the partial states in the same fixed order,
    so they give bitwise the same output."""
    q, segs = _values(21 + tokens, tokens, (1024, 512, 256), gpu_device)
    plan = prepare_segmented_gqa(q, segs)
    torch.cuda.synchronize()
    assert plan.splits_workspace_bytes > 0
    first = plan.output.clone()
    _check(first, q, segs)
    for _ in range(4):
        plan.run()
    torch.cuda.synchronize()
    assert torch.equal(plan.output.view(torch.int16), first.view(torch.int16))


def test_rejects_bad_inputs(gpu_device):
    q, segs = _values(1, 8, (4, 0, 2), gpu_device)
    with pytest.raises(ValueError):
        prepare_segmented_gqa(q, segs[:-1] + [(segs[-1][0][:4], segs[-1][1][:4])])
    with pytest.raises(TypeError):
        prepare_segmented_gqa(q, [(k.float(), v) for k, v in segs])
    for bad in (0.0, -1.0, float("inf"), float("nan")):
        with pytest.raises(ValueError):
            prepare_segmented_gqa(q, segs, scale=bad)


def test_out_aliasing_rejected(gpu_device):
    """An output sharing storage with q or a K/V segment is rejected
    (attention_cuda_compact.py:175-177)."""
    from llm_gpu_kernels_amd import prepare_cuda_gqa_compact
    q = torch.randn(32, 32, 128, device=gpu_device).to(torch.bfloat16)
    kv = torch.randn(2, 64, 8, 128, device=gpu_device).to(torch.bfloat16)
    cur = torch.randn(2, 32, 8, 128, device=gpu_device).to(torch.bfloat16)
    segs = [(kv[0], kv[1]), (cur[0], cur[1])]
    with pytest.raises(ValueError, match="share storage"):
        prepare_cuda_gqa_compact(q, segs, out=q)
    big = torch.empty(2, 32, 32, 128, device=gpu_device, dtype=torch.bfloat16)
    segs_alias = [(kv[0], kv[1]), (big[1, :, :8], cur[1])]
    with pytest.raises(ValueError):
        prepare_cuda_gqa_compact(q, segs_alias, out=big[0])
    prepare_cuda_gqa_compact(q, segs)
