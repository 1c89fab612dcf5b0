"""C ABI checks that need no GPU: exports, validation, host-side W4 functions."""
import ctypes
import re
from pathlib import Path

import pytest
import torch

from llm_gpu_kernels_amd import _native as N
from llm_gpu_kernels_amd import quantize_gate_up, tile_gate_up
from oracle import moe_oracle as O

INCLUDE = Path(__file__).resolve().parents[1] / "include"


def _declared_functions():
    names = set()
    for header in INCLUDE.glob("*.h"):
        text = re.sub(r"/\*.*?\*/", "", header.read_text(), flags=re.S)
        for m in re.finditer(r"^[A-Za-z_][\w\s\*]*?\b(\w+)\s*\([^;{]*\)\s*;", text, flags=re.M):
            if not m.group(0).lstrip().startswith(("typedef", "#")):
                names.add(m.group(1))
    return names


def test_library_exports_every_declared_function():
    lib = N.lib()
    declared = _declared_functions()
    assert declared, "no declarations parsed"
    assert declared <= set(N.SIGNATURES), declared - set(N.SIGNATURES)
    for name in declared:
        assert hasattr(lib, name), name
    assert lib.moe_abi_version() == 2


def test_struct_sizes_match_header():
    # 10 int32 + 10 pointers + size_t; 14 size_t + 4 int32.
    assert ctypes.sizeof(N.MoeDesc) == 40 + 8 * 10 + 8
    assert ctypes.sizeof(N.MoeLayout) == 8 * 14 + 16
    # 9 int32 (+pad) + 2 + 8 pointers + 8 int64 + float (+pad) + pointer + size_t.
    assert ctypes.sizeof(N.GqaDesc) == 40 + 16 + 64 + 64 + 8 + 8 + 8


def _desc(**kw):
    d = N.MoeDesc()
    d.T, d.H, d.I, d.E, d.K = kw.get("T", 17), kw.get("H", 2048), kw.get("I", 768), \
        kw.get("E", 128), kw.get("K", 8)
    d.weight_format = kw.get("fmt", N.WEIGHTS_BF16)
    d.id_dtype = kw.get("ids", N.IDS_INT32)
    d.route_mode = kw.get("route", N.ROUTE_FIXED)
    d.token_block = kw.get("tb", 0)
    return d


def _layout(d):
    lay = N.MoeLayout()
    rc = N.lib().moe_workspace_layout(ctypes.byref(d), ctypes.byref(lay))
    return rc, lay


def test_layout_for_qwen_shape():
    rc, lay = _layout(_desc())
    assert rc == 0
    r = 17 * 8
    assert lay.token_block == 16 and lay.fast_path == 1 and lay.launches == 4
    assert lay.task_capacity == (r + 15) // 16 + 128
    assert lay.act % 256 == 0 and lay.routed % 256 == 0
    assert lay.total >= lay.routed + r * 2048 * 2
    rc, lay = _layout(_desc(T=1024))
    assert lay.token_block == 64 and lay.fast_path == 2
    rc, lay = _layout(_desc(T=300))
    assert lay.token_block == 32 and lay.fast_path == 1
    rc, lay = _layout(_desc(T=0))
    assert rc == 0 and lay.launches == 0
    # One multi-workgroup launch routes and plans (16 tokens per workgroup).
    rc, lay = _layout(_desc(route=N.ROUTE_LOGITS, T=1024))
    assert lay.launches == 4
    rc, lay = _layout(_desc(route=N.ROUTE_LOGITS, T=193))
    assert lay.launches == 4
    assert lay.partials % 256 == 0 and lay.act >= lay.partials + 13 * 129 * 4 + 4
    rc, lay = _layout(_desc(route=N.ROUTE_LOGITS, T=16 * 256))
    assert lay.launches == 4
    rc, lay = _layout(_desc(route=N.ROUTE_LOGITS, T=16 * 256 + 1))
    assert lay.launches == 5  # more workgroups than CUs: separate router launch
    rc, lay = _layout(_desc(route=N.ROUTE_LOGITS, T=16))
    assert lay.launches == 3
    rc, lay = _layout(_desc(route=N.ROUTE_LOGITS, T=17))
    assert lay.launches == 3  # bf16: routing and planning in the gate/up launch
    rc, lay = _layout(_desc(route=N.ROUTE_LOGITS, T=32))
    assert lay.launches == 3
    rc, lay = _layout(_desc(route=N.ROUTE_LOGITS, T=17, fmt=N.WEIGHTS_W4G128))
    assert lay.launches == 3  # W4: routing and planning in the gate/up launch too
    rc2, lay2 = _layout(_desc(route=N.ROUTE_LOGITS, T=17, fmt=N.WEIGHTS_W4G128_FOLD))
    assert rc2 == 0 and (lay2.total, lay2.launches, lay2.fast_path) == (lay.total, lay.launches, lay.fast_path)
    rc, lay = _layout(_desc(route=N.ROUTE_LOGITS, T=17, H=4096))
    assert lay.launches == 4
    rc, lay = _layout(_desc(route=N.ROUTE_LOGITS, T=33))
    assert lay.launches == 4
    rc, lay = _layout(_desc(route=N.ROUTE_LOGITS, T=17, E=256))
    assert lay.launches == 4
    rc, lay = _layout(_desc(H=33, I=19, E=8, K=2))
    assert rc == 0 and lay.fast_path == 0


def _choice(cus=256, **kw):
    out = (ctypes.c_int32 * 4)()
    assert N.lib().moe_gemm_choice(ctypes.byref(_desc(**kw)), cus, out) == 0, N.last_error()
    return list(out)


@pytest.mark.parametrize("fmt", [N.WEIGHTS_BF16, N.WEIGHTS_W4G128])
@pytest.mark.parametrize("experts", [1, 8, 16, 32, 128])
def test_tiled_units_fill_idle_cus(experts, fmt):
    """While the units of the mean expert leave half the CUs idle, lower ones
    that make more of them are taken: never fewer units with more rows, also
    where one block holds the whole expert (a mean of 128 rows)."""
    def units(inter, mean, rows):
        return experts * (-(-inter // 128)) * (-(-mean // rows))
    for inter in (96, 256, 512, 768, 1536):
        for mean in list(range(97, 170)) + [192, 256, 320, 321]:
            kernel, rows, _, _ = _choice(T=mean * experts, K=1, E=experts, H=1152, I=inter, fmt=fmt, tb=64)
            assert kernel == N.GEMM_TILED and rows in (32, 64, 96, 128, 160)
            n = units(inter, mean, rows)
            assert 2 * n >= 256 or n == units(inter, mean, 32), (inter, mean, rows)
    # 16 experts, gate/up and down (six and eight weight tiles).
    rows = {t: _choice(T=t, K=1, E=16, fmt=fmt)[1::2] for t in (1024, 1400, 1600, 1800, 2032, 2048, 2049, 4096)}
    assert rows == {1024: [64, 64], 1400: [64, 96], 1600: [64, 96], 1800: [96, 96], 2032: [96, 96],
                    2048: [96, 160], 2049: [128, 160], 4096: [160, 160]}
    shape = dict(K=4, E=16, H=1152, I=512, fmt=fmt, tb=64)  # four gate/up tiles: half of the CUs, or three quarters
    assert [_choice(T=t, **shape)[1] for t in (400, 500, 512, 600, 700)] == [64] * 5
    assert _choice(T=2048, fmt=fmt)[1] == 160  # every CU has units: the fewest weight reads


@pytest.mark.parametrize("kw", [dict(E=0), dict(E=257), dict(K=0), dict(K=33), dict(H=0),
                                dict(I=-1), dict(T=-1), dict(fmt=7), dict(ids=9), dict(tb=8), dict(tb=48),
                                dict(route=N.ROUTE_LOGITS, ids=N.IDS_INT64),
                                dict(route=N.ROUTE_LOGITS, E=4, K=8),
                                dict(fmt=N.WEIGHTS_W4G128, H=192), dict(fmt=N.WEIGHTS_W4G128, H=512, I=48),
                                dict(fmt=N.WEIGHTS_W4G128_FOLD, H=192), dict(fmt=3),
                                dict(T=2 ** 27, K=16)])
def test_layout_rejects_invalid_descriptors(kw):
    rc, _ = _layout(_desc(**kw))
    assert rc == N.MOE_EINVAL
    assert N.last_error()


def test_tiled_matrix_size():
    """The tiled kernels take matrices whose byte offsets, the rows of the last tile
    past the end included, fit 32 bits: neither smaller ones are refused nor do
    long rows wrap."""
    for h, i in ((32768, 32768), (34816, 32800), (65024, 32768), (32768, 65024)):
        assert _choice(T=40, E=1, K=1, H=h, I=i)[::2] == [N.GEMM_TILED, N.GEMM_TILED], (h, i)
    for h, i in ((65536, 32768), (1 << 24, 32), (32, 1 << 23)):  # 127 rows of 32 MiB, 255 of 16 MiB
        assert _choice(T=40, E=1, K=1, H=h, I=i)[::2] == [N.GEMM_RUNTIME_K, N.GEMM_RUNTIME_K], (h, i)


@pytest.mark.parametrize("tokens,experts,hidden,inter,kernel", [
    (256, 8, 256, 96, N.GEMM_DECODE_ONCE), (256, 8, 512, 96, N.GEMM_DECODE_ONCE),  # small matrices
    (2560, 64, 512, 480, N.GEMM_DECODE_ONCE), (2560, 64, 1024, 96, N.GEMM_DECODE_ONCE),
    (512, 64, 1536, 768, N.GEMM_DECODE_ONCE), (767, 64, 1536, 768, N.GEMM_DECODE_ONCE),  # below 48 rows per expert
    (768, 64, 1536, 768, N.GEMM_TILED), (1024, 32, 2560, 1024, N.GEMM_TILED), (1024, 64, 1024, 512, N.GEMM_TILED),
    (256, 8, 1792, 32, N.GEMM_RUNTIME_K), (256, 8, 128, 512, N.GEMM_TILED), (256, 8, 384, 96, N.GEMM_RUNTIME_K),
    (1024, 64, 2048, 768, N.GEMM_DECODE_ONCE), (2048, 64, 2048, 768, N.GEMM_TILED),  # H = 2048: the pair kernel
])
def test_w4_64_row_choice(tokens, experts, hidden, inter, kernel):
    """The gate/up kernel of W4 64-row tasks (K = 4): each where it measured
    fastest of decode-once, tiled and run-time-K."""
    kw = dict(T=tokens, E=experts, H=hidden, I=inter, K=4, fmt=N.WEIGHTS_W4G128)
    assert _layout(_desc(**kw))[1].token_block == 64
    assert _choice(**kw)[0] == kernel


def _gqa_choice(tokens, history, hq, hkv, cus=256):
    d = N.GqaDesc()
    d.T, d.Hq, d.Hkv, d.D, d.num_segments = tokens, hq, hkv, 128, len(history) + 1
    for i, length in enumerate((*history, tokens)):
        d.len[i], d.k[i], d.v[i] = length, 1 << 20, 1 << 20
        d.k_stride[i] = d.v_stride[i] = hkv * 128
    d.q = d.out = 1 << 20
    out = (ctypes.c_int32 * 2)()
    assert N.lib().gqa_seg_choice(ctypes.byref(d), cus, out) == 0, N.last_error()
    return tuple(out)


def test_long_chunk_attention_choice():
    """The long-chunk kernel where it measured faster (tokens x history keys, query /
    KV heads), the short-chunk kernel where that one did: few stages, and splits
    whose further rounds cost more than they save."""
    short, long_, mid, most = (16, 0, 1), (8192, 2049, 575), (1024, 512, 256), (4000, 64, 32)
    for hq, hkv in ((32, 8), (16, 8), (8, 8), (64, 8), (8, 1), (4, 4)):
        for tokens in (1, 32, 255):
            assert _gqa_choice(tokens, long_, hq, hkv)[0] == 0
        for history in ((), (1,), short, (100, 50, 50), (500, 0, 0)):
            assert _gqa_choice(256, history, hq, hkv)[0] == 0, (hq, hkv, history)
    assert _gqa_choice(512, mid, 32, 8)[0] == _gqa_choice(1024, mid, 32, 8)[0] == 0
    assert _gqa_choice(3000, short, 16, 8)[0] == _gqa_choice(3000, (300, 0, 7), 8, 8)[0] == 0
    assert _gqa_choice(4096, (500, 0, 0), 4, 4) == (1, 4)
    assert _gqa_choice(2048, short, 32, 8) == _gqa_choice(2048, long_, 32, 8) == (1, 1)
    assert _gqa_choice(1024, long_, 32, 8) == (1, 2) and _gqa_choice(512, long_, 32, 8) == (1, 4)
    assert _gqa_choice(2048, long_, 16, 8) == (1, 2) and _gqa_choice(1024, short, 64, 8) == (1, 1)


def test_plan_create_rejects_null_pointers():
    d = _desc()
    handle = ctypes.c_void_p()
    rc = N.lib().moe_plan_create(ctypes.byref(handle), ctypes.byref(d))
    assert rc == N.MOE_EINVAL and not handle.value
    with pytest.raises(ValueError):
        N.check(rc, "prepare")


@pytest.mark.parametrize("shape", [(2, 16, 128), (3, 32, 384), (1, 48, 1024)])
def test_quantize_matches_oracle_bit_exact(shape):
    g = torch.Generator().manual_seed(sum(shape))
    w = (torch.randn(shape, generator=g) * 0.02).to(torch.bfloat16)
    w[0, 0, :128] = 0
    w[0, 1, :8] = torch.tensor([7.0, -7.0, 3.5, 4.5, -3.5, 0.5, 1.5, -0.5]).to(torch.bfloat16) * 1e-2
    p = quantize_gate_up(w.contiguous())
    ow, os_ = O.quantize_w4(w)
    assert torch.equal(p.words, ow)
    assert torch.equal(p.scales.view(torch.int16), os_.view(torch.int16))


def test_quantize_rejects_nonfinite():
    w = torch.zeros((1, 16, 128), dtype=torch.bfloat16)
    w[0, 3, 5] = float("nan")
    with pytest.raises(ValueError):
        quantize_gate_up(w)


def test_tile_layout_index_map():
    """words_t[e][rb][grp][lane][j] == v1 word 16*grp + 4*j + lane//16 of row 16*rb + lane%16."""
    e, n, k = 2, 32, 256
    words = torch.arange(e * n * k // 8, dtype=torch.int32).reshape(e, n, k // 8)
    scales = torch.arange(e * n * k // 128, dtype=torch.int16).view(torch.bfloat16).reshape(e, n, k // 128)
    t = tile_gate_up(O_packed(words, scales))
    for ei, rb, grp, lane, j in [(0, 0, 0, 0, 0), (1, 1, 1, 63, 3), (0, 1, 0, 17, 2), (1, 0, 1, 40, 1)]:
        r, g = lane % 16, lane // 16
        assert t.words[ei, rb, grp, lane, j] == words[ei, rb * 16 + r, 16 * grp + 4 * j + g]
        assert t.scales[ei, rb, grp, r].view(torch.int16) == scales[ei, rb * 16 + r, grp].view(torch.int16)
    assert sorted(t.words.reshape(-1).tolist()) == list(range(e * n * k // 8))


def O_packed(words, scales):
    from llm_gpu_kernels_amd.weight_quant import PackedGateUp
    return PackedGateUp(words, scales, {})


def _decode_word_like_kernel(word, s):
    """Host restatement of the kernel's w4_decode8 (llm_gpu_kernels_amd/csrc/common.h):
    nibble n at mantissa position p of 2^23 -> fma(2^23 + n*16^p, s*16^-p,
    -(2^(23-4p)+8)*s), evaluated exactly in float64, rounded once to fp32."""
    import struct
    def fl(b):
        return struct.unpack("<f", struct.pack("<I", b & 0xFFFFFFFF))[0]
    lo, hi = (word << 8) & 0xFFFFFFFF, word >> 12
    plan = [(lo, 2), (lo, 3), (word, 2), (word, 3), (word, 4), (hi, 2), (hi, 3), (hi, 4)]
    out = []
    for src, p in plan:
        v = fl(0x4B000000 | (src & (0xF << (4 * p))))
        sp = float(torch.tensor(s * 2.0 ** (-4 * p), dtype=torch.float32))
        cp = float(torch.tensor(-s * float(2 ** (23 - 4 * p) + 8), dtype=torch.float32))
        out.append(float(torch.tensor(v * sp + cp, dtype=torch.float32)))
    return out


def test_tile_emulated_decode_matches_oracle_dequant():
    """Host emulation of the kernel decode on the tiled layout == oracle dequant."""
    g = torch.Generator().manual_seed(11)
    w = (torch.randn((1, 32, 256), generator=g) * 0.03).to(torch.bfloat16)
    w[0, 5, :128] = 0  # scale 1 group
    p = quantize_gate_up(w)
    t = tile_gate_up(p)
    ref = O.dequantize_w4(p.words, p.scales)
    e, n, k = 1, 32, 256
    out = torch.empty((e, n, k), dtype=torch.bfloat16)
    wt = t.words.to(torch.int64) & 0xFFFFFFFF
    st = t.scales.float()
    for rb in range(n // 16):
        for grp in range(k // 128):
            for lane in range(64):
                r, gg = lane % 16, lane // 16
                s = float(st[0, rb, grp, r])
                for j in range(4):
                    vals = _decode_word_like_kernel(int(wt[0, rb, grp, lane, j]), s)
                    base = grp * 128 + 32 * j + 8 * gg
                    out[0, rb * 16 + r, base:base + 8] = torch.tensor(vals).to(torch.bfloat16)
    assert torch.equal(out.view(torch.int16), ref.view(torch.int16))


def test_cuda_variant_names_validated():
    """prepare_cuda_moe accepts the reference's variant names only
    (moe_cuda.py:17,57-58); the check precedes any device work."""
    from llm_gpu_kernels_amd import moe as M
    assert M.CUDA_VARIANTS == ("sync", "async", "async_skip")
    with pytest.raises(ValueError, match="unsupported CUDA variant"):
        M.prepare_cuda_moe(None, None, None, None, None, variant="mfma")


def test_attention_out_storage_check():
    """Output aliasing q or any K/V segment storage is rejected (views of one
    storage included); empty tensors never alias."""
    from llm_gpu_kernels_amd.attention import check_out_storage
    q = torch.zeros(4, 32, 128, dtype=torch.bfloat16)
    kv = torch.zeros(2, 4, 8, 128, dtype=torch.bfloat16)
    out = torch.zeros_like(q)
    check_out_storage(out, [q, kv[0], kv[1]])
    with pytest.raises(ValueError, match="share storage"):
        check_out_storage(q, [q, kv[0], kv[1]])
    with pytest.raises(ValueError, match="share storage"):
        check_out_storage(kv[1], [q, kv[0]])
    check_out_storage(torch.empty(0, 32, 128), [torch.empty(0, 8, 128)])


def test_status_bit_values():
    """Status bits of the header, as the Python layer reads them."""
    text = (INCLUDE / "moe_mi355x.h").read_text()
    for name, value in (("BAD_ID", 1), ("BAD_WEIGHT", 2), ("BAD_LOGIT", 4), ("DIRTY_COUNTERS", 8), ("STALLED", 16)):
        assert re.search(rf"#define MOE_STATUS_{name} {value}u", text), name
        assert getattr(N, f"STATUS_{name}") == value


def test_static_workspace_size_matches_header():
    text = (INCLUDE / "moe_mi355x.h").read_text()
    assert re.search(r"#define MOE_STATIC_WORKSPACE_BYTES \(16u << 20\)", text)
    assert N.STATIC_WORKSPACE_BYTES == 16 << 20
