"""GPU parity of the decode attention (attention.py:1040-1262) against the
oracle: the new cache rows (rotated k within one bf16 ulp -- the kernel rotates
in fp32, the oracle in fp64 --, v exact), untouched rows elsewhere, and the
output within 2^-7 relative plus 1e-3 of the row's largest value (bf16
operands and output, fp32 accumulation, the exp of the hardware)."""

import numpy as np
import pytest
import torch

import helpers as H
from bitnet_tt import _native as N
from bitnet_tt.layers.attention import DecodeAttention

pytestmark = pytest.mark.gpu


def run(orc, B, Hq, Hkv, S, pos, adjacent, seed, scale=None):
    rng = np.random.default_rng(seed)
    D = 128
    qkv = orc.f32_to_bf16(rng.standard_normal((B, (Hq + 2 * Hkv) * D)).astype(np.float32))
    kc = orc.f32_to_bf16(rng.standard_normal((B, Hkv, S, D)).astype(np.float32))
    vc = orc.f32_to_bf16(rng.standard_normal((B, Hkv, S, D)).astype(np.float32))
    att = DecodeAttention(Hq, Hkv, D, S, H.dev(), rope_theta=500000.0, use_fused_rope=adjacent, scale=scale)
    cache = att.new_cache(B)
    cache.key_cache.copy_(H.to_dev_bf16(kc).view(B, Hkv, S, D))
    cache.value_cache.copy_(H.to_dev_bf16(vc).view(B, Hkv, S, D))
    out = att(H.to_dev_bf16(qkv), cache, torch.tensor(pos, dtype=torch.int32, device=H.dev()))
    torch.cuda.synchronize()
    cos, sin = orc.rope_tables(D, S, 500000.0)
    ref, kc2, vc2 = orc.decode_attention(qkv, kc, vc, np.asarray(pos), Hq, Hkv, cos, sin, adjacent, att.scale)
    return att, cache, H.bits_of(out).astype(np.uint16), ref, kc, vc, kc2, vc2


def check(orc, got_bits, ref, cache, kc2, vc2):
    got = orc.bf16_to_f32(got_bits.view(np.uint16)).astype(np.float64)
    tol = 2.0 ** -7 * np.abs(ref) + 1e-3 * np.abs(ref).max(axis=-1, keepdims=True)
    assert np.all(np.abs(got - ref) <= tol), np.max(np.abs(got - ref) - tol)
    kgot = H.bits_of(cache.key_cache).reshape(kc2.shape).astype(np.int32)
    assert np.all(np.abs(kgot - kc2.astype(np.int32)) <= 1)  # 1 bf16 ulp (same sign here)
    assert np.array_equal(H.bits_of(cache.value_cache).reshape(vc2.shape), vc2)


@pytest.mark.parametrize("adjacent", [False, True])
@pytest.mark.parametrize("B,Hq,Hkv,S,pos", [(3, 4, 1, 256, [0, 130, 255]), (2, 4, 2, 128, [5, 127]),
                                           (4, 2, 2, 384, [383, 0, 129, 256]), (1, 1, 1, 64, [63])])
def test_small_shapes(orc, B, Hq, Hkv, S, pos, adjacent):
    print(f"attention B={B} H={Hq} Hkv={Hkv} S={S} adjacent={adjacent}", flush=True)
    att, cache, out, ref, kc, vc, kc2, vc2 = run(orc, B, Hq, Hkv, S, pos, adjacent, seed=B * 31 + S)
    check(orc, out, ref, cache, kc2, vc2)


@pytest.mark.parametrize("full", [True, False])
def test_2b_shape(orc, full):
    """32 users, 20 query / 5 key-value heads, context 512 (4 chunks per
    user and head group): every user at the last position, or at spread
    positions."""
    B, Hq, Hkv, S = 32, 20, 5, 512
    pos = [511] * B if full else list(np.random.default_rng(9).integers(0, S, size=B))
    print(f"attention 2B shape full={full}", flush=True)
    att, cache, out, ref, kc, vc, kc2, vc2 = run(orc, B, Hq, Hkv, S, pos, True, seed=77 + full)
    check(orc, out, ref, cache, kc2, vc2)


def test_graph_replay_advances_position(orc):
    """A captured call reads the position from the device: replays after an
    increment of pos write the next cache rows and match the eager results."""
    B, Hq, Hkv, S, D = 4, 4, 1, 256, 128
    rng = np.random.default_rng(5)
    att = DecodeAttention(Hq, Hkv, D, S, H.dev())
    cache = att.new_cache(B)
    qkv = H.to_dev_bf16(orc.f32_to_bf16(rng.standard_normal((B, (Hq + 2 * Hkv) * D)).astype(np.float32)))
    pos = torch.zeros(B, dtype=torch.int32, device=H.dev())
    out = torch.empty((B, Hq * D), dtype=torch.bfloat16, device=H.dev())
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    eager = []
    with torch.cuda.stream(s):
        for t in range(3):
            pos.fill_(t)
            att(qkv, cache, pos, out=out)
            eager.append(H.bits_of(out).copy())
    torch.cuda.synchronize()
    k_eager = H.bits_of(cache.key_cache).copy()
    cache.key_cache.zero_()
    cache.value_cache.zero_()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        att(qkv, cache, pos, out=out)
    for t in range(3):
        with torch.cuda.stream(s):
            pos.fill_(t)
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert np.array_equal(H.bits_of(out), eager[t]), f"replay {t}"
    assert np.array_equal(H.bits_of(cache.key_cache), k_eager)
    with torch.cuda.stream(s):
        assert att.error_word(B=B) == 0


def test_position_out_of_range_is_flagged(orc):
    B, Hq, Hkv, S, D = 2, 4, 1, 128, 128
    att = DecodeAttention(Hq, Hkv, D, S, H.dev())
    cache = att.new_cache(B)
    qkv = torch.ones((B, (Hq + 2 * Hkv) * D), dtype=torch.bfloat16, device=H.dev())
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        out = att(qkv, cache, torch.tensor([3, S], dtype=torch.int32, device=H.dev()))
        torch.cuda.synchronize()
        assert att.error_word(B=B) != 0
    # check() surfaces the sticky word as RuntimeError and resets the workspace
    with pytest.raises(RuntimeError, match="error word"):
        att.check()
    with torch.cuda.stream(s):
        assert att.error_word(B=B) == 0
    att.check()
    assert torch.all(out[1] == 0) and torch.isfinite(out[0].float()).all()
    assert not cache.key_cache[1].any()  # nothing written for the bad row


def test_full_layer_chain(orc):
    """One mini layer through step_full: QKV (bit-exact), attention (oracle
    tolerance), then o_proj, gate||up and down from the kernel's attention
    output (bit-exact), and the cache rows at the position."""
    from bitnet_tt.config import BitNetMiniConfig
    from bitnet_tt.decode import BitLinearDecodeStep

    cfg = BitNetMiniConfig(num_layers=1, num_attention_heads=4, num_key_value_heads=1, hidden_size=512,
                           intermediate_size=512)
    print("mini layer with attention", flush=True)
    step = BitLinearDecodeStep.random_init(cfg, H.dev(), seed=81, batch=8).alloc_buffers(seed=82)
    step.alloc_attention(max_seq_len=256, pos=200)
    kc0 = H.bits_of(step.kv[0].key_cache).reshape(8, 1, 256, 128).copy()
    vc0 = H.bits_of(step.kv[0].value_cache).reshape(8, 1, 256, 128).copy()
    hid = H.bits_of(step.hidden).copy()
    step.step_full()
    torch.cuda.synchronize()
    w = step.layers[0]

    def wkn(pw):
        return orc.devlayout_decode(pw.data.cpu().numpy().view(np.uint32), pw.in_features, pw.out_features)

    qkv = orc.bitlinear(hid, wkn(w.qkv), list(w.qkv.segment_scales), list(w.qkv.segment_ends),
                        gamma_bf16=H.bits_of(w.input_layernorm), norm_eps=step.eps)["out"]
    assert np.array_equal(H.bits_of(step.qkv_out), qkv)
    cos, sin = orc.rope_tables(128, 256, cfg.rope_theta)
    ref, kc2, vc2 = orc.decode_attention(qkv, kc0, vc0, np.full(8, 200), 4, 1, cos, sin, False, step.attention.scale)
    attn = H.bits_of(step.attn_out)
    check(orc, attn, ref, step.kv[0], kc2, vc2)
    h = orc.bitlinear(attn, wkn(w.o_proj), list(w.o_proj.segment_scales), gamma_bf16=H.bits_of(w.attn_sub_norm),
                      norm_eps=step.eps, residual_bf16=hid)["out"]
    r = orc.gate_up_relu2(h, wkn(w.gate_up), w.gate_up.segment_scales[0], w.gate_up.segment_scales[1],
                          gamma_bf16=H.bits_of(w.post_attention_layernorm), norm_eps=step.eps)
    h = orc.bitlinear(r["h"], wkn(w.down), list(w.down.segment_scales), gamma_bf16=H.bits_of(w.ffn_sub_norm),
                      norm_eps=step.eps, residual_bf16=h)["out"]
    assert np.array_equal(H.bits_of(step.hidden), h)


def _full_state(step):
    return (step.hidden.clone(), [(kv.key_cache.clone(), kv.value_cache.clone()) for kv in step.kv])


def _restore(step, state):
    hid, caches = state
    step.hidden.copy_(hid)
    for kv, (k, v) in zip(step.kv, caches):
        kv.key_cache.copy_(k)
        kv.value_cache.copy_(v)
    torch.cuda.synchronize()


def _outputs(step):
    torch.cuda.synchronize()
    return {"hidden": H.bits_of(step.hidden).copy(), "qkv": H.bits_of(step.qkv_out).copy(),
            "attn": H.bits_of(step.attn_out).copy(), "ffn_h": H.bits_of(step.ffn_h).copy(),
            "k": [H.bits_of(kv.key_cache).copy() for kv in step.kv],
            "v": [H.bits_of(kv.value_cache).copy() for kv in step.kv]}


def _compare(a, b, what):
    for key in ("hidden", "qkv", "attn", "ffn_h"):
        bad = int((a[key] != b[key]).sum())
        assert bad == 0, f"{what}: {key} differs in {bad} of {a[key].size} values"
    for i, (ka, kb, va, vb) in enumerate(zip(a["k"], b["k"], a["v"], b["v"])):
        assert np.array_equal(ka, kb) and np.array_equal(va, vb), f"{what}: layer {i} cache differs"


@pytest.mark.parametrize("layers,batch,pos", [(2, 8, 200), (3, 5, None)])
def test_persistent_full_step_matches_step_full_mini(orc, layers, batch, pos):
    """The one-launch step with the decode attention (btl_decode_step_full)
    against step_full (QKV, attention and the other BitLinears as separate
    launches, each pinned to the oracle elsewhere): hidden, the last layer's
    qkv / attention / FFN rows and every layer's cache, bit for bit; spread
    positions per user in the second case."""
    from bitnet_tt.config import BitNetMiniConfig
    from bitnet_tt.decode import BitLinearDecodeStep

    cfg = BitNetMiniConfig(num_layers=layers, num_attention_heads=4, num_key_value_heads=1, hidden_size=512,
                           intermediate_size=512)
    print(f"persistent full step mini layers={layers} batch={batch} pos={pos}", flush=True)
    step = BitLinearDecodeStep.random_init(cfg, H.dev(), seed=91 + layers, batch=batch).alloc_buffers(seed=92)
    step.alloc_attention(max_seq_len=256, pos=pos if pos is not None else 0)
    if pos is None:
        step.pos.copy_(torch.from_numpy(np.random.default_rng(3).integers(0, 256, batch).astype(np.int32)))
    state = _full_state(step)
    step.step_full()
    step.check()
    ref = _outputs(step)
    _restore(step, state)
    step.step_persistent_full()
    step.check()
    _compare(_outputs(step), ref, "persistent full step")


def test_persistent_full_step_attention_on_qkv_units(orc):
    """More attention items than GEMM units without QKV work (26 users x 8
    key-value heads = 208 items; 64 QKV units of 224), so that units 16-63
    run a QKV unit and then an attention item in each layer: the one-launch
    step against step_full, bit for bit."""
    from bitnet_tt.config import BitNetMiniConfig
    from bitnet_tt.decode import BitLinearDecodeStep

    cfg = BitNetMiniConfig(num_layers=2, num_attention_heads=16, num_key_value_heads=8, hidden_size=2048,
                           intermediate_size=512)
    print("persistent full step, attention on QKV units: batch 26, 8 kv heads", flush=True)
    step = BitLinearDecodeStep.random_init(cfg, H.dev(), seed=97, batch=26).alloc_buffers(seed=98)
    step.alloc_attention(max_seq_len=128, pos=0)
    step.pos.copy_(torch.from_numpy(np.random.default_rng(5).integers(0, 128, 26).astype(np.int32)))
    state = _full_state(step)
    step.step_full()
    step.check()
    ref = _outputs(step)
    _restore(step, state)
    step.step_persistent_full()
    step.check()
    _compare(_outputs(step), ref, "persistent full step, attention on QKV units")


def test_persistent_full_step_2b_layer_against_oracle(orc):
    """One 2B layer (20 query / 5 key-value heads, batch 32, every user at
    position 511 of a 512 context) through the one-launch step with the
    attention, against the oracle: QKV bit-exact, the attention within the
    oracle tolerance (with the new cache rows), and o_proj, gate||up and down
    from the kernel's attention output bit-exact."""
    from bitnet_tt.config import BitNet2B4TConfig
    from bitnet_tt.decode import BitLinearDecodeStep

    cfg = BitNet2B4TConfig()
    print("persistent full step, one 2B layer against the oracle", flush=True)
    step = BitLinearDecodeStep.random_init(cfg, H.dev(), seed=99, num_layers=1).alloc_buffers(seed=100)
    step.alloc_attention(max_seq_len=512)
    B, Hq, Hkv, S = 32, cfg.num_attention_heads, cfg.num_key_value_heads, 512
    kc0 = H.bits_of(step.kv[0].key_cache).reshape(B, Hkv, S, 128).copy()
    vc0 = H.bits_of(step.kv[0].value_cache).reshape(B, Hkv, S, 128).copy()
    hid = H.bits_of(step.hidden).copy()
    pos = step.pos.cpu().numpy().astype(np.int64)
    step.step_persistent_full()
    step.check()
    w = step.layers[0]

    def wkn(pw):
        return orc.devlayout_decode(pw.data.cpu().numpy().view(np.uint32), pw.in_features, pw.out_features)

    qkv = orc.bitlinear(hid, wkn(w.qkv), list(w.qkv.segment_scales), list(w.qkv.segment_ends),
                        gamma_bf16=H.bits_of(w.input_layernorm), norm_eps=step.eps)["out"]
    assert np.array_equal(H.bits_of(step.qkv_out), qkv)
    cos, sin = orc.rope_tables(128, S, cfg.rope_theta)
    ref, kc2, vc2 = orc.decode_attention(qkv, kc0, vc0, pos, Hq, Hkv, cos, sin, False, step.attention.scale)
    attn = H.bits_of(step.attn_out)
    check(orc, attn, ref, step.kv[0], kc2, vc2)
    h = orc.bitlinear(attn, wkn(w.o_proj), list(w.o_proj.segment_scales), gamma_bf16=H.bits_of(w.attn_sub_norm),
                      norm_eps=step.eps, residual_bf16=hid)["out"]
    r = orc.gate_up_relu2(h, wkn(w.gate_up), w.gate_up.segment_scales[0], w.gate_up.segment_scales[1],
                          gamma_bf16=H.bits_of(w.post_attention_layernorm), norm_eps=step.eps)
    assert np.array_equal(H.bits_of(step.ffn_h), r["h"])
    h = orc.bitlinear(r["h"], wkn(w.down), list(w.down.segment_scales), gamma_bf16=H.bits_of(w.ffn_sub_norm),
                      norm_eps=step.eps, residual_bf16=h)["out"]
    assert np.array_equal(H.bits_of(step.hidden), h)


def test_persistent_full_step_matches_step_full_2b(orc):
    """The 2B model (30 layers, 20 query / 5 key-value heads, batch 32, every
    user at position 511 of a 512 context), the one-launch step with
    attention against step_full, bit for bit; then graph replays of the
    one-launch step from the same state give the same bits again (three
    compared in full, 100 more on the hidden state), and once more with every
    GEMM unit forced onto the sentinel check's re-read path."""
    from bitnet_tt.config import BitNet2B4TConfig
    from bitnet_tt.decode import BitLinearDecodeStep

    print("persistent full step 2B", flush=True)
    step = BitLinearDecodeStep.random_init(BitNet2B4TConfig(), H.dev(), seed=95).alloc_buffers(seed=96)
    step.alloc_attention(max_seq_len=512)
    state = _full_state(step)
    step.step_full()
    step.check()
    ref = _outputs(step)
    _restore(step, state)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        step.step_persistent_full()
    s.synchronize()
    step.check()
    _compare(_outputs(step), ref, "persistent full step")
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        step.step_persistent_full()
    for rep in range(3):
        _restore(step, state)
        g.replay()
        torch.cuda.synchronize()
        _ = torch.ones(1024, device=H.dev()).sum().item()  # eager work between replays
        _compare(_outputs(step), ref, f"graph replay {rep}")
    step.check()
    # 100 more replays, the hidden state compared on the device: the hand-offs
    # of the attention units (QKV words in, attention words out) every layer
    ref_h = torch.from_numpy(ref["hidden"].view(np.int16)).to(H.dev())
    bad = []
    for rep in range(100):
        _restore(step, state)
        g.replay()
        torch.cuda.synchronize()
        if not torch.equal(step.hidden.view(torch.int16), ref_h):
            bad.append(rep)
    step.check()
    assert not bad, f"replays {bad[:10]} differ"
    # Every GEMM unit on the sentinel check's rare path (it waits for its
    # operand pieces, reads them and its weights again and redoes its MFMAs),
    # forced through the step workspace's test word: the attention instance's
    # own register allocation of that path gives the same bits.
    with torch.cuda.stream(s):
        ws = H.step_workspace(step)
    off = int(N.lib().btl_decode_step_error_offset()) + 64
    ws[off:off + 4] = torch.tensor([1, 0, 0, 0], dtype=torch.uint8, device=ws.device)
    try:
        _restore(step, state)
        torch.cuda.synchronize()
        with torch.cuda.stream(s):
            step.step_persistent_full()
        s.synchronize()
        step.check()
        _compare(_outputs(step), ref, "persistent full step, every unit on the re-read path")
    finally:
        ws[off:off + 4] = 0
        torch.cuda.synchronize()


# (users, query heads, kv heads, cache length, positions): the edges of one
# round (511..513 cached positions), of the blocks of 64, of the splits'
# ranges and of the contexts that stay whole (896 and 1280 positions at 13 and 20
# users); 8, 5, 3, 2 and 1 splits per pair.
SPLIT_SHAPES = [
    (1, 4, 1, 4096, [4095]),
    (4, 20, 5, 4096, [0, 511, 512, 4095]),
    (6, 6, 3, 2048, [513, 575, 576, 577, 1023, 1024]),
    (3, 8, 8, 1000, [999, 640, 513]),
    (16, 20, 5, 1024, [1023 - 37 * i for i in range(16)]),
    (23, 20, 5, 640, [639 - i for i in range(23)]),
    (13, 20, 5, 1024, [895, 896, 897, 960, 961, 1023, 512, 513, 0, 1, 700, 64, 1000]),
    (20, 20, 5, 1400, [1279, 1280, 1281, 1399, 1344, 1345, 640, 513, 512, 0] + [1390 - 70 * i for i in range(10)]),
]


@pytest.mark.parametrize("B,Hq,Hkv,S,pos", SPLIT_SHAPES)
def test_split_contexts(orc, B, Hq, Hkv, S, pos):
    """Contexts split over several workgroups against the oracle, twice on the
    same workspace (the arrival counters are left clean)."""
    print(f"split attention B={B} Hq={Hq} Hkv={Hkv} S={S}", flush=True)
    for seed in (51, 52):
        att, cache, got, ref, kc, vc, kc2, vc2 = run(orc, B, Hq, Hkv, S, pos, seed == 52, seed)
        att.check()
        check(orc, got, ref, cache, kc2, vc2)


@pytest.mark.parametrize("B,Hq,Hkv,S,pos", [SPLIT_SHAPES[1], SPLIT_SHAPES[2], (4, 20, 5, 4096, [4095, -1, 4096, 700])])
def test_split_contexts_around_bad_rows(orc, B, Hq, Hkv, S, pos):
    """Cache rows past each user's position hold NaN and infinities, which
    nothing of the output may take up (another split reads the row that split
    0 writes); users outside the range among split ones give zeros, leave
    their caches as they are and are flagged, and the same call with every
    user in range is right after it."""
    print(f"split attention, bad rows B={B} Hq={Hq} Hkv={Hkv} S={S}", flush=True)
    rng = np.random.default_rng(57)
    D = 128
    qkv = orc.f32_to_bf16(rng.standard_normal((B, (Hq + 2 * Hkv) * D)).astype(np.float32))
    kv = [orc.f32_to_bf16(rng.standard_normal((B, Hkv, S, D)).astype(np.float32)) for _ in "kv"]
    bad = [p < 0 or p >= S for p in pos]
    for c in kv:
        for b, p in enumerate(pos):
            c[b, :, max(p, 0):, 0::2] = 0x7FC0  # NaN
            c[b, :, max(p, 0):, 1::2] = 0xFF80  # -inf
    att = DecodeAttention(Hq, Hkv, D, S, H.dev())
    cache = att.new_cache(B)
    assert cache.split is not None
    cache.key_cache.copy_(H.to_dev_bf16(kv[0]).view(B, Hkv, S, D))
    cache.value_cache.copy_(H.to_dev_bf16(kv[1]).view(B, Hkv, S, D))
    x = H.to_dev_bf16(qkv)
    cos, sin = orc.rope_tables(D, S, 500000.0)
    cur = list(pos)
    for rep in range(2):
        got = orc.bf16_to_f32(H.bits_of(att(x, cache, torch.tensor(cur, dtype=torch.int32, device=H.dev()))))
        if rep == 0 and any(bad):
            with pytest.raises(RuntimeError, match="out of range"):
                att.check()
        else:
            att.check()
        for b in range(B):
            if rep == 0 and bad[b]:
                assert not got[b].any()
                assert np.array_equal(H.bits_of(cache.key_cache[b]).reshape(Hkv, S, D), kv[0][b])
                assert np.array_equal(H.bits_of(cache.value_cache[b]).reshape(Hkv, S, D), kv[1][b])
                continue
            ref = orc.decode_attention(qkv[b:b + 1], kv[0][b:b + 1], kv[1][b:b + 1], np.asarray(cur[b:b + 1]), Hq, Hkv,
                                       cos, sin, False, att.scale)[0]
            tol = 2.0 ** -7 * np.abs(ref) + 1e-3 * np.abs(ref).max()
            assert np.all(np.abs(got[b] - ref) <= tol), b
        # the users that were outside: at the start of their cache
        cur = [0 if f else p for f, p in zip(bad, pos)]


@pytest.mark.parametrize("positions", [
    ([4095, 4096, 900, 64, 3000], [-1, 2000, 4095, 600, 513], [4095, 4000, 900, 64, 3000]),
    ([4096], [4000], [-1], [100]),  # one user: its own kernel
])
def test_split_step_with_a_position_out_of_range(orc, positions):
    """The one-launch step with split contexts and one user outside the range:
    the others' layer as step_full's, that user's attention zero, flagged; the
    next step, every user in range, is right."""
    from bitnet_tt.config import BitNet2B4TConfig
    from bitnet_tt.decode import BitLinearDecodeStep

    step = BitLinearDecodeStep.random_init(BitNet2B4TConfig(), H.dev(), seed=89, batch=len(positions[0]), num_layers=1)
    step.alloc_buffers(seed=90).alloc_attention(max_seq_len=4096)
    for pos in positions:
        step.pos.copy_(torch.tensor(pos, dtype=torch.int32))
        bad = [b for b, p in enumerate(pos) if p < 0 or p >= 4096]
        state = _full_state(step)
        outs = []
        for run_step in (step.step_full, step.step_persistent_full):
            _restore(step, state)
            run_step()
            if bad:
                with pytest.raises(RuntimeError, match="out of range"):
                    step.check()
            step.check()
            outs.append(_outputs(step))
        _compare(outs[1], outs[0], f"positions {pos}")
        attn = step.attn_out.float()
        assert all(bool((attn[b] == 0).all()) for b in bad)


def test_whole_context_entry_needs_one_zero_word(orc):
    """btl_decode_attention at a shape whose contexts the split entry would
    split: a 256-byte workspace of which only the error word is zero."""
    B, Hq, Hkv, S, D = 2, 20, 5, 2048, 128
    pos = [2047, 1300]
    att, cache, _, ref, kc, vc, kc2, vc2 = run(orc, B, Hq, Hkv, S, pos, False, 53)
    rng = np.random.default_rng(53)
    qkv = H.to_dev_bf16(orc.f32_to_bf16(rng.standard_normal((B, (Hq + 2 * Hkv) * D)).astype(np.float32)))
    ws = torch.full((256,), 0xA5, dtype=torch.uint8, device=H.dev())
    ws[:4] = 0
    p = torch.tensor(pos, dtype=torch.int32, device=H.dev())
    out = torch.full((B, Hq * D), 7.0, dtype=torch.bfloat16, device=H.dev())
    N.check(N.lib().btl_decode_attention(
        N.ptr(qkv), B, Hq, Hkv, D, S, N.ptr(p), N.ptr(att.rope_cos), N.ptr(att.rope_sin), 0, att.scale,
        N.ptr(cache.key_cache), N.ptr(cache.value_cache), N.ptr(out), N.ptr(ws), 256, N.stream_of(H.dev())), "attention")
    torch.cuda.synchronize()
    assert int(ws[:4].view(torch.int32).item()) == 0 and bool((ws[4:] == 0xA5).all())
    check(orc, H.bits_of(out), ref, cache, kc2, vc2)
    # a cache object without a split scratch: the same whole contexts
    cache.split = None
    assert np.array_equal(H.bits_of(att(qkv, cache, p)), H.bits_of(out))


def test_split_call_recovers_from_left_over_arrivals(orc):
    """Arrivals that an earlier call left in the scratch do not keep a later
    call from merging: the same bits as on a clean scratch, and the counts are
    zero again."""
    B, Hq, Hkv, S = 3, 20, 5, 4096
    rng = np.random.default_rng(54)
    att = DecodeAttention(Hq, Hkv, 128, S, H.dev())
    cache = att.new_cache(B)
    cache.key_cache.normal_()
    cache.value_cache.normal_()
    qkv = H.to_dev_bf16(orc.f32_to_bf16(rng.standard_normal((B, (Hq + 2 * Hkv) * 128)).astype(np.float32)))
    pos = torch.tensor([4095, 700, 2000], dtype=torch.int32, device=H.dev())
    ref = att(qkv, cache, pos)
    words = cache.split[: 8 * B * Hkv].view(torch.int64)
    words += torch.arange(B * Hkv, device=H.dev()) % 9
    for rep in range(3):
        out = torch.full_like(ref, 7.0)
        att(qkv, cache, pos, out=out)
        assert torch.equal(out, ref), rep
        assert int((words % 16).abs().max().item()) == 0, rep


def test_graphs_of_one_stream_replayed_at_once(orc):
    """Two graphs captured on one stream, each with its own cache, replayed on
    two streams at once give what each gives alone."""
    B, Hq, Hkv, S = 2, 20, 5, 4096
    att = DecodeAttention(Hq, Hkv, 128, S, H.dev())
    s = torch.cuda.Stream()
    calls = []
    for i in range(2):
        cache = att.new_cache(B)
        cache.key_cache.normal_()
        cache.value_cache.normal_()
        qkv = torch.randn((B, (Hq + 2 * Hkv) * 128), device=H.dev()).bfloat16()
        pos = torch.tensor([4000 - 900 * i, 3000], dtype=torch.int32, device=H.dev())
        out = torch.empty((B, Hq * 128), dtype=torch.bfloat16, device=H.dev())
        torch.cuda.synchronize()
        with torch.cuda.stream(s):
            att(qkv, cache, pos, out=out)
        s.synchronize()
        ref = out.clone()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            for _ in range(8):
                att(qkv, cache, pos, out=out)
        calls.append((g, out, ref, cache, qkv, pos, torch.cuda.Stream()))
    for rep in range(20):
        for g, out, *_ in calls:
            out.zero_()
        torch.cuda.synchronize()
        for g, *_, st in calls:
            with torch.cuda.stream(st):
                g.replay()
        torch.cuda.synchronize()
        for i, (g, out, ref, *_) in enumerate(calls):
            assert torch.equal(out, ref), (rep, i)
    att.check()


@pytest.mark.parametrize("batch,kv,S", [(1, 1, 4096), (5, 2, 1024), (26, 1, 640)])
def test_persistent_full_step_split_contexts(orc, batch, kv, S):
    """The one-launch step with split contexts against step_full, bit for bit,
    three steps in a row at moving positions (the partials' words are reused by
    every layer and launch)."""
    from bitnet_tt.config import BitNetMiniConfig
    from bitnet_tt.decode import BitLinearDecodeStep

    cfg = BitNetMiniConfig(num_layers=2, num_attention_heads=4, num_key_value_heads=kv, hidden_size=512,
                           intermediate_size=512)
    print(f"persistent full step, split contexts: batch {batch} kv {kv} S {S}", flush=True)
    step = BitLinearDecodeStep.random_init(cfg, H.dev(), seed=93, batch=batch).alloc_buffers(seed=94)
    step.alloc_attention(max_seq_len=S)
    for back in (1, S // 2 - 60, 2):
        step.pos.copy_(torch.tensor([max(0, S - back - 13 * i) for i in range(batch)], dtype=torch.int32))
        state = _full_state(step)
        step.step_full()
        step.check()
        ref = _outputs(step)
        _restore(step, state)
        step.step_persistent_full()
        step.check()
        _compare(_outputs(step), ref, f"split contexts, back {back}")


@pytest.mark.parametrize("batch", [5, 11, 13, 22])
def test_persistent_full_step_split_contexts_on_qkv_units(orc, batch):
    """Batches at the 2B shape whose attention items reach units that also run
    QKV (200, 220, 195 and 220 items of 224 units, 60 of them QKV's), users at short,
    middle and long contexts: the one-launch step against step_full."""
    from bitnet_tt.config import BitNet2B4TConfig
    from bitnet_tt.decode import BitLinearDecodeStep

    print(f"persistent full step, split contexts at the 2B shape: batch {batch}", flush=True)
    step = BitLinearDecodeStep.random_init(BitNet2B4TConfig(), H.dev(), seed=87, batch=batch, num_layers=2)
    step.alloc_buffers(seed=88).alloc_attention(max_seq_len=4096)
    for first in (4095, 700):
        step.pos.copy_(torch.tensor([max(0, first - 190 * i) for i in range(batch)], dtype=torch.int32))
        state = _full_state(step)
        step.step_full()
        step.check()
        ref = _outputs(step)
        for rep in range(2):
            _restore(step, state)
            step.step_persistent_full()
            step.check()
            _compare(_outputs(step), ref, f"batch {batch}, first position {first}, rep {rep}")


# Batch 1, whose step has a kernel of its own: whole and split contexts, two
# chunks of F per thread, and a shape whose 216 units and 64 attention items do
# not fit 256 workgroups (the two-hop kernel).
ONE_USER_FULL = [
    (dict(num_layers=2, num_attention_heads=4, num_key_value_heads=1, hidden_size=512, intermediate_size=512), 256),
    (dict(num_layers=3, num_attention_heads=16, num_key_value_heads=8, hidden_size=2048, intermediate_size=512), 1000),
    (dict(num_layers=2, num_attention_heads=20, num_key_value_heads=5, hidden_size=2560, intermediate_size=6912), 4096),
    (dict(num_layers=1, num_attention_heads=16, num_key_value_heads=8, hidden_size=2048, intermediate_size=6912), 4096),
]


@pytest.mark.parametrize("shape,S", ONE_USER_FULL)
def test_one_user_full_step_matches_step_full(orc, shape, S):
    """The one-launch step with attention at batch 1 against step_full, bit for
    bit, at an early, a middle and the last position."""
    from bitnet_tt.config import BitNetMiniConfig
    from bitnet_tt.decode import BitLinearDecodeStep

    print(f"one-user full step {shape} S={S}", flush=True)
    step = BitLinearDecodeStep.random_init(BitNetMiniConfig(**shape), H.dev(), seed=83, batch=1).alloc_buffers(seed=84)
    step.alloc_attention(max_seq_len=S)
    for pos in (0, S // 2 + 3, S - 1):
        step.pos.fill_(pos)
        state = _full_state(step)
        step.step_full()
        step.check()
        ref = _outputs(step)
        for rep in range(3):
            _restore(step, state)
            step.step_persistent_full()
            step.check()
            _compare(_outputs(step), ref, f"one user, pos {pos}, rep {rep}")
