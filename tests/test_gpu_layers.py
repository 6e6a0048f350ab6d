"""GPU parity of the reference-API layers (Linear, FeedForward, fused QKV) and
of the decode-step chain, on the BitLinear configurations of the 2B model:

  C1  single BitLinear 2560->2560, x ~N(0,1) with 1 % outlier channels x20,
      W ~N(0,0.02) absmean-quantised;
  C2  fused RMSNorm + QKV 2560->3840 (20 Q / 5 KV heads of 128), three scales;
  C3  FFN block: gate||up 2560->2x6912, relu^2*up, ffn_sub_norm, down 6912->2560;
  C4  decode-step chain: all 30 layers at full size bit-exact against the
      oracle chain for both launch structures (120 fused launches and the
      one-launch step, its sentinel re-read path forced too), the mini model
      and graph replays likewise;
  C5  prefill BitLinear through the layer API (M = 512).

Integer results and bf16 outputs are compared bit for bit with the oracle
(RMSNorm in its fixed fp32 order); against the float64 reading of the
reference formula the bf16 output is within 1e-2 relative.
"""

import numpy as np
import pytest
import torch

import helpers as H
from bitnet_tt.config import BitNet2B4TConfig, BitNetMiniConfig
from bitnet_tt.decode import BitLinearDecodeStep
from bitnet_tt.layers.attention import QKVProjection
from bitnet_tt.layers.bitlinear import Linear
from bitnet_tt.layers.ffn import FeedForward
from bitnet_tt.ternary_matmul import ternary_matmul
from bitnet_tt import _native as N

pytestmark = pytest.mark.gpu


def rel_err(out_bits, ref64, orc):
    out = orc.bf16_to_f32(out_bits).astype(np.float64)
    return np.max(np.abs(out - ref64)) / np.max(np.abs(ref64))


def test_c1_single_bitlinear(orc):
    m, k, n = 32, 2560, 2560
    xb = H.activations(orc, m, k, seed=101)
    w = H.latent(n, k, seed=102)
    lin = Linear(k, n, H.dev())
    lin.load_weights(w)
    out = lin(H.to_dev_bf16(xb))
    q, s = orc.weight_quant_ternary(w)
    assert lin.weight_scale == float(s)
    ref = orc.bitlinear(xb, np.ascontiguousarray(q.T), [float(s)])
    assert np.array_equal(H.bits_of(out), ref["out"])
    # float64 reading of quant -> matmul -> scale
    xf = orc.bf16_to_f32(xb).astype(np.float64)
    a = np.abs(xf).max(1, keepdims=True)
    ref64 = np.clip(np.round(xf * (127 / a)), -128, 127) @ q.T.astype(np.float64) * float(s) * a / 127
    assert rel_err(H.bits_of(out), ref64, orc) < 1e-2
    split = [(q == 1).mean(), (q == 0).mean(), (q == -1).mean()]
    print(f"C1 ternary split +1/0/-1 = {split[0]:.3f}/{split[1]:.3f}/{split[2]:.3f}")


def test_c1_device_weight_load_matches_host(orc):
    k, n = 2560, 2560
    w = H.latent(n, k, seed=102)
    a, b = Linear(k, n, H.dev()), Linear(k, n, H.dev())
    a.load_weights(w)
    b.load_weights(H.to_dev(w))
    assert a.weight_scale == b.weight_scale
    assert torch.equal(a.weight.data, b.weight.data)


def test_c2_fused_rmsnorm_qkv(orc):
    c = BitNet2B4TConfig()
    H_, qd, kvd = c.hidden_size, c.num_attention_heads * c.head_dim, c.num_kv_heads * c.head_dim
    xb = H.activations(orc, 32, H_, seed=201)
    gb = H.gamma(orc, H_, seed=202)
    wq, wk, wv = H.latent(qd, H_, 203), H.latent(kvd, H_, 204), H.latent(kvd, H_, 205)
    proj = QKVProjection(H_, c.num_attention_heads, c.num_kv_heads, c.head_dim, H.dev())
    proj.load_weights(wq, wk, wv)
    out = proj(H.to_dev_bf16(xb), norm_weight=H.to_dev_bf16(gb), norm_epsilon=c.rms_norm_eps)
    qs = [orc.weight_quant_ternary(w) for w in (wq, wk, wv)]
    w_kn = np.ascontiguousarray(np.concatenate([q for q, _ in qs]).T)
    ends = [qd, qd + kvd, qd + 2 * kvd]
    ref = orc.bitlinear(xb, w_kn, [float(s) for _, s in qs], ends, gamma_bf16=gb, norm_eps=c.rms_norm_eps)
    assert out.shape == (32, 3840)
    assert np.array_equal(H.bits_of(out), ref["out"])
    # RMSNorm in double precision (reference formula) -> output within 1e-2
    ref0 = orc.bitlinear(xb, w_kn, [float(s) for _, s in qs], ends, gamma_bf16=gb, norm_eps=c.rms_norm_eps, order=0)
    assert rel_err(H.bits_of(out), orc.bf16_to_f32(ref0["out"]).astype(np.float64), orc) < 1e-2


def test_c2_rope_permutation_and_unscaled(orc):
    hd, nh, nkv, hid = 16, 4, 2, 64
    rng_w = [H.latent(nh * hd, hid, 1), H.latent(nkv * hd, hid, 2), H.latent(nkv * hd, hid, 3)]
    xb = H.activations(orc, 8, hid, seed=4, outliers=False)
    gb = H.gamma(orc, hid, seed=5)
    proj = QKVProjection(hid, nh, nkv, hd, H.dev(), use_fused_rope=True)
    proj.load_weights(*rng_w, apply_scales=False)
    out = proj(H.to_dev_bf16(xb), norm_weight=H.to_dev_bf16(gb), norm_epsilon=1e-5)
    qs = [orc.weight_quant_ternary(w) for w in rng_w]
    qt = orc.permute_halfsplit_to_adjacent(np.ascontiguousarray(qs[0][0].T), nh, hd)
    kt = orc.permute_halfsplit_to_adjacent(np.ascontiguousarray(qs[1][0].T), nkv, hd)
    w_kn = np.ascontiguousarray(np.concatenate([qt, kt, qs[2][0].T], axis=1))
    ref = orc.bitlinear(xb, w_kn, [1.0, 1.0, 1.0], [64, 96, 128], gamma_bf16=gb, norm_eps=1e-5)
    assert np.array_equal(H.bits_of(out), ref["out"])


def test_c3_ffn_block(orc):
    c = BitNet2B4TConfig()
    Hh, F = c.hidden_size, c.intermediate_size
    xb = H.activations(orc, 32, Hh, seed=301)
    g_post = H.gamma(orc, Hh, seed=302)
    sub = orc.bf16_to_f32(H.gamma(orc, F, seed=303))
    gate, up, down = H.latent(F, Hh, 304), H.latent(F, Hh, 305), H.latent(Hh, F, 306)
    ffn = FeedForward(Hh, F, H.dev(), eps=c.rms_norm_eps)
    ffn.load_weights(gate, up, down, sub)
    res = orc.f32_to_bf16(np.random.default_rng(307).standard_normal((32, Hh)).astype(np.float32))
    y = ffn(H.to_dev_bf16(xb), mode="decode", norm_weight=H.to_dev_bf16(g_post), norm_epsilon=c.rms_norm_eps,
            residual=H.to_dev_bf16(res))
    gq, gs = orc.weight_quant_ternary(gate)
    uq, us = orc.weight_quant_ternary(up)
    dq, ds = orc.weight_quant_ternary(down)
    r1 = orc.gate_up_relu2(xb, np.ascontiguousarray(np.concatenate([gq, uq]).T), float(gs), float(us),
                           gamma_bf16=g_post, norm_eps=c.rms_norm_eps)
    r2 = orc.bitlinear(r1["h"], np.ascontiguousarray(dq.T), [float(ds)], gamma_bf16=orc.f32_to_bf16(sub),
                       norm_eps=c.rms_norm_eps, residual_bf16=res)
    assert np.array_equal(H.bits_of(y), r2["out"])


def test_c5_prefill_linear(orc):
    m, k, n = 512, 2560, 2560
    xb = H.activations(orc, m, k, seed=501)
    gb = H.gamma(orc, k, seed=502)
    w = H.latent(n, k, seed=503)
    lin = Linear(k, n, H.dev())
    lin.load_weights(w)
    out = H.bits_of(lin(H.to_dev_bf16(xb), norm_weight=H.to_dev_bf16(gb), norm_epsilon=1e-5))
    q, s = orc.weight_quant_ternary(w)
    rows = [0, 1, 77, 255, 256, 511]
    ref = orc.bitlinear(np.ascontiguousarray(xb[rows]), np.ascontiguousarray(q.T), [float(s)], gamma_bf16=gb,
                        norm_eps=1e-5)
    assert np.array_equal(out[rows], ref["out"])


def test_ternary_matmul_op_signature(orc):
    """The reference call form: ternary_matmul(x, W, use_packed_ternary=True,
    norm_weight=..., norm_epsilon=...) with [1, 1, M, K] activations."""
    k, n = 256, 96
    xb = H.activations(orc, 32, k, seed=601).reshape(1, 1, 32, k)
    gb = H.gamma(orc, k, seed=602)
    w = H.latent(n, k, seed=603)
    lin = Linear(k, n, H.dev())
    lin.load_weights(w)
    out = ternary_matmul(H.to_dev_bf16(xb), lin.weight, use_packed_ternary=True,
                         norm_weight=H.to_dev_bf16(gb).reshape(1, 1, 1, k), norm_epsilon=1e-5)
    assert out.shape == (1, 1, 32, n)
    q, s = orc.weight_quant_ternary(w)
    ref = orc.bitlinear(xb.reshape(32, k), np.ascontiguousarray(q.T), [float(s)], gamma_bf16=gb, norm_eps=1e-5)
    assert np.array_equal(H.bits_of(out).reshape(32, n), ref["out"])
    with pytest.raises(RuntimeError, match="Weights not loaded"):
        Linear(k, n, H.dev())(H.to_dev_bf16(xb))


def oracle_layer(orc, step, i, hidden, attn):
    """One decode layer of the chain on the CPU, from the device weights."""
    w = step.layers[i]
    eps = step.eps
    c = step.config

    def wkn(pw):
        dev = pw.data.cpu().numpy().view(np.uint32)
        return orc.devlayout_decode(dev, pw.in_features, pw.out_features)

    g = lambda t: H.bits_of(t)  # noqa: E731
    qkv = orc.bitlinear(hidden, wkn(w.qkv), list(w.qkv.segment_scales), list(w.qkv.segment_ends),
                        gamma_bf16=g(w.input_layernorm), norm_eps=eps)["out"]
    hidden = orc.bitlinear(attn, wkn(w.o_proj), list(w.o_proj.segment_scales), gamma_bf16=g(w.attn_sub_norm),
                           norm_eps=eps, residual_bf16=hidden)["out"]
    r = orc.gate_up_relu2(hidden, wkn(w.gate_up), w.gate_up.segment_scales[0], w.gate_up.segment_scales[1],
                          gamma_bf16=g(w.post_attention_layernorm), norm_eps=eps)
    hidden = orc.bitlinear(r["h"], wkn(w.down), list(w.down.segment_scales), gamma_bf16=g(w.ffn_sub_norm),
                           norm_eps=eps, residual_bf16=hidden)["out"]
    assert c.qkv_dim == qkv.shape[1]
    return hidden, qkv


def test_c4_mini_decode_chain_exact(orc):
    cfg = BitNetMiniConfig(num_layers=2)
    step = BitLinearDecodeStep.random_init(cfg, H.dev(), seed=7).alloc_buffers(seed=8)
    hid, attn = H.bits_of(step.hidden), H.bits_of(step.attn_out)
    step.step()
    torch.cuda.synchronize()
    for i in range(2):
        hid, qkv = oracle_layer(orc, step, i, hid, attn)
    assert np.array_equal(H.bits_of(step.hidden), hid)
    assert np.array_equal(H.bits_of(step.qkv_out), qkv)


def test_c4_graph_replay_matches_eager(orc):
    cfg = BitNetMiniConfig(num_layers=3)
    step = BitLinearDecodeStep.random_init(cfg, H.dev(), seed=9).alloc_buffers(seed=10)
    step.step()  # warm-up: workspaces exist before capture
    step.reset_hidden()
    step.step()
    torch.cuda.synchronize()
    eager = H.bits_of(step.hidden)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        step.reset_hidden()
        step.step()
    torch.cuda.current_stream().wait_stream(s)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):  # the stream whose workspaces the warm-up made
        step.step()
    for rep in range(4):
        step.reset_hidden()
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert np.array_equal(H.bits_of(step.hidden), eager), f"replay {rep} differs"
        _ = torch.ones(1024, device=H.dev()).sum().item()  # eager work between replays


@pytest.fixture(scope="module")
def c4_model(orc):
    """The 2B model (30 layers, seeded random init, outlier activations) on the
    device, and the oracle's 30-layer chain from the same device weights and
    inputs: (step, hidden after layer i for every i, qkv of the last layer)."""
    cfg = BitNet2B4TConfig()
    step = BitLinearDecodeStep.random_init(cfg, H.dev(), seed=11).alloc_buffers(seed=12)
    assert len(step.layers) == 30
    pos, zero, neg = step.ternary_split
    print(f"C4 ternary split +1/0/-1 = {pos:.4f}/{zero:.4f}/{neg:.4f}", flush=True)
    assert abs(zero - 0.31) < 0.01
    hid, attn = H.bits_of(step.hidden0), H.bits_of(step.attn_out)
    hiddens = []
    for i in range(len(step.layers)):
        hid, qkv = oracle_layer(orc, step, i, hid, attn)
        hiddens.append(hid)
        print(f"oracle layer {i} done", flush=True)
    return step, hiddens, qkv


def test_c4_full_model_per_call_chain_exact(orc, c4_model):
    """All 120 fused launches of the 30-layer step (step_per_call) against the
    oracle chain: the final hidden state and the last QKV output bit for bit;
    a second step from the same input gives the same bits."""
    step, hiddens, ref_qkv = c4_model
    step.reset_hidden()
    step.step_per_call()
    step.check()
    got = H.bits_of(step.hidden)
    bad = int((got != hiddens[-1]).sum())
    assert bad == 0, f"{bad} of {got.size} hidden values differ after 30 layers"
    assert np.array_equal(H.bits_of(step.qkv_out), ref_qkv)
    step.reset_hidden()
    step.step_per_call()
    step.check()
    assert np.array_equal(H.bits_of(step.hidden), got)


# Agreement with the reference's own CPU order (torch HF RMSNorm statistic,
# numpy quantiser).  The GPU follows a fixed fp32 order for the RMS statistic
# (bit-exact with the oracle above); the reference order differs from it in the
# last bit of 1/rms now and then, which flips ~1e-5 of the normalised bf16
# values and ~1.6e-7 of the int8 codes per BitLinear: ~2.3 flipped codes in the
# 14 M codes of a 30-layer batch-32 step.  One flipped code moves a whole output
# row by one quantisation step, and the chain carries that on: on the CPU, a
# single flipped code in layer 0 ends the 30-layer chain 2.2 % apart normwise,
# 4.0 % in the largest element (relative to the largest magnitude), PCC 0.99975.
# Bounds: each single BitLinear within 1e-2 of the largest reference magnitude
# (the per-BitLinear bar); the 30-layer chain within what a few early flipped
# codes give: normwise 5e-2, largest element 1e-1, PCC >= 0.999.
CHAIN_REL_FRO, CHAIN_MAX_REL, CHAIN_PCC, ONE_BITLINEAR_MAX_REL = 5e-2, 1e-1, 0.999, 1e-2


def test_c4_persistent_step_against_reference_order_chain(orc, c4_model):
    step, _, _ = c4_model
    h0, attn = H.bits_of(step.hidden0), H.bits_of(step.attn_out)
    step.reset_hidden()
    step.step_persistent()
    step.check()
    got_h, got_qkv = H.bits_of(step.hidden), H.bits_of(step.qkv_out)
    # one BitLinear: layer 0's QKV from the step's input (the mini chain of one layer)
    step.reset_hidden()
    step.layer(0, step.hidden, step.attn_out, step.qkv_out, step.ffn_h)
    step.check()
    _, ref_qkv1 = H.reference_order_chain(orc, step, h0, attn, layers=1)
    one = H.chain_agreement(orc, H.bits_of(step.qkv_out), ref_qkv1)
    ref_h, ref_qkv = H.reference_order_chain(orc, step, h0, attn)
    chain = H.chain_agreement(orc, got_h, ref_h)
    qkv = H.chain_agreement(orc, got_qkv, ref_qkv)
    print(f"one BitLinear (layer 0 QKV) {one}; 30-layer hidden {chain}; last QKV {qkv}", flush=True)
    assert one["max_rel"] <= ONE_BITLINEAR_MAX_REL, one
    assert chain["rel_fro"] <= CHAIN_REL_FRO, chain
    assert chain["max_rel"] <= CHAIN_MAX_REL, chain
    assert chain["pcc"] >= CHAIN_PCC, chain


@pytest.mark.parametrize("batch,layers", [(32, 2), (5, 3), (17, 1)])
def test_persistent_step_mini_matches_per_call(orc, batch, layers):
    """btl_decode_step (every BitLinear of the step in one launch) against the
    120-launch chain and the oracle: hidden, the last QKV output and the last
    FFN intermediate bit for bit, over three launches in a row (the launch
    epochs advance; nothing is cleared between launches)."""
    cfg = BitNetMiniConfig(num_layers=layers)
    step = BitLinearDecodeStep.random_init(cfg, H.dev(), seed=31 + batch, batch=batch).alloc_buffers(seed=32)
    hid, attn = H.bits_of(step.hidden0), H.bits_of(step.attn_out)
    for i in range(layers):
        hid, qkv = oracle_layer(orc, step, i, hid, attn)
    step.step_per_call()
    step.check()
    ref_ffn = H.bits_of(step.ffn_h)
    assert np.array_equal(H.bits_of(step.hidden), hid)
    for rep in range(3):
        print(f"persistent step batch={batch} layers={layers} launch {rep}", flush=True)
        step.reset_hidden()
        step.qkv_out.zero_()
        step.ffn_h.zero_()
        step.step_persistent()
        step.check()
        assert np.array_equal(H.bits_of(step.hidden), hid), f"launch {rep}: hidden"
        assert np.array_equal(H.bits_of(step.qkv_out), qkv), f"launch {rep}: qkv_out"
        assert np.array_equal(H.bits_of(step.ffn_h), ref_ffn), f"launch {rep}: ffn_h"


def test_handoff_floor_interleaves_with_the_step(orc):
    """btl_decode_step_floor (the persistent step's waits and hand-off stores
    with no arithmetic) runs on the step's workspace without a timed-out
    wait, and persistent steps launched after it on that workspace still
    equal the oracle chain bit for bit."""
    cfg = BitNetMiniConfig(num_layers=2)
    step = BitLinearDecodeStep.random_init(cfg, H.dev(), seed=51).alloc_buffers(seed=52)
    hid, attn = H.bits_of(step.hidden0), H.bits_of(step.attn_out)
    for i in range(2):
        hid, qkv = oracle_layer(orc, step, i, hid, attn)
    step.step_persistent()
    step.check()
    assert np.array_equal(H.bits_of(step.hidden), hid)
    for rep in range(3):
        print(f"hand-off floor launch {rep}", flush=True)
        before = H.bits_of(step.hidden)
        step.step_floor()
        step.check()
        assert np.array_equal(H.bits_of(step.hidden), before), "the floor launch changed hidden"
        step.reset_hidden()
        step.step_persistent()
        step.check()
        assert np.array_equal(H.bits_of(step.hidden), hid), f"step after floor launch {rep}"
        assert np.array_equal(H.bits_of(step.qkv_out), qkv), f"qkv after floor launch {rep}"


def test_persistent_step_graph_replay(orc):
    """The one-launch step captured in a HIP graph: every replay, with eager
    work between replays, equals the eager launch."""
    cfg = BitNetMiniConfig(num_layers=3)
    step = BitLinearDecodeStep.random_init(cfg, H.dev(), seed=41).alloc_buffers(seed=42)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        step.reset_hidden()
        step.step_persistent()  # prepares this stream's workspace
    torch.cuda.synchronize()
    eager = H.bits_of(step.hidden)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        step.step_persistent()
    for rep in range(4):
        step.reset_hidden()
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert np.array_equal(H.bits_of(step.hidden), eager), f"replay {rep} differs"
        _ = torch.ones(1024, device=H.dev()).sum().item()
    step.check()


def test_c4_full_model_persistent_step_exact(orc, c4_model):
    """The 2B 30-layer step as one btl_decode_step launch against the oracle
    chain, twice in a row."""
    step, hiddens, ref_qkv = c4_model
    for rep in range(2):
        step.reset_hidden()
        step.step_persistent()
        step.check()
        got = H.bits_of(step.hidden)
        bad = int((got != hiddens[-1]).sum())
        assert bad == 0, f"run {rep}: {bad} of {got.size} hidden values differ after 30 layers"
        assert np.array_equal(H.bits_of(step.qkv_out), ref_qkv), f"run {rep}: last QKV output"


def test_c4_persistent_step_reread_path(orc, c4_model):
    """The rare path of the step's sentinel check (a GEMM unit that found
    operand bytes not yet landed waits for them, reads its tile and weights
    again and redoes its MFMAs), forced for every unit through the step
    workspace's test word: the same bits as the oracle chain."""
    step, hiddens, ref_qkv = c4_model
    step.reset_hidden()
    step.step_persistent()  # prepares this stream's step workspace
    step.check()
    ws = H.step_workspace(step)
    off = int(N.lib().btl_decode_step_error_offset()) + 64
    ws[off:off + 4] = torch.tensor([1, 0, 0, 0], dtype=torch.uint8, device=ws.device)
    try:
        step.reset_hidden()
        step.step_persistent()
        step.check()
        got = H.bits_of(step.hidden)
        assert int((got != hiddens[-1]).sum()) == 0, "hidden differs with every unit on the re-read path"
        assert np.array_equal(H.bits_of(step.qkv_out), ref_qkv)
    finally:
        ws[off:off + 4] = 0
        torch.cuda.synchronize()


def test_c4_persistent_step_many_replays(orc, c4_model):
    """The 2B one-launch step replayed 300 times from a HIP graph, the inputs
    restored between replays: every replay gives the oracle chain's bits and
    no bounded wait runs out.  The hand-off protocol (flags behind unacknowledged
    operand stores, sentinel bytes between uses, epochs as tags) is exercised
    at every BitLinear of every replay, so a rare ordering gap would show as a
    replay that differs or an error word."""
    step, hiddens, _ = c4_model
    ref = torch.from_numpy(np.ascontiguousarray(hiddens[-1]).view(np.int16)).to(H.dev())
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        step.reset_hidden()
        step.step_persistent()  # prepares this stream's workspace
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        step.reset_hidden()
        step.step_persistent()
    bad = []
    for rep in range(300):
        g.replay()
        s.synchronize()
        if not torch.equal(step.hidden.view(torch.int16), ref):
            bad.append(rep)
        if rep % 100 == 99:
            print(f"persistent step replay {rep + 1}", flush=True)
    step.check()
    assert not bad, f"replays {bad[:10]} differ from the oracle chain"


@pytest.mark.parametrize("device", ["cuda", None, "cuda:0"])
def test_load_weights_one_pass_however_the_device_is_named(orc, monkeypatch, device):
    """A weight on the layer's device takes the one-pass load, also where the
    device was given without an index; the same bytes as the host's."""
    from bitnet_tt.layers import bitlinear as B

    calls = []
    real = B.quantize_for_gemm
    monkeypatch.setattr(B, "quantize_for_gemm", lambda w: calls.append(1) or real(w))
    w = (np.random.default_rng(11).standard_normal((96, 160)) * 0.02).astype(np.float32)
    lin, ref = B.Linear(160, 96, device), B.Linear(160, 96, H.dev())
    lin.load_weights(H.to_dev(w))
    assert calls == [1]
    ref.load_weights(w)
    assert calls == [1] and lin.weight_scale == ref.weight_scale
    assert torch.equal(lin.weight.data, ref.weight.data)


def test_models_taking_turns_keep_their_own_step_workspace(orc):
    """Two models' one-launch steps in turn on one stream, with graph replays of
    the first between them, give what each gives alone; a model's workspaces
    go with it."""
    import gc

    from bitnet_tt import _native as N
    from bitnet_tt.config import BitNetMiniConfig
    from bitnet_tt.decode import BitLinearDecodeStep

    cfg = BitNetMiniConfig(num_layers=2, num_attention_heads=2)
    print("two models in turn", flush=True)
    models = [BitLinearDecodeStep.random_init(cfg, H.dev(), seed=61 + i, batch=8 + i).alloc_buffers(seed=71 + i)
              for i in range(2)]
    refs = []
    for m in models:
        m.step_per_call()
        refs.append(m.hidden.clone())
        m.reset_hidden()
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    g = torch.cuda.CUDAGraph()
    with torch.cuda.stream(s):
        for m in models:
            m.step_persistent()
    s.synchronize()
    with torch.cuda.graph(g, stream=s):
        models[0].step_persistent()
    for rep in range(3):
        for m, ref in zip(models, refs):
            m.reset_hidden()
            m.step_persistent()
            assert torch.equal(m.hidden, ref)
        models[0].reset_hidden()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(models[0].hidden, refs[0])
        m.check()
    owners = [N.owner_id(m) for m in models]
    assert {k[3] for k in N._workspaces if len(k) == 4} >= set(owners)
    del g, m, models
    gc.collect()
    assert not {k[3] for k in N._workspaces if len(k) == 4} & set(owners)


# Batches of one run the kernel whose units do the row work themselves: more
# QKV units than gate||up units and the reverse, one and two chunks of F per
# thread, the 2B shape.
ONE_USER_CONFIGS = [
    dict(num_layers=3, num_attention_heads=2),
    dict(num_layers=1, num_attention_heads=2, intermediate_size=128),
    dict(num_layers=2, num_attention_heads=4, hidden_size=512, intermediate_size=4224),
    dict(num_layers=2, num_attention_heads=20, num_key_value_heads=5, hidden_size=2560, intermediate_size=6912),
]


@pytest.mark.parametrize("shape", ONE_USER_CONFIGS)
def test_one_user_step_matches_per_call(orc, shape):
    """hidden, qkv and FFN rows of the one-launch step at batch 1 equal the
    per-call chain's (pinned to the oracle elsewhere), over 50 graph replays
    with the hand-off floor's launches on the same workspace between them."""
    from bitnet_tt.config import BitNetMiniConfig
    from bitnet_tt.decode import BitLinearDecodeStep

    print(f"one-user step {shape}", flush=True)
    step = BitLinearDecodeStep.random_init(BitNetMiniConfig(**shape), H.dev(), seed=81, batch=1).alloc_buffers(seed=82)
    step.step_per_call()
    ref = [t.clone() for t in (step.hidden, step.qkv_out, step.ffn_h)]
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    g = torch.cuda.CUDAGraph()
    with torch.cuda.stream(s):
        step.step_persistent()
    s.synchronize()
    with torch.cuda.graph(g, stream=s):
        step.step_persistent()
    for rep in range(50):
        step.reset_hidden()
        torch.cuda.synchronize()
        if rep % 10 == 3:
            with torch.cuda.stream(s):
                step.step_floor()
        with torch.cuda.stream(s):
            g.replay()
        s.synchronize()
        for got, want in zip((step.hidden, step.qkv_out, step.ffn_h), ref):
            assert torch.equal(got, want), rep
    step.check()
