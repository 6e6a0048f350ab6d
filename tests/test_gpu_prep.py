"""GPU parity of the load-time kernels: absmean weight quantisation, the
reference tile format (pack / unpack) and the repack into the GEMM layout.
All integer/byte work: bit-exact against the oracle."""

import numpy as np
import pytest
import torch

import helpers as H
from bitnet_tt.kernels import pack as P
from bitnet_tt.utils import quantization as Q

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(7,), (64, 128), (300, 301), (640, 2560), (6912, 2560)])
def test_weight_quant_device_matches_numpy(orc, shape):
    w = H.latent(int(np.prod(shape[:-1])) if len(shape) > 1 else 1, shape[-1], seed=sum(shape))
    w = w.reshape(shape)
    print(f"weight quant shape={shape}", flush=True)
    q_d, s_d = Q.weight_quant_ternary(H.to_dev(w))
    q_h, s_h = orc.weight_quant_ternary(w)
    assert np.float32(s_d) == s_h
    assert np.array_equal(q_d.cpu().numpy(), q_h)


def test_weight_quant_device_unaligned_and_partial(orc):
    """Full 8192-blocks plus a partial last block, from a buffer that is not
    16-byte aligned (the one-thread block sums) and from an aligned one (one
    wave per full block): the scale and codes equal numpy's either way."""
    w = H.latent(1, 3 * 8192 + 12, seed=41).reshape(-1)
    d = H.to_dev(w)
    print("weight quant unaligned / aligned, n=%d" % (w.size - 1), flush=True)
    for view, host in ((d[1:], w[1:]), (d[:-1], w[:-1])):
        q_d, s_d = Q.weight_quant_ternary(view)
        q_h, s_h = orc.weight_quant_ternary(np.ascontiguousarray(host))
        assert np.float32(s_d) == s_h
        assert np.array_equal(q_d.cpu().numpy(), q_h)


def test_weight_quant_device_special_cases(orc):
    z = torch.zeros((4, 64), dtype=torch.float32, device=H.dev())
    q, s = Q.weight_quant_ternary(z)
    assert np.float32(s) == np.float32(1e-5) and int(q.abs().sum()) == 0
    w = np.array([0.5, 1.5, -0.5, -1.5, 0.0, 2.0], np.float32)
    q, s = Q.weight_quant_ternary(H.to_dev(w))
    assert s == 1.0 and q.cpu().tolist() == [0, 1, 0, -1, 0, 1]


@pytest.mark.parametrize("out_f,in_f", [(32, 32), (64, 128), (50, 100), (33, 65), (3840, 2560)])
def test_pack_unpack_device(orc, out_f, in_f):
    print(f"pack out={out_f} in={in_f}", flush=True)
    q = H.ternary(out_f, in_f, seed=out_f + in_f)
    packed = P.pack_ternary_tilized_device(H.to_dev(q))
    ref, _ = orc.pack_ternary_tilized(q, 1.0)
    assert np.array_equal(packed.cpu().numpy(), ref)
    un = P.unpack_ternary_tilized_device(packed, in_f, out_f)
    assert np.array_equal(un.cpu().numpy(), q.T)


def test_unpack_device_reads_reserved_code_as_zero(orc):
    packed = torch.full((1, 256), 0xFF, dtype=torch.uint8, device=H.dev())
    un = P.unpack_ternary_tilized_device(packed, 32, 32)
    assert int(un.abs().sum()) == 0


@pytest.mark.parametrize("k,n", [(32, 32), (96, 64), (128, 96), (224, 32), (2560, 3840), (6912, 2560)])
def test_repack_matches_oracle_layout(orc, k, n):
    print(f"repack K={k} N={n}", flush=True)
    w_kn = H.ternary(k, n, seed=k * 7 + n)
    packed, _ = orc.pack_ternary_tilized(np.ascontiguousarray(w_kn.T), 1.0)
    wdev = P.repack_for_gemm(H.to_dev(packed), k, n)
    got = wdev.cpu().numpy().view(np.uint32)
    assert np.array_equal(got, orc.devlayout_encode(w_kn))
    assert np.array_equal(orc.devlayout_decode(got, k, n), w_kn)


@pytest.mark.parametrize("n", [1, 7, 8, 9, 127, 128, 129, 135, 136, 137, 263, 1031, 4103, 6000, 8184, 8191, 8193, 16383])
def test_weight_scale_of_every_block_length(orc, n):
    """Partial blocks around the leaves of numpy's split tree, aligned and not:
    the scale is numpy's to the bit."""
    w = H.latent(1, n + 1, seed=43 + n).reshape(-1)
    d = H.to_dev(w)
    for view, host in ((d[:n], w[:n]), (d[1:], w[1:])):
        q_d, s_d = Q.weight_quant_ternary(view)
        q_h, s_h = orc.weight_quant_ternary(np.ascontiguousarray(host))
        assert np.float32(s_d) == s_h and np.array_equal(q_d.cpu().numpy(), q_h)


@pytest.mark.parametrize("n,k,special", [(32, 32, False), (64, 96, False), (96, 160, True), (160, 128, True),
                                         (2560, 6912, False), (1440, 4064, True)])
def test_quantize_for_gemm_matches_the_three_passes(orc, n, k, special):
    """The one-pass load against quantise, tiles and repack, bit for bit; with
    `special`, ties at half the scale, zeros, a NaN (the scale is then eps) and,
    in a second weight, an infinity (an infinite scale)."""
    from bitnet_tt.kernels.pack import pack_ternary_tilized_device, quantize_for_gemm, repack_for_gemm

    print(f"quantize_for_gemm {n}x{k}", flush=True)
    w = H.latent(n, k, seed=n + k)
    ws = [w]
    if special:
        t = np.float32(0.5) * np.mean(np.abs(w), dtype=np.float32)
        w2, w3, w4 = w.copy(), w.copy(), w.copy()
        w2[::3, ::5] = t
        w2[1::3, ::7] = np.nextafter(-t, np.float32(-1))
        w2[2, :] = 0.0
        w3[0, 0] = np.nan
        w3[3, 1:9] = [5e-6, -5e-6, 5.1e-6, -5.1e-6, 0.0, 1.0, -0.0, np.nan]
        w4[n // 2, k // 2] = -np.inf
        ws += [w2, w3, w4]
    for x in ws:
        d = H.to_dev(x)
        q, s = Q.weight_quant_ternary(d)
        ref = repack_for_gemm(pack_ternary_tilized_device(q), k, n)
        got, s2 = quantize_for_gemm(d)
        assert s == s2 and torch.equal(got, ref)
