"""The online softmax: running maxima that climb, small and large V, waves without scores."""
import math

import pytest
import torch

from oracle import torch_oracle as T
from tests import helpers as H

pytestmark = pytest.mark.gpu

P_MAX = {4: 4.0, 2: 1.0}      # decode.hip: 2^p_shift


def _exact(q, k, v, S, bits, gs, scale):
    """One sequence in 64 bits over what the packed cache and the window hold: (scores [kv head, group head, token], V
    [kv head, token, 128], error of a score as the kernel sums it).  A score's fp32 sums hold 1024 + code in place of the
    code, so their terms reach 1024 * sum |q_c s_c|; two roundings (hi and lo) of that, and those of the score itself."""
    z = T.quantize_kv(k[None, :S].float(), v[None, :S].float(), bits, gs, torch.float16)
    h_k = k.shape[1]
    kh = (z.k_codes.double().reshape(S // gs, gs, h_k, 128) * z.k_scale[0].double()[:, None] + z.k_zero[0].double()[:, None])
    vh = (z.v_codes.double().reshape(S, h_k, 128 // gs, gs) * z.v_scale[0].double()[..., None] + z.v_zero[0].double()[..., None])
    kh = torch.cat([kh.reshape(S, h_k, 128), k[S:].double()]).transpose(0, 1)
    vh = torch.cat([vh.reshape(S, h_k, 128), v[S:].double()]).transpose(0, 1)
    q = q.double().reshape(h_k, -1, 128)
    s = q @ kh.transpose(1, 2) * scale
    terms = 1024 * (q.abs() @ z.k_scale[0].double().permute(1, 2, 0)).max().item()
    return s, vh, abs(scale) * terms * 2 ** -23 + s.abs().max().item() * 2 ** -21


@pytest.mark.parametrize("rise", [0.0, 0.2, 0.3, 0.45, 0.6, 2.2, 30.0])
@pytest.mark.parametrize("bits,gs,scale", [(4, 128, 0.09), (4, 32, -0.09), (2, 128, 0.09), (2, 64, 3.0), (4, 64, 1e-30), (2, 32, -0.5)])
def test_scores_that_climb_from_step_to_step(device, bits, gs, scale, rise):
    """`rise` (in nats) from one unit of a wave to its next, up and (second kv head) down; one split, so that a wave sees several
    units (the waves take them in turn: 16 units on one level), a window behind them.  Rise 0: scores as they come, elsewhere they deviate by 0.05.  Tolerance: fp16 probabilities
    (2^-11 of each, of outputs below 4) and the rounding of the output, and the scores' own error."""
    from bitladder_amd import fwd_kvcache_int, kvcache_pack_int
    level, R, h_k, g = 16 * (64 if bits == 4 else 128), 37, 2, 4
    S = 8 * level
    gen = torch.Generator(device=device).manual_seed(int(10 * rise) + bits + gs)
    q = torch.randn((1, 1, h_k * g, 128), generator=gen, device=device).half()
    k, v = (torch.randn((1, S + R, h_k, 128), generator=gen, device=device).half() for _ in range(2))
    if rise and abs(scale) > 1e-3:
        k *= 0.05 / (abs(scale) * math.sqrt(128))
    # a common direction of q and k carries the climb: channel 7 of k is constant over each level
    q[..., 7] = 1.0
    n = torch.arange(S + R, device=device) // level
    step = rise / abs(scale) if abs(scale) > 1e-3 else rise
    climb = ((n - n.max() / 2) * step * (1 if scale >= 0 else -1)).clamp(-3e4, 3e4)
    k[0, :, 0, 7] = climb.half()
    k[0, :, 1, 7] = -climb.half()
    cache = H.alloc_cache(1, S, h_k, bits, gs, device)
    kvcache_pack_int(k[:, :S], cache[0], cache[1], v[:, :S], cache[2], cache[3], None, None, S, "k-channel", gs, bits)
    s, vh, err = _exact(q[0, 0], k[0], v[0], S, bits, gs, scale)
    if rise and abs(scale) > 1e-3:      # a wave's maxima do climb as said: 64 tokens after 64 tokens of one wave
        tops = s[0, 0, :S].reshape(8, 16, -1).amax(2)
        assert ((tops[1:] - tops[:-1]) - rise).abs().max() < 0.16 + 2 ** -10 * 4 * rise
    want, want_lse = (torch.softmax(s, -1) @ vh).reshape(-1, 128), torch.logsumexp(s, -1).reshape(-1)
    for ns in (1, 0, 3):
        out, lse = fwd_kvcache_int(q, *cache, None, scale, "k-channel", gs, bits, k_residual=k[:, S:].contiguous(),
                                   v_residual=v[:, S:].contiguous(), num_splits=ns, return_lse=True)
        assert (out[0, 0].double() - want).abs().max() < 4e-3 + 4 * err, ns
        assert (lse[0].reshape(-1).double() - want_lse).abs().max() < 5e-4 + err, ns


@pytest.mark.parametrize("rows", [1, 4])
@pytest.mark.parametrize("bits,gs", [(4, 128), (4, 32), (2, 128), (2, 64)])
@pytest.mark.parametrize("size", [1.0, 0.1, 0.01, 0.003, 0.001, 1e-4])
def test_small_values_keep_their_bits(device, bits, gs, size, rows):
    """V of small magnitude, scores of deviation 3: products p * (V scale) below 2^-14 are held to 2^-24.  Every unit of 128
    tokens has a score at the maximum, so that each wave's probabilities are 2^p_shift * exp(s - max).

    Bound: a product's pair is off by 2^-24 / sqrt(12), times the code (rms below 9 of 15, 2.2 of 3), p by as much or 2^-12 of itself, over
    the sum L of the p; fp16 rounding of the output; four times the relative error at V of 1 (7e-4 of the norm for p and the
    fp32 sums) covers neither."""
    from bitladder_amd import fwd_kvcache_int, kvcache_pack_int
    from tests.test_gpu_rows import _blocks
    S, h_k, g = 128 * 64, 2, 8 // rows
    b = 1 if rows == 1 else 72
    gen = torch.Generator(device=device).manual_seed(bits + gs)
    q = torch.randn((1, 1, h_k * g, 128), generator=gen, device=device).half()
    k = torch.randn((1, S, h_k, 128), generator=gen, device=device)
    v = (torch.randn((1, S, h_k, 128), generator=gen, device=device) * size).half()
    best = (q[0, 0].float().reshape(h_k, g, 128) / q[0, 0].float().reshape(h_k, g, 128).norm(dim=-1, keepdim=True)).sum(1) * (4 * 11.3 / 8)
    k[0, ::128] = best
    k = k.half()
    scale = 3 / math.sqrt(128)
    cache = H.alloc_cache(1, S, h_k, bits, gs, device)
    kvcache_pack_int(k, cache[0], cache[1], v, cache[2], cache[3], None, None, S, "k-channel", gs, bits)
    s, vh, err = _exact(q[0, 0], k[0], v[0], S, bits, gs, scale)
    p = P_MAX[bits] * torch.exp(s - s.amax(-1, keepdim=True))
    want = (torch.softmax(s, -1) @ vh).reshape(-1, 128)
    if rows == 1:
        args = (q, *cache)
    else:       # the same sequence often enough for blocks of sixteen pairs, with as many equal rows
        args = (q.expand(b, 2 * rows, -1, -1).contiguous(), *(t.expand(b, *t.shape[1:]).contiguous() for t in cache))
        assert _blocks(b, h_k, 2 * rows * g, S, 0, bits, gs, False, S, 1) == 1      # of sixteen
    out = fwd_kvcache_int(*args, None, scale, "k-channel", gs, bits, num_splits=1)
    rms_code = 9 if bits == 4 else 2.2
    slip = 2 ** -24 / math.sqrt(12) * math.sqrt(S) / p.sum(-1).reshape(-1, 1) * (rms_code + 2 * size)
    bound = ((slip ** 2 + 2 ** -48 / 12) * 128).sum().sqrt() * 1.2 + (8e-4 + err) * want.norm()
    got = (out[0, 0].double() - want).norm()
    assert got < bound, (got / want.norm(), bound / want.norm())
    assert (out == out[:1, :1]).all()


@pytest.mark.parametrize("bits,gs", [(4, 128), (4, 32), (2, 128), (2, 64)])
def test_values_at_the_end_of_the_range(device, bits, gs):
    """V of +-65504, the largest V scale there is, times the largest p: no product overflows."""
    from bitladder_amd import fwd_kvcache_int, kvcache_pack_int
    level, h_k, g = 16 * (64 if bits == 4 else 128), 2, 8
    S = 4 * level
    gen = torch.Generator(device=device).manual_seed(bits + gs)
    q = torch.randn((1, 1, h_k * g, 128), generator=gen, device=device).half()
    k = torch.randn((1, S, h_k, 128), generator=gen, device=device).half() * 0.005
    v = 65504.0 * (torch.randint(0, 2, (1, S, h_k, 128), generator=gen, device=device) * 2 - 1).half()
    q[..., 7] = 1.0
    k[0, :, :, 7] = (((torch.arange(S, device=device) // level) % 2) * 5.0)[:, None].half()
    cache = H.alloc_cache(1, S, h_k, bits, gs, device)
    kvcache_pack_int(k, cache[0], cache[1], v, cache[2], cache[3], None, None, S, "k-channel", gs, bits)
    s, vh, err = _exact(q[0, 0], k[0], v[0], S, bits, gs, 0.09)
    want = (torch.softmax(s, -1) @ vh).reshape(-1, 128)
    for ns in (1, 0):
        out = fwd_kvcache_int(q, *cache, None, 0.09, "k-channel", gs, bits, num_splits=ns)
        assert (out[0, 0].double() - want).abs().max() < 65504 * (1e-3 + err), ns


def test_windows_alone_and_idle_waves(device):
    """No packed tokens: most waves have no score at all, and the reference of those that have comes from a tile."""
    from bitladder_amd import fwd_kvcache_int
    gen = torch.Generator(device=device).manual_seed(1)
    for R in (1, 15, 16, 17, 128):
        q = torch.randn((2, 1, 8, 128), generator=gen, device=device).half()
        k, v = (torch.randn((2, R, 2, 128), generator=gen, device=device).half() for _ in range(2))
        k *= 20
        for bits, gs in ((4, 128), (4, 32), (2, 64)):
            cache = H.alloc_cache(2, 128, 2, bits, gs, device)
            out = fwd_kvcache_int(q, *cache, None, 0.3, "k-channel", gs, bits, seqlen_k=0, k_residual=k, v_residual=v)
            qq = q[:, 0].double().reshape(2, 2, 4, 128)
            p = torch.softmax(qq @ k.double().permute(0, 2, 3, 1) * 0.3, -1)
            want = (p @ v.double().transpose(1, 2)).reshape(2, 1, 8, 128)
            assert (out.double() - want).abs().max() < 4e-3, (R, bits, gs)
