"""The reference of the online softmax: it moves only when a score exceeds it, and then leaves headroom above the score."""
import math

import pytest
import torch

from oracle import torch_oracle as T
from tests import helpers as H

pytestmark = pytest.mark.gpu


def _exact(q, k, v, S, bits, gs, scale):
    """One sequence in 64 bits over what the packed cache and the window hold."""
    z = T.quantize_kv(k[None, :S].float(), v[None, :S].float(), bits, gs, torch.float16)
    h_k = k.shape[1]
    kh = (z.k_codes.double().reshape(S // gs, gs, h_k, 128) * z.k_scale[0].double()[:, None] + z.k_zero[0].double()[:, None])
    vh = (z.v_codes.double().reshape(S, h_k, 128 // gs, gs) * z.v_scale[0].double()[..., None] + z.v_zero[0].double()[..., None])
    kh = torch.cat([kh.reshape(S, h_k, 128), k[S:].double()]).transpose(0, 1)
    vh = torch.cat([vh.reshape(S, h_k, 128), v[S:].double()]).transpose(0, 1)
    s = q.double().reshape(h_k, -1, 128) @ kh.transpose(1, 2) * scale
    return (torch.softmax(s, -1) @ vh).reshape(-1, 128), torch.logsumexp(s, -1).reshape(-1)


@pytest.mark.parametrize("rise", [0.0, 0.4, 1.9, 2.2, 30.0])
@pytest.mark.parametrize("bits,gs,scale", [(4, 128, 0.09), (4, 32, -0.09), (2, 128, 0.09), (2, 64, 3.0), (4, 64, 1e-30), (2, 32, -0.5)])
def test_scores_that_climb_from_step_to_step(device, bits, gs, scale, rise):
    """`rise` (in units of the exponent) from 64 tokens to the next, below and above the headroom of 3 * ln 2 = 2.08, up and
    (second kv head) down; one split, so that a wave sees several steps, a window behind them.  Tolerance: fp16
    probabilities (2^-11 of each, of outputs below 4) and the rounding of the output."""
    from bitladder_amd import fwd_kvcache_int, kvcache_pack_int
    S, R, h_k, g = 64 * 70, 37, 2, 4
    S = S // 128 * 128
    gen = torch.Generator(device=device).manual_seed(int(10 * rise) + bits + gs)
    q = torch.randn((1, 1, h_k * g, 128), generator=gen, device=device).half()
    k, v = (torch.randn((1, S + R, h_k, 128), generator=gen, device=device).half() for _ in range(2))
    # a common direction of q and k carries the climb: channel 7 of k is constant over each block of 64 tokens
    q[..., 7] = 1.0
    n = torch.arange(S + R, device=device) // 64
    step = rise / abs(scale) if abs(scale) > 1e-3 else rise
    climb = ((n - n.max() / 2) * step * (1 if scale >= 0 else -1)).clamp(-3e4, 3e4)
    k[0, :, 0, 7] = climb.half()
    k[0, :, 1, 7] = -climb.half()
    cache = H.alloc_cache(1, S, h_k, bits, gs, device)
    kvcache_pack_int(k[:, :S], cache[0], cache[1], v[:, :S], cache[2], cache[3], None, None, S, "k-channel", gs, bits)
    want, want_lse = _exact(q[0, 0], k[0], v[0], S, bits, gs, scale)
    for ns in (1, 0, 3):
        out, lse = fwd_kvcache_int(q, *cache, None, scale, "k-channel", gs, bits, k_residual=k[:, S:].contiguous(),
                                   v_residual=v[:, S:].contiguous(), num_splits=ns, return_lse=True)
        assert (out[0, 0].double() - want).abs().max() < 4e-3, ns
        # (a score of magnitude s carries the rounding of its fp32 sum, whose terms reach 1024 times a code's share)
        tol = 1e-3 + 2 ** -20 * abs(scale) * 3e4 * 16 * (abs(scale) > 1e-3)
        assert (lse[0].reshape(-1).double() - want_lse).abs().max() < tol, ns


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
