"""Launches that are split although every compute unit has a workgroup without it keep the accuracy of one split."""
import math

import pytest
import torch

from oracle import torch_oracle as T
from tests import helpers as H

pytestmark = pytest.mark.gpu

SCALE = 1.0 / math.sqrt(128)


def _setup(device, b, h_k, S, R, gs, seed):
    from bitladder_amd import kvcache_pack_int
    g = torch.Generator(device=device).manual_seed(seed)
    q = torch.randn((b, 1, 2 * h_k, 128), generator=g, device=device).half()
    k, v = (torch.randn((b, S + R, h_k, 128), generator=g, device=device).half() for _ in range(2))
    k[..., [5, 40, 99]] *= 10      # outlier channels: few keys carry the softmax, and outputs are as large as values
    cache = H.alloc_cache(b, S, h_k, 4, gs, device)
    kvcache_pack_int(k[:, :S], cache[0], cache[1], v[:, :S], cache[2], cache[3], None, None, S, "k-channel", gs, 4)
    return q, k, v, cache


def _exact(q, k, v, S, gs, i):
    """Sequence i in 64 bits over what the packed cache holds: the quantizer's codes, scales and zeros."""
    z = T.quantize_kv(k[i:i + 1, :S].float(), v[i:i + 1, :S].float(), 4, gs, torch.float16)
    h_k = k.shape[2]
    kh = (z.k_codes.double().reshape(S // gs, gs, h_k, 128) * z.k_scale[0].double()[:, None] + z.k_zero[0].double()[:, None])
    vh = (z.v_codes.double().reshape(S, h_k, 128 // gs, gs) * z.v_scale[0].double()[..., None] + z.v_zero[0].double()[..., None])
    kh = torch.cat([kh.reshape(S, h_k, 128), k[i, S:].double()]).transpose(0, 1)
    vh = torch.cat([vh.reshape(S, h_k, 128), v[i, S:].double()]).transpose(0, 1)
    qq = q[i, 0].double().reshape(h_k, -1, 128)
    return torch.stack([torch.softmax(qq[j] @ kh[j].t() * SCALE, -1) @ vh[j] for j in range(h_k)]).reshape(-1, 128)


@pytest.mark.parametrize("b,S,gs", [(33, 4096, 128), (48, 4096, 128), (33, 8192, 32), (48, 8192, 64)])
def test_more_pairs_than_compute_units_lose_no_precision_to_the_split(device, b, S, gs):
    """264 and 384 pairs: the error of two and three splits against 64 bits is that of one split or less."""
    from bitladder_amd import fwd_kvcache_int
    q, k, v, cache = _setup(device, b, 8, S, 64, gs, b)
    seqs = (0, b // 2, b - 1)
    ref = torch.stack([_exact(q, k, v, S, gs, i) for i in seqs])
    err = []
    for ns in (1, 0, 2, 3):
        out = fwd_kvcache_int(q, *cache, None, SCALE, "k-channel", gs, 4, k_residual=k[:, S:].contiguous(),
                              v_residual=v[:, S:].contiguous(), num_splits=ns)[list(seqs), 0].double()
        err.append(float((out - ref).norm() / ref.norm()))
    assert max(err) == err[0], err


def test_records_of_splits_without_keys_beside_ones_with_residual_words(device):
    """Splits that have no keys (short and empty sequences) send no residual words; launch after launch on one workspace,
    with other queries and lengths in turn, equals a workspace of its own."""
    from bitladder_amd import fwd_kvcache_int, plan_fwd_kvcache_int
    b, h_k, S = 65, 8, 1024
    q, k, v, cache = _setup(device, b, h_k, S, 0, 128, 5)
    lens = [torch.tensor([128 * ((5 * i + 3 * j) % 9) for i in range(b)], dtype=torch.int32, device=device) for j in range(3)]
    args = (*cache, None, SCALE, "k-channel", 128, 4)
    for step in range(7):
        qs, ls = q.roll(step, 0).contiguous(), lens[step % 3]
        got = fwd_kvcache_int(qs, *args, seqlens_k=ls, max_seqlen_k=S, num_splits=7)
        plan = plan_fwd_kvcache_int(qs, *args, seqlens_k=ls, max_seqlen_k=S, num_splits=7)
        assert torch.equal(got, plan.run()), step
        one = fwd_kvcache_int(qs, *args, seqlens_k=ls, max_seqlen_k=S, num_splits=1)
        # (one rounding of the output to fp16 each, and the order of the sums)
        assert (got.float() - one.float()).abs().max() < 2e-3, step
        assert not got[ls == 0].any()


def test_residual_words_in_the_step_and_with_several_rows(device):
    from bitladder_amd import BitKVCache, fwd_kvcache_int
    b, h_k, S = 33, 8, 512
    q, k, v, cache = _setup(device, b, h_k, S, 8, 128, 6)
    lens = torch.tensor([128 * (i % 5) for i in range(b)], dtype=torch.int32, device=device)
    rows = torch.cat([q, q.roll(1, 0), q.roll(2, 0)], 1)
    args = (*cache, None, SCALE, "k-channel", 128, 4)
    for _ in range(3):
        got = fwd_kvcache_int(rows, *args, seqlens_k=lens, max_seqlen_k=S, num_splits=5)
        for r in range(3):
            one = fwd_kvcache_int(rows[:, r:r + 1].contiguous(), *args, seqlens_k=lens, max_seqlen_k=S, num_splits=1)
            assert (got[:, r:r + 1].float() - one.float()).abs().max() < 2e-3
    caches = [BitKVCache(b, h_k, 640, device=device) for _ in range(2)]
    for c in caches:
        c.prefill(k[:, :500], v[:, :500], [(41 * i) % 450 for i in range(b)])
    for t in range(6):
        new = (k[:, 500 + t:501 + t], v[:, 500 + t:501 + t])
        many, one = (c.step(q, *new, SCALE, num_splits=ns) for c, ns in zip(caches, (5, 1)))
        assert (many.float() - one.float()).abs().max() < 2e-3
        assert torch.equal(caches[0].k_res, caches[1].k_res) and torch.equal(caches[0].total, caches[1].total)


@pytest.mark.parametrize("b,S,gs", [(18, 4096, 128), (17, 8192, 64)])
def test_several_rows_lose_no_precision_to_the_split(device, b, S, gs):
    """Sixteen (row, head) pairs of each of 144 or 136 (sequence, kv head) pairs: more blocks of eight than compute units, fewer of
    sixteen.  The error of the library's own split count is that of one split or less, as with one row."""
    from bitladder_amd import fwd_kvcache_int
    from tests.test_gpu_rows import _blocks
    q, k, v, cache = _setup(device, b, 8, S, 64, gs, b)
    assert {_blocks(b, 8, 16, S, 64, 4, gs, False, S, ns) for ns in (0, 1, 2, 3)} == {1}      # of sixteen
    rows = torch.cat([q.roll(j, 0) for j in range(8)], 1)
    seqs = (0, b // 2, b - 1)
    ref = torch.stack([torch.stack([_exact(rows[:, j:j + 1], k, v, S, gs, i) for j in range(8)]) for i in seqs])
    err = []
    for ns in (1, 0, 2, 3):
        out = fwd_kvcache_int(rows, *cache, None, SCALE, "k-channel", gs, 4, k_residual=k[:, S:].contiguous(),
                              v_residual=v[:, S:].contiguous(), num_splits=ns)[list(seqs)].double()
        err.append(float((out - ref).norm() / ref.norm()))
    assert max(err) == err[0], err
