"""The pack kernel's workgroup per chunk and its two workgroups per chunk (one each for K and V) give the same bytes: a call
of n chunks against the same chunks packed one call at a time, at the sizes where the choice changes."""
import pytest
import torch

from tests import helpers as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bits,gs,dtype,mode", [(4, 128, torch.float16, "k-channel"), (4, 64, torch.bfloat16, "k-tensor"),
                                                (2, 32, torch.float16, "k-channel"), (2, 128, torch.bfloat16, "k-channel")])
@pytest.mark.parametrize("chunks,h_k", [(1, 1), (73, 7), (64, 8), (767, 1), (96, 8)])
def test_chunks_packed_together_and_one_by_one(device, bits, gs, dtype, mode, chunks, h_k):
    from bitladder_amd import kvcache_pack_int
    g = torch.Generator(device=device).manual_seed(chunks)
    n = 128 * chunks
    k, v = (torch.randn((1, n, h_k, 128), generator=g, device=device).to(dtype) for _ in range(2))
    pn = 16 // bits
    params = (1, 128 // gs, h_k, n)
    make = lambda: [torch.zeros((1, n // pn, h_k, 128), dtype=torch.uint16, device=device),
                    torch.zeros(params if mode == "k-tensor" else (1, n // gs, h_k, 128), dtype=torch.float32, device=device),
                    torch.zeros((1, n, h_k, 128 // pn), dtype=torch.uint16, device=device),
                    torch.zeros(params, dtype=torch.float32, device=device)]
    whole, parts = make(), make()
    kvcache_pack_int(k, whole[0], whole[1], v, whole[2], whole[3], None, None, n, mode, gs, bits)
    step = max(1, chunks // 8)      # at most 96 chunks a call
    for c in range(0, chunks, step):
        t = slice(128 * c, 128 * min(chunks, c + step))
        kvcache_pack_int(k[:, t], parts[0], parts[1], v[:, t], parts[2], parts[3], None, None, 0, mode, gs, bits,
                         dst_offset=128 * c)
    for a, b in zip(whole, parts):
        assert torch.equal(a.view(torch.int16), b.view(torch.int16))
    if chunks == 1:      # both forms agree with each other above; the small one with the oracle here
        from oracle import bitdecode_oracle as O
        if mode == "k-channel":
            H.assert_cache_equals_oracle(H.cache_to_numpy(*whole), O.quantize_kv_ref(
                k.float().cpu().numpy(), v.float().cpu().numpy(), bits, gs, "bf16" if dtype == torch.bfloat16 else "fp16"))
