"""BitKVCache's one-launch prefill and append against the same work done with the pack entry point and torch copies:
every byte a decode can read is the same, and so are the device's lengths."""
import pytest
import torch

pytestmark = pytest.mark.gpu

CASES = [  # bits, group, dtype, mode, kv heads, prompt lengths
    (4, 128, torch.float16, "k-channel", 2, [0, 1, 127, 128, 129, 300, 256, 383]),
    (4, 64, torch.bfloat16, "k-channel", 1, [255, 511, 20]),
    (4, 32, torch.float16, "k-tensor", 3, [127, 400]),
    (2, 128, torch.bfloat16, "k-channel", 8, [1000, 4096, 126]),      # 3 x 32 x 8 chunks packed: streamed
    (2, 64, torch.float16, "k-channel", 16, [4223 // 2, 127]),        # 2 x 16 x 16: the smallest streamed size
    (4, 128, torch.bfloat16, "k-channel", 15, [2100, 127]),           # just below it
    (2, 32, torch.float16, "k-channel", 1, [127 + (i % 3) for i in range(130)]),      # more sequences than one launch takes
]


def _pair(bits, gs, dtype, mode, h_k, b, capacity, device):
    from bitladder_amd import BitKVCache
    one, ref = (BitKVCache(b, h_k, capacity, num_bits=bits, group_size=gs, dtype=dtype, device=device, quant_mode=mode)
                for _ in range(2))
    ref._write = lambda *a: False      # the torch path
    return one, ref


def _live(cache):
    """What a decode can read: whole packed blocks of every sequence and the live rows of its window."""
    blocks, held = cache.capacity // 128, []
    packed = [t.view(torch.int16).reshape(cache.b, cache.h_k, blocks, -1)
              for t in (cache.k_pack, cache.k_params, cache.v_pack, cache.v_params)]
    for i, (p, r) in enumerate(zip(cache.packed_len, cache.res_len)):
        held += [t[i, :, :p // 128] for t in packed] + [cache.k_res[i, :r], cache.v_res[i, :r]]
    return held


def _same(one, ref):
    assert one.lengths == ref.lengths and one.packed_len == ref.packed_len
    assert one.total.tolist() == ref.total.tolist() == one.lengths
    for x, y in zip(_live(one), _live(ref)):
        assert torch.equal(x.contiguous().view(torch.int16), y.contiguous().view(torch.int16))
    assert one._published is not None
    packed, res = one._device_lengths()
    assert packed is one._published[0] and packed.tolist() == one.packed_len and res.tolist() == one.res_len


@pytest.mark.parametrize("bits,gs,dtype,mode,h_k,lengths", CASES)
def test_prefill_and_append_match_the_separate_calls(device, bits, gs, dtype, mode, h_k, lengths):
    g = torch.Generator(device=device).manual_seed(bits * 1000 + gs)
    b, n = len(lengths), max(lengths) + 5
    one, ref = _pair(bits, gs, dtype, mode, h_k, b, n + 8, device)
    # rows of a tensor laid out by heads, and a V with padding between tokens
    k = torch.randn((b, h_k, n, 128), generator=g, device=device).to(dtype).transpose(1, 2)
    v = torch.randn((b, n, h_k, 136), generator=g, device=device).to(dtype)[..., :128]
    for c in (one, ref):
        c.prefill(k, v, lengths)
    _same(one, ref)
    for step in range(4):
        kn = torch.randn((b, 1, h_k, 128), generator=g, device=device).to(dtype)
        vn = torch.randn((b, h_k, 128), generator=g, device=device).to(dtype)[:, None]
        for c in (one, ref):
            c.append(kn, vn) if step % 2 else c.append(kn[:, 0], vn[:, 0])
        _same(one, ref)
        q = torch.randn((b, 1, h_k, 128), generator=g, device=device).to(dtype)
        assert torch.equal(one.decode(q), ref.decode(q))
    # what the kernels do not take goes the old way, and the lengths on the device are not the old ones then
    kn = torch.randn((b, 1, h_k, 128), generator=g, device=device)
    for c in (one, ref):
        c.append(kn, kn)
    assert one._device_lengths()[1].tolist() == one.res_len
    for x, y in zip(_live(one), _live(ref)):
        assert torch.equal(x.contiguous().view(torch.int16), y.contiguous().view(torch.int16))
    q = torch.randn((b, 1, h_k, 128), generator=g, device=device).to(dtype)
    assert torch.equal(one.decode(q), ref.decode(q))


def test_prefill_of_whole_tensors_restarts_the_cache(device):
    from bitladder_amd import BitKVCache
    cache = BitKVCache(2, 2, 256, device=device)
    k = torch.randn((2, 200, 2, 128), device=device).half()
    cache.prefill(k, k)
    cache.prefill(k[:, :64], k[:, :64])
    assert cache.lengths == [64, 64] and cache.total.tolist() == [64, 64] and torch.equal(cache.k_res[:, :64], k[:, :64])
    with pytest.raises(ValueError):
        cache.prefill(torch.zeros((2, 300, 2, 128), device=device).half(), torch.zeros((2, 300, 2, 128), device=device).half())


def test_a_cache_per_layer_finds_its_decode_calls_again(device):
    """The device lengths of a cache keep their place from token to token, so a call is another one only when the bound of
    its packed length changes; on another stream they are other arrays."""
    from bitladder_amd import BitKVCache, interface
    layers, tokens = 6, 40
    k, q = torch.randn((2, 110, 2, 128), device=device).half(), torch.randn((2, 1, 4, 128), device=device).half()
    caches = [BitKVCache(2, 2, 256, device=device) for _ in range(layers)]
    interface._plan_cache().clear()
    for c in caches:
        c.prefill(k, k, [110, 30])
    for t in range(tokens):
        outs = []
        for c in caches:
            c.append(k[:, t:t + 1], k[:, t:t + 1])
            outs.append(c.decode(q))
            assert [x.tolist() for x in c._device_lengths()] == [c.packed_len, c.res_len]
        assert all(torch.equal(o, outs[0]) for o in outs)
    assert len(interface._plan_cache()) == 2 * layers      # below and from 128 tokens on
    first = caches[0]._device_lengths()[0]
    side = torch.cuda.Stream(device)
    side.wait_stream(torch.cuda.current_stream(device))
    with torch.cuda.stream(side):
        assert caches[0]._device_lengths()[0] is not first
        caches[0].append(k[:, :1], k[:, :1])
        assert caches[0]._device_lengths()[0] is not first
        got = caches[0].decode(q)
    side.synchronize()
    caches[1].append(k[:, :1], k[:, :1])
    assert first.tolist() == [128, 0] and torch.equal(got, caches[1].decode(q))


def test_a_copy_of_a_cache_keeps_its_own_lengths(device):
    """A shallow copy shares the tensors: the writes of one leave the other's decode at its own lengths."""
    import copy
    from bitladder_amd import BitKVCache
    k, q = torch.randn((2, 110, 2, 128), device=device).half(), torch.randn((2, 1, 4, 128), device=device).half()
    cache = BitKVCache(2, 2, 256, device=device)
    cache.prefill(k, k, [90, 30])
    before, fork = cache.decode(q), copy.copy(cache)
    for t in range(3):
        cache.append(k[:, t:t + 1], k[:, t:t + 1])
        assert torch.equal(fork.decode(q), before)
    after, deep = cache.decode(q), copy.deepcopy(cache)
    cache.append(k[:, :1], k[:, :1])
    assert torch.equal(deep.decode(q), after) and deep.lengths == [93, 33]


def test_caches_that_the_kernels_do_not_take_are_written_by_torch_operations(device):
    """More sequences than the kernels' limit, no capacity, and formats without a decode, whose windows can be filled."""
    from bitladder_amd import BitKVCache
    many = BitKVCache(70000, 1, 128, device=device)
    k = torch.randn((70000, 1, 1, 128), device=device).half()
    many.append(k, k)
    assert many.lengths == [1] * 70000 and torch.equal(many.k_res[:, :1], k)
    # (one key: the output is its value, rounded once more)
    assert (many.decode(k).float() - k.float()).abs().max() < 2 ** -9
    empty = BitKVCache(2, 1, 0, device=device)
    empty.prefill(k[:2], k[:2], [0, 0])
    assert empty.lengths == [0, 0] and not empty.decode(k[:2]).any()
    with pytest.raises(ValueError):
        empty.append(k[:2], k[:2])
    for options in (dict(dtype=torch.float32), dict(num_bits=8), dict(group_size=16)):
        c = BitKVCache(2, 1, 128, device=device, **options)
        x = k[:2].to(c.dtype)
        c.prefill(x, x)
        c.append(x, x)
        assert c.lengths == [2, 2] == c.total.tolist() and torch.equal(c.k_res[:, 1:2], x)
