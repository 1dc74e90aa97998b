"""The drop-in calls whose argument blocks are found again by native code (csrc/hostpath.cpp): what counts as another call,
and what goes the long way round, with the same results."""
import ctypes
import math

import pytest
import torch

from oracle import bitdecode_oracle as O
from tests import helpers as H

pytestmark = pytest.mark.gpu

SCALE = 1.0 / math.sqrt(128)


def _setup(device, b=2, S=512):
    from bitladder_amd import kvcache_pack_int
    q, k, v = O.make_inputs(b, 8, 2, S, 64, seed=5)
    kd, vd = H.to_dev(k, "fp16", device), H.to_dev(v, "fp16", device)
    cache = H.alloc_cache(b, S, 2, 4, 128, device)
    kvcache_pack_int(kd[:, :S], cache[0], cache[1], vd[:, :S], cache[2], cache[3], None, None, S, "k-channel", 128, 4)
    return H.to_dev(q, "fp16", device), kd, vd, cache


def test_every_option_is_part_of_the_call(device):
    from bitladder_amd import fwd_kvcache_int, interface, plan_fwd_kvcache_int
    q, kd, vd, cache = _setup(device)
    kr, vr = kd[:, 512:].contiguous(), vd[:, 512:].contiguous()
    lens = torch.tensor([512, 128], dtype=torch.int32, device=device)
    args = (None, SCALE, "k-channel", 128, 4)
    interface._plan_cache().clear()
    variants = [dict(), dict(seqlen_k=256), dict(seqlens_k=lens), dict(seqlens_k=lens, max_seqlen_k=512),
                dict(k_residual=kr, v_residual=vr), dict(k_residual=kr, v_residual=vr, residual_len=7),
                dict(num_splits=2), dict(num_splits=1), dict(return_lse=True), dict(return_lse=False)]
    for _ in range(3):
        for kw in variants:
            plan = plan_fwd_kvcache_int(q, *cache, *args, **kw)
            got = fwd_kvcache_int(q, *cache, *args, **kw)
            plan.run()
            if kw.get("return_lse"):
                assert torch.equal(got[1], plan.lse)
                got = got[0]
            assert torch.equal(got, plan.out), kw
    assert len(interface._plan_cache()) == len(variants)
    assert not torch.equal(fwd_kvcache_int(q, *cache, None, SCALE, "k-channel", 128, 4),
                           fwd_kvcache_int(q, *cache, None, 2 * SCALE, "k-channel", 128, 4))
    with pytest.raises(ValueError):
        fwd_kvcache_int(q, *cache, None, SCALE, "k-channels", 128, 4)
    # a device error code raises as from the long way round: an entry whose block is made invalid
    key, entry = next(iter(interface._plan_cache().items()))
    bad = type(entry[0].args)()
    ctypes.memmove(ctypes.byref(bad), ctypes.byref(entry[0].args), ctypes.sizeof(bad))
    bad.num_splits = -1
    interface._plan_cache()[key] = (bad, ctypes.addressof(bad)) + entry[2:]
    with pytest.raises(interface._lib.BitDecodeError):
        fwd_kvcache_int(q, *cache, *args)
    interface._plan_cache().clear()


def test_other_kinds_of_argument_take_the_long_way(device):
    from bitladder_amd import fwd_kvcache_int, interface

    class Sub(torch.Tensor):
        pass

    q, kd, vd, cache = _setup(device)
    args = (None, SCALE, "k-channel", 128, 4)
    want = fwd_kvcache_int(q, *cache, *args)
    n = len(interface._plan_cache())
    assert torch.equal(fwd_kvcache_int(q.as_subclass(Sub), *cache, *args).as_subclass(torch.Tensor), want)
    assert len(interface._plan_cache()) == n
    p = torch.nn.Parameter(q)
    for _ in range(2):
        got = fwd_kvcache_int(p, *cache, *args)
        assert torch.equal(got, want) and not got.requires_grad


def test_pack_calls_found_again_and_captured(device):
    from bitladder_amd import kvcache_pack_int
    q, kd, vd, cache = _setup(device)
    other = H.alloc_cache(2, 512, 2, 4, 128, device)
    off = torch.tensor([0, 128], dtype=torch.int32, device=device)

    def pack(dst):
        kvcache_pack_int(kd[:, :384], dst[0], dst[1], vd[:, :384], dst[2], dst[3], None, None, 384, "k-channel", 128, 4,
                         dst_offsets=off)

    pack(other)
    other2 = H.alloc_cache(2, 512, 2, 4, 128, device)
    for t in other2:
        t.zero_()
    pack(other2)
    kd.mul_(0.5)          # new contents of the same tensors
    off.copy_(torch.tensor([128, 0], dtype=torch.int32))
    pack(other)
    fresh = H.alloc_cache(2, 512, 2, 4, 128, device)
    pack(fresh)
    # sequence 0: tokens 0-127 are from the first call, the rest from the second
    for a, b in zip(other, fresh):
        x = a.view(torch.int16).reshape(2, 2, 4, -1)
        y = b.view(torch.int16).reshape(2, 2, 4, -1)
        assert torch.equal(x[0, :, 1:], y[0, :, 1:]) and torch.equal(x[1, :, :3], y[1, :, :3])
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        pack(other2)
    for _ in range(3):
        for t in other2:
            t.zero_()
        g.replay()
        torch.cuda.synchronize()
        for a, b in zip(other2, fresh):
            x, y = (t.view(torch.int16).reshape(2, 2, 4, -1) for t in (a, b))
            assert torch.equal(x[0, :, 1:], y[0, :, 1:]) and torch.equal(x[1, :, :3], y[1, :, :3])
    with pytest.raises(RuntimeError):
        kvcache_pack_int(kd[:, :100], *other[:2], vd[:, :100], *other[2:], None, None, 100, "k-channel", 128, 4)


def test_numbers_given_as_tensors_are_read_with_every_call(device):
    """A number may be a tensor of one element; another value at the same address is another call."""
    import numpy as np
    from bitladder_amd import fwd_kvcache_int, fwd_kvcache_int_append, kvcache_pack_int
    q, kd, vd, cache = _setup(device)
    number, whole = np.zeros(1), np.zeros(1, dtype=np.int64)

    def given(x):      # a new tensor object over the same memory
        (whole if isinstance(x, int) else number)[0] = x
        return torch.from_numpy(whole if isinstance(x, int) else number).reshape(())

    for scale in (SCALE, 2 * SCALE):
        assert torch.equal(fwd_kvcache_int(q, *cache, None, given(scale), "k-channel", 128, 4),
                           fwd_kvcache_int(q, *cache, None, scale, "k-channel", 128, 4))
        assert torch.equal(fwd_kvcache_int(q.repeat(1, 3, 1, 1), *cache, None, given(scale), "k-channel", 128, 4),
                           fwd_kvcache_int(q.repeat(1, 3, 1, 1), *cache, None, scale, "k-channel", 128, 4))
    for n in (256, 512):
        assert torch.equal(fwd_kvcache_int(q, *cache, None, SCALE, "k-channel", 128, 4, seqlen_k=given(n)),
                           fwd_kvcache_int(q, *cache, None, SCALE, "k-channel", 128, 4, seqlen_k=n))
    got, want = H.alloc_cache(2, 512, 2, 4, 128, device), H.alloc_cache(2, 512, 2, 4, 128, device)
    for offset in (128, 256):
        for dst, x in ((got, given(offset)), (want, offset)):
            kvcache_pack_int(kd[:, :128], dst[0], dst[1], vd[:, :128], dst[2], dst[3], None, None, 0, "k-channel", 128, 4,
                             dst_offset=x)
    for a, b in zip(got, want):
        assert torch.equal(a.view(torch.int16), b.view(torch.int16))
    new = kd[:, :1].contiguous()
    window = torch.zeros((2, 128, 2, 128), dtype=torch.float16, device=device)
    for bound in (384, 512):
        outs = []
        for x in (given(bound), bound):
            lengths = torch.tensor([300, 130], dtype=torch.int32, device=device)
            outs.append(fwd_kvcache_int_append(q, new, new, *cache, window, window, lengths, x, None, SCALE, "k-channel",
                                               128, 4))
        assert torch.equal(*outs)


def test_numbers_of_other_libraries_are_found_again_by_value(device):
    import enum
    import numpy as np
    from bitladder_amd import fwd_kvcache_int, interface

    class Mode(str, enum.Enum):
        CHANNEL = "k-channel"

    q, kd, vd, cache = _setup(device)
    for kind in (np.float32, np.float16):
        interface._plan_cache().clear()
        for _ in range(3):
            for scale in (0.125, 0.25):
                got = fwd_kvcache_int(q, *cache, None, kind(scale), Mode.CHANNEL, np.int64(128), np.int32(4), seqlen_k=np.int64(256))
                assert torch.equal(got, fwd_kvcache_int(q, *cache, None, scale, "k-channel", 128, 4, seqlen_k=256))
        assert len(interface._plan_cache()) == 4      # two scales, each in two types
    with pytest.raises((TypeError, ValueError)):
        fwd_kvcache_int(q, *cache, None, 1j, "k-channel", 128, 4)
