"""Several query rows per sequence in one launch: the (row, head) pairs of a kv head run in blocks of eight or sixteen."""
import math

import pytest
import torch

from oracle import bitdecode_oracle as O
from tests import helpers as H

pytestmark = pytest.mark.gpu

SCALE = 1.0 / math.sqrt(128)


def _blocks(b, h_k, pairs, max_s, max_r, bits, gs, ragged, capacity, ns):
    """Blocks of row and head pairs per kv head that a call runs in."""
    import ctypes

    from bitladder_amd import _lib
    n = ctypes.c_int32()
    _lib.lib().bitdecode_rows_splits(b, h_k, pairs, max_s, max_r, 256, bits, gs, ragged, capacity, ns, ctypes.byref(n))
    return n.value


@pytest.mark.parametrize("h,h_k,m,bits,gs,mode,dtype,ns,paged", [
    (6, 2, 5, 4, 128, "k-channel", "fp16", 3, False),      # 15 pairs: a row is cut by the block boundary, last block of 7
    (3, 3, 9, 2, 64, "k-channel", "fp16", 2, False),       # 9 pairs: last block of 1
    (16, 2, 2, 4, 32, "k-channel", "bf16", 1, True),       # 16 pairs, one block per row, one split
    (8, 1, 3, 4, 64, "k-tensor", "fp16", 4, False),
    (7, 1, 300, 2, 128, "k-channel", "fp16", 0, True),     # many blocks, more workgroups than compute units
])
def test_rows_equal_the_calls_for_each_row(device, h, h_k, m, bits, gs, mode, dtype, ns, paged):
    """Every row of one launch equals a call with that row alone: both take the same scores and differ by the split
    count at most, so by the rounding of the fp16 records and of the output (2^-11 of |out| < 2 each: 1e-3, and a bf16
    output by its rounding, 2^-8 of |out|)."""
    from bitladder_amd import fwd_kvcache_int, kvcache_pack_int
    b, S, R = 3, 128 * 10, 53
    _, k, v = O.make_inputs(b, h, h_k, S, R, seed=m, dtype=dtype)
    tdt = H.torch_dtype(dtype)
    kd, vd = H.to_dev(k, dtype, device), H.to_dev(v, dtype, device)
    g = torch.Generator(device=device).manual_seed(m)
    wide = torch.randn((b, h, m, 128), generator=g, device=device).to(tdt)
    q = wide.transpose(1, 2)                                # rows are not the slowest index in memory
    table = None
    if paged:
        table = torch.randperm(b * S // 256, generator=g, device=device).to(torch.int32).reshape(b, -1)
        cache = H.alloc_cache(b * S // 256, 256, h_k, bits, gs, device, k_tensor=mode == "k-tensor")
    else:
        cache = H.alloc_cache(b, S, h_k, bits, gs, device, k_tensor=mode == "k-tensor")
    kvcache_pack_int(kd[:, :S], cache[0], cache[1], vd[:, :S], cache[2], cache[3], table, None, S, mode, gs, bits)
    lens = torch.tensor([S, 128 * 3, 0], dtype=torch.int32, device=device)
    res = torch.tensor([R, 1, 17], dtype=torch.int32, device=device)
    kw = dict(seqlens_k=lens, k_residual=kd[:, S:], v_residual=vd[:, S:], residual_len=res, return_lse=True)
    args = (*cache, table, SCALE, mode, gs, bits)
    given = torch.full((b, m, h, 128), float("nan"), dtype=tdt, device=device)
    for _ in range(2):                                      # the second launch finds the workspace as the first left it
        out, lse = fwd_kvcache_int(q, *args, num_splits=ns, out=given, **kw)
    assert out is given and lse.shape == (b, m, h)
    for r in sorted({0, 1, m // 2, m - 1}):
        one, lse1 = fwd_kvcache_int(q[:, r:r + 1].contiguous(), *args, num_splits=ns, **kw)
        err = (out[:, r:r + 1].float() - one.float()).abs()
        assert (err <= 1e-3 + (2 ** -8 * one.float().abs() if dtype == "bf16" else 0)).all(), (r, err.max().item())
        assert (lse[:, r] - lse1).abs().max().item() < 1e-4, r


@pytest.mark.parametrize("m,h,num_splits", [(4100, 1, 0), (1030, 4, 512)])
def test_more_rows_than_one_launch_takes(device, m, h, num_splits):
    """More rows than a launch accepts, and more records than its workspace may hold: several launches, the same rows."""
    from bitladder_amd import fwd_kvcache_int, kvcache_pack_int
    g = torch.Generator(device=device).manual_seed(m)
    k, v = (torch.randn((1, 256, 1, 128), generator=g, device=device).half() for _ in range(2))
    cache = H.alloc_cache(1, 256, 1, 4, 128, device)
    kvcache_pack_int(k, cache[0], cache[1], v, cache[2], cache[3], None, None, 256, "k-channel", 128, 4)
    q = torch.randn((1, m, h, 128), generator=g, device=device).half()
    out, lse = fwd_kvcache_int(q, *cache, None, 0.09, "k-channel", 128, 4, num_splits=num_splits, return_lse=True)
    assert out.shape == q.shape and lse.shape == (1, m, h)
    for r0 in (0, m // 2, m - 8):
        want, wlse = fwd_kvcache_int(q[:, r0:r0 + 8].contiguous(), *cache, None, 0.09, "k-channel", 128, 4,
                                     num_splits=min(num_splits, 2), return_lse=True)
        # (other split counts round the partial outputs differently: one fp16 rounding of a mean of unit normals)
        assert (out[:, r0:r0 + 8].float() - want.float()).abs().max() < 2e-3
        assert (lse[:, r0:r0 + 8] - wlse).abs().max() < 1e-4


def test_rows_of_any_stride_and_alignment(device):
    """q as the reference's own reshape takes it: whatever the strides, also those of dimensions of one."""
    from bitladder_amd import fwd_kvcache_int, kvcache_pack_int
    g = torch.Generator(device=device).manual_seed(3)
    k, v = (torch.randn((1, 256, 2, 128), generator=g, device=device).half() for _ in range(2))
    cache = H.alloc_cache(1, 256, 2, 4, 128, device)
    kvcache_pack_int(k, cache[0], cache[1], v, cache[2], cache[3], None, None, 256, "k-channel", 128, 4)
    args = (*cache, None, SCALE, "k-channel", 128, 4)
    want = None
    data = torch.randn((1, 3, 4, 128), generator=g, device=device).half()
    flat = torch.zeros(8192, dtype=torch.float16, device=device)
    for offset, strides in ((0, (1536, 512, 128, 1)), (0, (1541, 512, 128, 1)), (1, (1536, 512, 128, 1)),
                            (0, (1536, 516, 129, 1)), (0, (1536, 1024, 256, 2)), (0, (1536, 128, 384, 1))):
        q = flat.as_strided(data.shape, strides, offset)
        q.copy_(data)
        out = fwd_kvcache_int(q, *args)
        want = out if want is None else want
        assert torch.equal(out, want), (offset, strides)
        held = torch.full((8192,), 7.0, dtype=torch.float16, device=device)
        given = held.as_strided(data.shape, strides, offset)
        assert fwd_kvcache_int(q, *args, out=given) is given and torch.equal(given, want)
        given.fill_(7.0)
        assert (held == 7.0).all()


def test_many_sequences_take_their_rows_in_one_launch(device):
    """Eight rows of 4096 sequences of 8 heads: one launch reads the cache once."""
    from bitladder_amd import fwd_kvcache_int, interface, kvcache_pack_int
    b, h = 4096, 8
    g = torch.Generator(device=device).manual_seed(8)
    k, v = (torch.randn((b, 128, h, 128), generator=g, device=device).half() for _ in range(2))
    cache = H.alloc_cache(b, 128, h, 4, 128, device)
    kvcache_pack_int(k, cache[0], cache[1], v, cache[2], cache[3], None, None, 128, "k-channel", 128, 4)
    q = torch.randn((b, 8, h, 128), generator=g, device=device).half()
    interface._plan_cache().clear()
    out = fwd_kvcache_int(q, *cache, None, SCALE, "k-channel", 128, 4)
    assert len(interface._plan_cache()) == 1
    for r in (0, 5, 7):
        assert torch.equal(out[:, r:r + 1], fwd_kvcache_int(q[:, r:r + 1].contiguous(), *cache, None, SCALE, "k-channel", 128, 4))


@pytest.mark.parametrize("b,h,h_k,m,S,bits,gs,mode,dtype,ns", [
    (8, 6, 2, 3, 128 * 130, 4, 128, "k-channel", "fp16", 5),      # 9 pairs: a block of sixteen with seven empty columns
    (7, 8, 1, 4, 128 * 260, 2, 64, "k-channel", "bf16", 33),      # 32 pairs, more splits than a round of the merge takes
    (9, 5, 5, 17, 128 * 36, 4, 32, "k-channel", "bf16", 1),       # 17 pairs: last block of one, one split
    (16, 8, 2, 5, 128 * 65, 4, 64, "k-tensor", "fp16", 0),        # 20 pairs
    (24, 16, 2, 4, 128 * 33, 2, 128, "k-channel", "fp16", 17),
    (24, 16, 2, 2, 128 * 50, 2, 32, "k-channel", "fp16", 2),
])
def test_blocks_of_sixteen_equal_the_calls_for_each_row(device, b, h, h_k, m, S, bits, gs, mode, dtype, ns):
    """As above, at sizes that run in blocks of sixteen: unequal lengths, windows, an empty sequence, outputs large enough for
    the residual words in one sequence.  The LSE bound is that of the scores' fp32 sums, the output's the rounding of two
    records and an output (2^-11 each of the sequence's values)."""
    from bitladder_amd import _lib, fwd_kvcache_int, kvcache_pack_int
    assert _lib.lib().bitdecode_row_blocks(b, h_k, m * (h // h_k), S, 256, bits) == -(-m * (h // h_k) // 16)
    R, tdt = 53, H.torch_dtype(dtype)
    g = torch.Generator(device=device).manual_seed(m)
    k, v = (torch.randn((b, S + R, h_k, 128), generator=g, device=device).to(tdt) for _ in range(2))
    k[..., [5, 40, 99]] *= 6
    v[1] *= 40                                              # residual words
    q = torch.randn((b, h, m, 128), generator=g, device=device).to(tdt).transpose(1, 2)
    cache = H.alloc_cache(b, S, h_k, bits, gs, device, k_tensor=mode == "k-tensor")
    kvcache_pack_int(k[:, :S], cache[0], cache[1], v[:, :S], cache[2], cache[3], None, None, S, mode, gs, bits)
    lens = torch.full((b,), S, dtype=torch.int32, device=device)
    res = torch.full((b,), R, dtype=torch.int32, device=device)
    lens[2], lens[3], res[3], res[4] = 384, 0, 0, 1
    kw = dict(seqlens_k=lens, k_residual=k[:, S:], v_residual=v[:, S:], residual_len=res, return_lse=True)
    args = (*cache, None, SCALE, mode, gs, bits)
    for flip in (1, -1, 1):                                 # launch after launch on one workspace, other queries in between
        out, lse = fwd_kvcache_int(q * flip, *args, num_splits=ns, **kw)
    assert torch.isinf(lse[3]).all() and not out[3].any()
    scale_of = v.float().abs().amax((1, 2, 3)).reshape(b, 1, 1, 1) / 4
    for r in sorted({0, 1, m // 2, m - 1}):
        one, lse1 = fwd_kvcache_int(q[:, r:r + 1].contiguous(), *args, num_splits=min(ns, 4), **kw)
        err = (out[:, r:r + 1].float() - one.float()).abs()
        bound = 1.5e-3 * scale_of + (2 ** -7 * one.float().abs() if dtype == "bf16" else 0)
        assert (err <= bound).all(), (r, (err - bound).max().item())
        ok = lens + res > 0
        assert (lse[ok, r] - lse1[ok]).abs().max().item() < 5e-4, r


def test_few_rows_stay_in_blocks_of_eight(device):
    """Where eight pairs a workgroup are the faster choice the row blocks say so, whatever the sizes."""
    from bitladder_amd import _lib
    blocks = lambda *a: _lib.lib().bitdecode_row_blocks(*a)
    assert [blocks(2, 8, p, 8192, 256, 4) for p in (1, 8, 9, 32)] == [1, 1, 2, 2]
    assert blocks(1, 8, 32, 4096, 256, 4) == 4 and blocks(3, 8, 32, 4096, 256, 2) == 4 and blocks(4, 8, 64, 2048, 256, 2) == 4
    assert blocks(1, 1, 64, 65536, 256, 4) == 8 and blocks(1, 1, 64, 131072, 256, 4) == 4 and blocks(1, 1, 64, 131072, 256, 2) == 8


def test_count_left_to_the_library_fits_a_workspace_sized_for_blocks_of_eight(device):
    """The C entry with num_splits = 0: a workspace for the count of blocks of eight is taken, a smaller one refused."""
    import ctypes

    from bitladder_amd import _lib, fwd_kvcache_int, interface, kvcache_pack_int
    g = torch.Generator(device=device).manual_seed(4)
    k, v = (torch.randn((2, 8192, 8, 128), generator=g, device=device).half() for _ in range(2))
    cache = H.alloc_cache(2, 8192, 8, 4, 128, device)
    kvcache_pack_int(k, cache[0], cache[1], v, cache[2], cache[3], None, None, 8192, "k-channel", 128, 4)
    q = torch.randn((2, 8, 32, 128), generator=g, device=device).half()
    want = fwd_kvcache_int(q, *cache, None, SCALE, "k-channel", 128, 4)
    plan = interface.plan_fwd_kvcache_int(q, *cache, None, SCALE, "k-channel", 128, 4, _rows=True)
    L, a = _lib.lib(), plan.args
    n8 = L.bitdecode_num_splits_for(2, 8 * 4, 8192, 0, 0, 4, 128, 0)
    assert plan.args.fwd.num_splits > n8 > 1
    stream = torch.cuda.current_stream().cuda_stream
    for splits, ok in ((n8, True), (n8 + 1, True), (n8 - 1, False)):
        nbytes = L.bitdecode_fwd_workspace_bytes(2, 8 * 32, splits)
        ws = torch.zeros(nbytes, dtype=torch.uint8, device=device)
        a.fwd.num_splits, a.fwd.workspace, a.fwd.workspace_bytes = 0, ws.data_ptr(), nbytes
        plan.out.zero_()
        assert (L.bitdecode_fwd_rows(ctypes.byref(a), stream) == 0) is ok
        torch.cuda.synchronize()
        if ok:      # (another split count: the rounding of the records)
            assert (plan.out.float() - want.float()).abs().max() < 1e-3


@pytest.mark.parametrize("bits,gs,mode,dtype,ns", [(4, 128, "k-channel", "fp16", 5), (2, 64, "k-channel", "bf16", 9),
                                                   (4, 64, "k-tensor", "fp16", 17)])
def test_splits_without_work_have_some_in_the_next_launch(device, bits, gs, mode, dtype, ns):
    """One workspace, lengths and windows that change from launch to launch: splits of a short or empty sequence have neither a unit nor a
    tile, the same splits have both one launch later.  Bounds as for `test_blocks_of_sixteen_equal_the_calls_for_each_row`."""
    from bitladder_amd import fwd_kvcache_int, kvcache_pack_int
    from bitladder_amd.interface import plan_fwd_kvcache_int
    b, h, h_k, m, S, R, tdt = 8, 16, 2, 6, 128 * 130, 128, H.torch_dtype(dtype)
    assert _blocks(b, h_k, m * (h // h_k), S, R, bits, gs, True, S + 128, ns) == 3      # of sixteen
    g = torch.Generator(device=device).manual_seed(ns)
    k, v = (torch.randn((b, S + R, h_k, 128), generator=g, device=device).to(tdt) for _ in range(2))
    q = torch.randn((b, m, h, 128), generator=g, device=device).to(tdt)
    cache = H.alloc_cache(b, S + 128, h_k, bits, gs, device, k_tensor=mode == "k-tensor")
    kvcache_pack_int(k[:, :S], cache[0], cache[1], v[:, :S], cache[2], cache[3], None, None, S, mode, gs, bits)
    lens, res = (torch.zeros(b, dtype=torch.int32, device=device) for _ in range(2))
    args = (q, *cache, None, SCALE, mode, gs, bits)
    kw = dict(seqlens_k=lens, max_seqlen_k=S, k_residual=k[:, S:], v_residual=v[:, S:], residual_len=res, return_lse=True)
    plan = plan_fwd_kvcache_int(*args, num_splits=ns, _rows=True, **kw)
    launches = [([0, 128, 256, S, 0, 128, 512, S - 128], [0, 0, 1, 0, 17, 128, 0, 3]),
                ([S, S, S - 256, 0, 256, 0, 128, 128], [1, 0, 0, 0, 0, 16, 1, 0]),
                ([128, 0, 0, 384, S, S, 0, 0], [0, 128, 0, 33, 0, 0, 0, 1])]
    for _ in range(2):
        for n_s, n_r in launches:
            lens.copy_(torch.tensor(n_s, dtype=torch.int32))
            res.copy_(torch.tensor(n_r, dtype=torch.int32))
            out = plan.run()
            for r in (0, m - 1):
                one, lse1 = fwd_kvcache_int(q[:, r:r + 1].contiguous(), *args[1:], num_splits=1, **kw)
                err = (out[:, r:r + 1].float() - one.float()).abs()
                assert (err <= 1.5e-3 + (2 ** -7 * one.float().abs() if dtype == "bf16" else 0)).all(), (n_s, r, err.max().item())
                some = lens + res > 0
                assert torch.isinf(plan.lse[~some]).all() and not out[~some].any()
                assert (plan.lse[some, r] - lse1[some]).abs().max().item() < 5e-4


@pytest.mark.parametrize("b,h,m,S", [(10, 32, 8, 8192), (32, 8, 16, 2048)])
@pytest.mark.parametrize("bits,gs", [(4, 128), (4, 32), (2, 128), (2, 64)])
@pytest.mark.parametrize("size,deviation", [(1.0, 1.0), (1.0, 3.0), (0.003, 3.0)])
def test_blocks_of_sixteen_are_as_accurate_as_calls_for_each_row(device, bits, gs, size, deviation, b, h, m, S):
    """Error against 64 bits over one split, many fp32 additions per sum: no more than calls with one row have, whose
    hi and lo parts are summed apart by 16 (2 bits; 12 at group 64) or 8 waves; 10 % for the order of the sums, over 32K outputs and more."""
    from bitladder_amd import fwd_kvcache_int, kvcache_pack_int
    from oracle import torch_oracle as T
    h_k, n = 8, 2
    assert _blocks(b, h_k, m * (h // h_k), S, 0, bits, gs, False, S, 1) == m * (h // h_k) // 16      # of sixteen
    g = torch.Generator(device=device).manual_seed(bits + gs)
    q = torch.randn((b, m, h, 128), generator=g, device=device).half()
    k, v = (torch.randn((b, S, h_k, 128), generator=g, device=device) for _ in range(2))
    k, v = k.half(), (v * size).half()
    cache = H.alloc_cache(b, S, h_k, bits, gs, device)
    kvcache_pack_int(k, cache[0], cache[1], v, cache[2], cache[3], None, None, S, "k-channel", gs, bits)
    z = T.quantize_kv(k[:n].float(), v[:n].float(), bits, gs, torch.float16)      # (of the first n sequences)
    kh = (z.k_codes.double().reshape(n, S // gs, gs, h_k, 128) * z.k_scale.double()[:, :, None] + z.k_zero.double()[:, :, None])
    vh = (z.v_codes.double().reshape(n, S, h_k, 128 // gs, gs) * z.v_scale.double()[..., None] + z.v_zero.double()[..., None])
    kh, vh = (t.reshape(n, S, h_k, 128).transpose(1, 2).contiguous() for t in (kh, vh))
    scale = deviation * SCALE
    qq = q[:n].double().reshape(n, m, h_k, h // h_k, 128).permute(0, 2, 1, 3, 4).reshape(n, h_k, -1, 128)
    ref = torch.softmax(qq @ kh.transpose(2, 3).contiguous() * scale, -1) @ vh
    ref = ref.reshape(n, h_k, m, h // h_k, 128).transpose(1, 2).reshape(n, m, h, 128)
    args = (*cache, None, scale, "k-channel", gs, bits)
    ones = torch.cat([fwd_kvcache_int(q[:, r:r + 1].contiguous(), *args, num_splits=1) for r in range(m)], 1)
    err, one = ((t[:n].double() - ref).norm().item() for t in (fwd_kvcache_int(q, *args, num_splits=1), ones))
    assert err < 1.1 * one, (err / ref.norm().item(), one / ref.norm().item())


@pytest.mark.parametrize("b,h,h_k,m,S,bits,gs,mode,dtype,ns", [
    (8, 6, 2, 3, 128 * 130, 4, 128, "k-channel", "fp16", 9),      # 9 pairs: a block of sixteen with seven empty columns
    (7, 8, 1, 4, 128 * 260, 2, 64, "k-channel", "bf16", 33),      # more splits than a round of the merge takes
    (16, 5, 5, 32, 128 * 16, 4, 32, "k-channel", "bf16", 1),      # one split
    (16, 8, 2, 5, 128 * 64, 4, 64, "k-tensor", "fp16", 0),        # 20 pairs
    (24, 16, 2, 4, 128 * 72, 2, 128, "k-channel", "fp16", 17),
    (70, 16, 2, 2, 128 * 50, 2, 32, "k-channel", "fp16", 1),      # more sequences than are dealt out by length
    (9, 16, 2, 7, 128 * 64, 2, 128, "k-channel", "fp16", 0),      # 56 pairs: a last block of eight
])
def test_blocks_of_sixteen_with_unequal_lengths(device, b, h, h_k, m, S, bits, gs, mode, dtype, ns):
    """Calls that do run in blocks of sixteen, each row against a call of its own; bounds as for `test_blocks_of_sixteen_equal_the_calls_for_each_row`."""
    from bitladder_amd import fwd_kvcache_int, kvcache_pack_int
    R, tdt, pairs = 53, H.torch_dtype(dtype), m * (h // h_k)
    assert _blocks(b, h_k, pairs, S, R, bits, gs, True, S + 128, ns) == -(-pairs // 16) < -(-pairs // 8)
    g = torch.Generator(device=device).manual_seed(m)
    k, v = (torch.randn((b, S + R, h_k, 128), generator=g, device=device, dtype=tdt) for _ in range(2))
    k[..., [5, 40, 99]] *= 6
    v[1] *= 40                                              # residual words
    q = torch.randn((b, h, m, 128), generator=g, device=device).to(tdt).transpose(1, 2)
    cache = H.alloc_cache(b, S + 128, h_k, bits, gs, device, k_tensor=mode == "k-tensor")
    kvcache_pack_int(k[:, :S], cache[0], cache[1], v[:, :S], cache[2], cache[3], None, None, S, mode, gs, bits)
    lens = torch.tensor([S - 128 * ((5 * i) % 9) for i in range(b)], dtype=torch.int32, device=device)
    res = torch.full((b,), R, dtype=torch.int32, device=device)
    lens[2], lens[3], res[3], res[4] = 384, 0, 0, 1
    args = (*cache, None, SCALE, mode, gs, bits)
    kw = dict(seqlens_k=lens, max_seqlen_k=S, k_residual=k[:, S:], v_residual=v[:, S:], residual_len=res, return_lse=True)
    for flip in (1, -1, 1):                                 # launch after launch on one workspace, other queries in between
        out, lse = fwd_kvcache_int(q * flip, *args, num_splits=ns, **kw)
    assert torch.isinf(lse[3]).all() and not out[3].any()
    scale_of = v[:8].float().abs().amax((1, 2, 3)).reshape(-1, 1, 1, 1) / 4
    for r in sorted({0, 1, m // 2, m - 1}):
        one, lse1 = fwd_kvcache_int(q[:, r:r + 1].contiguous(), *args, num_splits=min(ns, 4), **kw)
        err = (out[:8, r:r + 1].float() - one[:8].float()).abs()
        assert (err <= 1.5e-3 * scale_of[:b] + (2 ** -7 * one[:8].float().abs() if dtype == "bf16" else 0)).all(), (r, err.max().item())
        ok = lens + res > 0
        assert (lse[ok, r] - lse1[ok]).abs().max().item() < 5e-4, r
