"""Cache management around the two kernels: a packed low-bit prefix plus an fp16 residual window per
sequence, kept in step with the tokens a decode loop appends.

This is the bookkeeping the reference's figures describe (imgs/overview.png, imgs/scheme.png: the most
recent `L mod N_r` tokens stay fp16 and are attended in fp16; when the window reaches `N_r` tokens it is
quantize-packed and appended to the cache) and that its kernel traits still name
(csrc/bit_decode/src/include/kernel_traits.h:76,85: residual_block_size).  The reference's main branch
ships no code for it; here it is host logic over `kvcache_pack_int(dst_offsets=...)` and
`fwd_kvcache_int(seqlens_k=..., residual_len=...)`, or one launch per token with
`fwd_kvcache_int_append` (`step`).  Lengths are tracked on the host (they are a pure function of the
calls made) and mirrored in a device counter that `step` advances, so nothing is read back from the
device.
"""
from __future__ import annotations

import ctypes
import math
from typing import Optional, Sequence

import torch

from . import _lib
from .interface import (_check_cache, _dtype_code, _on_device, _stream_ptr, fwd_kvcache_int, fwd_kvcache_int_append,
                        kvcache_pack_int, plan_fwd_kvcache_int_append)

BLOCK = 128          # tokens per packed block = residual window size N_r


class BitKVCache:
    """One attention layer's KV cache: `k_pack/k_params/v_pack/v_params` with the reference's tensor
    contract (evaluation/test.py:74-83) and `k_res/v_res [b, 128, h_k, 128]` for the window.

    Sequences may have different lengths.  `packed_len[i]` is always a multiple of 128 and
    `res_len[i] < 128` after every call.
    """

    # packed and window lengths on the device as the last write left them: [packed, window, stream, and the host's lists of
    # the same lengths] (_write, _device_lengths); of the class, for caches that were saved before there were any
    _published: Optional[list] = None

    def __init__(self, batch: int, kv_heads: int, max_tokens: int, *, num_bits: int = 4, group_size: int = 128,
                 dtype: torch.dtype = torch.float16, device="cuda", head_dim: int = 128,
                 quant_mode: str = "k-channel"):
        if head_dim != 128:
            raise NotImplementedError("head_dim must be 128")
        if quant_mode not in ("k-channel", "k-tensor"):
            raise ValueError(f"quant_mode must be 'k-channel' or 'k-tensor', got {quant_mode!r}")
        if quant_mode == "k-tensor" and num_bits != 4:
            raise NotImplementedError("quant_mode 'k-tensor' is implemented for num_bits=4 only")
        self.b, self.h_k, self.bits, self.gs, self.dtype = batch, kv_heads, num_bits, group_size, dtype
        self.quant_mode = quant_mode
        self.device = torch.device(device)
        self.capacity = (max_tokens + BLOCK - 1) // BLOCK * BLOCK
        pn, S, d = 16 // num_bits, self.capacity, head_dim
        dev = self.device
        self.k_pack = torch.zeros((batch, S // pn, kv_heads, d), dtype=torch.uint16, device=dev)
        # "k-tensor": one (scale, zero) per token and channel group for K as well, shaped like V's
        k_params_shape = (batch, d // group_size, kv_heads, S) if quant_mode == "k-tensor" \
            else (batch, S // group_size, kv_heads, d)
        self.k_params = torch.zeros(k_params_shape, dtype=torch.float32, device=dev)
        self.v_pack = torch.zeros((batch, S, kv_heads, d // pn), dtype=torch.uint16, device=dev)
        self.v_params = torch.zeros((batch, d // group_size, kv_heads, S), dtype=torch.float32, device=dev)
        self.k_res = torch.zeros((batch, BLOCK, kv_heads, d), dtype=dtype, device=dev)
        self.v_res = torch.zeros_like(self.k_res)
        self.packed_len = [0] * batch
        self.res_len = [0] * batch
        self.total = torch.zeros(batch, dtype=torch.int32, device=dev)     # tokens held, as `step` needs them
        self._rows = torch.arange(batch, device=dev)

    # ------------------------------------------------------------------ lengths
    @property
    def lengths(self) -> list[int]:
        return [p + r for p, r in zip(self.packed_len, self.res_len)]

    def _i32(self, values: Sequence[int]) -> torch.Tensor:
        return torch.tensor(list(values), dtype=torch.int32, device=self.device)

    # ------------------------------------------------------------------ writes
    def _write(self, entry: str, k: torch.Tensor, v: torch.Tensor, lengths: list[int]) -> bool:
        """`prefill` or `append` in one launch: tokens k / v [b, n, h_k, 128], lengths per sequence, to the packed cache,
        the window, `total` and a new pair of device length arrays.  False if the tensors are not what the kernels take
        (another element type than the cache's, unaligned or strided rows, a capture in progress, no GPU) or the cache is one
        that they do not: the caller then works with torch operations."""
        kr, vr = self.k_res, self.v_res
        if (not kr.is_cuda or self.b < 1 or k.dim() != 4 or k.shape != v.shape or k.shape[0] != self.b or
                k.shape[2] != self.h_k or k.shape[3] != 128 or kr.shape != (self.b, BLOCK, self.h_k, 128) or
                vr.shape != kr.shape or self.total.dtype != torch.int32 or self.total.shape != (self.b,) or
                self.total.stride(0) != 1):
            return False
        device, dtype = kr.device, kr.dtype
        if (self.b > 65535 or not 0 < self.h_k <= 65535 or self.capacity == 0 or self.bits not in (2, 4) or
                self.gs not in (32, 64, 128) or dtype not in (torch.float16, torch.bfloat16)):
            return False
        args = (k, v, kr, vr)
        for t in args:
            st = t.stride()
            if (t.dtype != dtype or t.device != device or st[3] != 1 or (st[0] | st[1] | st[2]) % 8 or
                    t.data_ptr() % 16):
                return False
        if self.total.device != device or torch.cuda.is_current_stream_capturing():
            return False
        b, S, h_k = _check_cache(self.k_pack, self.k_params, self.v_pack, self.v_params, self.bits, self.gs, device,
                                 self.quant_mode == "k-tensor")
        if (b, S, h_k) != (self.b, self.capacity, self.h_k):
            return False
        a = _lib.CacheArgs()
        a.k, a.v, a.k_res, a.v_res = (t.data_ptr() for t in args)
        a.k_stride_b, a.k_stride_t, a.k_stride_h = k.stride()[:3]
        a.v_stride_b, a.v_stride_t, a.v_stride_h = v.stride()[:3]
        a.kres_stride_b, a.kres_stride_t, a.kres_stride_h = kr.stride()[:3]
        a.vres_stride_b, a.vres_stride_t, a.vres_stride_h = vr.stride()[:3]
        a.k_pack, a.k_params = self.k_pack.data_ptr(), self.k_params.data_ptr()
        a.v_pack, a.v_params = self.v_pack.data_ptr(), self.v_params.data_ptr()
        a.total = self.total.data_ptr()
        a.lengths = (ctypes.c_int32 * b)(*lengths)
        a.b, a.n_tokens, a.h_k, a.d = b, k.shape[1], h_k, 128
        a.cache_tokens = S
        a.bits, a.group_size, a.dtype = self.bits, self.gs, _dtype_code(kr)
        a.quant_mode = _lib.K_TENSOR if self.quant_mode == "k-tensor" else _lib.K_CHANNEL
        with _on_device(device):
            stream = _stream_ptr(device)
            # The same arrays from write to write: a cache per layer then finds its `decode` calls again, whose key holds
            # the addresses.  Only calls on the stream that writes them read them (_device_lengths), so they may be
            # written over; another stream gets arrays of its own.  The record is one list, changed in place, for all
            # copies of the cache that share the arrays.
            record = self._published
            if record is None or record[2] != stream or record[0].device != device or record[0].shape != (b,):
                record = self._published = [torch.empty(b, dtype=torch.int32, device=device),
                                            torch.empty(b, dtype=torch.int32, device=device), stream, None, None]
            a.packed_lens, a.res_lens = record[0].data_ptr(), record[1].data_ptr()
            record[3] = record[4] = None      # (until the caller says which lengths they are)
            _lib.check(getattr(_lib.lib(), entry)(ctypes.byref(a), stream))
        return True

    def _publish(self) -> None:
        """The arrays of the write just made hold the host's lengths."""
        self._published[3:] = [list(self.packed_len), list(self.res_len)]

    def _device_lengths(self):
        """Packed and window lengths as device tensors: those the last write left if the host's lengths are still theirs
        and the stream is the one that wrote them (their memory belongs to it), else uploaded.  Not under capture: a
        graph would keep the addresses of arrays that later writes free or change, and an upload cannot be recorded."""
        if self.total.is_cuda and torch.cuda.is_current_stream_capturing():
            raise RuntimeError("decode takes its lengths from the host and cannot be captured: capture a plan_step plan")
        if self._published is not None:
            packed, res, stream, host_packed, host_res = self._published
            if host_packed == self.packed_len and host_res == self.res_len and _stream_ptr(packed.device) == stream:
                return packed, res
        return self._i32(self.packed_len), self._i32(self.res_len)

    def prefill(self, k: torch.Tensor, v: torch.Tensor, lengths: Optional[Sequence[int]] = None) -> None:
        """Start the cache from prompt K/V `[b, L, h_k, 128]` (`lengths[i] <= L` valid tokens per sequence,
        default L): whole 128-token blocks are quantize-packed in one launch, each sequence's last
        `length mod 128` tokens go to its fp16 window."""
        b, L = k.shape[0], k.shape[1]
        lengths = [L] * b if lengths is None else [int(x) for x in lengths]
        if b != self.b or len(lengths) != b or max(lengths) > L or min(lengths) < 0:
            raise ValueError("prefill: batch or lengths do not match")
        if max(lengths) > self.capacity:
            raise ValueError(f"prefill: {max(lengths)} tokens exceed the capacity of {self.capacity}")
        self.packed_len = [x // BLOCK * BLOCK for x in lengths]
        self.res_len = [x - p for x, p in zip(lengths, self.packed_len)]
        if self._write("bitdecode_cache_prefill", k, v, lengths):
            self._publish()
            return
        n_pack = max(self.packed_len)
        if n_pack:
            # sequences shorter than n_pack get blocks of padding packed behind their prefix; decode never
            # reads them (seqlens_k) and later appends overwrite them
            kvcache_pack_int(k[:, :n_pack], self.k_pack, self.k_params, v[:, :n_pack], self.v_pack, self.v_params,
                             None, None, n_pack, self.quant_mode, self.gs, self.bits)
        for i, (p, r) in enumerate(zip(self.packed_len, self.res_len)):
            if r:
                self.k_res[i, :r].copy_(k[i, p:p + r])
                self.v_res[i, :r].copy_(v[i, p:p + r])
        self.total.copy_(self._i32(lengths))

    def append(self, k_new: torch.Tensor, v_new: torch.Tensor) -> None:
        """Append one token per sequence, `[b, 1, h_k, 128]` (or `[b, h_k, 128]`).  A window that reaches 128
        tokens is quantize-packed behind its sequence's prefix in the same call (one launch for all
        sequences that filled up; the others are skipped through a negative offset)."""
        if any(p + r + 1 > self.capacity for p, r in zip(self.packed_len, self.res_len)):
            raise ValueError("append: cache capacity exceeded")
        if all(p % BLOCK == 0 and 0 <= r < BLOCK for p, r in zip(self.packed_len, self.res_len)):
            k1, v1 = (k_new[:, :1], v_new[:, :1]) if k_new.dim() == 4 else (k_new[:, None], v_new[:, None])
            if self._write("bitdecode_cache_append", k1, v1, self.lengths):
                self.packed_len = [p + BLOCK if r == BLOCK - 1 else p for p, r in zip(self.packed_len, self.res_len)]
                self.res_len = [(r + 1) % BLOCK for r in self.res_len]
                self._publish()
                return
        if k_new.dim() == 4:
            k_new, v_new = k_new[:, 0], v_new[:, 0]
        pos = self._i32(self.res_len).long()
        self.k_res[self._rows, pos] = k_new.to(self.dtype)
        self.v_res[self._rows, pos] = v_new.to(self.dtype)
        self.res_len = [r + 1 for r in self.res_len]
        if BLOCK in self.res_len:
            full = [r == BLOCK for r in self.res_len]
            offsets = self._i32([p if f else -1 for p, f in zip(self.packed_len, full)])
            kvcache_pack_int(self.k_res, self.k_pack, self.k_params, self.v_res, self.v_pack, self.v_params,
                             None, None, BLOCK, self.quant_mode, self.gs, self.bits, dst_offsets=offsets)
            self.packed_len = [p + BLOCK if f else p for p, f in zip(self.packed_len, full)]
            self.res_len = [0 if f else r for r, f in zip(self.res_len, full)]
        self.total += 1

    # ------------------------------------------------------------------ read
    def decode(self, q: torch.Tensor, softmax_scale: Optional[float] = None, **kw) -> torch.Tensor:
        """Attention of one query token per sequence, `q [b, 1, h, 128]`, over everything appended so far."""
        if softmax_scale is None:
            softmax_scale = 1.0 / math.sqrt(q.shape[-1])
        packed, res = self._device_lengths()
        # (the window's bound is its size, not the longest window of the moment: the same grid, and one call all along a block)
        return fwd_kvcache_int(q, self.k_pack, self.k_params, self.v_pack, self.v_params, None, softmax_scale,
                               self.quant_mode, self.gs, self.bits,
                               seqlens_k=packed, max_seqlen_k=max(self.packed_len),
                               k_residual=self.k_res, v_residual=self.v_res,
                               residual_len=res, max_residual_len=BLOCK, **kw)

    # ------------------------------------------------------------------ one launch per token
    def plan_step(self, q: torch.Tensor, k_new: torch.Tensor, v_new: torch.Tensor,
                  softmax_scale: Optional[float] = None, **kw):
        """A `DecodePlan` whose `run()` is one decode step in one launch: attend `q` over everything held
        plus the new token, append the token, pack the window if it became full.  The plan reads
        `q / k_new / v_new` in place and sizes its grid for the cache's capacity, so it can be run (or
        captured in a HIP graph and replayed) once per token.  Lengths advance on the device; the host
        copies do not follow a plan that is run directly: call `sync_lengths()` before mixing it with the
        other methods."""
        if softmax_scale is None:
            softmax_scale = 1.0 / math.sqrt(q.shape[-1])
        return plan_fwd_kvcache_int_append(q, k_new, v_new, self.k_pack, self.k_params, self.v_pack, self.v_params,
                                           self.k_res, self.v_res, self.total, self.capacity + BLOCK - 1, None,
                                           softmax_scale, self.quant_mode, self.gs, self.bits, **kw)

    def step(self, q: torch.Tensor, k_new: torch.Tensor, v_new: torch.Tensor,
             softmax_scale: Optional[float] = None, **kw) -> torch.Tensor:
        """`append` and `decode` in one launch, except that a window filled by this token is attended in
        fp16 once more before its packed form takes over.  A sequence that has no room left is attended
        but not extended."""
        if k_new.dim() == 3:
            k_new, v_new = k_new[:, None], v_new[:, None]
        if any(p + r + 1 > self.capacity for p, r in zip(self.packed_len, self.res_len)):
            raise ValueError("step: cache capacity exceeded")
        if softmax_scale is None:
            softmax_scale = 1.0 / math.sqrt(q.shape[-1])
        # (the plain entry point: its workspace comes from the per-stream cache and its argument block is
        # found again when the same buffers are passed step after step)
        out = fwd_kvcache_int_append(q, k_new.to(self.dtype), v_new.to(self.dtype), self.k_pack, self.k_params,
                                     self.v_pack, self.v_params, self.k_res, self.v_res, self.total,
                                     self.capacity + BLOCK - 1, None, softmax_scale, self.quant_mode, self.gs, self.bits,
                                     **kw)
        for i, (p, r) in enumerate(zip(self.packed_len, self.res_len)):
            if r + 1 < BLOCK:
                self.res_len[i] = r + 1
            elif p + BLOCK <= self.capacity:
                self.packed_len[i], self.res_len[i] = p + BLOCK, 0
        return out

    def sync_lengths(self) -> None:
        """Reads the device counter back (synchronises) and rebuilds the host copies from it."""
        totals = self.total.tolist()
        self.packed_len = [t // BLOCK * BLOCK for t in totals]
        self.res_len = [t - p for t, p in zip(totals, self.packed_len)]
