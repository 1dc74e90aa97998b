// Quantize-pack kernel: fp16/bf16 K,V -> 2/4-bit codes + scale/zero in the gfx950 layout of
// layout.h.  One workgroup (256 threads) packs one 128-token chunk of one (batch, kv-head) with the
// shared chunk routine of qpack_chunk.h, or two workgroups do where the chunks leave compute units idle.  HBM-bound:
// reads 64 KB, writes chunk_code_bytes*2 + params per chunk.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "kernels.h"
#include "layout.h"
#include "qpack_chunk.h"

namespace bitdecode {
namespace {

// How a launch cuts its chunks.  Up to three rounds of workgroups over the 256 compute units a chunk's K and V go to a
// workgroup each: twice as many in flight, and each a chain (fetch, statistics, codes, store) half as long.  Measured, us for one
// workgroup per chunk | two, 4 bits group 128 / 4 bits group 32 / 2 bits group 128:
//     8 chunks   6.6 | 4.5     7.6 | 5.1     6.5 | 4.4          128   8.2 | 6.2     8.9 | 6.8     7.7 | 6.0
//   256          9.5 | 8.1    10.0 | 8.5     8.6 | 7.8          384  10.8 | 9.8    12.5 | 10.3   11.2 | 9.4
//   512         12.9 | 11.4   14.4 | 13.5   12.8 | 11.1         640  14.0 | 13.1   16.8 | 15.8   14.9 | 12.7
// Beyond that they are within 3 % of each other either way ("k-tensor" 2-4 % slower with two at 768-1024 chunks) and
// one workgroup keeps its chunk.  From 512 chunks on input and output are streamed past the caches.
enum class Cut { kSides, kSidesStream, kStream };
Cut choose_cut(int64_t chunks) {
    return chunks < 512 ? Cut::kSides : chunks < 768 ? Cut::kSidesStream : Cut::kStream;
}

template <int BITS, int GS, bool BF16, bool KT, Cut CUT>
__global__ __launch_bounds__(qp::kPackThreads) void qpack_kernel(QpackParams P) {
    __shared__ qp::PackLds<GS> L;
    const int tid = threadIdx.x;
    const int ci_src = CUT != Cut::kStream ? blockIdx.x >> 1 : blockIdx.x, hk = blockIdx.y, bi = blockIdx.z;
    const int dst_base = P.dst_offsets ? P.dst_offsets[bi] : P.dst_offset;
    if (dst_base < 0) return;       // a negative per-sequence offset skips that sequence (whole workgroup)
    const int dst_tok = dst_base + ci_src * kChunk;
    // a device-side offset the host never saw: not on a chunk boundary, or past the cache -> nothing is written
    if ((dst_base & (kChunk - 1)) != 0 || dst_tok + kChunk > P.capacity) return;
    const ChunkPlace place = chunk_place(P.block_table, P.bt_stride, P.chunks_per_page, bi, hk, P.hk, dst_tok / kChunk);
    const qp::ChunkDst D = qp::chunk_dst<BITS, GS, KT>(P.k_pack, P.k_params, P.v_pack, P.v_params, P.kpack_bh, P.kparams_bh,
                                                   P.vpack_bh, P.vparams_bh, place);
    const uint16_t* ks = P.k + bi * P.k_sb + static_cast<int64_t>(ci_src) * kChunk * P.k_st + hk * P.k_sh;
    const uint16_t* vs = P.v + bi * P.v_sb + static_cast<int64_t>(ci_src) * kChunk * P.v_st + hk * P.v_sh;
    const int64_t k_st = P.k_st, v_st = P.v_st;
    if constexpr (CUT != Cut::kStream) {
        qp::pack_chunk_side<BITS, GS, BF16, KT, CUT == Cut::kSidesStream>(
            L, tid, blockIdx.x & 1, [=](int n) { return ks + n * k_st; }, [=](int n) { return vs + n * v_st; }, D);
        return;
    }
    // 4 bits, group 128: with the V tile prefetched the kernel needs 133 registers and only three
    // workgroups fit a CU; fetched after the K side it needs 114, a fourth workgroup fits (LDS: 40 KB
    // each) and the kernel is 10 % faster.  (At group 64 a fourth workgroup was measured 3 % slower.)
    qp::pack_chunk<BITS, GS, BF16, !(BITS == 4 && GS == 128), KT, true>(
        L, tid, true, [=](int n) { return ks + n * k_st; }, [=](int n) { return vs + n * v_st; }, D);
}

// Start of a cache from ragged prompts, one launch: workgroup (c, head, sequence) packs the c-th 128-token chunk, up to
// the longest prompt's last whole one (behind a shorter prompt that is padding, which no decode reads), and the one whose
// chunk the prompt ends in copies what lies behind the prompt's last whole chunk into the fp16 window.  Same bound and same
// chunk routine as qpack_kernel; what it saves are two copies per sequence for the windows and the upload of the lengths.
template <int BITS, int GS, bool BF16, bool KT, Cut CUT>
__global__ __launch_bounds__(qp::kPackThreads) void cache_prefill_kernel(CacheParams P) {
    __shared__ qp::PackLds<GS> L;
    const int tid = threadIdx.x;
    const int ci = CUT != Cut::kStream ? blockIdx.x >> 1 : blockIdx.x, hk = blockIdx.y, bi = P.first + blockIdx.z;
    const bool v_side = CUT != Cut::kStream && (blockIdx.x & 1);
    const int n = P.lengths[blockIdx.z], whole = n / kChunk, rest = n % kChunk;
    if (ci == 0 && hk == 0 && tid == 0 && !v_side) {
        P.total[bi] = n;
        if (P.packed_lens) {
            P.packed_lens[bi] = n - rest;
            P.res_lens[bi] = rest;
        }
    }
    const uint16_t* ks = P.k + bi * P.k_sb + static_cast<int64_t>(ci) * kChunk * P.k_st + hk * P.k_sh;
    const uint16_t* vs = P.v + bi * P.v_sb + static_cast<int64_t>(ci) * kChunk * P.v_st + hk * P.v_sh;
    const int64_t k_st = P.k_st, v_st = P.v_st;
    if (ci == whole && !v_side) {
        uint16_t* kw = P.k_res + bi * P.kres_sb + hk * P.kres_sh;
        uint16_t* vw = P.v_res + bi * P.vres_sb + hk * P.vres_sh;
        const int col = (tid & 15) * 8;
        for (int r = tid >> 4; r < rest; r += qp::kPackThreads / 16) {
            const qp::u4 kr = qp::ld16<false>(ks + r * k_st + col), vr = qp::ld16<false>(vs + r * v_st + col);
            qp::st16<false>(kw + r * P.kres_st + col, kr);
            qp::st16<false>(vw + r * P.vres_st + col, vr);
        }
    }
    if (ci >= P.pack_chunks) return;
    const qp::ChunkDst D = qp::chunk_dst<BITS, GS, KT>(P.k_pack, P.k_params, P.v_pack, P.v_params, P.kpack_bh, P.kparams_bh,
                                                   P.vpack_bh, P.vparams_bh, ChunkPlace{static_cast<int64_t>(bi) * P.hk + hk, ci});
    if constexpr (CUT != Cut::kStream) {
        qp::pack_chunk_side<BITS, GS, BF16, KT, CUT == Cut::kSidesStream>(
            L, tid, v_side, [=](int r) { return ks + r * k_st; }, [=](int r) { return vs + r * v_st; }, D);
        return;
    }
    qp::pack_chunk<BITS, GS, BF16, !(BITS == 4 && GS == 128), KT, true>(
        L, tid, true, [=](int r) { return ks + r * k_st; }, [=](int r) { return vs + r * v_st; }, D);
}

// One token per sequence: threads 0-31 of workgroup (head, sequence) copy its K and V into the window's next row and one
// thread per sequence counts it.  A few kilobytes: a launch and one round trip to memory, whatever the batch.  (As torch
// operations: two indexed stores of 5.5 us, an addition, and three uploads of integers that each wait for the stream.
// 8 prompts of 1K-8K tokens and 8 tokens each by append and decode: 911 us before, 300 with this and the prefill above;
// 4 prompts of 700-2000 tokens and 16 decode steps: 307 and 240; 247 and 158 with the native host path.)
__device__ __forceinline__ void append_token(const CacheParams& P, int hk, int bi, int n, int tid) {
    const int r = n % kChunk;
    if (tid < 32) {
        const int col = (tid & 15) * 8;
        if (tid < 16) {
            qp::st16<false>(P.k_res + bi * P.kres_sb + r * P.kres_st + hk * P.kres_sh + col,
                            qp::ld16<false>(P.k + bi * P.k_sb + hk * P.k_sh + col));
        } else {
            qp::st16<false>(P.v_res + bi * P.vres_sb + r * P.vres_st + hk * P.vres_sh + col,
                            qp::ld16<false>(P.v + bi * P.v_sb + hk * P.v_sh + col));
        }
    } else if (tid == 32 && hk == 0) {
        P.total[bi] += 1;
        if (P.packed_lens) {
            P.packed_lens[bi] = n - r + (r == kChunk - 1 ? kChunk : 0);
            P.res_lens[bi] = (r + 1) % kChunk;
        }
    }
}
__global__ __launch_bounds__(64) void cache_append_kernel(CacheParams P) {
    append_token(P, blockIdx.x, P.first + blockIdx.y, P.lengths[blockIdx.y], threadIdx.x);
}
// The same when some window becomes full: its workgroups, one for K and one for V, also pack it behind the prefix, 127 rows from the window and the
// last one from the new token.
template <int BITS, int GS, bool BF16, bool KT>
__global__ __launch_bounds__(qp::kPackThreads) void cache_append_pack_kernel(CacheParams P) {
    __shared__ qp::PackLds<GS> L;
    const int tid = threadIdx.x, hk = blockIdx.x, bi = P.first + blockIdx.y;
    const int n = P.lengths[blockIdx.y];
    const bool v_side = blockIdx.z != 0;
    if (!v_side) append_token(P, hk, bi, n, tid);
    if (n % kChunk != kChunk - 1) return;
    const uint16_t* kn = P.k + bi * P.k_sb + hk * P.k_sh;
    const uint16_t* vn = P.v + bi * P.v_sb + hk * P.v_sh;
    const uint16_t* kw = P.k_res + bi * P.kres_sb + hk * P.kres_sh;
    const uint16_t* vw = P.v_res + bi * P.vres_sb + hk * P.vres_sh;
    const int64_t k_st = P.kres_st, v_st = P.vres_st;
    const qp::ChunkDst D = qp::chunk_dst<BITS, GS, KT>(P.k_pack, P.k_params, P.v_pack, P.v_params, P.kpack_bh, P.kparams_bh,
                                                   P.vpack_bh, P.vparams_bh,
                                                   ChunkPlace{static_cast<int64_t>(bi) * P.hk + hk, n / kChunk});
    qp::pack_chunk_side<BITS, GS, BF16, KT>(
        L, tid, v_side, [=](int r) { return r == kChunk - 1 ? kn : kw + r * k_st; },
        [=](int r) { return r == kChunk - 1 ? vn : vw + r * v_st; }, D);
}

template <int BITS, int GS, bool BF16, bool KT>
hipError_t launch_cache_tt(const CacheParams& P, int n, bool append, hipStream_t stream) {
    if (append) {
        hipLaunchKernelGGL((cache_append_pack_kernel<BITS, GS, BF16, KT>), dim3(P.hk, n, 2), dim3(qp::kPackThreads), 0, stream, P);
        return hipGetLastError();
    }
    // (one workgroup more per head for the windows of the prompts that end behind the last packed chunk)
    const int across = P.pack_chunks + 1;
    switch (choose_cut(static_cast<int64_t>(P.pack_chunks) * P.hk * n)) {
        case Cut::kStream:
            hipLaunchKernelGGL((cache_prefill_kernel<BITS, GS, BF16, KT, Cut::kStream>), dim3(across, P.hk, n), dim3(qp::kPackThreads), 0, stream, P);
            break;
        case Cut::kSides:
            hipLaunchKernelGGL((cache_prefill_kernel<BITS, GS, BF16, KT, Cut::kSides>), dim3(2 * across, P.hk, n), dim3(qp::kPackThreads), 0, stream, P);
            break;
        default:
            hipLaunchKernelGGL((cache_prefill_kernel<BITS, GS, BF16, KT, Cut::kSidesStream>), dim3(2 * across, P.hk, n), dim3(qp::kPackThreads), 0, stream, P);
    }
    return hipGetLastError();
}
template <int BITS, int GS>
hipError_t launch_cache_t(const CacheParams& P, int n, bool append, hipStream_t stream) {
    if (P.ktensor) {
        if constexpr (BITS == 4) {
            return P.bf16 ? launch_cache_tt<BITS, GS, true, true>(P, n, append, stream)
                          : launch_cache_tt<BITS, GS, false, true>(P, n, append, stream);
        } else {
            return hipErrorInvalidValue;
        }
    }
    return P.bf16 ? launch_cache_tt<BITS, GS, true, false>(P, n, append, stream)
                  : launch_cache_tt<BITS, GS, false, false>(P, n, append, stream);
}
hipError_t launch_cache(const CacheParams& P, int n, bool append, hipStream_t stream) {
    switch (P.bits * 1000 + P.gs) {
        case 4128: return launch_cache_t<4, 128>(P, n, append, stream);
        case 4064: return launch_cache_t<4, 64>(P, n, append, stream);
        case 4032: return launch_cache_t<4, 32>(P, n, append, stream);
        case 2128: return launch_cache_t<2, 128>(P, n, append, stream);
        case 2064: return launch_cache_t<2, 64>(P, n, append, stream);
        case 2032: return launch_cache_t<2, 32>(P, n, append, stream);
    }
    return hipErrorInvalidValue;
}

template <int BITS, int GS, bool KT, Cut CUT>
hipError_t launch_qpack_tt(const QpackParams& P, dim3 grid, hipStream_t stream) {
    if (CUT != Cut::kStream) grid.x *= 2;
    if (P.bf16) {
        hipLaunchKernelGGL((qpack_kernel<BITS, GS, true, KT, CUT>), grid, dim3(256), 0, stream, P);
    } else {
        hipLaunchKernelGGL((qpack_kernel<BITS, GS, false, KT, CUT>), grid, dim3(256), 0, stream, P);
    }
    return hipGetLastError();
}
template <int BITS, int GS, bool KT>
hipError_t launch_qpack_cut(const QpackParams& P, hipStream_t stream) {
    const dim3 grid(P.n_tokens / kChunk, P.hk, P.b);
    switch (choose_cut(static_cast<int64_t>(grid.x) * grid.y * grid.z)) {
        case Cut::kStream: return launch_qpack_tt<BITS, GS, KT, Cut::kStream>(P, grid, stream);
        case Cut::kSides: return launch_qpack_tt<BITS, GS, KT, Cut::kSides>(P, grid, stream);
        default: return launch_qpack_tt<BITS, GS, KT, Cut::kSidesStream>(P, grid, stream);
    }
}

template <int BITS, int GS>
hipError_t launch_qpack_t(const QpackParams& P, hipStream_t stream) {
    if (P.ktensor) {      // K quantized per token like V: 4 bits only, as in the reference (qpack.h:385)
        if constexpr (BITS == 4) {
            return launch_qpack_cut<BITS, GS, true>(P, stream);
        } else {
            return hipErrorInvalidValue;
        }
    }
    return launch_qpack_cut<BITS, GS, false>(P, stream);
}

}  // namespace

hipError_t launch_qpack(const QpackParams& P, hipStream_t stream) {
    if (P.n_tokens == 0 || P.b == 0) return hipSuccess;
    switch (P.bits * 1000 + P.gs) {
        case 4128: return launch_qpack_t<4, 128>(P, stream);
        case 4064: return launch_qpack_t<4, 64>(P, stream);
        case 4032: return launch_qpack_t<4, 32>(P, stream);
        case 2128: return launch_qpack_t<2, 128>(P, stream);
        case 2064: return launch_qpack_t<2, 64>(P, stream);
        case 2032: return launch_qpack_t<2, 32>(P, stream);
    }
    return hipErrorInvalidValue;
}

hipError_t launch_cache_prefill(const CacheParams& P, int n, hipStream_t stream) { return launch_cache(P, n, false, stream); }
hipError_t launch_cache_append(const CacheParams& P, int n, bool fills, hipStream_t stream) {
    if (fills) return launch_cache(P, n, true, stream);
    hipLaunchKernelGGL(cache_append_kernel, dim3(P.hk, n), dim3(64), 0, stream, P);
    return hipGetLastError();
}

}  // namespace bitdecode
