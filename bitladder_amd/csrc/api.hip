// C ABI of libbitdecode.so: argument validation, split choice, workspace carving, launches.
// Host-side counterpart of csrc/bit_decode/decode_api.cpp:301-441 (decode) and :517-603 (pack)
// in the reference; unsupported configurations return an error instead of silently doing nothing
// (decode_api.cpp:190-202 leaves the output uninitialised there).
#include <hip/hip_runtime.h>
#include <stdarg.h>
#include <stdio.h>

#include <algorithm>
#include <atomic>
#include <cmath>

#include "../../include/bitdecode.h"
#include "kernels.h"
#include "layout.h"

namespace {

thread_local char g_err[512] = "";

int fail(int code, const char* fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof(g_err), fmt, ap);
    va_end(ap);
    return code;
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

// Scratch of bitdecode_fwd_static: device memory that belongs to the library's code object, so the call
// needs no allocation.  Every GPU that loads the library holds its own copy until the process ends.
// Layout: arrival counters for up to kStaticHeads (batch x query head) rows, one 256-byte block each,
// then the two record slots of the splits.  Calls of different shapes follow one another on this one
// array, and the decode kernel expects the part it uses to be zero when a shape starts on it: every
// call therefore clears its counters and record slots with a small fill kernel in front of the decode
// kernel (a kernel, not a memset node: the call may be recorded into a HIP graph).
constexpr size_t kStaticHeads = 4096;
constexpr size_t kStaticCounterBytes = kStaticHeads * bitdecode::kTicketStride * sizeof(int);     // 1 MiB
constexpr size_t kStaticScratchBytes = size_t(8) << 20;
static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];
// address of `scratch` on each device (the name itself is only a host-side handle)
std::atomic<unsigned char*> g_scratch_ptr[64] = {};

// 16-byte stores of zero over [p, p + n16 * 16)
__global__ void zero_fill_kernel(uint4* p, size_t n16) {
    const size_t stride = static_cast<size_t>(gridDim.x) * blockDim.x;
    for (size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n16; i += stride) p[i] = uint4{0, 0, 0, 0};
}
hipError_t zero_fill(void* p, size_t bytes, hipStream_t stream) {      // bytes: a multiple of 16
    const size_t n16 = bytes / 16;
    if (n16 == 0) return hipSuccess;
    const unsigned int blocks = static_cast<unsigned int>(std::min<size_t>((n16 + 255) / 256, 1024));
    hipLaunchKernelGGL(zero_fill_kernel, dim3(blocks), dim3(256), 0, stream, static_cast<uint4*>(p), n16);
    return hipGetLastError();
}

int check_quant(int bits, int gs, int dtype, int d) {
    if (d != bitdecode::kHeadDim) return fail(BITDECODE_EUNSUPPORTED, "head_dim %d unsupported (only 128)", d);
    if (bits != 2 && bits != 4) return fail(BITDECODE_EUNSUPPORTED, "num_bits %d unsupported (2 or 4)", bits);
    if (gs != 32 && gs != 64 && gs != 128)
        return fail(BITDECODE_EUNSUPPORTED, "group_size %d unsupported (32, 64 or 128)", gs);
    if (dtype != BITDECODE_FP16 && dtype != BITDECODE_BF16)
        return fail(BITDECODE_EUNSUPPORTED, "dtype %d unsupported (fp16=0, bf16=1)", dtype);
    return 0;
}

int check_mode(int quant_mode, int bits) {
    if (quant_mode != BITDECODE_K_CHANNEL && quant_mode != BITDECODE_K_TENSOR)
        return fail(BITDECODE_EINVAL, "quant_mode %d (k-channel=0, k-tensor=1)", quant_mode);
    if (quant_mode == BITDECODE_K_TENSOR && bits != 4)
        return fail(BITDECODE_EUNSUPPORTED, "quant_mode k-tensor is implemented for 4 bits only (as in the reference)");
    return 0;
}

int query_cus() {
    int dev = 0, n = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 256;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) return 256;
    return n;
}

// Number of workgroups ("splits") a (batch, kv-head) pair is cut into.
//
// By the machine: a launch is as long as its busiest compute unit, and a unit that gets a second workgroup takes
// twice as long as its neighbours.  So the grid holds at most one workgroup per unit: the largest n with n * pairs
// <= units.  One split more (n rounded up instead of down: a grid of 264 for 24 pairs, 288 for 48) measured, us at
// 8K tokens, 4 bits g128 | 2 bits g128 | 4 bits g32:
//   24 pairs, 11 and 10 splits: 10.6 and 10.0 | 9.3 (10 splits) | 15.4 and 12.1      48 pairs (10K), 6 and 5: 19.4 and 16.5 | 21.7 and 12.7 | 29.5 and 19.3
//   80 pairs,  4 and  3 splits: 22.8 and 18.6 | 23.1 and 15.6 | 34.4 and 23.7        160 pairs (4K), 2 and 1: 24.0 and 23.7 | 23.4 and 18.0 | 34.9 and 30.5
// With more pairs than half the units, one workgroup each leaves units idle; two or three splits then even that out at 4
// bits, where the waves of several workgroups overlap on a unit (at group 32, one workgroup per unit, the rounds even out),
// from 4K tokens on, where the extra merges pay.  us with 1 | 2 | 3 splits, 4 bits g128, 8K tokens: 136 pairs 38.9 | 40.9 | 31.7,
// 168 pairs 42.2 | 42.8 | 35.5, 200 pairs 43.6 | 45.8 | 47.4; g32 53.9 | 58.0 | 43.5, 57.2 | 60.4 | 45.3, 58.0 | 62.7 | 65.0.
// Above one workgroup per unit the splits also send residual words (decode.hip: kPartialLoFrom), and it pays up to one and
// a half, a third split from 6K tokens on, and at group 32 from 6K tokens on; 4K | 8K tokens, g128 / g64 / g32:
//   264 pairs, 1, 2 and 3 splits: 38.1 36.0 35.7 | 71.3 64.4 60.2 / 41.9 38.1 38.7 / 55.8 51.5 52.5 | 106 89.3 85.6
//   384 pairs, 1 and 2: 42.6 41.6 | 79.0 74.5 / 45.8 44.3 / 57.9 58.3 | 110 98      (32K tokens, g128: 306 and 266)
//   424 pairs, 1 and 3: 43.4 52.0 | 82.1 91.0 / 47.2 54.8 | 89.8 97.4 / 60.8 77.0 | 115 119      -- one split
//   600 pairs, 1 and 2: 64.5 65.5 | 125 120 / 69.5 68.4 | 132 124 / 89.9 93.7 | 169 163          -- one split
//   800 pairs, 1 and 2: 83.4 86.0 | 164 160 / 90.2 90.7 / 117 124 | 221 214                      -- one split
// At 2 bits (one workgroup of 16 waves per unit) it never paid below one per unit (200 pairs: 32.6 against 37.7 us).
//
// By the work: a workgroup wants a unit for every wave of the 8-wave kernels at 4 bits (a unit for each of 4 waves,
// one per SIMD, at 2 bits, up to 16 splits: the merging wave takes 16 records per round trip, and a wave's time per unit
// is bound by its SIMD's vector ALU; one sequence, 8 kv heads: 2K tokens 8.5 us with 2 splits, 8.0 with 4; 8K tokens
// 8.8 with 8, 8.6 with 16).  Without packed tokens, four fp16 tiles count as a unit.
int choose_splits(int b, int hk, int max_seqlen_k, int max_res_len, int num_cus, int bits, int gs) {
    const int packed_units = max_seqlen_k / bitdecode::unit_tokens(bits);
    const int tiles = (max_res_len + 15) / 16;
    const int units = packed_units > 0 ? packed_units : (tiles + 3) / 4;
    if (units <= 0) return 1;
    const int64_t pairs = std::max<int64_t>(1, static_cast<int64_t>(b) * hk);
    int by_machine = static_cast<int>(std::max<int64_t>(1, num_cus / pairs));
    const bool over = pairs > num_cus, long_enough = packed_units >= 96;
    if (bits == 4 && 2 * pairs > num_cus && packed_units >= 64 && (!over || (2 * pairs <= 3 * num_cus && (gs >= 64 || long_enough)))) {
        // share of the machine's time that the busiest unit uses: ceil(n * pairs / units) / n, against pairs / units
        double best = 0.0;
        for (int n = 1; n <= (over && !long_enough ? 2 : 3); ++n) {
            const int64_t wgs = n * pairs, rounds = (wgs + num_cus - 1) / num_cus;
            const double fill = static_cast<double>(wgs) / static_cast<double>(rounds * num_cus);
            if (fill > 1.1 * best) {
                best = fill;
                by_machine = n;
            }
        }
    }
    int by_work;
    if (bits == 4) {
        by_work = (units + bitdecode::kFewWaves - 1) / bitdecode::kFewWaves;
    } else {
        const int nw = bitdecode::decode_waves(bits, gs);
        // (up to 8 units in one workgroup; not more than 4 in the 8 waves of group 32 if the window has none or more than 4
        // tiles, whose waves then work one after the other: 6 units and 128 window tokens, 8 pairs, 9.7 us with one split and
        // 9.0 with two, no window 8.4 and 7.8, but 32 window tokens 8.5 and 8.7; 16 waves: 8.1 and 8.1)
        const bool one = units <= 8 && !(nw == 8 && units > 4 && (tiles == 0 || tiles > 4));
        by_work = one ? 1 : std::max(std::min((units + 3) / 4, 16), (2 * units + nw - 1) / nw);
    }
    int n = std::min(std::min(by_machine, std::max(1, by_work)), 256);
    // drop splits that would be empty: ceil(units / n) units per split
    const int ups = (units + n - 1) / n;
    n = (units + ups - 1) / ups;
    return std::max(1, n);
}

// The 4-bit kernels also exist with 8 waves per workgroup (decode.hip: launch_fwd_tt), used whenever the packed
// prefix is the bulk of the work.  With per-sequence lengths on the device the workgroups of the longest
// sequences can be left streaming alone at the end, where 16 waves keep more bytes in flight per compute
// unit: then only up to 32 units per workgroup (measured on a batch of 16 sequences of 1.9K-8K tokens: 26.2
// against 26.6 us; equal-length batches of every size measured gain 1-7 % from the 8 waves).
bool use_few_waves(int bits, int gs, int max_s, int max_r, int nsplit, bool device_lengths) {
    const int packed_units = max_s / bitdecode::unit_tokens(bits);
    const int units_per_wg = (packed_units + nsplit - 1) / nsplit;
    return bitdecode::few_waves_variant(bits, gs) && units_per_wg >= 1 && max_r <= 512 &&
           (!device_lengths || units_per_wg <= 32);
}

// Split count for a call; `ragged` = per-sequence lengths come from the device (the host only has their bound).
// Two workgroups of the 8-wave kernels fit a compute unit (78 KB of LDS and 125 registers each).  A batch of
// unequal sequences is better served by twice as many workgroups of half the size: the two that share a unit
// add up, and the kernel orders the sequences so that the longest shares with the shortest (decode.hip:
// sequence_of_position).  16 sequences of 1.9K-8K tokens: 62 units on the busiest unit with one workgroup
// per unit, 49.5 with two.  Only for batches that fill the machine with one to three splits: the host cannot tell a
// ragged batch from an equal one, and equal sequences lose by the doubling what the extra splits cost
// (32 x 8 heads: nothing; 16 x 8: 1.5 %; 8 x 8 and 4 x 8, where 4 and 8 splits would become 8 and 16: 9-12 %).
// Lengths drawn from 1K-8K, 8 kv heads, 4 bits: 9 sequences 16.3 us with 3 splits, 15.4 with 7; 12 sequences 21.7 with
// 2, 17.4 with 5.  Where the doubling does not apply, sequences that occupy more than half of the units are cut in two:
// the short ones end early anyway (20 sequences: 35.4 us with one split, 27.7 with two; 2 bits 28.5 and 23.2).
//
// Long sequences on a number of pairs that does not divide the units: rounded down, the grid leaves units idle while the
// longest sequence's workgroups are as long as ever; rounded up, a few units get two workgroups, which costs nothing if a short
// sequence's is among them and half the time again if all are equal.  Two full rounds are near the better of the two in
// either case, from 28 blocks per workgroup on (fewer: the merges and the second start cost more) and up to 16 splits (one
// round trip of the merge).  Six draws of lengths from S/8 to S, mean time with n rounded down and with two rounds as a
// multiple of that with n rounded up, and all sequences equal, two rounds as a multiple of n rounded down; 4 bits g128, g32, 2 bits g64:
//    96 pairs, 18K tokens   2: 1.12 1.18 1.12     5: 1.03 0.99 1.00     equal 1.07 1.02 1.02
//   104 pairs, 18K          2: 1.10 1.19 1.12     4: 1.05 1.05 1.00     equal 1.14 1.13 1.13
//    72 pairs, 28K          3: 1.11 1.15 1.17     7: 1.02 0.99 1.01     equal 1.12 1.02 0.99
//    88 pairs, 57K          2: 1.24 1.31 1.36     5: 0.94 0.93 0.93     equal 0.97 0.99 0.94
//    40 pairs, 57K          6: 1.05 1.09 1.08    12: 1.00 0.98 1.00     equal 1.08 1.11 1.17
//    56 pairs, 18K, below   4: 1.02 1.06 1.02     9: 0.90 1.14 1.09     equal 1.08 1.14 1.15
int choose_splits_for(int b, int hk, int max_s, int max_r, int num_cus, int bits, int gs, bool ragged) {
    int n1 = choose_splits(b, hk, max_s, max_r, num_cus, bits, gs);
    if (!ragged || b < 2) return n1;
    const int64_t pairs = static_cast<int64_t>(b) * hk;
    if (2 * pairs < num_cus && num_cus % pairs != 0) {
        const int rounds2 = choose_splits(b, hk, max_s, max_r, 2 * num_cus, bits, gs);
        if (rounds2 > n1 && rounds2 <= 16 && max_s / rounds2 >= 28 * bitdecode::kChunk) return rounds2;
    }
    if (n1 > 3) return n1;
    if (2 * pairs > num_cus) n1 = pairs < num_cus ? std::min(2, choose_splits(1, 1, max_s, max_r, num_cus, bits, gs)) : 1;
    // (the 8-wave kernel of group size 32 takes 95 KB of LDS: one workgroup per unit, 20.0 us with 3 splits against 23.5
    // with 7 for 9 sequences)
    if (gs < 64) return n1;
    const int n2 = choose_splits(b, hk, max_s, max_r, 2 * num_cus, bits, gs);
    if (n2 > n1 && n2 * pairs <= 2 * num_cus && use_few_waves(bits, gs, max_s, max_r, n2, true))
        return n2;
    return n1;
}

// Several query rows per sequence, in blocks of eight or sixteen (query row, query head) pairs.  A workgroup of sixteen unpacks the
// codes for twice as many pairs, at half the vector instructions per pair, but a wave takes longer over a unit and over the merge, and
// a compute unit holds one such workgroup.
struct RowsCall {
    int b, hk, pairs, max_s, max_r, cus, bits, gs;
    bool ragged;        // per-sequence lengths on the device
    bool open;          // ... and no bound of theirs but the cache's capacity
    int64_t blocks8() const { return (static_cast<int64_t>(pairs) + bitdecode::kMaxGroupHeads - 1) / bitdecode::kMaxGroupHeads; }
    int64_t blocks16() const { return (blocks8() + 1) / 2; }
    int64_t triples() const { return static_cast<int64_t>(b) * hk * blocks16(); }      // (sequence, kv head, block of sixteen)
};

// So sixteen pays with work: W = units of 64 tokens times blocks of eight pairs per compute unit.  us in blocks of eight | sixteen,
// 32 / 8 heads unless said, 4 bits g128, 4 bits g32, 2 bits g128:
//   1 x 4K, 8 rows            W  8:   8.6 |  9.9    9.4 | 10.5    9.2 | 10.3
//   1 x 8K, 8 rows            W 16:  10.9 | 11.3   12.7 | 12.0   10.1 | 11.6       16 x 1K, 4 rows  W 16:  10.1 | 10.1   11.5 | 10.8   9.0 | 9.4
//   1 x 12K, 8 rows           W 24:  12.9 | 11.9   14.8 | 12.8   11.9 | 12.2       3 x 4K, 8 rows   W 24:  14.7 | 12.3   17.2 | 13.7  13.1 | 10.9
//   4 x 2K, 64 / 8, 8 rows    W 32:  16.9 | 12.4   20.1 | 13.9   13.4 | 11.5       32 x 2K, 8 / 8, 16 rows  W 64:  29.1 | 18.0   37.7 | 21.6  25.7 | 15.2
// Where so few triples are left that filling the machine takes 32 splits and more, their merge outweighs it at 2 bits, and at 4 bits until
// W is larger:
//   1 x 64K, 8 / 1, 8 rows    W 32:  17.7 | 18.6   21.0 | 19.9   16.7 | 17.9       1 x 128K, 8 / 1  W 64:  31.2 | 24.0   37.0 | 27.1  22.8 | 21.1 (g64 23.7 | 24.9)
//   2 x 25K, 12 / 4, 4 rows   W 25:  13.3 | 14.3 (31 splits)                          1 x 33K, 16 / 8, 8 rows  W 32, 2 bits: 14.3 | 14.9 (29)
// (2 bits g128 before its blocks of sixteen summed the lo parts apart, 5-9 % of their time, decode.hip: lo_sums.  Since then, with 16 splits
// and more: 1 x 14K, 8 rows W 28 13.0 | 13.7, 1 x 16K W 32 and 1 x 18K W 36 13.2 | 13.2 and 14.2 | 14.2, 1 x 20K W 40 14.7 | 14.3; with fewer: 7 x 4K and 16 x 1.75K, 4
// rows W 28 13.2 | 12.3 and 13.6 | 12.2, 2 x 8K, 8 rows W 32 13.0 | 13.0.)
bool rows_work(const RowsCall& c) {
    if (c.pairs <= bitdecode::kMaxGroupHeads) return false;
    const bool many_splits = c.triples() * 32 <= c.cus;
    if (many_splits && c.bits == 2) return false;
    int from = many_splits ? 48 : c.bits == 4 ? 20 : c.gs == 128 && c.triples() * 16 <= c.cus ? 32 : 28;
    // (lengths of an eighth to a quarter of the capacity, the only bound: W by the bound 60 9.4 | 11.8, 66 9.6 | 10.9, 83 12.5 | 11.7 and 15.8 | 19.9, 98
    // 20.0 | 11.6, 115 17.1 | 11.4, 139 17.9 | 11.0)
    if (c.open) from = std::max(from, 96);
    return c.blocks8() * c.b * c.hk * (c.max_s / 64) >= static_cast<int64_t>(from) * c.cus;
}

// Whether a call of n splits runs in blocks of sixteen.  us in blocks of eight | sixteen over 1300 drawn calls, every bit width, group size, mode and element type among them:
//  * Up to half the units' number of workgroups of sixteen, blocks of eight fit the machine side by side and take less time each, at
//    every length (one split of 46K tokens, 21 triples, 2 bits: 128 | 174; 48 triples of 16K, 2 splits, 4 bits: 39.9 | 46.1; 128 triples 13.4 | 15.2), from
//    160 on they do not (160: 29.3 | 18.0, 174: 43.3 | 27.7, 168: 28.9 | 18.7).  The library's own counts are above that.
//  * A workgroup wants a unit of 64 tokens for each of its eight waves (5.5: 123 | 140).
//  * Three or five blocks of eight make two or three of sixteen, a quarter or a sixth of whose columns is idle: only where the workgroups
//    fill the machine (144 of 256 units: 15.5 | 18.1, 39.1 | 45.9; 176: 31.2 | 33.9; 1056 of 1280: 48.8 | 56.9; 240: 14.9 | 13.5, 53.8 | 35.6), and three blocks only
//    with few splits to merge (4 bits, 21 splits: 13.9 | 16.5, 16: 31.9 | 28.3; 2 bits, 16: 20.4 | 21.1, 10: 15.4 | 17.3, 8: 23.7 | 21.3).
//  * The 16-wave 4-bit kernel of blocks of eight (long sequences of unequal length, long windows) sums half as many tokens per wave: only
//    where there are twice as many splits, so that no sum is longer than it would be.
bool rows_wide(const RowsCall& c, int n) {
    if (!rows_work(c)) return false;
    const int64_t wgs = c.triples() * n;
    if (2 * wgs <= c.cus || c.max_s / 64 < 8 * n) return false;
    const int64_t slots = (wgs + c.cus - 1) / c.cus * c.cus;
    if (c.blocks8() == 3 && (8 * wgs < 7 * slots || n > (c.bits == 4 ? 16 : 8))) return false;
    if (c.blocks8() == 5 && 5 * wgs < 4 * slots) return false;
    if (bitdecode::few_waves_variant(c.bits, c.gs) && !use_few_waves(c.bits, c.gs, c.max_s, c.max_r, n, c.ragged))
        return n >= 2 * choose_splits_for(c.b, static_cast<int>(c.hk * c.blocks8()), c.max_s, c.max_r, c.cus, c.bits, c.gs, c.ragged);
    return true;
}

struct RowsPlan { int splits; bool wide; };
// Split count (num_splits, or the library's own if that is zero) and blocks of a call; no split count of its own whose workspace is
// larger than `fits` says, if a smaller one can do.
template <class Fits>
RowsPlan plan_rows(const RowsCall& c, int num_splits, const Fits& fits) {
    if (num_splits > 0) return {num_splits, rows_wide(c, num_splits)};
    // (as for equal lengths: choose_splits_for's doubling counts on two workgroups per unit; 16 sequences of up to 2560 tokens in doubled and
    // plain counts, blocks of eight: 17.6 and 12.6, 14.1; up to 896: 20.5 and 10.7, 12.7)
    const int n16 = choose_splits(c.b, static_cast<int>(c.hk * c.blocks16()), c.max_s, c.max_r, c.cus, c.bits, c.gs);
    if (rows_wide(c, n16) && fits(n16)) return {n16, true};
    int n = choose_splits_for(c.b, static_cast<int>(c.hk * c.blocks8()), c.max_s, c.max_r, c.cus, c.bits, c.gs, c.ragged);
    // a workspace sized by bitdecode_num_splits_for and bitdecode_row_blocks is taken
    const int least = std::min(n, rows_work(c) ? choose_splits_for(c.b, static_cast<int>(c.hk * c.blocks16()), c.max_s, c.max_r, c.cus, c.bits, c.gs, c.ragged) : n);
    while (n > least && !fits(n)) --n;
    return {n, false};
}
int row_blocks_of(const RowsCall& c, bool wide) { return static_cast<int>(wide ? c.blocks16() : c.blocks8()); }

}  // namespace

extern "C" {

int bitdecode_abi_version(void) { return BITDECODE_ABI_VERSION; }

const char* bitdecode_last_error(void) { return g_err; }

int bitdecode_num_splits(int32_t b, int32_t h_k, int32_t max_seqlen_k, int32_t max_res_len, int32_t num_cus,
                         int32_t bits, int32_t group_size) {
    if (num_cus <= 0) num_cus = query_cus();
    if (check_quant(bits, group_size, BITDECODE_FP16, bitdecode::kHeadDim)) return -1;
    return choose_splits(b, h_k, max_seqlen_k, max_res_len, num_cus, bits, group_size);
}

int bitdecode_num_splits_for(int32_t b, int32_t h_k, int32_t max_seqlen_k, int32_t max_res_len, int32_t num_cus,
                             int32_t bits, int32_t group_size, int32_t per_sequence_lengths) {
    if (num_cus <= 0) num_cus = query_cus();
    if (check_quant(bits, group_size, BITDECODE_FP16, bitdecode::kHeadDim)) return -1;
    return choose_splits_for(b, h_k, max_seqlen_k, max_res_len, num_cus, bits, group_size, per_sequence_lengths != 0);
}

int bitdecode_row_blocks(int32_t b, int32_t h_k, int32_t pairs, int32_t max_seqlen_k, int32_t num_cus, int32_t bits) {
    if (num_cus <= 0) num_cus = query_cus();
    if (check_quant(bits, 128, BITDECODE_FP16, bitdecode::kHeadDim)) return -1;
    if (b <= 0 || h_k <= 0 || pairs <= 0) return fail(BITDECODE_EINVAL, "batch, head and pair counts must be positive"), -1;
    const RowsCall c{b, h_k, pairs, max_seqlen_k, 0, num_cus, bits, 128, false, false};
    return row_blocks_of(c, rows_work(c));
}

int bitdecode_rows_splits(int32_t b, int32_t h_k, int32_t pairs, int32_t max_seqlen_k, int32_t max_res_len, int32_t num_cus, int32_t bits,
                          int32_t group_size, int32_t per_sequence_lengths, int32_t capacity, int32_t num_splits, int32_t* row_blocks) {
    if (num_cus <= 0) num_cus = query_cus();
    if (check_quant(bits, group_size, BITDECODE_FP16, bitdecode::kHeadDim)) return -1;
    if (b <= 0 || h_k <= 0 || pairs <= 0 || num_splits < 0) return fail(BITDECODE_EINVAL, "batch, head, pair and split counts must be positive"), -1;
    const RowsCall c{b, h_k, pairs, max_seqlen_k, max_res_len, num_cus, bits, group_size, per_sequence_lengths != 0,
                     per_sequence_lengths != 0 && max_seqlen_k >= capacity};
    const RowsPlan p = plan_rows(c, num_splits, [](int) { return true; });
    if (row_blocks) *row_blocks = row_blocks_of(c, p.wide);
    return p.splits;
}

// [tickets: one 256-byte block per (batch, query head)][o_part][ml_part]
static size_t ticket_bytes(int32_t b, int32_t h) { return static_cast<size_t>(b) * h * bitdecode::kTicketStride * sizeof(int); }

// two slots of records behind the counters (kernels.h: split_slot_words)
static size_t slots_bytes(int32_t b, int32_t h, int32_t num_splits) {
    return 2 * bitdecode::split_slot_words(static_cast<size_t>(b) * h, static_cast<size_t>(num_splits)) * sizeof(uint32_t);
}

size_t bitdecode_fwd_workspace_bytes(int32_t b, int32_t h, int32_t num_splits) {
    if (num_splits <= 1) return 0;
    return ticket_bytes(b, h) + slots_bytes(b, h, num_splits);
}

// paged cache: cache_tokens is the page size; the table must cover `tokens` per sequence
static int check_paging(const int32_t* block_table, int64_t stride, int32_t max_pages, int32_t num_pages,
                        int32_t page_tokens, int32_t tokens) {
    if (!block_table) return BITDECODE_OK;
    if (max_pages <= 0 || num_pages <= 0 || stride < max_pages)
        return fail(BITDECODE_EINVAL, "block_table: %d pages per sequence, stride %lld, pool of %d pages", max_pages,
                    static_cast<long long>(stride), num_pages);
    if (static_cast<int64_t>(tokens) > static_cast<int64_t>(max_pages) * page_tokens)
        return fail(BITDECODE_EINVAL, "block_table covers %d x %d tokens per sequence, %d needed", max_pages, page_tokens,
                    tokens);
    return BITDECODE_OK;
}

int bitdecode_qpack(const bitdecode_qpack_args* a, void* stream) {
    using namespace bitdecode;
    if (!a) return fail(BITDECODE_EINVAL, "args is null");
    if (int rc = check_quant(a->bits, a->group_size, a->dtype, a->d)) return rc;
    if (int rc = check_mode(a->quant_mode, a->bits)) return rc;
    if (a->b < 0 || a->h_k <= 0 || a->n_tokens < 0) return fail(BITDECODE_EINVAL, "negative size");
    if (a->n_tokens % kChunk) return fail(BITDECODE_EINVAL, "n_tokens %d is not a multiple of 128", a->n_tokens);
    if (a->cache_tokens % kChunk || a->cache_tokens <= 0)
        return fail(BITDECODE_EINVAL, "cache_tokens %d is not a positive multiple of 128", a->cache_tokens);
    // tokens one sequence can hold: the tensor capacity, or what its row of the block table covers
    const int64_t capacity = a->block_table ? static_cast<int64_t>(a->max_pages_per_seq) * a->cache_tokens
                                            : a->cache_tokens;
    if (!a->dst_offsets) {
        if (a->dst_offset < 0 || a->dst_offset % kChunk)
            return fail(BITDECODE_EINVAL, "dst_offset %d is not a multiple of 128", a->dst_offset);
        if (static_cast<int64_t>(a->dst_offset) + a->n_tokens > capacity)
            return fail(BITDECODE_EINVAL, "dst_offset %d + n_tokens %d exceeds cache capacity %lld", a->dst_offset,
                        a->n_tokens, static_cast<long long>(capacity));
    } else if (a->n_tokens > capacity) {
        return fail(BITDECODE_EINVAL, "n_tokens %d exceeds cache capacity %lld", a->n_tokens,
                    static_cast<long long>(capacity));
    }
    if (int rc = check_paging(a->block_table, a->block_table_stride, a->max_pages_per_seq, a->num_pages,
                              a->cache_tokens, 0))
        return rc;
    if (a->n_tokens == 0 || a->b == 0) return BITDECODE_OK;
    if (!a->k || !a->v || !a->k_pack || !a->k_params || !a->v_pack || !a->v_params)
        return fail(BITDECODE_EINVAL, "null tensor pointer");
    if (!aligned16(a->k) || !aligned16(a->v) || !aligned16(a->k_pack) || !aligned16(a->k_params) ||
        !aligned16(a->v_pack) || !aligned16(a->v_params))
        return fail(BITDECODE_EINVAL, "tensor pointers must be 16-byte aligned");
    const int64_t strides[6] = {a->k_stride_b, a->k_stride_t, a->k_stride_h, a->v_stride_b, a->v_stride_t, a->v_stride_h};
    for (int64_t s : strides)
        if (s % 8) return fail(BITDECODE_EINVAL, "K/V strides must be multiples of 8 elements");

    QpackParams P{};
    P.k = static_cast<const uint16_t*>(a->k);
    P.v = static_cast<const uint16_t*>(a->v);
    P.k_sb = a->k_stride_b; P.k_st = a->k_stride_t; P.k_sh = a->k_stride_h;
    P.v_sb = a->v_stride_b; P.v_st = a->v_stride_t; P.v_sh = a->v_stride_h;
    P.k_pack = static_cast<uint8_t*>(a->k_pack);
    P.k_params = static_cast<uint8_t*>(a->k_params);
    P.v_pack = static_cast<uint8_t*>(a->v_pack);
    P.v_params = static_cast<uint8_t*>(a->v_params);
    P.kpack_bh = code_region_bytes(a->cache_tokens, a->bits);
    P.vpack_bh = P.kpack_bh;
    P.ktensor = a->quant_mode == BITDECODE_K_TENSOR;
    P.kparams_bh = P.ktensor ? v_param_region_bytes(a->cache_tokens, a->group_size)
                             : k_param_region_bytes(a->cache_tokens, a->group_size);
    P.vparams_bh = v_param_region_bytes(a->cache_tokens, a->group_size);
    P.b = a->b; P.n_tokens = a->n_tokens; P.hk = a->h_k;
    P.dst_offset = a->dst_offset;
    P.dst_offsets = a->dst_offsets;
    P.capacity = static_cast<int>(std::min<int64_t>(capacity, INT32_MAX / 2));
    P.bits = a->bits; P.gs = a->group_size; P.bf16 = a->dtype == BITDECODE_BF16;
    P.block_table = a->block_table; P.bt_stride = a->block_table_stride;
    P.chunks_per_page = a->cache_tokens / kChunk;
    hipError_t e = launch_qpack(P, static_cast<hipStream_t>(stream));
    if (e != hipSuccess) return fail(BITDECODE_ELAUNCH, "qpack launch failed: %s", hipGetErrorString(e));
    return BITDECODE_OK;
}

// BitKVCache's prefill (append = false) and append of a token (append = true)
static int run_cache(const bitdecode_cache_args* a, bool append, void* stream) {
    using namespace bitdecode;
    if (!a) return fail(BITDECODE_EINVAL, "args is null");
    if (int rc = check_quant(a->bits, a->group_size, a->dtype, a->d)) return rc;
    if (int rc = check_mode(a->quant_mode, a->bits)) return rc;
    if (a->b <= 0 || a->b > 65535 || a->h_k <= 0 || a->h_k > 65535 || a->n_tokens < 0)
        return fail(BITDECODE_EINVAL, "batch %d, %d kv heads, %d tokens", a->b, a->h_k, a->n_tokens);
    if (a->cache_tokens % kChunk || a->cache_tokens <= 0)
        return fail(BITDECODE_EINVAL, "cache_tokens %d is not a positive multiple of 128", a->cache_tokens);
    if (append && a->n_tokens != 1) return fail(BITDECODE_EINVAL, "append of %d tokens (one per sequence)", a->n_tokens);
    if (!a->lengths || !a->total || !a->k_pack || !a->k_params || !a->v_pack || !a->v_params || !a->k_res || !a->v_res ||
        (a->n_tokens > 0 && (!a->k || !a->v)) || !a->packed_lens != !a->res_lens)
        return fail(BITDECODE_EINVAL, "null tensor pointer");
    if (!aligned16(a->k) || !aligned16(a->v) || !aligned16(a->k_pack) || !aligned16(a->k_params) || !aligned16(a->v_pack) ||
        !aligned16(a->v_params) || !aligned16(a->k_res) || !aligned16(a->v_res))
        return fail(BITDECODE_EINVAL, "tensor pointers must be 16-byte aligned");
    const int64_t strides[12] = {a->k_stride_b, a->k_stride_t, a->k_stride_h, a->v_stride_b, a->v_stride_t, a->v_stride_h,
                                 a->kres_stride_b, a->kres_stride_t, a->kres_stride_h,
                                 a->vres_stride_b, a->vres_stride_t, a->vres_stride_h};
    for (int64_t s : strides)
        if (s % 8) return fail(BITDECODE_EINVAL, "K/V strides must be multiples of 8 elements");
    int longest = 0;
    for (int i = 0; i < a->b; ++i) {
        const int n = a->lengths[i];
        longest = std::max(longest, n);
        // append: a window that this token fills needs room for its chunk
        const int64_t need = append && n % kChunk == kChunk - 1 ? static_cast<int64_t>(n) + 1 : n;
        if (n < 0 || need > a->cache_tokens || (!append && n > a->n_tokens))
            return fail(BITDECODE_EINVAL, "sequence %d: length %d (%d tokens given, capacity %d)", i, n, a->n_tokens,
                        a->cache_tokens);
    }
    CacheParams P{};
    P.k = static_cast<const uint16_t*>(a->k);
    P.v = static_cast<const uint16_t*>(a->v);
    P.k_sb = a->k_stride_b; P.k_st = a->k_stride_t; P.k_sh = a->k_stride_h;
    P.v_sb = a->v_stride_b; P.v_st = a->v_stride_t; P.v_sh = a->v_stride_h;
    P.k_pack = static_cast<uint8_t*>(a->k_pack);
    P.k_params = static_cast<uint8_t*>(a->k_params);
    P.v_pack = static_cast<uint8_t*>(a->v_pack);
    P.v_params = static_cast<uint8_t*>(a->v_params);
    P.kpack_bh = code_region_bytes(a->cache_tokens, a->bits);
    P.vpack_bh = P.kpack_bh;
    P.ktensor = a->quant_mode == BITDECODE_K_TENSOR;
    P.kparams_bh = P.ktensor ? v_param_region_bytes(a->cache_tokens, a->group_size)
                             : k_param_region_bytes(a->cache_tokens, a->group_size);
    P.vparams_bh = v_param_region_bytes(a->cache_tokens, a->group_size);
    P.k_res = static_cast<uint16_t*>(a->k_res);
    P.v_res = static_cast<uint16_t*>(a->v_res);
    P.kres_sb = a->kres_stride_b; P.kres_st = a->kres_stride_t; P.kres_sh = a->kres_stride_h;
    P.vres_sb = a->vres_stride_b; P.vres_st = a->vres_stride_t; P.vres_sh = a->vres_stride_h;
    P.total = a->total; P.packed_lens = a->packed_lens; P.res_lens = a->res_lens;
    P.b = a->b; P.hk = a->h_k;
    P.pack_chunks = longest / kChunk;
    P.bits = a->bits; P.gs = a->group_size; P.bf16 = a->dtype == BITDECODE_BF16;
    for (P.first = 0; P.first < a->b; P.first += kCacheSeqs) {
        const int n = std::min(kCacheSeqs, a->b - P.first);
        bool fills = false;
        for (int i = 0; i < n; ++i) {
            P.lengths[i] = a->lengths[P.first + i];
            fills = fills || P.lengths[i] % kChunk == kChunk - 1;
        }
        hipError_t e = append ? launch_cache_append(P, n, fills, static_cast<hipStream_t>(stream))
                              : launch_cache_prefill(P, n, static_cast<hipStream_t>(stream));
        if (e != hipSuccess) return fail(BITDECODE_ELAUNCH, "cache launch failed: %s", hipGetErrorString(e));
    }
    return BITDECODE_OK;
}

int bitdecode_cache_prefill(const bitdecode_cache_args* a, void* stream) { return run_cache(a, false, stream); }

int bitdecode_cache_append(const bitdecode_cache_args* a, void* stream) { return run_cache(a, true, stream); }

// bytes of the per-sequence step counters that lead a step workspace
static size_t step_ticket_bytes(int32_t b) { return static_cast<size_t>(b) * bitdecode::kTicketStride * sizeof(int); }

size_t bitdecode_fwd_append_workspace_bytes(int32_t b, int32_t h, int32_t num_splits) {
    return step_ticket_bytes(b) + bitdecode_fwd_workspace_bytes(b, h, num_splits);
}

// decode, or (step != null) decode step with append, or (rows_args != null) decode of several query rows
static int run_fwd(const bitdecode_fwd_args* a, const bitdecode_fwd_append_args* step, void* stream,
                   unsigned char* static_scratch = nullptr, const bitdecode_fwd_rows_args* rows_args = nullptr) {
    using namespace bitdecode;
    if (!a) return fail(BITDECODE_EINVAL, "args is null");
    if (int rc = check_quant(a->bits, a->group_size, a->dtype, a->d)) return rc;
    if (int rc = check_mode(a->quant_mode, a->bits)) return rc;
    if (a->b <= 0 || a->h <= 0 || a->h_k <= 0) return fail(BITDECODE_EINVAL, "batch and head counts must be positive");
    if (a->h % a->h_k) return fail(BITDECODE_EINVAL, "h %d is not a multiple of h_k %d", a->h, a->h_k);
    const int g = a->h / a->h_k;
    if (g > kMaxGroupHeads)
        return fail(BITDECODE_EUNSUPPORTED, "%d query heads per kv head unsupported (at most %d)", g, kMaxGroupHeads);
    const int rows = rows_args ? rows_args->rows : 1;
    if (rows < 1 || rows > 4096) return fail(BITDECODE_EINVAL, "%d query rows per sequence (1 to 4096)", rows);
    if (rows_args && rows_args->q_stride_row % 8)
        return fail(BITDECODE_EINVAL, "q and residual strides must be multiples of 8 elements");
    const int n_h = a->h * rows;        // workspace rows per sequence
    int max_s = a->seqlens_k ? a->max_seqlen_k : a->seqlen_k;
    int max_r = a->res_lens ? a->max_res_len : a->res_len;
    if (step) {
        // lengths live on the device; the host bound sizes the grid: up to max_len tokens before the
        // step, of which whole chunks are packed, and a window of up to 128 tokens with the new one
        if (!step->lengths || !step->k_new || !step->v_new)
            return fail(BITDECODE_EINVAL, "decode step: lengths, k_new and v_new are required");
        if (step->max_len < 0) return fail(BITDECODE_EINVAL, "decode step: max_len %d is negative", step->max_len);
        if (!a->k_res || !a->v_res || a->max_res_len < kChunk)
            return fail(BITDECODE_EINVAL, "decode step: a residual window of at least 128 tokens is required "
                                          "(max_res_len = its capacity, got %d)", a->max_res_len);
        if (!aligned16(step->k_new) || !aligned16(step->v_new))
            return fail(BITDECODE_EINVAL, "tensor pointers must be 16-byte aligned");
        const int64_t ns[4] = {step->knew_stride_b, step->knew_stride_h, step->vnew_stride_b, step->vnew_stride_h};
        for (int64_t s : ns)
            if (s % 8) return fail(BITDECODE_EINVAL, "k_new / v_new strides must be multiples of 8 elements");
        max_s = step->max_len / kChunk * kChunk;
        max_r = kChunk;
    }
    if (max_s < 0 || max_r < 0) return fail(BITDECODE_EINVAL, "negative length");
    const int cus = query_cus();
    if (max_s % kChunk) return fail(BITDECODE_EINVAL, "packed length %d is not a multiple of 128", max_s);
    if (!a->block_table && max_s > a->cache_tokens)
        return fail(BITDECODE_EINVAL, "packed length %d exceeds cache capacity %d", max_s, a->cache_tokens);
    if (a->block_table && (a->cache_tokens <= 0 || a->cache_tokens % kChunk))
        return fail(BITDECODE_EINVAL, "page size %d is not a positive multiple of 128", a->cache_tokens);
    if (int rc = check_paging(a->block_table, a->block_table_stride, a->max_pages_per_seq, a->num_pages,
                              a->cache_tokens, max_s))
        return rc;
    if (max_s > 0 && (a->cache_tokens % kChunk)) return fail(BITDECODE_EINVAL, "cache_tokens must be a multiple of 128");
    if (!a->q || !a->out) return fail(BITDECODE_EINVAL, "q/out is null");
    if ((max_s > 0 || step) && (!a->k_pack || !a->k_params || !a->v_pack || !a->v_params))
        return fail(BITDECODE_EINVAL, "null packed-cache pointer");
    if (step && (a->cache_tokens <= 0 || a->cache_tokens % kChunk))
        return fail(BITDECODE_EINVAL, "cache_tokens %d is not a positive multiple of 128", a->cache_tokens);
    if (max_r > 0 && (!a->k_res || !a->v_res)) return fail(BITDECODE_EINVAL, "null residual pointer");
    if (!aligned16(a->q) || !aligned16(a->k_pack) || !aligned16(a->k_params) || !aligned16(a->v_pack) ||
        !aligned16(a->v_params) || !aligned16(a->k_res) || !aligned16(a->v_res))
        return fail(BITDECODE_EINVAL, "tensor pointers must be 16-byte aligned");
    const int64_t strides[8] = {a->q_stride_b, a->q_stride_h, a->kres_stride_b, a->kres_stride_t, a->kres_stride_h,
                                a->vres_stride_b, a->vres_stride_t, a->vres_stride_h};
    for (int64_t s : strides)
        if (s % 8) return fail(BITDECODE_EINVAL, "q and residual strides must be multiples of 8 elements");

    int nsplit = a->num_splits;
    if (nsplit < 0) return fail(BITDECODE_EINVAL, "num_splits %d is negative", nsplit);
    if (nsplit > 512) return fail(BITDECODE_EINVAL, "num_splits %d is above the limit of 512", nsplit);
    bool wide = false;
    int row_blocks = 1, blocks8 = 1;
    if (rows > 1) {
        const int64_t cap = a->block_table ? static_cast<int64_t>(a->max_pages_per_seq) * a->cache_tokens : a->cache_tokens;
        const RowsCall c{a->b, a->h_k, rows * g, max_s, max_r, cus, a->bits, a->group_size, a->seqlens_k != nullptr, a->seqlens_k && max_s >= cap};
        const RowsPlan plan = plan_rows(c, nsplit, [&](int n) {
            return n <= 1 || (a->workspace && bitdecode_fwd_workspace_bytes(a->b, n_h, n) <= a->workspace_bytes); });
        nsplit = plan.splits;
        wide = plan.wide;
        row_blocks = row_blocks_of(c, wide);
        blocks8 = row_blocks_of(c, false);
    } else if (nsplit == 0) {
        nsplit = choose_splits_for(a->b, a->h_k, max_s, max_r, cus, a->bits, a->group_size, a->seqlens_k && !step);
    }
    // (the built-in scratch takes every call that leaves the count to the library: it chooses no more than fits)
    while (static_scratch && a->num_splits == 0 && nsplit > 1 && slots_bytes(a->b, n_h, nsplit) > kStaticScratchBytes - kStaticCounterBytes)
        --nsplit;
    if (nsplit > 1 && slots_bytes(a->b, n_h, nsplit) >= (size_t(1) << 31))
        return fail(BITDECODE_EUNSUPPORTED, "%d splits x %d x %d heads: partial outputs of 2 GiB or more", nsplit, a->b, n_h);
    // the kernel divides workgroup ids and unit counts by the split count and the head count with a
    // multiply (kernels.h: division_magic), exact while numerator x divisor stays below 2^32
    {
        const uint64_t wgs = static_cast<uint64_t>(nsplit) * a->b * a->h_k * row_blocks;
        // lengths read on the device are clamped to the capacity by the kernel, not to max_seqlen_k: that is the bound
        const uint64_t cap_tokens = a->block_table ? static_cast<uint64_t>(a->max_pages_per_seq) * a->cache_tokens
                                                   : static_cast<uint64_t>(a->cache_tokens);
        const uint64_t longest = (a->seqlens_k || step) ? std::max<uint64_t>(cap_tokens, max_s) : static_cast<uint64_t>(max_s);
        const uint64_t units = longest / 64 + static_cast<uint64_t>(nsplit);
        if (wgs * std::max(std::max(nsplit, a->h_k), row_blocks) >= (1ull << 32) || units * nsplit >= (1ull << 32))
            return fail(BITDECODE_EUNSUPPORTED, "%d splits x %d x %d kv heads: too many workgroups", nsplit, a->b, a->h_k);
    }
    if (static_scratch) {
        const size_t rows = static_cast<size_t>(a->b) * a->h;
        const size_t need = nsplit > 1 ? slots_bytes(a->b, a->h, nsplit) : 0;
        if (rows > kStaticHeads || need > kStaticScratchBytes - kStaticCounterBytes)
            return fail(BITDECODE_EWORKSPACE, "bitdecode_fwd_static: %d splits x %zu (batch x head) rows need %zu bytes; the "
                        "built-in scratch holds %zu rows and %zu bytes (use bitdecode_fwd with a workspace)", nsplit, rows,
                        need, kStaticHeads, kStaticScratchBytes - kStaticCounterBytes);
    } else if (nsplit > 1 || step) {
        const size_t need = step ? bitdecode_fwd_append_workspace_bytes(a->b, a->h, nsplit)
                                 : bitdecode_fwd_workspace_bytes(a->b, n_h, nsplit);
        if (!a->workspace || a->workspace_bytes < need)
            return fail(BITDECODE_EWORKSPACE, "workspace of %zu bytes needed for %d splits, got %zu", need, nsplit,
                        a->workspace ? a->workspace_bytes : size_t(0));
        if (!aligned16(a->workspace)) return fail(BITDECODE_EINVAL, "workspace must be 16-byte aligned");
    }

    FwdParams P{};
    P.q = static_cast<const uint16_t*>(a->q);
    P.q_sb = a->q_stride_b; P.q_sh = a->q_stride_h;
    P.k_pack = static_cast<const uint8_t*>(a->k_pack);
    P.k_params = static_cast<const uint8_t*>(a->k_params);
    P.v_pack = static_cast<const uint8_t*>(a->v_pack);
    P.v_params = static_cast<const uint8_t*>(a->v_params);
    P.kpack_bh = code_region_bytes(a->cache_tokens, a->bits);
    P.vpack_bh = P.kpack_bh;
    P.ktensor = a->quant_mode == BITDECODE_K_TENSOR;
    P.kparams_bh = P.ktensor ? v_param_region_bytes(a->cache_tokens, a->group_size)
                             : k_param_region_bytes(a->cache_tokens, a->group_size);
    P.vparams_bh = v_param_region_bytes(a->cache_tokens, a->group_size);
    P.k_res = static_cast<const uint16_t*>(a->k_res);
    P.v_res = static_cast<const uint16_t*>(a->v_res);
    P.kres_sb = a->kres_stride_b; P.kres_st = a->kres_stride_t; P.kres_sh = a->kres_stride_h;
    P.vres_sb = a->vres_stride_b; P.vres_st = a->vres_stride_t; P.vres_sh = a->vres_stride_h;
    P.seqlens = a->seqlens_k; P.reslens = a->res_lens;
    P.seqlen = a->seqlen_k; P.reslen = a->res_len;
    P.out = static_cast<uint16_t*>(a->out);
    P.out_sb = a->out_stride_b; P.out_sh = a->out_stride_h;
    P.lse = a->softmax_lse;
    P.b = a->b; P.h = n_h; P.hk = a->h_k; P.g = g; P.nsplit = nsplit;
    P.rows = rows; P.row_blocks = row_blocks; P.rows_wide = wide;
    P.row_blocks_magic = division_magic(static_cast<uint32_t>(row_blocks));
    P.g_magic = division_magic(static_cast<uint32_t>(g));
    if (rows_args) {
        P.q_sr = rows_args->q_stride_row;
        P.out_sr = rows_args->out_stride_row;
    }
    // (decode.hip: kPartialLoFrom)
    // (several query rows: counted in blocks of eight also where they run in blocks of sixteen, whose split counts are no reason to round more)
    if (nsplit > 1 && static_cast<int64_t>(a->b) * a->h_k * blocks8 > cus) P.h |= INT32_MIN;
    P.scale = a->softmax_scale;
    P.scale_log2 = fabsf(a->softmax_scale) * 1.4426950408889634f;   // decode_api.cpp:128-142
    P.neg_scale = a->softmax_scale < 0.0f;
    P.xcd_remap = (a->b * a->h_k) % 8 == 0 && nsplit > 1;
    P.few_waves = use_few_waves(a->bits, a->group_size, max_s, max_r, nsplit, a->seqlens_k != nullptr || step != nullptr);
    // more than one workgroup per compute unit and lengths that differ: the kernel deals the sequences out so
    // that long ones share a unit with short ones (a pure permutation of the batch index, from the lengths
    // on the device; not in the step with append, whose launch itself advances the lengths)
    P.seq_perm = a->seqlens_k && !step && a->b >= 2 && a->b <= 64 &&
                 static_cast<int64_t>(nsplit) * a->b * a->h_k * row_blocks > cus;
    P.nsplit_magic = division_magic(static_cast<uint32_t>(nsplit));
    P.hk_magic = division_magic(static_cast<uint32_t>(a->h_k));
    P.block_table = a->block_table; P.bt_stride = a->block_table_stride;
    P.chunks_per_page = a->block_table ? a->cache_tokens / kChunk : 1;
    P.bits = a->bits; P.gs = a->group_size; P.bf16 = a->dtype == BITDECODE_BF16;
    {
        const int64_t cap = a->block_table ? static_cast<int64_t>(a->max_pages_per_seq) * a->cache_tokens : a->cache_tokens;
        P.capacity = static_cast<int>(std::min<int64_t>(cap, INT32_MAX / 2));
        P.res_cap = max_r;
    }
    uint8_t* ws = static_cast<uint8_t*>(a->workspace);
    if (step) {
        P.lengths = step->lengths;
        P.seqlens = step->lengths;      // (decode.hip: step_length)
        P.step_tickets = reinterpret_cast<int*>(ws);
        ws += step_ticket_bytes(a->b);
        P.k_new = static_cast<const uint16_t*>(step->k_new);
        P.v_new = static_cast<const uint16_t*>(step->v_new);
        P.knew_sb = step->knew_stride_b; P.knew_sh = step->knew_stride_h;
        P.vnew_sb = step->vnew_stride_b; P.vnew_sh = step->vnew_stride_h;
    }
    if (nsplit > 1) {
        const size_t records = static_cast<size_t>(nsplit) * a->b * n_h;
        if (static_scratch) {
            P.tickets = reinterpret_cast<int*>(static_scratch);
            P.o_part = reinterpret_cast<uint32_t*>(static_scratch + kStaticCounterBytes);
        } else {
            P.tickets = reinterpret_cast<int*>(ws);
            P.o_part = reinterpret_cast<uint32_t*>(ws + ticket_bytes(a->b, n_h));
        }
        P.ml_part = reinterpret_cast<float*>(P.o_part + 2 * records * kPartialWords);
        if (static_scratch) {
            // another shape may have used the array before: counters and record slots of this call start at zero
            hipError_t e = zero_fill(P.tickets, ticket_bytes(a->b, a->h), static_cast<hipStream_t>(stream));
            if (e == hipSuccess) e = zero_fill(P.o_part, slots_bytes(a->b, a->h, nsplit), static_cast<hipStream_t>(stream));
            if (e != hipSuccess) return fail(BITDECODE_ELAUNCH, "decode launch failed: %s", hipGetErrorString(e));
        }
    }
    hipError_t e = launch_fwd(P, static_cast<hipStream_t>(stream));
    if (e != hipSuccess) return fail(BITDECODE_ELAUNCH, "decode launch failed: %s", hipGetErrorString(e));
    return BITDECODE_OK;
}

int bitdecode_fwd(const bitdecode_fwd_args* a, void* stream) { return run_fwd(a, nullptr, stream); }

int bitdecode_fwd_static(const bitdecode_fwd_args* a, void* stream) {
    int dev = 0;
    if (hipError_t e = hipGetDevice(&dev); e != hipSuccess || dev < 0 || dev >= 64)
        return fail(BITDECODE_ELAUNCH, "bitdecode_fwd_static: no current device (%s)", hipGetErrorString(e));
    unsigned char* ptr = g_scratch_ptr[dev].load(std::memory_order_acquire);
    if (!ptr) {
        // once per device, with that device current: where this device keeps its copy of the array
        if (hipError_t e = hipGetSymbolAddress(reinterpret_cast<void**>(&ptr), HIP_SYMBOL(scratch)); e != hipSuccess || !ptr)
            return fail(BITDECODE_ELAUNCH, "bitdecode_fwd_static: address of the built-in scratch: %s", hipGetErrorString(e));
        g_scratch_ptr[dev].store(ptr, std::memory_order_release);
    }
    return run_fwd(a, nullptr, stream, ptr);
}

int bitdecode_fwd_rows(const bitdecode_fwd_rows_args* a, void* stream) {
    if (!a) return fail(BITDECODE_EINVAL, "args is null");
    return run_fwd(&a->fwd, nullptr, stream, nullptr, a);
}

int bitdecode_fwd_append(const bitdecode_fwd_append_args* a, void* stream) {
    if (!a) return fail(BITDECODE_EINVAL, "args is null");
    return run_fwd(&a->fwd, a, stream);
}

#ifdef BITDECODE_PROF
int bitdecode_prof_set(void* p) { return bitdecode::set_prof_buffer(static_cast<unsigned long long*>(p)) != hipSuccess; }
#endif

}  // extern "C"
