// Kernel-shape selection for the softmax kernels.
//
// chunks = ceil(sk / 512) decides how a row is laid over waves.  Measured on MI355X, a
// wave that holds 2 chunks (1024 columns) is the sweet spot at every row length -- 4 chunks
// per wave cost 3-5 % of bandwidth, 1 chunk per wave 10-20 % -- so a row gets
// ceil(chunks / 2) waves:
//   chunks == 1    several rows per wave (packed kernels; causal rows that leave much of their lane group
//                  idle: with as many lanes as the rows see keys)    (sk <= 512)
//   chunks <= 4    full-row backward only: packed kernel, one wave per row, R x C = 4
//   chunks == 2    1 wave per row, 4 rows per 256-thread block      (sk <= 1024)
//   chunks <= 4    2 waves per row, 2 rows per block (4 rows at 4 chunks: 2-3 % faster in an
//                  interleaved comparison; at 3 chunks 2 rows are)   (sk <= 2048)
//   chunks <= 8    4 waves per row (2 rows per block: two_causal_rows)  (sk <= 4096)
//   chunks <= 16   8 waves per row, 512-thread block                 (sk <= 8192)
//   chunks <= 32   16 waves per row, 1024-thread block               (sk <= 16384)
//                  forward, in the lower 3/4 of each of these three ranges (7/8 of the last):
//                  half as many waves with 3 (4) chunks each; backward likewise, causal at 2049-3072 (if there
//                  are rows enough), 4097-6144 and 8193-12288 columns, full rows with dropout at 2049-3072 and
//                  4097-6144 (ragged ones to 5120), ragged full rows without at 2049-2304 (8192 rows and
//                  more) and 4097-4608; mask-tensor forward at 513-2048 columns (unless the call
//                  knows where its rows end) and causal forward at 1025-1408: packed kernel, two
//                  rows of two chunks or one row of three or four chunks per wave
//   chunks <= 64   16 waves per row with 3 or 4 chunks per wave      (sk <= 32768)
//   longer rows    staged in LDS, one 1024-thread block per row: in half of a CU's LDS, two
//                  blocks per CU (sk <= 40448), or in all of it       (sk <= 81408)
//   ragged rows    (sk % 8 != 0 or pointers not 16-byte aligned; 8 <= sk < 81408)
//                  the same packed, one- to sixteen-wave row and LDS-staged kernels with the kRagged flag; three and
//                  four chunks (causal forward: up to 1856 columns) in one wave, results of one-wave rows and of
//                  the backward pass in two waves staged in LDS where it pays (kStaged)
//   sliding window (kBand) the row kernels, aligned rows of 513-32768 columns: dispatch_band_rows
//   anything else  element-wise kernels (rows shorter than 8 columns or beyond 81408)
#pragma once

#include <algorithm>
#include <optional>
#include <type_traits>

#include "internal.hpp"

namespace neox {

// EXTRA is the feature set of a translation unit -- any combination of kAlibi, kBias, kDropout and
// kRagged for the forward pass, of kDropout and kRagged for the backward pass, or kBand alone -- and
// every kernel of the unit is compiled for exactly that set: the caller picks the unit by what the
// call brings along (slopes, a bias tensor, a dropout probability, unaligned rows).

// the output starts on a 4 KiB boundary (both outputs, with dropout)
static bool on_pieces(const SoftmaxArgs& a) {
    return (reinterpret_cast<uintptr_t>(a.out) & 4095u) == 0 && (a.out2 == nullptr || (reinterpret_cast<uintptr_t>(a.out2) & 4095u) == 0);
}
// rows of two 4 KiB pieces each, which several rows per block store in the order of with_xcd_mapping
[[maybe_unused]] static bool two_piece_rows(const SoftmaxArgs& a) { return a.sk * 2 == 8192 && on_pieces(a); }

// Switches the XCD-aware block -> unit mapping on (see xcd_slot) when the work units of a block
// -- `units` of them, `unit_bytes` each, consecutive in memory -- tile 4 KiB pieces exactly and
// the output starts on a 4 KiB boundary; and for rows of two pieces, several per block.
static SoftmaxArgs with_xcd_mapping(const SoftmaxArgs& a, uint64_t unit_bytes, uint32_t units, uint32_t blocks) {
    SoftmaxArgs b = a;
    b.piece_shift = 0;
    b.group_shift = 3;
    b.affine_blocks = 0;
    const bool aligned = on_pieces(a);
    if (aligned && unit_bytes > 0 && unit_bytes <= 4096 && 4096 % unit_bytes == 0 && blocks >= 8) {
        const uint32_t upp = (uint32_t)(4096 / unit_bytes);
        if (units % upp == 0 && units / upp >= 1) {
            b.piece_shift = (uint32_t)__builtin_ctz(upp);  // unit_bytes divides 4096: a power of two
            b.affine_blocks = blocks & ~7u;
        }
    }
    // Units of two pieces, several per block: blocks 4 apart run on XCDs that share two pieces in eight, and a
    // block takes every fourth unit of its group's run (sliding window over 4096 columns, [32,4096,4096]
    // window 1024, forward 226 -> 206 us, backward 274 -> 247).  Units of four pieces gain nothing that
    // way ([8,8192,8192] window 1024: 220 -> 220 and 241 -> 254).
    if (aligned && unit_bytes == 8192 && units > 1) {
        b.group_shift = 2;
        b.affine_blocks = blocks & ~3u;
    }
    return b;
}

template <typename T, Mask M, bool BWD, int EXTRA, int NCH, int WPR, int RPB>
static hipError_t launch_shape(const SoftmaxArgs& a0, hipStream_t st) {
    const dim3 grid((a0.rows + RPB - 1) / RPB);
    const dim3 block(kWave * WPR * RPB);
    // (one wave per row of two pieces: the order costs 2-5 %, sliding window of 256 over 4096 columns)
    const uint64_t unit_bytes = (uint64_t)a0.sk * 2;
    constexpr int FLAGS = kDefaultFlags | EXTRA;
    constexpr bool staged = (EXTRA & kStaged) != 0;  // a block's rows then are one run: rows in order
    const SoftmaxArgs a = with_xcd_mapping(a0, staged || (WPR == 1 && unit_bytes > 4096) ? 0 : unit_bytes, RPB, grid.x);
    const uint32_t lds = staged ? stage_bytes(RPB, (uint32_t)a0.sk) : 0;
    if constexpr (BWD) {
        hipLaunchKernelGGL((softmax_bwd_kernel<T, NCH, WPR, RPB, M, FLAGS>), grid, block, lds, st, a);
    } else {
        hipLaunchKernelGGL((softmax_fwd_kernel<T, NCH, WPR, RPB, M, FLAGS>), grid, block, lds, st, a);
    }
    return hipGetLastError();
}

template <typename T, Mask M, bool BWD, int EXTRA>
static hipError_t launch_generic(const SoftmaxArgs& a, hipStream_t st) {
    const dim3 grid(a.rows);
    const dim3 block(kGenericThreads);
    if constexpr (BWD) {
        hipLaunchKernelGGL((softmax_bwd_generic_kernel<T, M, EXTRA>), grid, block, 0, st, a);
    } else {
        hipLaunchKernelGGL((softmax_fwd_generic_kernel<T, M, EXTRA>), grid, block, 0, st, a);
    }
    return hipGetLastError();
}

template <typename T, Mask M, bool BWD, int EXTRA, int G, int R, int C>
static hipError_t launch_packed_shape(const SoftmaxArgs& a0, hipStream_t st) {
    const uint32_t per_block = Packed<G, R>::kRowsPerBlock;
    const dim3 grid((a0.rows + per_block - 1) / per_block);
    // the unit is a wave's run of rows: 4 waves per block.  Not for the full-row backward with
    // several chunks per lane group: two loads per store, and the order measured 0-2 % slower there.
    const uint64_t unit_bytes = (BWD && C > 1) ? 0 : (uint64_t)Packed<G, R>::kRowsPerWave * a0.sk * 2;
    const SoftmaxArgs a = with_xcd_mapping(a0, unit_bytes, 4, grid.x);
    constexpr int FLAGS = kDefaultFlags | EXTRA;
    if constexpr (BWD) {
        hipLaunchKernelGGL((softmax_bwd_packed_kernel<T, G, M, FLAGS, R, C>), grid, dim3(256), 0, st, a);
    } else {
        hipLaunchKernelGGL((softmax_fwd_packed_kernel<T, G, M, FLAGS, R, C>), grid, dim3(256), 0, st, a);
    }
    return hipGetLastError();
}

// causal rows that leave much of their group of GMAX lanes idle: see softmax_fwd_causal_packed_kernel
template <typename T, bool BWD, int EXTRA, int GMAX>
static hipError_t launch_causal_packed(const SoftmaxArgs& a0, hipStream_t st) {
    typedef Packed<GMAX, kPackedPasses> P;
    const dim3 grid((a0.rows + P::kRowsPerBlock - 1) / P::kRowsPerBlock);
    const SoftmaxArgs a = with_xcd_mapping(a0, (uint64_t)P::kRowsPerWave * a0.sk * 2, 4, grid.x);
    constexpr int FLAGS = kDefaultFlags | EXTRA;
    if constexpr (BWD) hipLaunchKernelGGL((softmax_bwd_causal_packed_kernel<T, GMAX, FLAGS>), grid, dim3(256), 0, st, a);
    else hipLaunchKernelGGL((softmax_fwd_causal_packed_kernel<T, GMAX, FLAGS>), grid, dim3(256), 0, st, a);
    return hipGetLastError();
}

// Whether causal rows of 65 to 447 columns go that way: those that fill less than three quarters of their lane group, with
// dropout, whose Philox rounds the idle lanes compute too, up to seven eighths and in both passes, and enough rows of them.
// The kernel's chain is longer by the zeroing, the staging and its bigger code, half a microsecond, which few rows do
// not win back.  us per launch, fp16, softmax_*_packed_kernel -> softmax_*_causal_packed_kernel, timed from 2^11 to 2^18 rows:
//   forward, 65-88 columns    aligned rows -6...+2 % up to 2^17, [3640,72,72] level, with ALiBi 16.8 -> 15.4; ragged [504,65,65] 4.3 -> 4.4,
//                             [1008,65,65] 5.8 -> 5.5
//     129-184                 [64,129,129] 4.0 -> 4.1, [127,129,129] 4.7 -> 4.6, [254,129,129] 6.5 -> 5.3, [46,177,177] 4.1 -> 4.2, [93,177,177] 5.4 -> 5.1
//     257-376                 [7,281,281] 3.7 -> 4.0, [29,281,281] 4.7 -> 4.6, [58,281,281] 6.3 -> 5.6, [1020,257,257] 54 -> 44; aligned
//                             [28,296,296] 4.8 -> 4.1, [14,296,296] +2 %, [14,304,304] -3 %
//   with dropout, 65-127      aligned [2731,96,96] 28.1 -> 27.0, -5...-15 % with fewer rows; ragged [504,65,65] 7.7 -> 7.9, [1008,65,65] 11.6 -> 10.1
//     129-192                 [64,129,129] 7.4 -> 6.2, [57,144,144] 5.4 -> 5.4; ragged [46,177,177] 5.9 -> 6.4, [93,177,177] 9.5 -> 8.8; aligned
//                             [341,192,192] 14.1 -> 16.2, [683,192,192] 26.9 -> 26.6
//     193-216                 aligned -28...+3 % throughout: never; ragged [78,209,209] 7.7 -> 8.7, [157,209,209] 12.7 -> 12.2
//     257-384                 [28,296,296] 7.2 -> 5.7, [11,376,376] 5.7 -> 5.3, ragged [7,281,281] 5.6 -> 6.1, [14,281,281] +16 %
//     385-440                 aligned [20,400,400] 6.0 -> 6.6, [82,400,400] 16.3 -> 15.9; ragged [20,401,401] 7.8 -> 8.9, [41,401,401] 13.1 -> 12.4
//   backward, with dropout    up to 192 and 384 columns -5...+92 % ([1020,257,257] 127 -> 66, [504,65,65] 8.0 -> 7.4); beyond, [78,209,209]
//                             7.4 -> 8.0, [157,209,209] 11.7 -> 11.2, [20,401,401] 7.4 -> 8.0, [41,401,401] 12.0 -> 10.3, [20,400,400] 5.7 -> 5.7
template <bool BWD, int EXTRA, int G>
static bool causal_lanes_pay(const SoftmaxArgs& a, int lanes) {
    constexpr bool rag = (EXTRA & kRagged) != 0;
    if constexpr ((EXTRA & kDropout) == 0) {
        if (lanes * 4 >= G * 3) return false;
        if (G == 16) return a.rows >= (rag ? 1u << 16 : 3u << 16);
        if (G == 32) return a.rows >= 1u << 14;
        return a.rows >= (rag ? 1u << 12 : lanes * 8 <= G * 5 ? 3u << 11 : 1u << 13);
    }
    if (G == 16) return a.sk != G * kVec && (BWD || a.rows >= (rag ? 1u << 16 : 3u << 16));
    if (lanes * 8 >= G * 7) return false;
    if (lanes * 4 > G * 3) {
        if (G == 32) return rag && a.rows >= 1u << 15;
        return a.rows >= (rag ? 1u << 14 : BWD ? 1u << 13 : 1u << 15);
    }
    if (BWD) return true;
    if (G == 64) return a.rows >= (rag ? 1u << 12 : 1u << 13);
    if (lanes * 8 <= G * 5) return a.rows >= (rag ? 1u << 13 : 1u << 14);
    return a.rows >= (rag ? 1u << 14 : 1u << 17);
}

template <typename T, Mask M, bool BWD, int EXTRA, int G>
static hipError_t launch_packed(const SoftmaxArgs& a, hipStream_t st) {
    const int lanes = (a.sk + kVec - 1) / kVec;
    if constexpr (M == Mask::Causal && G >= 16 && (!BWD || (EXTRA & kDropout) != 0)) {
        if (causal_lanes_pay<BWD, EXTRA, G>(a, lanes)) return launch_causal_packed<T, BWD, EXTRA, G>(a, st);
    }
    // passes per wave: 4, except for lane groups of 32 and 64 lanes in the causal kernels and the
    // full-row backward, which run faster with 2 when the rows fill their lane groups (causal forward
    // 15 %, causal backward up to 11 % at 512 columns, full-row backward 0-4 %).  With a quarter or
    // more of the lanes idle (129-192 and 257-384 columns) 4 passes are 4-12 % faster there too.
    constexpr int R = (M != Mask::Bytes && G >= 32) ? 2 : kPackedPasses;
    // (the dropout backward of causal rows that leave so many idle has gone above, see causal_lanes_pay)
    if constexpr (R != kPackedPasses && !(BWD && M == Mask::Causal && (EXTRA & kDropout) != 0)) {
        if (lanes * 4 <= G * 3) return launch_packed_shape<T, M, BWD, EXTRA, G, kPackedPasses, 1>(a, st);
    }
    return launch_packed_shape<T, M, BWD, EXTRA, G, R, 1>(a, st);
}

// sk <= 512: lane groups of G = pow2 >= sk/8 lanes per row
template <typename T, Mask M, bool BWD, int EXTRA>
static hipError_t dispatch_packed(const SoftmaxArgs& a, hipStream_t st) {
    const int lanes = (a.sk + kVec - 1) / kVec;
    if (lanes <= 1) return launch_packed<T, M, BWD, EXTRA, 1>(a, st);
    if (lanes <= 2) return launch_packed<T, M, BWD, EXTRA, 2>(a, st);
    if (lanes <= 4) return launch_packed<T, M, BWD, EXTRA, 4>(a, st);
    if (lanes <= 8) return launch_packed<T, M, BWD, EXTRA, 8>(a, st);
    if (lanes <= 16) return launch_packed<T, M, BWD, EXTRA, 16>(a, st);
    if (lanes <= 32) return launch_packed<T, M, BWD, EXTRA, 32>(a, st);
    return launch_packed<T, M, BWD, EXTRA, 64>(a, st);
}

// sk <= 512.  The packed forward kernels address the mask and the bias tensor through one buffer
// each; a call whose mask or bias tensor is beyond the 32-bit range of a buffer goes to the row
// kernel, which forms a 64-bit address per row.  (The backward pass reads neither.)
template <typename T, Mask M, bool BWD, int EXTRA>
static hipError_t dispatch_short_rows(const SoftmaxArgs& a, hipStream_t st) {
    constexpr bool side_tensor = !BWD && (M == Mask::Bytes || (EXTRA & kBias) != 0);
    if constexpr (side_tensor) {
        const bool fits32 = (M != Mask::Bytes || a.mask_bytes != 0) && (a.bias == nullptr || a.bias_bytes != 0);
        if (!fits32) return launch_shape<T, M, BWD, EXTRA, 1, 1, 4>(a, st);
    }
    return dispatch_packed<T, M, BWD, EXTRA>(a, st);
}

// Rows beyond the register budget, staged in LDS: in half of a CU's LDS when the row fits there,
// two blocks per CU, else in all of it.  Ragged rows need room for one position more.
static_assert(kMaxStagedRow == kMaxLdsRow, "the range the callers check is the range of the kernels");
template <typename T, Mask M, bool BWD, int EXTRA>
static hipError_t launch_lds(const SoftmaxArgs& a, hipStream_t st) {
    const int positions = a.sk + ((EXTRA & kRagged) != 0 ? 1 : 0);
    if (positions > kMaxLdsRow) return hipErrorInvalidValue;  // the caller checks
    const bool half = positions <= kMaxLdsHalfRow;
    const dim3 grid(a.rows), block(kLdsThreads);
    if constexpr (BWD) {
        // ragged rows with dropout need more than the 64 registers per lane that two blocks on a CU
        // leave each: all of the LDS, one block per CU, at any length
        constexpr bool half_fits = EXTRA != (kRagged | kDropout);
        if constexpr (half_fits) {
            if (half) {
                hipLaunchKernelGGL((softmax_bwd_lds_kernel<T, M, 5, kLdsHalf, EXTRA>), grid, block, 0, st, a);
                return hipGetLastError();
            }
        }
        hipLaunchKernelGGL((softmax_bwd_lds_kernel<T, M, 10, kLdsBytes, EXTRA>), grid, block, 0, st, a);
    } else {
        if (half) hipLaunchKernelGGL((softmax_fwd_lds_kernel<T, M, kLdsHalf, EXTRA>), grid, block, 0, st, a);
        else hipLaunchKernelGGL((softmax_fwd_lds_kernel<T, M, kLdsBytes, EXTRA>), grid, block, 0, st, a);
    }
    return hipGetLastError();
}

// The shapes that need 16-byte aligned rows: element-wise kernels when they are not, LDS-staged
// and packed kernels.  No value: none of them applies, the row kernels take the call.
template <typename T, Mask M, bool BWD, int EXTRA>
static std::optional<hipError_t> dispatch_aligned(const SoftmaxArgs& a, bool vec_ok, int chunks, hipStream_t st) {
    if (!vec_ok) return launch_generic<T, M, BWD, EXTRA>(a, st);
    if (a.sk > kMaxRegisterRow) {
        // beyond the register budget: the row is staged in LDS while it fits there
        if (a.sk <= kMaxLdsRow) return launch_lds<T, M, BWD, EXTRA>(a, st);
        return launch_generic<T, M, BWD, EXTRA>(a, st);
    }
    if (chunks == 1) return dispatch_short_rows<T, M, BWD, EXTRA>(a, st);
    if constexpr (!BWD && M == Mask::Bytes) {
        // mask-tensor forward, 513-2048 columns: the packed kernel -- two rows of two chunks, or one row of
        // three or four chunks per wave -- keeps four accesses per tensor in flight and fetches no score of
        // a lane whose keys are all hidden.  Against the row kernels (two waves with four chunk slots from
        // 1025 columns on): -17 % at 520-640 columns, -8 % at 768, -9 % at 1032 and 1152, -5 % at 1280, -1 %
        // at 1536 whatever the mask; at 769-1024 and 1537-2048 columns -5...-19 % under padding and causal
        // masks and +0...3 % under masks that hide nothing or hide at random.  With dropout folded in
        // the steps up to 1536 columns gain 4-11 %.  A call that knows where its rows end
        // (SoftmaxArgs::row_end, which the packed kernels do not look at) takes the row kernel at two
        // chunks, which ends the row there without waiting for the mask bytes and sums in the same order
        // (-16 % at 640 columns, -3...-7 % at 1024 against the packed kernel); at three and four chunks it
        // measured -3...+9 % and would sum in another order, so those stay with the packed kernel.
        const bool fits32 = a.mask_bytes != 0 && (a.bias == nullptr || a.bias_bytes != 0);
        if (fits32) {
            if (chunks == 2 && a.row_end == nullptr) return launch_packed_shape<T, M, BWD, EXTRA, kWave, 2, 2>(a, st);
            if (chunks == 3) return launch_packed_shape<T, M, BWD, EXTRA, kWave, 1, 3>(a, st);
            if (chunks == 4) return launch_packed_shape<T, M, BWD, EXTRA, kWave, 1, 4>(a, st);
        }
    }
    if constexpr (!BWD && M == Mask::Causal) {
        // causal forward, 1025-1408 columns: one row of three chunks per wave instead of two waves with
        // four slots (-11 % at 1032 and 1152 columns, -5 % at 1280, +1 % at 1536).  At two and at four
        // chunks, and in the causal backward at any, the packed kernel measured 2-16 % slower.  The
        // dropout variant follows (it loses 1-8 % here): its undropped output stays bit-equal to the
        // plain kernel's, which needs the same order of summation.
        const bool fits32 = a.bias == nullptr || a.bias_bytes != 0;
        if (chunks == 3 && a.sk <= 1408 && fits32) return launch_packed_shape<T, M, BWD, EXTRA, kWave, 1, 3>(a, st);
    }
    if constexpr (BWD && M == Mask::Causal && (EXTRA & kDropout) != 0) {
        // causal backward with dropout, 1025-1344 columns, many rows: one wave per row with three chunks, two rows per block; the Philox rounds
        // of a fourth chunk slot are work for nothing.  us per launch, fp16, two waves per row -> one: [113,1088,1088] 104.9 -> 93.0, [81,1280,1280]
        // 96.8 -> 90.7; % of two waves against one, by matrices, both kernels in turn in one process, buffers changing:
        //   fp16  1056: 5 +2.8, 6 +4.9, 8 +1.4, 12 +3.1, 16 +4.4; 1088: 6 +7.0, 8 +1.4, 14 +4.4; 1120: 5 +2.4, 7 -0.5, 8 -0.6, 14 +1.6; 1152: 6 +4.8, 8 -0.4, 14 +3.4;
        //         1184: 5 +3.9, 7 -2.2, 10 -0.3, 14 +1.4; 1248: 6 -3.8, 10 -2.2, 16 +0.1; 1304: 10 -3.1, 20 -2.1, 28 +1.8; 1336: 20 -2.5, 34 -1.5
        //   bf16  1032: 6 -6.3, 20 0, 28 +0.9; 1056: 6 -5.0, 14 +1.0, 20 +1.8, 28 +3.0; 1088: 6 -3.8, 20 +1.6, 28 +2.3; 1152: 6 -4.0, 20 +0.5, 28 +1.8; 1200: 10 -3.7, 28
        //         -1.0; 1248: 10 -4.1, 28 -0.7; 1336: 28 -3.8
        // above 1280 columns [40,1336,1336] -2.5 / -3.2, whole and half lines [40,1312,1312] +3.8 / -0.1, [64,1344,1344] +7.0 / +2.8; beyond [67,1408,1408]
        // 94.0 -> 90.3 us, but [8,1408,1408] 14.8 -> 15.3; without dropout one wave is 1-3 % slower throughout
        const bool f16 = std::is_same<T, F16>::value;
        const uint32_t least = a.sk <= 1152 ? (f16 ? 4608 : 20480) : f16 ? 18432 : 36864;
        if (chunks == 3 && a.rows >= least && a.sk <= (a.sk % (kLine / 4) == 0 ? 1344 : 1280)) return launch_shape<T, M, BWD, EXTRA, 3, 1, 2>(a, st);
    }
    if constexpr (BWD && M == Mask::None) {
        // full rows up to 2048 columns: straight-line packed kernel, R x C = 4 accesses per tensor
        if (chunks == 2) return launch_packed_shape<T, M, BWD, EXTRA, kWave, 2, 2>(a, st);
        if (chunks == 3) return launch_packed_shape<T, M, BWD, EXTRA, kWave, 1, 3>(a, st);
        if (chunks == 4) return launch_packed_shape<T, M, BWD, EXTRA, kWave, 1, 4>(a, st);
    }
    return std::nullopt;
}

// Whether causal rows of 7 or 8 chunks go two to a block (not the dropout backward: [16,4096,4096] 174 -> 175 us, [16,3840,3840]
// 156 -> 161).  It pays where neighbouring rows share a cache line, which one block then stores as a whole, and at 4096
// columns in the order of with_xcd_mapping.  us per launch forward / backward / forward with dropout (16 matrices), one row per
// block -> two, 32 matrices; alignment of the rows:
//   32 or 64 bytes   3248 186 -> 177 / 245 -> 233 / 159 -> 152, 3616 227 -> 215 / 307 -> 286 / 193 -> 183, 4000 279 -> 263 / 375 -> 351 /
//                    223 -> 213, 3088 158 -> 159 / 218 -> 218 / 139 -> 139
//   128 bytes        3200 165 -> 169 / 215 -> 222 / 140 -> 141, 3712 221 -> 221 / 292 -> 291 / 183 -> 182, 3968 245 -> 251 / 330 -> 332;
//                    4096 265 -> 254 / 346 -> 340 / 227 -> 217, but off the 4 KiB boundary 279 -> 275 / 373 -> 373
//   16 bytes         3080 159 -> 161 / 211 -> 219 / 139 -> 141, 3592 219 -> 219 / 292 -> 299, 4088 279 -> 287 / 376 -> 390 / 248 -> 257
//   8 bytes          3076 162 -> 172 / 220 -> 214, 3500 207 -> 213 / 283 -> 274 / 194 -> 184, 4004 269 -> 273 / 372 -> 361 / 251 -> 237
//   4 bytes          3130 168 -> 175 / 224 -> 218 / 153 -> 164, 3998 260 -> 268 / 361 -> 354 / 241 -> 256
//   2 bytes          3201 184 -> 187 / 245 -> 234, 3333 197 -> 198 / 265 -> 254 / 182 -> 182, 3689 237 -> 235 / 320 -> 306 / 220 -> 216,
//                    3999 277 -> 275 / 373 -> 358 / 254 -> 251
// (rows of 16 bytes and more on tensors off a 16-byte boundary were not measured: one row).  One or two matrices leave too few blocks
// for either: [1,3616,3616] forward 9.5 -> 9.9, [2,4096,4096] 18.8 -> 19.1, [4,3616,3616] 29.7 -> 29.5.
template <bool BWD, int EXTRA>
static bool two_causal_rows(const SoftmaxArgs& a, int chunks) {
    if (a.rows < 12288) return false;
    if constexpr ((EXTRA & kRagged) == 0) return (a.sk % 16 == 0 && a.sk % 64 != 0) || two_piece_rows(a);
    else if (BWD) return a.sk % 8 != 0;
    else if (a.sk % 2 != 0) return chunks == 8;
    else return (EXTRA & kDropout) != 0 && a.sk % 8 == 4;
}

// Ragged rows of two chunks: the block's results through LDS (see Rows) where the call is large enough to be bound by what its stores
// do to the lines; below, the barrier and the detour cost more.  Rows of an even length, which begin on whole dwords, gain earlier.
// % per launch of direct against staged by thousands of rows, both kernels in turn in one process, buffers changing, fp16 / bf16:
//   causal forward       945: 45 -1.4 / -0.2, 60 -0.2 / -0.5, 75 +0.7 / -0.2, 120 +1.4 / +1.1; 1001: 24 -1.4 / -1.8, 48 -0.5 / -0.7, 64 +1.1 / +1.1, 96 +1.7 / +1.5,
//                        128 +2.1 / +2.0; 946: 30 -0.5 / -2.0, 45 +1.9 / +0.5; 962: 46 -0.2 / +0.2, 61 +1.3 / +1.2; 1002: 24 -0.7 / 0, 48 +1.6 / +0.7
//   mask-tensor forward  945: 45 -0.5 / -0.5, 60 -1.2 / -1.2; 1001: 48 -2.3 / -2.2, 64 -1.6 / -1.6; 1021: 49 -3.9 / -3.5; 1022: 16 -0.2 / -1.0, 32 +1.1 / +1.0, 49 +1.6 /
//                        +1.2; 1023: 24 -0.4 / -1.6, 32 +0.7 / 0, 65 +2.7 / +2.4; other lengths from 65536 rows on, [128,945,945] +1.1 / +0.8, [200,1001,1001] +2.5 / +2.6
//   causal backward      673: 64 -0.1 / -0.7, 86 +0.8 / +0.3; 721: 57 +0.2 / -0.3, 92 +1.5 / +1.1; 769: 24 -0.5 / -1.3, 36 +1.3 / -0.9, 49 +1.4 / -0.6, 61 +1.7 / +0.8; 865: 20
//                        -1.1 / -2.0, 41 +0.8 / -0.9, 55 +1.3 / +1.0; 897: 21 -0.1 / -0.2, 28 +1.0 / +0.5; 1001: 16 +0.2 / +1.0, 24 +2.2 / +0.9, 32 +1.3 / +2.3; 674: 32 +0.3 /
//                        -0.1, 53 +0.6 / +0.8; 722: 23 -1.1 / -1.0, 46 +1.1 / +1.0; 802: 25 +0.8 / +0.3, 38 +0.8 / +1.3
//   full-row backward    673: 16 -0.3 / -2.6, 32 +0.5 / -0.3; 721: 23 +1.4 / -0.1, 34 +2.5 / -0.6; 674: 10 +0.2 / +2.1, 16 +2.6 / -1.0, 32 +2.6 / +1.7; 746: 11 +2.4 / +1.0, 35 +3.2 /
//                        +2.8; from
//                        768 columns on [24,901,901] +1.2 / +0.9, [16,805,805] -0.2 / -1.2, [32,1001,1001] +2.9 / +1.9
// Aligned rows that come here (through_lds, 32768 of them and more) begin and end on 16 bytes: causal forward [34,968,968] -0.6, [80,1000,1000]
// +2.5, backward [52,776,776] +1.5, [140,840,840] +2.9, [52,648,648] 0.
// With dropout behind throughout ([96,1001,1001] 94.2 -> 96.1 us and 86.6 -> 90.0).
template <Mask M, bool BWD>
static bool staged_two_chunks(const SoftmaxArgs& a, bool vec_ok) {
    if (vec_ok) return a.sk >= (BWD ? 672 : 944);
    const bool odd = (a.sk & 1) != 0;
    uint32_t least;
    if constexpr (!BWD) {
        if (a.sk < 944) return false;
        least = M == Mask::Causal ? (odd ? 64000 : 45000) : a.sk >= 1022 ? 32768 : 65536;
    } else {
        if (a.sk < 672) return false;
        if constexpr (M == Mask::Causal) {
            least = a.sk >= 960 ? 20480 : a.sk >= 896 ? 27648 : a.sk >= 760 ? (odd ? 45056 : 32768) : odd ? 81920 : 49152;
        } else {
            least = a.sk >= 768 ? 18432 : odd ? 28672 : 8192;
        }
    }
    return a.rows >= least;
}

// Ragged rows of three or four chunks: one wave per row instead of two, four rows per block, the results through LDS.
// (Two waves leave a quarter of their slots empty at three chunks and meet at barriers; staged on top, they lose 5-13 %.)  us per
// launch, fp16, 2^27 elements, two waves -> one, forward / backward / mask-tensor forward with padding / its backward:
//   [127,1025,1025] 87.1 -> 70.4 / 95.2 -> 93.3 / 99.1 -> 80.9 / 102.1 -> 99.4, [93,1201,1201] 79.0 -> 69.6 / 95.4 -> 92.6 / 84.6 -> 74.4 /
//   114.4 -> 112.8, [56,1535,1535] 70.6 -> 68.6 / 91.7 -> 91.1 / 79.8 -> 77.5 / 110.9 -> 112.2, [52,1601,1601] 72.3 -> 69.8 / 94.5 -> 91.2 /
//   80.2 -> 78.9 / 96.8 -> 94.8, [41,1801,1801] 70.7 -> 70.3 / 93.2 -> 90.6 / 81.2 -> 80.0 / 101.2 -> 99.2; causal forward [37,1901,1901]
//   70.3 -> 70.9, [33,2001,2001] 69.3 -> 74.7, the others there 0...-4 %
// with ALiBi [60,1049,1049] 44.8 -> 36.3, [20,1801,1801] 36.4 -> 36.1, with a bias 47.7 -> 41.2 and 41.2 -> 40.6, with dropout 76.9 ->
// 67.0 and 64.3 -> 64.7, its backward 65.4 -> 58.7 and 56.1 -> 53.9.  All feature sets take the same shape: the same sums.
// The backward pass with few rows keeps two waves: full rows [1,1601,1601] 6.0 -> 6.3, [4,1601,1601] 13.8 -> 14.1, causal [1,1601,1601]
// 4.9 -> 5.1, [2,1601,1601] 7.5 -> 6.8, [1,1301,1301] level; with dropout [2,1868,1868] +3.8 %, [2,1900,1900] +3.5 %, [3,1868,1868] -14 %, [2,1707,1707] -10 %.
template <Mask M, bool BWD>
static bool one_wave_ragged(const SoftmaxArgs& a, int chunks, bool dropout) {
    if constexpr (!BWD) return M != Mask::Causal || a.sk <= 1856;
    return M == Mask::None ? a.rows >= 8192 : chunks == 3 || a.rows >= (dropout && a.sk > 1792 ? 4096u : 2048u);
}

template <typename T, Mask M, bool BWD, int EXTRA>
static hipError_t dispatch_rows(const SoftmaxArgs& a, bool vec_ok, hipStream_t st) {
    int chunks = (a.sk + kChunk - 1) / kChunk;
    if constexpr ((EXTRA & kRagged) != 0) {
        // rows at any alignment: the packed kernels up to 512 columns, the row kernels below beyond
        if (a.sk < kVec || a.sk >= kMaxLdsRow) return hipErrorInvalidValue;  // the caller checks
        if (a.sk >= kMaxRegisterRow) return launch_lds<T, M, BWD, EXTRA>(a, st);
        if (chunks > 1) {
            // rows of odd length: the row kernels lay those that start on an odd element one
            // position later on their lanes
            chunks = (a.sk + (a.sk & 1) + kChunk - 1) / kChunk;
        }
        if (chunks == 1) return dispatch_short_rows<T, M, BWD, EXTRA>(a, st);
    } else {
        if (const auto done = dispatch_aligned<T, M, BWD, EXTRA>(a, vec_ok, chunks, st)) return *done;
    }
    // (the aligned full-row backward has taken 2 to 4 chunks with its packed kernel above)
    if constexpr (!(BWD && M == Mask::None && (EXTRA & kRagged) == 0)) {
        if (chunks == 2) {
            if constexpr (EXTRA == kRagged) {
                if (staged_two_chunks<M, BWD>(a, vec_ok)) return launch_shape<T, M, BWD, EXTRA | kStaged, 2, 1, 4>(a, st);
            }
            if constexpr (M == Mask::Causal && (EXTRA & kRagged) == 0) {
                // Both chunks' loads in front of the first one's arithmetic.  us per launch, fp16, without -> with: forward [4,960,960] 5.0 -> 3.8,
                // [16,640,640] 6.7 -> 5.9, [404,576,576] 74.2 -> 72.0, [128,1024,1024] 65.6 -> 64.5; with dropout [8,832,832] 8.2 -> 6.4, its
                // backward [4,768,768] 5.2 -> 4.6, [227,768,768] 104.6 -> 101.8; backward [4,832,832] 5.0 -> 4.1, [64,640,640] 21.8 -> 20.0,
                // [404,576,576] 97.5 -> 92.0, [193,832,832] 90.6 -> 89.8, but [8,896,896] 6.7 -> 7.0, [128,1024,1024] 86.0 -> 87.9 (two input
                // streams, more of their loads at once); [4,1024,1024] 5.5 -> 5.4.  (With a mask tensor or a window 0...+6 %: not there.)
                const bool early = !BWD || (EXTRA & kDropout) != 0 || a.sk <= 880 || a.rows <= 4608;
                if (early) return launch_shape<T, M, BWD, EXTRA | kEarly, 2, 1, 4>(a, st);
            }
            if constexpr (!(M == Mask::Causal && (EXTRA & kRagged) == 0) || (BWD && (EXTRA & kDropout) == 0))
                return launch_shape<T, M, BWD, EXTRA, 2, 1, 4>(a, st);
        }
        constexpr bool ragged = (EXTRA & kRagged) != 0;
        if constexpr (ragged) {
            // not staged: the backward pass with dropout, [60,1049,1049] 58.7 us against 61.5, [26,1601,1601] 55.9 and 56.4, and the
            // mask-tensor forward with dropout, [8,7,1049,1049] 95.4 and 99.3, [8,3,1601,1601] 84.2 and 88.0
            constexpr bool staged = (EXTRA & kDropout) == 0 || (!BWD && M == Mask::Causal);
            constexpr int FL = EXTRA | (staged ? kStaged : 0);
            if (chunks <= 4 && one_wave_ragged<M, BWD>(a, chunks, (EXTRA & kDropout) != 0)) {
                // with dropout, few rows: [3,1701,1701] 13.1 us with two waves, 11.2 staged, 10.2 not; [4,1801,1801] 17.3, 15.4, 18.1;
                // [1,1601,1601] 7.2, 7.8, 6.7
                if constexpr (staged && (EXTRA & kDropout) != 0) {
                    if (a.rows < 6400) return chunks == 3 ? launch_shape<T, M, BWD, EXTRA, 3, 1, 4>(a, st) : launch_shape<T, M, BWD, EXTRA, 4, 1, 4>(a, st);
                }
                return chunks == 3 ? launch_shape<T, M, BWD, FL, 3, 1, 4>(a, st) : launch_shape<T, M, BWD, FL, 4, 1, 4>(a, st);
            }
        }
        if constexpr (!ragged || (BWD && M == Mask::None)) {
            if (chunks == 3) return launch_shape<T, M, BWD, EXTRA, 2, 2, 2>(a, st);
        }
        if constexpr (!ragged || BWD || M == Mask::Causal) {
            if (chunks == 4) {
                // the causal forward with two output streams (dropout) measured 3 % faster with 2 rows
                if constexpr (!BWD && M == Mask::Causal && (EXTRA & kDropout) != 0)
                    return launch_shape<T, M, BWD, EXTRA, 2, 2, 2>(a, st);
                return launch_shape<T, M, BWD, EXTRA, 2, 2, 4>(a, st);
            }
        }
    }
    if constexpr (!BWD) {
        // Forward, rows that would leave a quarter or more of the 2-chunk shape's slots empty:
        // half as many waves with 3 or 4 chunks each.  Measured in an interleaved comparison:
        // +20-50 % just above a power of two (2056, 4104, 8200 columns), +4-15 % up to 3/4 (7/8 with
        // 4 chunks) of the range, while full rows lose 2-3 % with 4 chunks per wave.
        if (chunks <= 6) return launch_shape<T, M, BWD, EXTRA, 3, 2, 2>(a, st);
        if (chunks > 8 && chunks <= 12) return launch_shape<T, M, BWD, EXTRA, 3, 4, 1>(a, st);
        if (chunks > 16 && chunks <= 24) return launch_shape<T, M, BWD, EXTRA, 3, 8, 1>(a, st);
        if (chunks > 24 && chunks <= 28) return launch_shape<T, M, BWD, EXTRA, 4, 8, 1>(a, st);
    }
    if constexpr (BWD) {
        // Backward likewise, where it gains: rows of five and six chunks in two waves, rows of nine and more in four.  us per launch,
        // fp16, 2^27 elements, two chunks per wave -> three, causal / full rows / both with dropout:
        //   [30,2112,2112] 88.9 -> 88.1 / 87.8 -> 81.6 / 102.7 -> 90.4 / 119.6 -> 104.4, [20,2560,2560] 87.9 -> 86.5 / 82.2 -> 82.6 /
        //     93.3 -> 87.8 / 102.0 -> 96.3, [14,3072,3072] 88.6 -> 86.7 / 61.7 -> 61.1 / 90.6 -> 87.5 / 70.2 -> 67.7; ragged [31,2051,2051]
        //     93.9 -> 92.1, its results staged 89.9, with dropout 118.6 -> 106.7; [14,3071,3071] 91.5 -> 93.2, staged 89.6
        //   [7,4160,4160] 88.5 -> 80.1 / 98.3 -> 83.1 / 95.8 -> 83.5 / 135.6 -> 114.2, [5,5120,5120] 89.8 -> 87.5 / 103.8 -> 102.9 / 95.8 -> 88.7 /
        //     126.2 -> 110.5, [3,6144,6144] 75.6 -> 74.8 / 88.8 -> 91.1 / 78.6 -> 75.5 / 110.3 -> 107.6
        //   full rows with dropout to the end of the range, [2,5600,5600] -5.4 %, [1,5888,5888] -5 %, [4,5632,5632] 120.9 -> 110.1, but ragged ones
        //     beyond ten chunks [2,5131,5131] +0.6 %, [1,5635,5635] +1.3 %, [3,5891,5891] -1.6 %
        //   with few rows: causal [1,2112,2112] 5.9 -> 6.1, with dropout [2,2112,2112] 10.0 -> 10.9, [3,2192,2192] +3.4 % (fp16), +5.4 % (bf16),
        //     [4,2432,2432] -2.8 and -0.7 %, [3,2728,2728] +2 %, [6,2728,2728] -1 %; without dropout [2,2688,2688] 0 and +2 %, [3,2496,2496] -0.6 %;
        //     full rows [1,2112,2112] 8.0 -> 7.5, ragged [1,2901,2901] 11.7 -> 11.9, [4,2901,2901] 35.2 -> 35.7
        //   aligned causal rows that nearly fill six chunks, where the smaller number of waves is all that is left of it, by what part of a
        //     line they end on, fp16 / bf16: [6,2848,2848] and [6,2912,2912] (half a line) -1...-3 %, [6,2984,2984] and [6,3048,3048] +1.7...+3.5 / +0.4...+2,
        //     whole lines [6,2944,2944] +1.9 / -0.4 and [6,3008,3008] +1.9 / 0, full [6,3072,3072] -1.6 / -2.7; with dropout +0.5...+2.3 on parts of a
        //     line, -0.7...-4 on halves and whole lines (from 32768 rows on they go to the ragged unit, -2...-7 %)
        // Aligned full rows without dropout: not at all.  They gain where the padding hides much of a sample (the figures above) and lose where
        // nothing is hidden, [1,30,2112,2112] 124.7 -> 127.5, [1,8,4608,4608] 158.3 -> 163.7, [1,8,5120,5120] 194.1 -> 203.9, and a call
        // that knows where its rows end must sum in the order of one that does not.
        if constexpr (M == Mask::Causal || EXTRA != 0) {
            constexpr bool drop = (EXTRA & kDropout) != 0;
            bool enough = EXTRA != kRagged || (a.rows >= 8192 && a.sk <= 2304);
            if constexpr (M == Mask::Causal) {
                enough = a.rows >= 4608;
                if constexpr ((EXTRA & kRagged) == 0) {
                    const bool ends = a.sk % (kLine / 4) == 0 && (drop || a.sk % (kLine / 2) != 0 || a.sk == 6 * kChunk);
                    enough = a.rows >= (drop ? 9216u : 6144u) && (a.sk <= 2816 || ends);
                }
            }
            if (chunks <= 6 && enough) return launch_shape<T, M, BWD, EXTRA | (EXTRA == kRagged ? kStaged : 0), 3, 2, 2>(a, st);
            //   likewise aligned causal rows of eleven and twelve chunks, fp16 / bf16: [2,5440,5440] -1.8 / -7.0, [2,5888,5888] -0.7 / -6.2, [2,6144,6144] -0.3 / -5.1
            //     (whole lines), [2,5328,5328] +1.5 / -3.4, [3,5840,5840] +1.6 / -1.5, [2,6008,6008] +2.1 / -1.7, [2,6112,6112] +0.9 / -1.9; with dropout [2,5440,5440] -4.6 /
            //     -4.7, [2,5344,5344] -0.7 / -1.4, [2,5744,5744] +1.6 / +0.9, [1,5840,5840] +2.6 / +2.3, [2,6032,6032] +1.8 / +0.4
            constexpr int most = M == Mask::Causal || EXTRA == kDropout ? 12 : EXTRA == kRagged ? 9 : 10;
            bool pays = true;
            if constexpr (M == Mask::Causal && (EXTRA & kRagged) == 0 && (drop || std::is_same<T, F16>::value))
                pays = a.sk <= (drop ? 5632 : 5120) || a.sk % (kLine / 2) == 0;
            if (chunks > 8 && chunks <= most && pays) return launch_shape<T, M, BWD, EXTRA, 3, 4, 1>(a, st);
        }
    }
    if constexpr (BWD && M == Mask::Causal) {
        // Causal backward just above 8192 columns: 8 waves with 3 chunks each instead of 16 with 2, of
        // which up to half would hold nothing (-13 % at 8200 columns, -8 % at 10240, -4 % at 12288).
        if (chunks > 16 && chunks <= 24) return launch_shape<T, M, BWD, EXTRA, 3, 8, 1>(a, st);
    }
    if constexpr (M == Mask::Causal && !(BWD && (EXTRA & kDropout) != 0)) {
        if (chunks >= 7 && chunks <= 8 && two_causal_rows<BWD, EXTRA>(a, chunks)) return launch_shape<T, M, BWD, EXTRA, 2, 4, 2>(a, st);
    }
    if (chunks <= 8) return launch_shape<T, M, BWD, EXTRA, 2, 4, 1>(a, st);
    if (chunks <= 16) return launch_shape<T, M, BWD, EXTRA, 2, 8, 1>(a, st);
    if (chunks <= 32) return launch_shape<T, M, BWD, EXTRA, 2, 16, 1>(a, st);
    if (chunks <= 48) return launch_shape<T, M, BWD, EXTRA, 3, 16, 1>(a, st);
    return launch_shape<T, M, BWD, EXTRA, 4, 16, 1>(a, st);
}

// Sliding-window causal softmax: aligned causal rows of two chunks or more.  The shape goes by the chunks the band can
// touch -- w + 1 keys lie in at most w / 512 + 2 of them, `chunks` -- and by those of the row: the waves hold the band, the rest of the
// row is zeros, which they store as well (band_zero_fill).  TB/s by algorithmic bytes, bf16, 2^27 elements, [columns, window], the shape
// of the rule against the one that the band alone would call for (chunks / 2 waves with two chunks, from 4097 columns on
// chunks waves with one).  With few rows other shapes lose 2-10 %, in the forward pass those with fewer waves per row, in the backward pass
// those with one chunk per wave ([1,2048,2048] window 256 backward 3.6 -> 3.9 us, [4,1536,1536] 384 forward 5.5 -> 5.9): `many`.
//   forward   rows of three chunks: one wave, [1152,576] 4.54 -> 5.82, [1536,768] 5.55 -> 5.89, [1536,256] 5.37 -> 5.46, [1152,288] 5.46 -> 5.50
//     of four: two waves with two rows per block, [2048,1024] 5.99 -> 6.14, [2048,600] 5.74 -> 5.97
//     of five to eight: one wave at two chunks, [2560,256] 5.08 -> 5.29, [3072,400] 5.19 -> 5.30, with four chunks up to 2560 columns or for
//       windows of 256 and more (us, four -> two: [5,3072,3072] 142 -2 %, [5,3584,3584] 180 -2 %, [8,3072,3072] 256 +1 %); two waves with
//       three chunks each at three to six, [3072,1000] 5.67 -> 5.78, [3072,1400] 5.70 -> 5.97, [3072,1600] 5.43 -> 6.03, [2560,1600] 5.16 -> 5.96, but [2560,700]
//       5.63 -> 5.61; with four from 3073 columns on at five and six, [3584,1792] 5.56 -> 5.82
//   backward  one chunk per wave: [2048,384] 5.88 -> 6.17, [2560,400] 5.41 -> 5.52, [1472,368] 5.45 -> 5.59, [1536,128] level (rows of three chunks
//       that end on half or whole lines, window 200: [12,1472,1472] +4 %, [24,1504,1504] +4 %, [12,1536,1536] +3 %; 300 0...-2 %, [12,1512,1512] 200 -1.7 %); [3072,768]
//     5.63 -> 5.72, [3584,896] 5.52 -> 5.76, [3072,1100] 5.70 -> 5.89, [2560,1280] 5.84 -> 5.92, but [2560,700] 5.69 -> 5.5; [8192,1600] 5.62 -> 5.81,
//     [8192,3000] 5.73 -> 5.93, [7168,1792] 5.55 -> 5.72, [6144,3072] 5.83 -> 5.94, but [5120,2560] 5.87 -> 5.79
//   4096 columns, rows of two 4 KiB pieces, two per block in the order of with_xcd_mapping: [4096,256] 5.4 -> 5.78 and backward 5.32 -> 5.80,
//     [4096,1024] 5.86 -> 5.96 (forward), [4096,2048] 5.65 -> 6.15 and 5.99 -> 6.13, [4096,2560] 5.81 -> 6.21 and 6.13 -> 6.22; three waves' worth
//     at three chunks [4096,1000] 5.86 -> 5.97, [4096,512] -1 %.  Off the 4 KiB boundary that order does not apply: as other lengths.
//   beyond 4096 columns one chunk per wave up to four chunks, [8192,256] 5.36 -> 5.68 (forward), [5000,1250] 252 -> 236 us and 294 -> 274,
//     (forward at two chunks: from 16 chunks of the row on, [4608,400] 46.2 -> 52.4; backward at two chunks up to 16 only where rows end inside a
//     line, us, fp16, window 256: [2,5000,5000] -12 %, [2,6160,6160] -12 %, but [2,5088,5088] +6 %, [2,6144,6144] +7 %, [2,7136,7136] +9 %, [2,8192,8192]
//     +5 %; [2,9216,9216] -10 %; five to eight chunks in the backward pass with few rows too, [1,7680,7680] 3000 -5 %, [1,8184,8184] 2600 -8 %),
//     up to 28 chunks of the row: [15360,1024] 200 -> 204 us, [16384,1500] 210 -> 232, [32768,1024] 408 -> 446
template <typename T, bool BWD>
static hipError_t dispatch_band_rows(const SoftmaxArgs& a, hipStream_t st) {
    constexpr Mask M = Mask::Causal;
    constexpr int B = kBand;
    const int row = (a.sk + kChunk - 1) / kChunk, chunks = std::min(a.window / kChunk + 2, row);
    const bool many = a.rows >= 8192;
    if (row <= 2) return launch_shape<T, M, BWD, B, 2, 1, 4>(a, st);
    if (two_piece_rows(a) && (chunks > 2 || many)) {
        if (chunks == 2) return launch_shape<T, M, BWD, B, 1, 2, 2>(a, st);
        if (chunks == 3 && a.window < 640) return launch_shape<T, M, BWD, B, 2, 2, 2>(a, st);
        if (chunks <= 4 && (BWD || (chunks == 4 && !many))) return launch_shape<T, M, BWD, B, 2, 2, 4>(a, st);
        if constexpr (!BWD) {
            if (chunks == 3) return launch_shape<T, M, BWD, B, 3, 2, 2>(a, st);
        }
        return launch_shape<T, M, BWD, B, 4, 2, 2>(a, st);
    }
    if (row <= 8) {
        if constexpr (!BWD) {
            if (row == 3 && (chunks == 3 || (a.window >= 256 && a.rows >= 32768))) return launch_shape<T, M, BWD, B, 3, 1, 4>(a, st);
            if (chunks == 2 && (row <= 4 || !many || (row > 5 && a.window < 256))) return launch_shape<T, M, BWD, B, 2, 1, 4>(a, st);
            if (chunks == 2) return launch_shape<T, M, BWD, B, 4, 1, 4>(a, st);
            if (row == 4 || (chunks == 3 && (row == 5 || !many))) return launch_shape<T, M, BWD, B, 2, 2, 2>(a, st);
            if (chunks == 4 && !many) return launch_shape<T, M, BWD, B, 2, 2, 4>(a, st);
            if (chunks <= 4 || (chunks <= 6 && row <= 6)) return launch_shape<T, M, BWD, B, 3, 2, 2>(a, st);
            if (chunks <= 6 && row == 7) return launch_shape<T, M, BWD, B, 4, 2, 2>(a, st);
        } else {
            const int narrow = row == 3 && a.sk % (kLine / 4) == 0 ? 256 : 192;
            if (chunks == 2 && a.sk > 1408 && a.window >= narrow && many) return launch_shape<T, M, BWD, B, 1, 2, 2>(a, st);
            if (chunks == 2) return launch_shape<T, M, BWD, B, 2, 1, 4>(a, st);
            if (many && ((chunks == 3 && row >= 6) || (chunks == 4 && row >= 5))) return launch_shape<T, M, BWD, B, 1, 4, 1>(a, st);
            if (chunks == 3) return launch_shape<T, M, BWD, B, 2, 2, 2>(a, st);
            if (chunks == 4) return launch_shape<T, M, BWD, B, 2, 2, 4>(a, st);
        }
        return launch_shape<T, M, BWD, B, 2, 4, 1>(a, st);
    }
    if (chunks <= 4) {
        const bool two = BWD ? many && (row > 16 || a.sk % (kLine / 4) != 0) : row >= 16;
        if (row <= 28 && (chunks > 2 || two)) return launch_shape<T, M, BWD, B, 1, 4, 1>(a, st);
        if (chunks == 2) return launch_shape<T, M, BWD, B, 2, 1, 4>(a, st);
        return chunks == 3 ? launch_shape<T, M, BWD, B, 2, 2, 2>(a, st) : launch_shape<T, M, BWD, B, 2, 2, 4>(a, st);
    }
    if constexpr (BWD) {
        if (chunks <= 8 && row >= 12 && row <= 16) return launch_shape<T, M, BWD, B, 1, 8, 1>(a, st);
        if (chunks > 16 && chunks <= 24) return launch_shape<T, M, BWD, B, 3, 8, 1>(a, st);
    }
    if (chunks <= 8) return launch_shape<T, M, BWD, B, 2, 4, 1>(a, st);
    if (chunks <= 16) return launch_shape<T, M, BWD, B, 2, 8, 1>(a, st);
    if (chunks <= 32) return launch_shape<T, M, BWD, B, 2, 16, 1>(a, st);
    if (chunks <= 48) return launch_shape<T, M, BWD, B, 3, 16, 1>(a, st);
    return launch_shape<T, M, BWD, B, 4, 16, 1>(a, st);
}

template <bool BWD>
static hipError_t dispatch_band(const SoftmaxArgs& a, int dtype, bool vec_ok, hipStream_t st) {
    if (!vec_ok || a.sk <= kChunk || a.sk > kMaxRegisterRow) return hipErrorInvalidValue;  // the caller checks
    return dtype == NEOX_F16 ? dispatch_band_rows<F16, BWD>(a, st) : dispatch_band_rows<BF16, BWD>(a, st);
}

template <bool BWD, int EXTRA = 0>
static hipError_t dispatch_softmax(const SoftmaxArgs& a, Mask mask, int dtype, bool vec_ok,
                                   hipStream_t st) {
    const bool f16 = (dtype == NEOX_F16);
    switch (mask) {
        case Mask::Causal:
            return f16 ? dispatch_rows<F16, Mask::Causal, BWD, EXTRA>(a, vec_ok, st)
                       : dispatch_rows<BF16, Mask::Causal, BWD, EXTRA>(a, vec_ok, st);
        case Mask::Bytes:
            if constexpr (!BWD) {
                return f16 ? dispatch_rows<F16, Mask::Bytes, BWD, EXTRA>(a, vec_ok, st)
                           : dispatch_rows<BF16, Mask::Bytes, BWD, EXTRA>(a, vec_ok, st);
            }
            [[fallthrough]];  // the backward pass needs no mask: masked probabilities are 0
        case Mask::None:
            if constexpr (BWD) {
                return f16 ? dispatch_rows<F16, Mask::None, BWD, EXTRA>(a, vec_ok, st)
                           : dispatch_rows<BF16, Mask::None, BWD, EXTRA>(a, vec_ok, st);
            }
            break;
    }
    return hipErrorInvalidValue;
}

}  // namespace neox
