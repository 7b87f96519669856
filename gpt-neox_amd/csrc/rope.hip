// Rotary embedding kernels and their launcher.
#include "internal.hpp"

namespace neox {

// LDS for the cos/sin values a block evaluates from angles: 2 x d_rot floats (at most 32 KiB)
template <typename CS>
static size_t angle_lds_bytes(const RopeArgs& a) {
    return std::is_same<CS, Angles>::value ? (size_t)a.half * 4 * sizeof(float) : 0;
}

template <typename T, typename CS, int W, bool BWD>
static hipError_t launch_rope_shape(const RopeArgs& a, int s, int n_outer, hipStream_t st) {
    const int lpv = a.lpv;
    const int vpb = (256 / lpv) > 0 ? (256 / lpv) : 1;  // vectors per block iteration
    int nmax = a.t[0].n_inner;
    if (a.nt > 1 && a.t[1].n_inner > nmax) nmax = a.t[1].n_inner;
    const int iters = (nmax + vpb - 1) / vpb;
    // split the vector loop over blockIdx.z until the grid has a few thousand blocks
    long long blocks = (long long)s * n_outer;
    int zsplit = 1;
    if (blocks < 4096) {
        zsplit = (int)((4096 + blocks - 1) / blocks);
        if (zsplit > iters) zsplit = iters;
        if (zsplit > 65535) zsplit = 65535;
        if (zsplit < 1) zsplit = 1;
    }
    const dim3 grid(s, n_outer, zsplit);
    const dim3 block(lpv, vpb);
    hipLaunchKernelGGL((rope_kernel<T, CS, W, BWD>), grid, block, angle_lds_bytes<CS>(a), st, a);
    return hipGetLastError();
}

template <typename T, typename CS, int W, bool BWD>
static bool try_launch_rope_piece(const RopeArgs& a, int s, int n_outer, hipStream_t st, hipError_t* err);

template <typename T, typename CS, int W, bool BWD>
static hipError_t launch_rope_span(const RopeArgs& a, int s, int n_outer, hipStream_t st) {
    RopeArgs b = a;
    b.lph = a.lpv * 2 + a.pad_slots;
    b.lph_magic = (65536 + b.lph - 1) / b.lph;
    b.spw = kWave / b.lph;
    if constexpr (!std::is_same<CS, Angles>::value) {
        hipError_t err = hipSuccess;
        if (try_launch_rope_piece<T, CS, W, BWD>(b, s, n_outer, st, &err)) return err;
    }
    const int vpb = (256 / kWave) * b.spw * kSpanIters;  // vectors per block iteration
    int nmax = a.t[0].n_inner;
    if (a.nt > 1 && a.t[1].n_inner > nmax) nmax = a.t[1].n_inner;
    // one loop iteration per block: many short-lived blocks measured faster than fewer blocks
    // that loop (the cos/sin values a block reloads come from L2)
    long long zsplit = (nmax + vpb - 1) / vpb;
    const long long pairs = (long long)s * n_outer;
    if (pairs * zsplit > 0x7fffffffLL) zsplit = 0x7fffffffLL / pairs;  // grid.x limit: blocks loop instead
    if (zsplit < 1) return hipErrorInvalidValue;
    b.zsplit = (int)zsplit;
    b.outer_grid = n_outer;
    b.share = (int)((nmax + zsplit - 1) / zsplit);
    hipLaunchKernelGGL((rope_span_kernel<T, CS, W, BWD>), dim3((unsigned)(pairs * zsplit)), dim3(256),
                       angle_lds_bytes<CS>(a), st, b);
    return hipGetLastError();
}

// Dense tensors laid out alike: the XCD-aware piece kernel (see rope_piece_kernel).  `a` comes
// from launch_rope_span's preparation (lph, spw set).  Returns false if the shape does not qualify.
template <typename T, typename CS, int W, bool BWD>
static bool try_launch_rope_piece(const RopeArgs& a, int s, int n_outer, hipStream_t st, hipError_t* err) {
    if (std::is_same<CS, Angles>::value) return false;
    const RopeTensor& q = a.t[0];
    // [s, b, h, d] dense: head vectors `vec` elements apart in one run, in and out, q and k
    const int64_t vec = q.in_stride[2];
    const int64_t vecs_per_pos = (int64_t)n_outer * q.n_inner;
    auto dense = [&](const RopeTensor& t) {
        for (int i = 0; i < 3; ++i)
            if (t.in_stride[i] != q.in_stride[i] || t.out_stride[i] != q.in_stride[i]) return false;
        return t.n_inner == q.n_inner && t.n_outer == q.n_outer;
    };
    if (vec < (int64_t)(a.lpv * 2 + a.pad_slots) * W || vec > 0x7fffffff) return false;
    if (q.in_stride[0] != vecs_per_pos * vec) return false;
    if (n_outer > 1 && q.in_stride[1] != (int64_t)q.n_inner * vec) return false;
    if (!dense(q) || (a.nt > 1 && !dense(a.t[1]))) return false;
    if (vecs_per_pos % a.spw != 0 || vecs_per_pos > 0x7fffffff) return false;
    if ((int64_t)a.spw * vec * 2 > 0x7fffffffLL) return false;  // a unit is addressed through one 32-bit buffer
    const int64_t units = (int64_t)s * vecs_per_pos / a.spw;
    if (units > 0x7fffffffLL || (int64_t)s * vecs_per_pos > 0xffffffffLL) return false;
    RopeArgs b = a;
    b.vec_elems = (int32_t)vec;
    b.vecs_per_pos = (uint32_t)vecs_per_pos;
    b.n_units = (uint32_t)units;
    constexpr int ITERS = kSpanIters;
    const uint32_t U = 4 * ITERS;
    const uint32_t blocks = (uint32_t)((units + U - 1) / U);
    // XCD-aware order where the units tile 4 KiB pieces and the tensors start on a piece boundary
    const int64_t unit_bytes = (int64_t)a.spw * vec * 2;
    auto aligned = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 4095u) == 0; };
    b.units_per_piece = 0;
    b.affine_blocks = 0;
    bool on_pieces = unit_bytes <= 4096 && 4096 % unit_bytes == 0 && blocks >= 8 && aligned(q.out) &&
                     (a.nt < 2 || aligned(a.t[1].out));
    if (on_pieces) {
        const uint32_t upp = (uint32_t)(4096 / unit_bytes);
        if (U % upp == 0) {
            b.units_per_piece = upp;
            b.affine_blocks = blocks & ~7u;
        }
    }
    // without that order the kernel has nothing over rope_span_kernel, which loads its cos/sin
    // values once per block (20B shape, 192-byte heads: 45.6 against 42.6 us)
    if (b.units_per_piece == 0) return false;
    hipLaunchKernelGGL((rope_piece_kernel<T, CS, W, BWD, ITERS>), dim3(blocks), dim3(256), 0, st, b);
    *err = hipGetLastError();
    return true;
}

// the rotated span, with the slots stored as loaded behind it, is at most 64 slots of w >= 2 dims:
// the contiguous-span kernel applies (a pass-through copy must be covered by those slots)
static bool span_shape(const RopeArgs& a, int w) {
    return w >= 2 && a.lpv * 2 + a.pad_slots <= kWave && (a.copy_dims == 0 || a.pad_slots * w == a.copy_dims);
}

// Whether dense heads with angles go to the run kernel rather than to launch_rope_w's: `rounds` sine and cosine
// evaluations per lane, at most, in a wave of the run kernel, whose 1024 dims no other wave shares them with.
// A block of rope_span_kernel evaluates a position's angles once for up to 4096 dims, on the other hand with as many
// of its lanes idle as its head vectors leave.  us per launch, that kernel -> the run kernel:
//   up to two rounds, any fill: [2048,2,64,96] d_rot 24 27.7 -> 18.6, [2048,1,32,128] d_rot 128 9.1 -> 8.6, [2048,2,64,96]
//     d_rot 96 20.4 -> 20.0, [2048,2,32,256] d_rot 64 25.1 -> 23.1; the one behind: [2048,2,64,112] d_rot 112 22.7 -> 23.1
//   more, blocks at most 3/4 filled with head vectors, and the share of lanes at work times the rounds at most 3:
//     [32768,1,2,256] d_rot 256 78 -> 23, [8192,1,8,256] 22.6 -> 17.0, [8192,1,20,256] 43 -> 36, [8192,1,24,256] 44.0 -> 41.8,
//     [8192,1,2,512] d_rot 512 23.3 -> 14.3; beyond 3, behind: [8192,1,4,512] (8 rounds, half the lanes) 24.1 -> 26.2,
//     [8192,1,16,160] (5 rounds, 5/8) 19.9 -> 20.7
//   more, fuller blocks, all behind: [2048,2,16,256] d_rot 256 14.8 -> 17.0, [2048,2,8,512] d_rot 512 15.8 -> 26.1, [4096,1,32,112]
//     d_rot 112 13.3 -> 14.4, [2048,1,40,96] d_rot 96 8.8 -> 9.1, [2048,2,32,160] d_rot 160 17.9 -> 19.4
//   8- and 4-byte slots, which rope_span_kernel moves one by one: [2048,1,40,88] d_rot 88 12.0 -> 8.9, [2048,2,24,168] 22.3 -> 17.9,
//     [8192,1,8,168] 15.3 -> 14.6; beyond 192 dims where few waves straddle positions, [2048,2,32,200] 29.4 -> 25.9, or the
//     blocks are as empty as above, [8192,1,4,200] 13.8 -> 11.2; behind: [8192,1,8,200] 15.9 -> 16.6
//   heads of more than 64 slots, element by element there: [2048,2,16,520] d_rot 256 61 -> 30, [2048,2,8,1024] d_rot 512 57 -> 49;
//     with nothing to pass through rope_kernel is as wide: [2048,2,16,264] d_rot 264 17.9 -> 21.1
static bool angles_in_runs(const RopeArgs& a, int w, int rounds) {
    if (!span_shape(a, w)) return a.copy_dims > 0;
    if (rounds <= 2) return true;
    const int lph = a.lpv * 2 + a.pad_slots;
    const int64_t per_block = (int64_t)(256 / kWave) * (kWave / lph) * kSpanIters;  // head vectors, as in launch_rope_span
    const int64_t n = a.nt > 1 && a.t[1].n_inner > a.t[0].n_inner ? a.t[1].n_inner : a.t[0].n_inner;
    const int64_t blocks = (n + per_block - 1) / per_block, used = n * lph, lanes = blocks * (256 * kSpanIters);
    const bool idle = n * 4 <= blocks * per_block * 3;
    if (w < kVec) return a.half <= 96 || idle || n * (2 * a.half + a.copy_dims) >= 8 * kRunSlots * kVec;
    return idle && used * rounds <= lanes * 3;
}

template <typename T, typename CS, int PW, bool BWD>
static hipError_t launch_rope_run(const RopeRunArgs& r, int nt, hipStream_t st) {
    const uint32_t slots = nt > 1 && r.slots[1] > r.slots[0] ? r.slots[1] : r.slots[0];
    const uint32_t units = (slots + kRunSlots - 1) / kRunSlots;
    hipLaunchKernelGGL((rope_run_kernel<T, CS, PW, BWD>), dim3((units + 3) / 4, nt), dim3(256),
                       4 * r.wave_floats * sizeof(float), st, r);
    return hipGetLastError();
}

// Whole heads of dense tensors, out of place: the run kernel (see rope_run_kernel).  Returns false if the
// call does not qualify.
template <typename T, typename CS, bool BWD>
static bool try_launch_rope_run(const RopeArgs& a, int s, int n_outer, int w, hipStream_t st, hipError_t* err) {
    const int d_rot = 2 * a.half, d = d_rot + a.copy_dims;
    if (n_outer != 1 || d % kVec != 0 || a.half % 2 != 0) return false;
    // Tables: where the half span is no multiple of 8 dims the other kernels move 8 or 4 bytes per access; where it is,
    // or where the whole head rotates, rope_piece_kernel reads nothing twice.  us per launch, fp16, that kernel or
    // rope_span_kernel -> this: [2048,2,64,96] d_rot 24 25.7 -> 18.8, [2048,2,40,80] d_rot 20 24.5 -> 12.2, [2048,2,8,256]
    // d_rot 24 9.0 -> 7.8; against it: [2048,2,64,128] d_rot 32 23.3 -> 23.7, d_rot = d = 128 13.3 -> 14.6, d_rot = d = 40
    // 18.3 -> 19.1 (bf16, q and k).  Angles: angles_in_runs.
    if (!std::is_same<CS, Angles>::value && (a.half % kVec == 0 || a.copy_dims == 0)) return false;
    RopeRunArgs r{};
    uint32_t positions = 0;  // that a piece can touch
    const uint32_t spv = (uint32_t)(d / kVec);
    uintptr_t in_lo[2], in_hi[2], out_lo[2], out_hi[2];
    for (int i = 0; i < a.nt; ++i) {
        const RopeTensor& t = a.t[i];
        const int64_t per_pos = (int64_t)t.n_inner * d;
        if (t.in_stride[2] != d || t.out_stride[2] != d || t.in_stride[0] != per_pos || t.out_stride[0] != per_pos) return false;
        in_lo[i] = reinterpret_cast<uintptr_t>(t.in), out_lo[i] = reinterpret_cast<uintptr_t>(t.out);
        if (in_lo[i] % 16 != 0 || out_lo[i] % 16 != 0) return false;
        const int64_t slots = (int64_t)t.n_inner * spv * s;
        if ((int64_t)t.n_inner * spv > 0x7fffffffLL || slots > 0x7fffffffLL) return false;
        in_hi[i] = in_lo[i] + (uintptr_t)slots * 16, out_hi[i] = out_lo[i] + (uintptr_t)slots * 16;
        r.in[i] = t.in, r.out[i] = t.out;
        r.slots[i] = (uint32_t)slots;
        r.by_vpp[i] = FastDiv::by((uint32_t)t.n_inner);
        const uint32_t vecs = (kRunSlots - 2) / spv + 2;  // head vectors that the slots of a wave can touch
        const uint32_t p = (vecs - 2 + (uint32_t)t.n_inner) / (uint32_t)t.n_inner + 1;
        if (p > positions) positions = p;
    }
    // a lane's partner is read from memory, so nothing that is read may be written
    for (int i = 0; i < a.nt; ++i)
        for (int o = 0; o < a.nt; ++o)
            if (in_lo[i] < out_hi[o] && out_lo[o] < in_hi[i]) return false;
    r.by_spv = FastDiv::by(spv);
    r.by_rot = FastDiv::by((uint32_t)d_rot);
    r.cos = a.cos, r.sin = a.sin;
    r.cs_stride = a.cs_stride;
    r.pos_offset = a.pos_offset;
    r.half = a.half;
    r.row = (uint32_t)(d_rot + kVec - 1) & ~(uint32_t)(kVec - 1);
    r.wave_floats = positions * 2 * r.row;
    if (r.wave_floats > 2048) return false;  // 32 KiB a block: heads of few bytes per position touch many positions
    if constexpr (std::is_same<CS, Angles>::value) {
        uint32_t evaluated = 0;  // positions whose angles a wave evaluates: one where every position is whole waves
        for (int i = 0; i < a.nt; ++i) {
            const uint32_t per_pos = (uint32_t)a.t[i].n_inner * spv;
            const uint32_t p = per_pos % kRunSlots == 0 ? 1u : kRunSlots % per_pos == 0 ? kRunSlots / per_pos : positions;
            if (p > evaluated) evaluated = p;
        }
        if (!angles_in_runs(a, w, (int)((evaluated * (uint32_t)d_rot + kWave - 1) / kWave))) return false;
    }
    if constexpr (std::is_same<CS, Angles>::value) {
        if (a.half % 8 == 0) {
            *err = launch_rope_run<T, CS, 8, BWD>(r, a.nt, st);
            return true;
        }
    }
    if (a.half % 4 == 0) *err = launch_rope_run<T, CS, 4, BWD>(r, a.nt, st);
    else *err = launch_rope_run<T, CS, 2, BWD>(r, a.nt, st);
    return true;
}

// q and k in place in a fused projection whose parts tile 4 KiB pieces: the cell kernel (see rope_cell_kernel).
// Returns false if the call does not qualify.
template <typename T, typename CS, bool BWD>
static bool try_launch_rope_cell(const RopeArgs& a, int s, int n_outer, int w, hipStream_t st, hipError_t* err) {
    if (std::is_same<CS, Angles>::value || n_outer != 1 || a.nt != 2 || w != kVec || a.copy_dims != 0) return false;
    const RopeTensor &q = a.t[0], &k = a.t[1];
    const int64_t cell = q.in_stride[2], hn = cell / 3;
    // Parts of one cache line, or of two that are rotated whole: the lanes of this kernel pass over what does not
    // move.  us per launch, rope_span_kernel -> this: bf16 [8192,1,32,3*128] d_rot 128 52.5 -> 47.1, [2048,4,32,3*128]
    // 53.3 -> 45.7, fp16 [2048,4,16,3*64] d_rot 64 14.7 -> 13.5, d_rot 16 12.8 -> 11.9; against it: bf16 [8192,1,32,3*128]
    // d_rot 64 27.4 -> 35.6, fp16 [2048,2,16,3*256] d_rot 256 25.1 -> 25.7, d_rot 64 9.7 -> 16.9.
    const bool pays = hn == 64 || (hn == 128 && a.half == 64);
    if (cell % 3 != 0 || !pays || k.in != q.in + hn * 2 || k.n_inner != q.n_inner) return false;
    for (const RopeTensor* t : {&q, &k}) {
        if (t->in != t->out || t->in_stride[2] != cell || t->out_stride[2] != cell) return false;
        if (t->in_stride[0] != t->n_inner * cell || t->out_stride[0] != t->in_stride[0]) return false;
    }
    const int64_t per_pos = q.n_inner * cell / kVec;
    if (reinterpret_cast<uintptr_t>(q.in) % 4096 != 0 || per_pos % kRunSlots != 0 || per_pos * s > 0x7fffffffLL) return false;
    if ((a.lpv * 2 + a.pad_slots) * kVec > hn) return false;
    RopeCellArgs r{};
    r.mixed = q.out;
    r.cos = a.cos, r.sin = a.sin;
    r.cs_stride = a.cs_stride;
    r.pos_offset = a.pos_offset;
    r.slots = (uint32_t)(per_pos * s);
    r.by_pos = FastDiv::by((uint32_t)per_pos);
    r.by_part = FastDiv::by((uint32_t)(hn / kVec));
    r.lps = a.lpv * 2;
    r.moved = a.lpv * 2 + a.pad_slots;
    hipLaunchKernelGGL((rope_cell_kernel<T, CS, BWD>), dim3((r.slots / kRunSlots + 3) / 4), dim3(256), 0, st, r);
    *err = hipGetLastError();
    return true;
}

template <typename T, typename CS, bool BWD>
static hipError_t launch_rope_w(const RopeArgs& a, int s, int n_outer, int w, hipStream_t st) {
    if (span_shape(a, w)) {
        switch (w) {
            case 8: return launch_rope_span<T, CS, 8, BWD>(a, s, n_outer, st);
            case 4: return launch_rope_span<T, CS, 4, BWD>(a, s, n_outer, st);
            default: return launch_rope_span<T, CS, 2, BWD>(a, s, n_outer, st);
        }
    }
    switch (w) {
        case 8: return launch_rope_shape<T, CS, 8, BWD>(a, s, n_outer, st);
        case 4: return launch_rope_shape<T, CS, 4, BWD>(a, s, n_outer, st);
        case 2: return launch_rope_shape<T, CS, 2, BWD>(a, s, n_outer, st);
        case 1: return launch_rope_shape<T, CS, 1, BWD>(a, s, n_outer, st);
        default: return hipErrorInvalidValue;
    }
}

template <typename T, typename CS>
static hipError_t launch_rope_dir(const RopeArgs& a, int s, int n_outer, int w, bool backward,
                                  hipStream_t st) {
    hipError_t err = hipSuccess;
    if (backward ? try_launch_rope_run<T, CS, true>(a, s, n_outer, w, st, &err)
                 : try_launch_rope_run<T, CS, false>(a, s, n_outer, w, st, &err)) return err;
    if constexpr (!std::is_same<CS, Angles>::value) {
        if (backward ? try_launch_rope_cell<T, CS, true>(a, s, n_outer, w, st, &err)
                     : try_launch_rope_cell<T, CS, false>(a, s, n_outer, w, st, &err)) return err;
    }
    return backward ? launch_rope_w<T, CS, true>(a, s, n_outer, w, st)
                    : launch_rope_w<T, CS, false>(a, s, n_outer, w, st);
}

hipError_t launch_rope(const RopeArgs& a, int s, int n_outer, int w, int dtype, int cs_dtype,
                       bool backward, hipStream_t stream) {
    if (cs_dtype == kRopeAngles) {
        return dtype == NEOX_F16 ? launch_rope_dir<F16, Angles>(a, s, n_outer, w, backward, stream)
                                 : launch_rope_dir<BF16, Angles>(a, s, n_outer, w, backward, stream);
    }
    const bool cs32 = (cs_dtype == NEOX_F32);
    if (dtype == NEOX_F16) {
        return cs32 ? launch_rope_dir<F16, float>(a, s, n_outer, w, backward, stream)
                    : launch_rope_dir<F16, F16>(a, s, n_outer, w, backward, stream);
    }
    return cs32 ? launch_rope_dir<BF16, float>(a, s, n_outer, w, backward, stream)
                : launch_rope_dir<BF16, BF16>(a, s, n_outer, w, backward, stream);
}

}  // namespace neox
