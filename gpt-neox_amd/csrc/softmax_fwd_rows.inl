// The forward pass of a wave's rows row0 .. row0 + rows_here - 1: the statements of softmax_fwd_rows and, once
// more, of softmax_fwd_packed_kernel itself.  Not a function for both: the compiler simplifies a function before
// it inlines it, and the kernels then come out different, some with half of their loads behind the first row's
// arithmetic.  Given: T, G, MASK, FLAGS, R, C, Sink; a, lane, row0, rows_here, stage, stage2.  Leaves `summed`.
    static_assert(C == 1 || G == kWave, "several chunks per row need a whole wave per row");
    constexpr int RPP = Packed<G, R>::kRowsPerPass;
    constexpr bool kLdNt = (FLAGS & kNtLoad) != 0, kStNt = (FLAGS & kNtStore) != 0;
    constexpr bool kRag = (FLAGS & kRagged) != 0;
    static_assert(!kRag || C == 1, "ragged rows: one chunk per lane group");
    const int sk = a.sk;
    const int grp = lane / G;
    const int back = ragged_back<kRag>((lane % G) * kVec, sk);  // kRagged: see ragged_back
    const int col0 = (lane % G) * kVec - back;                  // first column of the lane's accesses
    DropoutArgs drop = a.drop;
    if constexpr ((FLAGS & kDropout) != 0) drop = resolve(drop);
    const float ninf = -__builtin_inff();

    const rsrc_t rx = make_rsrc(static_cast<const char*>(a.in0) + (size_t)row0 * sk * 2, rows_here * sk * 2);
    const Sink out = Sink::at(a.out, (size_t)row0 * sk * 2, rows_here * sk * 2, stage);
    const rsrc_t rm = make_rsrc(a.mask, a.mask_bytes);
    Sink out2 = out;
    if constexpr ((FLAGS & kDropout) != 0) out2 = Sink::at(a.out2, (size_t)row0 * sk * 2, rows_here * sk * 2, stage2);
    const rsrc_t rb = make_rsrc(a.bias, a.bias_bytes);  // kBias: the whole bias tensor

    bool summed = true;
    u32x4 raw[R][C];
    u32x4 rawb[R][C];
    u32x2 mk[R][C];
    int len[R];
    int ipos[R];       // row position inside its matrix (ALiBi)
    float slope2[R];   // slope[head] * scale of the lane's row (ALiBi)
    const uint32_t i0 = a.by_sq.mod(row0);  // wave-uniform
#pragma unroll
    for (int p = 0; p < R; ++p) {
        const uint32_t lr = p * RPP + grp;  // row of this lane group inside the wave
        const uint32_t row = row0 + lr;
        const uint32_t i = wrap_row(i0 + lr, a.by_sq);
        len[p] = (MASK == Mask::Causal) ? min((int)i + 1, sk) : sk;
        if (lr >= rows_here) len[p] = 0;
        ipos[p] = alibi_row_position<MASK>(i, a);
        slope2[p] = 0.f;
        if constexpr ((FLAGS & kAlibi) != 0) {
            const uint32_t safe_row = lr < rows_here ? row : row0;
            slope2[p] = a.slopes[a.by_np.mod(a.by_sq.div(safe_row))] * a.scale;
        }
        if constexpr (MASK == Mask::Bytes) {
#pragma unroll
            for (int c = 0; c < C; ++c) {
                const int col = col0 + c * kChunk;
                const uint32_t mb = a.mask_bcast ? 0u : a.by_mask_batch.div(row);
                const uint32_t moff = (mb * (uint32_t)a.sq + i) * sk + col;
                mk[p][c] = packed_ld_mask(rm, moff, col < len[p]);
            }
        }
    }
    // the scores (and the bias) after the mask bytes: a lane whose 8 keys are all hidden fetches neither
#pragma unroll
    for (int p = 0; p < R; ++p) {
        const uint32_t lr = p * RPP + grp;
#pragma unroll
        for (int c = 0; c < C; ++c) {
            const int col = col0 + c * kChunk;
            bool active = col < len[p];
            // (SoftmaxArgs::row_end is not looked at here: it spared nothing more and cost a load per row)
            if constexpr (MASK == Mask::Bytes && kSkipHidden && !kRag) active = active && !all_hidden(mk[p][c]);
            raw[p][c] = packed_ld<kLdNt>(rx, (lr * sk + col) * 2u, active);
            if constexpr ((FLAGS & kBias) != 0) {
                const uint32_t boff = (bias_row(row0 + lr, a) * (uint32_t)sk + col) * 2u;
                rawb[p][c] = packed_ld<false>(rb, boff, active);
            }
        }
    }

#pragma unroll
    for (int p = 0; p < R; ++p) {
        float v[C][8];
        float mx = ninf;
#pragma unroll
        for (int c = 0; c < C; ++c) {
            const int col = col0 + c * kChunk;
            unpack8<T>(raw[p][c], v[c]);
            if constexpr ((FLAGS & kBias) != 0) {
                float bv[8];
                unpack8<T>(rawb[p][c], bv);
#pragma unroll
                for (int k = 0; k < 8; ++k) v[c][k] += bv[k];
            }
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                bool keep = (col + k) < len[p];
                if constexpr (MASK == Mask::Bytes) {
                    const uint32_t w = (k < 4) ? mk[p][c].x : mk[p][c].y;
                    keep = keep && (((w >> (8 * (k & 3))) & 0xffu) == 0);
                }
                float bias = 0.f;
                if constexpr ((FLAGS & kAlibi) != 0) bias = slope2[p] * alibi_distance<MASK>(col + k, ipos[p]);
                v[c][k] = keep ? fmaf(v[c][k], a.scale, bias) : ninf;
                mx = fmaxf(mx, v[c][k]);
            }
        }
        mx = group_reduce<OpMax, G>(mx);
        float sum = 0.f;
#pragma unroll
        for (int c = 0; c < C; ++c)
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                v[c][k] = fast_exp2(v[c][k] - mx);
                sum += (kRag && k < back) ? 0.f : v[c][k];  // columns the lane before counts
            }
        if constexpr (MASK == Mask::Bytes) {
            // rows with every key hidden (rare): uniform over the sk columns
            const bool all_masked = (mx == ninf) && len[p] > 0;
            if (__builtin_amdgcn_ballot_w64(all_masked) != 0) {
                if (all_masked) {
                    sum = 0.f;
#pragma unroll
                    for (int c = 0; c < C; ++c)
#pragma unroll
                        for (int k = 0; k < 8; ++k) {
                            v[c][k] = ((col0 + c * kChunk + k) < len[p]) ? 1.f : 0.f;
                            sum += (kRag && k < back) ? 0.f : v[c][k];
                        }
                }
            }
        }
        sum = group_reduce<OpSum, G>(sum);
        const float inv = 1.0f / sum;
        const uint32_t lr = p * RPP + grp;
        if constexpr (!std::is_same<Sink, DirectSink>::value) summed = summed && (lr >= rows_here || sum == sum);
#pragma unroll
        for (int c = 0; c < C; ++c) {
            const int col = col0 + c * kChunk;
#pragma unroll
            for (int k = 0; k < 8; ++k) v[c][k] *= inv;  // lanes of absent rows hold NaN and store nothing
            const bool st = lr < rows_here && col < sk;
            const u32x4 o = pack8<T>(v[c]);
            out.template put<kStNt>(o, (lr * sk + col) * 2u, st);
            if constexpr ((FLAGS & kDropout) != 0) {
                const uint32_t bits = keep_bits_row8<kRag>(drop, row0 + lr, sk, col);
                out2.template put<kStNt>(dropout8<T>(o, bits, drop.scale), (lr * sk + col) * 2u, st);
            }
        }
    }
