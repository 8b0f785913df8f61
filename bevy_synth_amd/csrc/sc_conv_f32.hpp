// f32 tile of the submanifold conv and the dense linear.  Included by
// sc_conv_kernels.hpp.
#pragma once

// Tile = 32 kB query rows x 32 kB output channels of one group, 4 waves in 2
// x 2, each kB x kB blocks of v_mfma_f32_16x16x4_f32 (transposed product:
// lane (l16, q4) ends with channels 4 q4 + e of row l16 of each block).  A
// slice is 64 bytes (16 channels) of the rows at one used offset; the tile
// walks them offset by offset, channels ascending, one FMA chain per value.
// Rows and weights [Cout][K][Cin] are DMA'd into a ring of kBuf LDS stages of
// kSl slices, kBuf - 1 stages ahead, 4 lanes to a row's 64 bytes (loads
// straight into the operand layout, 16 bytes a lane from 16 rows, ran at a
// quarter of the rate and left the kernel bound by the load path), absent
// neighbours, rows and channels past the end reading zero; one barrier a
// stage.  Operand reads are XOR-swizzled per row (wslot).
//
// Bound: the matrix cores (128 kB^2 cycles a slice and wave, 16 to 64 B/clk
// of LDS), so the tile is as small as fills the chip (f32_tile).  27 offsets,
// against a 256 x 128 tile that gathered its rows into registers:
//   rows      64 -> 64 channels     128 -> 128
//   600       230 -> 18.5 us        440 -> 33.5 us
//   14,648    233 -> 38.9           449 -> 124
//   120,000   428 -> 228            837 -> 825
// (7.3 TFLOP/s of the 64-channel conv of 14,648 rows before, 43 after; the
// largest 101, of 155 that a large f32 matrix product reaches here, 27
// offsets computed for 21.6 neighbours).
template <int kB>
struct F32Tile {
    static constexpr int kRows = 32 * kB, kCols = 32 * kB;
    static constexpr int kSl = kB == 1 ? 2 : 1;                // slices per stage
    static constexpr int kBuf = kB == 4 ? 3 : 4;               // stages in the ring
    static constexpr int kSlice = (kRows + kCols) * 64;        // bytes
    static constexpr int kStage = kSl * kSlice;
    static constexpr int kPer = kStage / 4096;                 // 1 KB DMA instructions per wave and stage
    static constexpr int kWgs = kB == 1 ? 4 : (kB == 2 ? 3 : 2);  // workgroups per CU
};

template <typename TO, int kB>
__global__ __launch_bounds__(kThreads, F32Tile<kB>::kWgs) void conv_f32_kernel(ConvArgs args)
{
    using T = F32Tile<kB>;
    constexpr int kRows = T::kRows, kBuf = T::kBuf, kPer = T::kPer;
    constexpr int kQ = kThreads / kRows;        // threads per row in the prologue
    constexpr int kEnt = kMaxTableK / kQ;       // map entries per thread
    __shared__ __attribute__((aligned(16))) unsigned char s_buf[kBuf * T::kStage];
    __shared__ uint32_t s_off[kMaxTableK][kRows];  // byte offset of the neighbour's input row
    __shared__ uint32_t s_mask;
    __shared__ float s_red[2][kRows];

    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int l16 = lane & 15, q4 = lane >> 4;
    const int wr = wave >> 1, wc = wave & 1;
    const int wave_u = __builtin_amdgcn_readfirstlane(wave);
    const int K = args.K;

    const int64_t row0 = (int64_t)tile_for_block(blockIdx.x, gridDim.x) * kRows;
    const int o0 = blockIdx.y * T::kCols;  // within the group
    const int g = blockIdx.z;
    const int64_t in_col0 = (int64_t)g * args.cin_g;
    const int64_t out_col0 = (int64_t)g * args.cout_g;
    const uint32_t row_bytes = (uint32_t)(args.cin * 4);

    // ---- prologue: neighbour offsets of the tile's rows, offsets in use
    if (tid == 0) s_mask = 0u;
    __syncthreads();
    {
        const int r = tid % kRows, kq = tid / kRows;
        const int64_t q = row0 + r;
        uint32_t m = 0;
        int32_t v[kEnt];
#pragma unroll
        for (int u = 0; u < kEnt; ++u) {
            const int k = kq + kQ * u;
            v[u] = -1;
            if (q < args.n_q && k < K) v[u] = args.map ? args.map[q * K + k] : (int32_t)q;  // no map: dense linear
        }
#pragma unroll
        for (int u = 0; u < kEnt; ++u) {
            const int k = kq + kQ * u;
            const bool ok = v[u] >= 0 && v[u] < args.n_in;
            if (k < K) s_off[k][r] = ok ? (uint32_t)v[u] * row_bytes : kOobOffset;
            m |= ok ? 1u << k : 0u;
        }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) m |= __shfl_xor(m, off, 64);
        if (lane == 0 && m) atomicOr(&s_mask, m);
    }
    __syncthreads();
    const uint32_t mask = __builtin_amdgcn_readfirstlane(s_mask);

    f32x4 acc[kB][kB];
#pragma unroll
    for (int i = 0; i < kB; ++i)
#pragma unroll
        for (int j = 0; j < kB; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    const int nkc = args.cin_g / 16;
    const int S = __builtin_popcount(mask) * nkc;    // slices
    const int n_st = (S + T::kSl - 1) / T::kSl;      // stages
    if (n_st > 0) {
        const i32x4_rsrc a_rsrc = rsrc_words(static_cast<const float *>(args.input) + in_col0,
                                             (uint32_t)(args.n_in * row_bytes - in_col0 * 4));
        const i32x4_rsrc w_rsrc =
            rsrc_words(args.weight, (uint32_t)(args.cout * (int64_t)K * args.cin_g * 4));
        const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)s_buf;
        // DMA instruction t of this wave fills LDS bytes [1 KB * (wave + 4 t),
        // +1 KB) of a stage: in each slice 2 kB instructions of rows, then 2
        // kB of channels, 16 of them an instruction; lane L moves, for row
        // (channel) L / 4, the 16-byte piece that slot L % 4 holds.
        int src[kPer];       // tile row, or byte offset of the channel's weights
#pragma unroll
        for (int t = 0; t < kPer; ++t) {
            const int in = (wave + 4 * t) % (4 * kB), n = 16 * (in % (2 * kB)) + (lane >> 2);
            const int o = o0 + n;
            src[t] = in < 2 * kB ? n
                                 : (int)(o < args.cout_g ? (uint32_t)((out_col0 + o) * (int64_t)K * args.cin_g * 4)
                                                         : kOobOffset);
        }
        const uint32_t piece = (uint32_t)wslot<64>(lane >> 2, lane & 3) * 16u;  // (16 n' + m)'s slot is m's
        uint32_t rem = mask;  // the next slice to load: its offset (lowest bit) and channel chunk
        int c = 0, left = S;
        auto dma = [&](int buf) {
            int k[T::kSl], cc[T::kSl];
            bool live[T::kSl];
#pragma unroll
            for (int s = 0; s < T::kSl; ++s) {
                live[s] = left > 0;
                k[s] = live[s] ? __builtin_ctz(rem) : 0;
                cc[s] = c;
                --left;
                if (++c == nkc) {
                    c = 0;
                    rem &= rem - 1u;
                }
            }
#pragma unroll
            for (int t = 0; t < kPer; ++t) {
                const int in = wave_u + 4 * t, s = kB == 1 ? t : 0;
                const bool is_row = kB == 1 ? wave_u < 2 : t < kPer / 2;  // uniform
                const uint32_t step = (uint32_t)cc[s] * 64u + piece;
                const uint32_t lds = lds0 + (uint32_t)(buf * T::kStage) + 1024u * (uint32_t)in;
                if (is_row) {
                    const uint32_t off = s_off[k[s]][src[t]];
                    lds_dma16(a_rsrc, live[s] ? off + step : kOobOffset, lds);
                } else {
                    lds_dma16(w_rsrc, live[s] ? (uint32_t)src[t] + (uint32_t)k[s] * (uint32_t)(args.cin_g * 4) + step
                                              : kOobOffset, lds);
                }
            }
        };
        // fragment offsets in a slice (blocks 1 KB apart; opaque, so that each
        // address is one of these plus a constant)
        int xoff = 16 * kB * wr * 64 + l16 * 64 + wslot<64>(l16, q4) * 16;
        int woff = kRows * 64 + 16 * kB * wc * 64 + l16 * 64 + wslot<64>(l16, q4) * 16;
        asm("" : "+v"(xoff));
        asm("" : "+v"(woff));
        auto step = [&](int u, int t) {
            uint4 x[T::kSl][kB], w[T::kSl][kB];
#pragma unroll
            for (int s = 0; s < T::kSl; ++s) {
                const unsigned char *base = s_buf + u * T::kStage + s * T::kSlice;
#pragma unroll
                for (int i = 0; i < kB; ++i) x[s][i] = *reinterpret_cast<const uint4 *>(base + xoff + 1024 * i);
#pragma unroll
                for (int j = 0; j < kB; ++j) w[s][j] = *reinterpret_cast<const uint4 *>(base + woff + 1024 * j);
            }
            __builtin_amdgcn_sched_barrier(0);
            if (t + kBuf - 1 < n_st) dma((u + kBuf - 1) % kBuf);
            __builtin_amdgcn_sched_barrier(0);
            // lane q4 holds channels 4 q4 .. 4 q4 + 3 of both operands:
            // element e of all four lanes is one MFMA's reduction
#pragma unroll
            for (int s = 0; s < T::kSl; ++s)
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int j = 0; j < kB; ++j)
#pragma unroll
                        for (int i = 0; i < kB; ++i) {
                            const uint32_t wv[4] = {w[s][j].x, w[s][j].y, w[s][j].z, w[s][j].w};
                            const uint32_t xv[4] = {x[s][i].x, x[s][i].y, x[s][i].z, x[s][i].w};
                            acc[i][j] =
                                __builtin_amdgcn_mfma_f32_16x16x4f32(u2f(wv[e]), u2f(xv[e]), acc[i][j], 0, 0, 0);
                        }
        };
        // Stage t uses buffer t % kBuf; at its top, stages t .. min(t + kBuf -
        // 2, n_st - 1) are in flight (in order; no other vector memory
        // operation is): wait until only the younger ones are, then the
        // barrier (every wave's share of t has landed, and every wave is done
        // with t - 1's buffer, which the stage's DMA refills).  Reading the
        // next stage's operands a stage ahead measured 2-3 % slower.
        auto sync = [&]() {
            __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
            __builtin_amdgcn_s_barrier();
        };
#pragma unroll
        for (int t = 0; t < kBuf - 1; ++t)
            if (t < n_st) dma(t);
        int t0 = 0;
        for (; t0 + 2 * kBuf - 2 <= n_st; t0 += kBuf) {
#pragma unroll
            for (int u = 0; u < kBuf; ++u) {
                wait_vmcnt<(kBuf - 2) * kPer>();
                sync();
                step(u, t0 + u);
            }
        }
#pragma unroll
        for (int u = 0; u < 2 * kBuf - 2; ++u) {
            const int t = t0 + u;
            if (t >= n_st) break;
            const int younger = min(kBuf - 2, n_st - 1 - t);
            if (younger >= 2)
                wait_vmcnt<2 * kPer>();
            else if (younger == 1)
                wait_vmcnt<kPer>();
            else
                wait_vmcnt<0>();
            sync();
            step(u % kBuf, t);
        }
    }

    // ---- epilogue: bias -> LayerNorm over the row -> SiLU -> + residual (or
    //      the C2S forms); lane l holds channels oc0 + 16 j + 4 q4 + e of tile
    //      row trow + 16 i.
    TO *__restrict__ out = static_cast<TO *>(args.out);
    const TO *__restrict__ res = static_cast<const TO *>(args.residual);
    const bool vec_ok = args.vec_out != 0;
    const int oc0 = o0 + 16 * kB * wc, trow = 16 * kB * wr + l16;
#pragma unroll
    for (int j = 0; j < kB; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int o = oc0 + j * 16 + 4 * q4 + e;
            const bool ok = o < args.cout_g;
            const float bias = (args.bias && ok) ? args.bias[out_col0 + o] : 0.f;
#pragma unroll
            for (int i = 0; i < kB; ++i) acc[i][j][e] = ok ? acc[i][j][e] + bias : 0.f;
        }
    if (args.ln) {
        // two-pass f32 statistics over the row's channels, all of them in the
        // tile (the host's choice): the two column waves meet in LDS
        const float inv_c = 1.0f / (float)args.cout_g;
        float part[kB], mean[kB];
        auto row_total = [&]() {
#pragma unroll
            for (int i = 0; i < kB; ++i) {
                part[i] += __shfl_xor(part[i], 16, 64);
                part[i] += __shfl_xor(part[i], 32, 64);
            }
            __syncthreads();
#pragma unroll
            for (int i = 0; i < kB; ++i)
                if (q4 == 0) s_red[wc][trow + 16 * i] = part[i];
            __syncthreads();
#pragma unroll
            for (int i = 0; i < kB; ++i) part[i] = s_red[0][trow + 16 * i] + s_red[1][trow + 16 * i];
        };
#pragma unroll
        for (int i = 0; i < kB; ++i) {
            part[i] = 0.f;
#pragma unroll
            for (int j = 0; j < kB; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e) part[i] += acc[i][j][e];
        }
        row_total();
#pragma unroll
        for (int i = 0; i < kB; ++i) {
            mean[i] = part[i] * inv_c;
            part[i] = 0.f;
#pragma unroll
            for (int j = 0; j < kB; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float d = acc[i][j][e] - mean[i];
                    part[i] += oc0 + j * 16 + 4 * q4 + e < args.cout_g ? d * d : 0.f;
                }
        }
        row_total();
#pragma unroll
        for (int j = 0; j < kB; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int o = oc0 + j * 16 + 4 * q4 + e;
                const bool ok = o < args.cout_g;
                const float lw = (args.ln_w && ok) ? args.ln_w[o] : 1.f;
                const float lb = (args.ln_b && ok) ? args.ln_b[o] : 0.f;
#pragma unroll
                for (int i = 0; i < kB; ++i)
                    acc[i][j][e] = (acc[i][j][e] - mean[i]) * rsqrt_f32(part[i] * inv_c + args.ln_eps) * lw + lb;
            }
    }
#pragma unroll
    for (int i = 0; i < kB; ++i) {
        const int64_t qrow = row0 + trow + 16 * i;
        if (qrow >= args.n_q) continue;
        const int64_t rowbase = qrow * args.cout + out_col0;
        const bool c2s = args.scatter_rows || args.skip_idx;
        const C2SRow crow = c2s ? c2s_row<TO>(args, qrow) : C2SRow{nullptr};
#pragma unroll
        for (int j = 0; j < kB; ++j) {
            const int oc = oc0 + j * 16 + 4 * q4;
            if (oc >= args.cout_g) continue;
            float v[4] = {acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]};
            if (args.silu) {
#pragma unroll
                for (int cc = 0; cc < 4; ++cc) v[cc] = silu_f32(v[cc]);
            }
            if (c2s) {
                c2s_store4<TO>(args, crow, qrow, (int)(out_col0 + oc), min(4, args.cout_g - oc), v, vec_ok);
            } else if (vec_ok && oc + 3 < args.cout_g) {
                if (res) {
                    float r4[4];
                    Out4<TO>::unpack(*reinterpret_cast<const typename Out4<TO>::V *>(res + rowbase + oc), r4);
#pragma unroll
                    for (int cc = 0; cc < 4; ++cc) v[cc] += r4[cc];
                }
                *reinterpret_cast<typename Out4<TO>::V *>(out + rowbase + oc) = Out4<TO>::pack(v);
            } else {
#pragma unroll
                for (int cc = 0; cc < 4; ++cc) {
                    if (oc + cc >= args.cout_g) continue;
                    float z = v[cc];
                    if (res) z += load_as_f32<TO>(res, rowbase + oc + cc);
                    store_from_f32<TO>(out, rowbase + oc + cc, z);
                }
            }
        }
    }
}

template <typename TO>
int launch_f32(const ConvArgs &a, int groups, hipStream_t s)
{
    int kB = f32_tile(a.n_q, a.cout_g, groups);
    if (a.ln || a.in_place) kB = std::max(kB, f32_row_tile(a.cout_g));
    while (kB < 4 && (a.cout_g + 32 * kB - 1) / (32 * kB) > 65535) kB *= 2;
    const int64_t gx = (a.n_q + 32 * kB - 1) / (32 * kB), gy = (a.cout_g + 32 * kB - 1) / (32 * kB);
    if (gx > INT32_MAX || gy > 65535 || groups > 65535) return fail(SC_ERR_OVERFLOW, "sparse conv grid overflow");
    const dim3 grid((unsigned)gx, (unsigned)gy, (unsigned)groups);
    if (kB == 1)
        conv_f32_kernel<TO, 1><<<grid, kThreads, 0, s>>>(a);
    else if (kB == 2)
        conv_f32_kernel<TO, 2><<<grid, kThreads, 0, s>>>(a);
    else
        conv_f32_kernel<TO, 4><<<grid, kThreads, 0, s>>>(a);
    SC_LAUNCH_CHECK("conv_f32_kernel launch");
    return SC_OK;
}
