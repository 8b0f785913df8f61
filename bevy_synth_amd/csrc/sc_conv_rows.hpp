// Row-block tile of the submanifold conv and the dense linear: small tiles
// whose operands go straight from global memory to registers.  Included by
// sc_conv_kernels.hpp.
#pragma once

// 16-bit calls whose 256-row tiles would leave most of the chip idle run here
// (rows_cut).
//
// A wave owns 16 kI rows x 64 output channels as kI x 4 blocks of
// v_mfma_f32_16x16x32 (transposed product: lane (l16, q4) holds channels 16 j
// + 4 q4 + e of row 16 i + l16).  A stage is one 64-byte slice (32 channels)
// of the input rows at one offset; its operands (kI row slices, 4 weight
// fragments, one 16-byte load per lane each) are loaded kDepth - 1 stages
// ahead straight into registers: LDS holds only the rows' neighbour offsets.
// kSplit waves of the workgroup share a block, wave s taking offset k of chunk
// c when (k + c) % kSplit == s, and add their partial sums through LDS: a
// 27-offset conv of 64 channels is 54 stages, which one wave would run one
// after the other.  The other waves take the 64-channel columns of the
// kNT-channel tile, then row blocks.  A wave walks only the offsets that its
// own rows use; the deal goes by the offset itself and not by its place in
// that list, so that a row's value does not depend on which rows share its
// block.
//
// Bound, measured: the load path, 16 bytes a lane from 16 different rows
// taking 64 cycles a fragment (packed weights, whole lines per 4 lanes, 16),
// so a workgroup moves 16-30 B/clk whatever the prefetch depth (4 or 6
// stages: the same).  Hence many small workgroups while the chip is not full,
// and tiles that share operands once it is.  bf16, 64 -> 64 channels, 27
// offsets, against the 256-row tiles:
//   rows      without a plan      with a plan
//   600       43.9 -> 11.8 us     22.7 ->  8.5 us
//   14,648    47.4 -> 17.7        23.8 -> 13.9
//   30,000    47.8 -> 29.9        24.4 -> 21.9
template <int kI, int kNT, int kSplit>
struct RowsTile {
    static constexpr int kColWaves = kNT / 64;
    static constexpr int kRowWaves = 4 / (kColWaves * kSplit);
    static constexpr int kRows = 16 * kI * kRowWaves;
    static constexpr int kDepth = kI == 1 ? 6 : (kI == 2 ? 4 : 3);  // operand sets: stages t .. t + kDepth - 1
    static constexpr int kE = kI >= kSplit ? kI / kSplit : 1;       // row blocks per wave in the epilogue
};

// args.wpack set: packed weights (16-bit activations; int8 weights are widened
// there, TW = uint16_t), else the reference layout; args.perm set: tile rows from a child plan's lists; args.plan_hdr
// set: a planned call, whose plan (and packed weights) must match it.
template <typename TA, typename TW, typename TO, int kI, int kNT, int kSplit>
__global__ __launch_bounds__(kThreads, kI == 1 ? 3 : 2) void conv_rows_kernel(ConvArgs args)
{
    using T = RowsTile<kI, kNT, kSplit>;
    constexpr int kRows = T::kRows, kDepth = T::kDepth, kE = T::kE;
    constexpr int kEl = 64 / (int)sizeof(TA);       // reduction elements per stage
    constexpr bool kI8 = sizeof(TW) == 1;
    constexpr int kWPiece = kI8 ? 8 : 16;           // weight bytes per lane and fragment
    constexpr int kQ = kRows >= kThreads ? 1 : kThreads / kRows;  // threads per row in the prologue
    constexpr int kPer = kMaxTableK / kQ;           // map entries per thread
    __shared__ uint32_t s_off[kMaxTableK][kRows];   // byte offset of the neighbour's input row
    __shared__ uint32_t s_mask[kRows / 16];
    __shared__ int32_t s_row[kRows];
    __shared__ float s_red[2][kRows];
    // partial sums of the waves that share a block (kSplit > 1)
    __shared__ f32x4 s_part[kSplit > 1 ? 4 : 1][kSplit > 1 ? kI * 4 * 64 : 1];

    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int l16 = lane & 15, q4 = lane >> 4;
    const int sp = __builtin_amdgcn_readfirstlane(wave) % kSplit;  // the wave's share of the stages
    const int ch = wave / kSplit % T::kColWaves;    // its 64 channels
    const int rw = wave / (kSplit * T::kColWaves);  // and its row blocks
    const int trow = 16 * kI * rw;                  // first tile row of the wave
    const int K = args.K;

    // ---- which rows and channels
    int64_t row0 = (int64_t)tile_for_block(blockIdx.x, gridDim.x) * kRows;
    int o0 = blockIdx.y * kNT;
    if (args.plan_hdr) {
        const PlanHeader *h = args.plan_hdr;
        bool w_ok = true;
        if (args.wpack) {
            const PackHeader *wh = static_cast<const PackHeader *>(args.wpack);
            w_ok = wh->magic == kPackMagic && wh->groups == (int)gridDim.z && wh->cout_g == args.cout_g &&
                   wh->cin_g == args.cin_g && wh->K == K && (wh->src_dtype == SC_DTYPE_F16) == __is_same(TA, _Float16);
        }
        const bool plan_ok = plan_matches(h, args);
        if (!plan_ok || !w_ok) {
            flag_plan_status(h, (plan_ok ? 0u : kPlanStatusMapMismatch) | (w_ok ? 0u : kPlanStatusWeightMismatch));
            return;
        }
        if (h->status != 0u) return;
        if (args.tile_child) {
            // the list tiles in use, then the spares, kRows rows at a time
            // (the grid covers the layout's bound)
            constexpr int kSub = kPlanTileRows / kRows;
            const int n_used = h->n_unique, n_real = (n_used + h->n_extras) * kSub;
            if ((int)blockIdx.x >= n_real) return;
            const int b = tile_for_block(blockIdx.x, n_real), lt = b / kSub;
            const int tile = lt < n_used ? lt : h->list_tiles + (lt - n_used);
            const int child = args.tile_child[tile];
            if (child < 0) return;
            o0 += child * args.child_ch;
            row0 = (int64_t)tile * kPlanTileRows + (b % kSub) * kRows;
        }
    }
    const int g = blockIdx.z;
    const int64_t in_col0 = (int64_t)g * args.cin_g;
    const int64_t out_col0 = (int64_t)g * args.cout_g;
    const uint32_t row_bytes = (uint32_t)(args.cin * (int64_t)sizeof(TA));

    // ---- prologue: the rows' neighbour offsets and each 16-row block's mask
    if (tid < kRows / 16) s_mask[tid] = 0u;
    __syncthreads();
    bool any;
    {
        const int r = tid % kRows, kq = tid / kRows;
        int64_t q = row0 + r;
        if (args.perm) {
            const int32_t p = args.perm[q];
            q = p >= 0 && p < args.n_q ? p : -1;
        } else if (q >= args.n_q) {
            q = -1;
        }
        uint32_t m = 0;
        int32_t v[kPer];
#pragma unroll
        for (int u = 0; u < kPer; ++u) {
            const int k = kq + kQ * u;
            v[u] = -1;
            if (q >= 0 && k < K) v[u] = args.map ? args.map[q * K + k] : (int32_t)q;  // no map: the dense linear
        }
#pragma unroll
        for (int u = 0; u < kPer; ++u) {
            const int k = kq + kQ * u;
            const bool ok = v[u] >= 0 && v[u] < args.n_in;
            if (k < K) s_off[k][r] = ok ? (uint32_t)v[u] * row_bytes : kOobOffset;
            m |= ok ? 1u << k : 0u;
        }
        if (kq == 0) s_row[r] = (int32_t)q;
        m |= __shfl_xor(m, 1, 64);
        m |= __shfl_xor(m, 2, 64);
        m |= __shfl_xor(m, 4, 64);
        m |= __shfl_xor(m, 8, 64);
        if (l16 == 0 && m) atomicOr(&s_mask[r >> 4], m);
        any = __syncthreads_or(q >= 0) != 0;
    }
    if (!any) return;  // a list tile's padding
    uint32_t wmask = 0;
#pragma unroll
    for (int i = 0; i < kI; ++i) wmask |= s_mask[kI * rw + i];
    wmask = __builtin_amdgcn_readfirstlane(wmask);

    f32x4 acc[kI][4];
#pragma unroll
    for (int i = 0; i < kI; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    const int oc0 = o0 + 64 * ch;
    const int nkc = args.cin_g / kEl;
    // the wave's offsets in chunk c, and its stages over all chunks
    constexpr uint32_t kDeal = kSplit == 4 ? 0x11111111u : (kSplit == 2 ? 0x55555555u : 0xffffffffu);
    auto share = [&](int c) { return wmask & (kDeal << ((sp - c) & (kSplit - 1))); };
    int S = 0;
#pragma unroll
    for (int c = 0; c < kSplit; ++c) S += __builtin_popcount(share(c)) * ((nkc - c + kSplit - 1) / kSplit);
    if (S > 0) {
        const __amdgpu_buffer_rsrc_t a_rsrc =
            make_rsrc(static_cast<const TA *>(args.input) + in_col0,
                      (uint32_t)(args.n_in * row_bytes - in_col0 * (int64_t)sizeof(TA)));
        // Weight fragment (offset k, chunk c, block j): base[j] + k w_k + c w_c.
        uint32_t wb[4], w_k, w_c;
        __amdgpu_buffer_rsrc_t w_rsrc;
        if (args.wpack) {
            const int n_ot = (args.cout_g + kBN - 1) / kBN;
            const uint32_t tile_bytes = (uint32_t)K * (uint32_t)nkc * 8u * 1024u;
            w_rsrc = make_rsrc(static_cast<const char *>(args.wpack) + kPackHeaderBytes,
                               (uint32_t)((int64_t)args.cin / args.cin_g * n_ot) * tile_bytes);
            w_c = 8u * 1024u;
            w_k = (uint32_t)nkc * w_c;
#pragma unroll
            for (int j = 0; j < 4; ++j)
                wb[j] = (oc0 >> 7) < n_ot ? (uint32_t)(g * n_ot + (oc0 >> 7)) * tile_bytes +
                                                (uint32_t)((oc0 & 127) / 16 + j) * 1024u + (uint32_t)lane * 16u
                                          : kOobOffset;
        } else {
            w_rsrc = make_rsrc(args.weight, (uint32_t)(args.cout * (int64_t)K * args.cin_g * (int64_t)sizeof(TW)));
            w_c = (uint32_t)(kEl * (int)sizeof(TW));
            w_k = (uint32_t)(args.cin_g * (int)sizeof(TW));
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int o = oc0 + 16 * j + l16;
                wb[j] = o < args.cout_g
                            ? (uint32_t)((out_col0 + o) * (int64_t)K * args.cin_g * (int64_t)sizeof(TW)) + q4 * kWPiece
                            : kOobOffset;
            }
        }
        const uint32_t *offs = &s_off[0][trow + l16];
        uint32_t rem = share(0);  // offsets left in the chunk of the next stage to load
        int c = 0;
        auto settle = [&]() {  // past the last chunk: offset 0, never loaded
            while (rem == 0u) rem = ++c < nkc ? share(c) : 1u;
        };
        settle();
        int k = __builtin_ctz(rem);
        uint32_t ro[kI];
        auto read_off = [&]() {
#pragma unroll
            for (int i = 0; i < kI; ++i) ro[i] = offs[k * kRows + 16 * i];
        };
        uint4 x[kDepth][kI], w[kDepth][4];
        auto issue = [&](int s) {
            const bool live = c < nkc;
            const uint32_t xc = (uint32_t)(c * 64 + q4 * 16);
            const uint32_t wo = (uint32_t)k * w_k + (uint32_t)c * w_c;
#pragma unroll
            for (int i = 0; i < kI; ++i) x[s][i] = bload16(a_rsrc, live ? ro[i] + xc : kOobOffset);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const uint32_t off = live ? wb[j] + wo : kOobOffset;
                if constexpr (kI8) {
                    const uint2 q = bload8(w_rsrc, off);
                    w[s][j].x = q.x;
                    w[s][j].y = q.y;
                } else {
                    w[s][j] = bload16(w_rsrc, off);
                }
            }
            rem &= rem - 1u;
            settle();
            k = __builtin_ctz(rem);
            read_off();
        };
        auto compute = [&](int s) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                uint4 f = w[s][j];
                if constexpr (kI8) {
                    f.w = i8pair_to_bf16x2(w[s][j].y, 16);
                    f.z = i8pair_to_bf16x2(w[s][j].y, 0);
                    f.y = i8pair_to_bf16x2(w[s][j].x, 16);
                    f.x = i8pair_to_bf16x2(w[s][j].x, 0);
                }
#pragma unroll
                for (int i = 0; i < kI; ++i) acc[i][j] = mfma_16x16x32<TA>(f, x[s][i], acc[i][j]);
            }
        };
        read_off();
#pragma unroll
        for (int s = 0; s < kDepth - 1; ++s) issue(s);
        int t = 0;
        for (; t + kDepth <= S; t += kDepth) {
#pragma unroll
            for (int u = 0; u < kDepth; ++u) {
                issue((u + kDepth - 1) % kDepth);
                __builtin_amdgcn_sched_barrier(0);
                compute(u);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
#pragma unroll
        for (int u = 0; u < kDepth - 1; ++u)
            if (t + u < S) compute(u);
    }

    // Waves that share a block add their partial sums (in share order); wave
    // sp then finishes row blocks [kE sp, kE sp + kE) (none past kI).
    f32x4 sum[kE][4];
    const int eb = kSplit > 1 ? kE * sp : 0;
    const bool idle = eb >= kI;
    const int erow = trow + 16 * (idle ? 0 : eb);
    if constexpr (kSplit > 1) {
        __syncthreads();
#pragma unroll
        for (int i = 0; i < kI; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) s_part[wave][(i * 4 + j) * 64 + lane] = acc[i][j];
        __syncthreads();
#pragma unroll
        for (int i = 0; i < kE; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int at = (((idle ? 0 : eb) + i) * 4 + j) * 64 + lane;
                f32x4 t = s_part[wave - sp][at];
#pragma unroll
                for (int u = 1; u < kSplit; ++u) t += s_part[wave - sp + u][at];
                sum[i][j] = t;
            }
    } else {
#pragma unroll
        for (int i = 0; i < kE; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) sum[i][j] = acc[i][j];
    }

    // ---- epilogue: * int8 scale + bias -> LayerNorm -> SiLU -> + residual
    //      (or the C2S forms), the halo-staged kernel's layout and order.
    TO *__restrict__ out = static_cast<TO *>(args.out);
    const TO *__restrict__ res = static_cast<const TO *>(args.residual);
    const bool vec_ok = args.vec_out != 0;
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int o = oc0 + j * 16 + 4 * q4 + e;
            const bool ok = o < args.cout_g;
            const float bias = (args.bias && ok) ? args.bias[out_col0 + o] : 0.f;
            const float scale = (args.w_scale && ok) ? args.w_scale[out_col0 + o] : 1.f;  // int8 weights
#pragma unroll
            for (int i = 0; i < kE; ++i) sum[i][j][e] = ok ? sum[i][j][e] * scale + bias : 0.f;
        }
    if (args.ln) {
        // two-pass f32 statistics over the row (or one child's channels); the
        // two 64-channel columns of a 128-channel row meet in LDS
        const bool exchange = kNT == 128 && args.ln_group != 64;
        const float inv_c = 1.0f / (float)args.ln_group;
        auto row_total = [&](float(&part)[kE]) {
            __syncthreads();
#pragma unroll
            for (int i = 0; i < kE; ++i)
                if (q4 == 0 && !idle) s_red[ch][erow + 16 * i + l16] = part[i];
            __syncthreads();
#pragma unroll
            for (int i = 0; i < kE; ++i) part[i] = s_red[0][erow + 16 * i + l16] + s_red[1][erow + 16 * i + l16];
        };
        float mean[kE], part[kE];
#pragma unroll
        for (int i = 0; i < kE; ++i) {
            float t = 0.f;
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e) t += sum[i][j][e];
            t += __shfl_xor(t, 16, 64);
            t += __shfl_xor(t, 32, 64);
            part[i] = t;
        }
        if (exchange) row_total(part);
#pragma unroll
        for (int i = 0; i < kE; ++i) {
            mean[i] = part[i] * inv_c;
            float qv = 0.f;
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float d = sum[i][j][e] - mean[i];
                    qv += oc0 + j * 16 + 4 * q4 + e < args.cout_g ? d * d : 0.f;
                }
            qv += __shfl_xor(qv, 16, 64);
            qv += __shfl_xor(qv, 32, 64);
            part[i] = qv;
        }
        if (exchange) row_total(part);
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int o = oc0 + j * 16 + 4 * q4 + e;
                const bool ok = o < args.cout_g;
                const int og = o % args.ln_group;
                const float lw = (args.ln_w && ok) ? args.ln_w[og] : 1.f;
                const float lb = (args.ln_b && ok) ? args.ln_b[og] : 0.f;
#pragma unroll
                for (int i = 0; i < kE; ++i)
                    sum[i][j][e] = (sum[i][j][e] - mean[i]) * rsqrt_f32(part[i] * inv_c + args.ln_eps) * lw + lb;
            }
    }
#pragma unroll
    for (int i = 0; i < kE; ++i) {
        const int32_t qrow = s_row[erow + 16 * i + l16];
        if (qrow < 0 || idle) continue;
        const int64_t rowbase = (int64_t)qrow * args.cout + out_col0;
        const bool c2s = args.scatter_rows || args.skip_idx;
        const C2SRow crow = c2s ? c2s_row<TO>(args, qrow) : C2SRow{nullptr};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int oc = oc0 + j * 16 + 4 * q4;
            if (oc >= args.cout_g) continue;
            float v[4] = {sum[i][j][0], sum[i][j][1], sum[i][j][2], sum[i][j][3]};
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

// How a 16-bit call over `rows` rows, `cols` output channels and `groups`
// groups is cut: {16-row blocks per wave, waves sharing a block}; {0, 0}: the
// 256-row tiles, which share operands through LDS, take it.  By the number of
// 16 x 64 blocks: up to one workgroup per CU with kI as small as that allows
// (2,000 rows x 128 channels, 250 blocks, planned bf16: kI = 1 12.0 us, 2
// 14.4, 4 20.8; 2,000 x 256, 500 blocks: 32.8, 25.0, 35.7; 6,000 x 128, 750
// blocks: 26.2, 24.1, 21.7), and kI = 4 up to two: planned 1,831 blocks 37.9
// against 52.1 us on the 256-row tiles, 3,662 blocks 124 against 99; without
// a plan 54.6 against 81.0, 189 against 164; linears 256 -> 1024 at 2,000
// blocks 9.7 against 12.0, at 6,000 23.8 against 13.4.
struct RowsCut {
    int kI, split;
};
inline RowsCut rows_cut(int64_t rows, int64_t cols, int groups)
{
    const int64_t blocks = (rows + 15) / 16 * ((cols + 63) / 64) * groups;
    if (blocks <= 256) return {1, 4};
    if (blocks <= 512) return {2, 4};
    if (blocks <= 2048) return {4, 4};
    return {0, 0};
}

// n_rows: query rows, or a child plan's tiles x 256; cols: output channels
// one row spans there.
template <typename TA, typename TW, typename TO>
int launch_rows(const ConvArgs &a, RowsCut cut, int64_t n_rows, int64_t cols, int groups, hipStream_t s)
{
    // 128-channel tiles, two waves a block: a LayerNorm row of 65-128
    // channels in one workgroup
    const bool wide = cols > 64 && a.ln;
    if (wide) cut.split = 2;
    const int nt = wide ? 128 : 64;
    const int64_t per = (int64_t)16 * cut.kI * 4 / (cut.split * (nt / 64));
    const int64_t gx = (n_rows + per - 1) / per, gy = (cols + nt - 1) / nt;
    if (gx > INT32_MAX || gy > 65535 || groups > 65535) return fail(SC_ERR_OVERFLOW, "sparse conv grid overflow");
    const dim3 grid((unsigned)gx, (unsigned)gy, (unsigned)groups);
    if (cut.kI == 1) {
        if (wide)
            conv_rows_kernel<TA, TW, TO, 1, 128, 2><<<grid, kThreads, 0, s>>>(a);
        else
            conv_rows_kernel<TA, TW, TO, 1, 64, 4><<<grid, kThreads, 0, s>>>(a);
    } else if (cut.kI == 2) {
        if (wide)
            conv_rows_kernel<TA, TW, TO, 2, 128, 2><<<grid, kThreads, 0, s>>>(a);
        else
            conv_rows_kernel<TA, TW, TO, 2, 64, 4><<<grid, kThreads, 0, s>>>(a);
    } else {
        if (wide)
            conv_rows_kernel<TA, TW, TO, 4, 128, 2><<<grid, kThreads, 0, s>>>(a);
        else
            conv_rows_kernel<TA, TW, TO, 4, 64, 4><<<grid, kThreads, 0, s>>>(a);
    }
    SC_LAUNCH_CHECK("conv_rows_kernel launch");
    return SC_OK;
}
