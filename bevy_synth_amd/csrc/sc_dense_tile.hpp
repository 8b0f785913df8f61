// Persistent 256 x 256 tile of the dense linear (16-bit).  Included by
// sc_conv_kernels.hpp.
#pragma once

// The dense linear out = x W^T + b for calls of many 256 x 256 tiles
// (dense_tile_takes): one workgroup of 8 waves per CU walks its tiles, k-steps
// of 32 input channels flowing through a ring of four 32 KB LDS stages (rows
// 256 x 64 B, channels 256 x 64 B, DMA'd three steps ahead) without a break
// between tiles: the next tile's first steps are in flight while a tile's
// epilogue runs, and the epilogue's stores drain under the next tile's MFMAs.
// It needs no LDS: the weight rows are dealt to the MFMA blocks so that a lane
// ends with 8 consecutive channels of a row per pair of blocks, and 4 lanes
// with 64 bytes of 16-bit output.
//
// Waves 2 x 4, 128 rows x 64 channels each (8 x 4 blocks of
// v_mfma_f32_16x16x32), as dense_gemm_kernel; a value's sum is the same there
// and here.  dense_gemm_kernel spent its time on bytes (a 256 x 128 tile reads
// 24 KB per k-step for half of this tile's MFMAs) and on a ring that starts and
// drains once per tile.  Measured, bf16, per call, there -> here: 113,857 rows
// 512 -> 2048 336 -> 288 us, 256 -> 1024 117 -> 99 us, 1024 -> 256 81 -> 77 us;
// the transposed upsample 512 -> 8 x 256 of 113,857 parents 378 -> 293 us.
// Bound now: 64-byte requests from L1 to L2 (the texture data path is busy 86 %
// of the time, the matrix cores 36 %; without the MFMAs 269 of 288 us remain).
// Stages of 64 channels, which halve the requests, leave one step of lead and
// do not fit the registers beside the accumulators: 320 us.
//
// Waits.  Vector memory operations complete in order, stores included: at a
// step's top its own DMA must have landed, with those of the next two steps
// (2 kPer operations) and, in the three steps after an epilogue, its kStores
// stores behind it.  The stores are issued without branches (a row or channel
// past the end gets an offset past the buffer), the DMAs past the last tile
// read zero, so the counts are exact; an operation not counted (the row
// list's DMA) only makes a wait stricter.  Buffer (k + 3) % 4, filled in step
// k, was read in step k - 1, which every wave has left at step k's barrier.
constexpr int kDenseBias = 4096;  // channels whose bias the tile keeps in LDS

template <typename TO>
__device__ inline void buf_store8(__amdgpu_buffer_rsrc_t r, uint32_t off, const float *v)
{
    if constexpr (sizeof(TO) == 2) {
        const uint4 u = Out8<TO>::pack(v);
        __builtin_amdgcn_raw_buffer_store_b128(u32x4{u.x, u.y, u.z, u.w}, r, off, 0, 0);
    } else {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const float *w = v + 4 * h;
            __builtin_amdgcn_raw_buffer_store_b128(
                u32x4{__builtin_bit_cast(uint32_t, w[0]), __builtin_bit_cast(uint32_t, w[1]),
                      __builtin_bit_cast(uint32_t, w[2]), __builtin_bit_cast(uint32_t, w[3])},
                r, off + 16u * h, 0, 0);
        }
    }
}

// kListed: rows and channels from a linear child plan (perm, child_base), the
// output scattered to the child rows.
template <typename TA, typename TO, bool kListed>
__global__ __launch_bounds__(512, 1) void dense_tile_kernel(ConvArgs args)
{
    constexpr int kI = 8, kBuf = 4, kStage = 32768, kPer = 4;
    constexpr int kStores = kI * 2 * (int)sizeof(TO) / 2;
    __shared__ __attribute__((aligned(16))) unsigned char s_buf[kBuf * kStage];
    __shared__ __attribute__((aligned(16))) float s_bias[kDenseBias];
    __shared__ __attribute__((aligned(16))) int32_t s_rows[2][kListed ? kTileRows : 4];  // by tile parity

    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int l16 = lane & 15, q4 = lane >> 4;
    const int rh = wave >> 2, qc = wave & 3;
    const int cin = (int)args.cin, nk = cin / 32;
    // This XCD's share of the tiles, its workgroups interleaved in it: a
    // contiguous range of row tile x column tile (columns fastest), so that a
    // row tile's columns meet in its L2; listed, an eighth of every child's
    // list, child fastest (len tiles from tile lo on), since the lists hold
    // the same parents in the same order (child after child, as the list
    // tiles lie, the rows come from HBM once per child).
    const int xcd = blockIdx.x & 7, per = gridDim.x >> 3;
    const int n_ct = ((kListed ? args.child_ch : args.cout_g) + 255) / 256;
    int lo[8], len[8];
    int row_tiles, first, n_mine = 0;
    if constexpr (kListed) {
        const PlanHeader *h = args.plan_hdr;
        if (!plan_matches(h, args)) {
            flag_plan_status(h, kPlanStatusMapMismatch);
            return;
        }
        row_tiles = __builtin_amdgcn_readfirstlane(h->status == 0u ? h->n_unique : 0);
        if (row_tiles == 0) return;
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            const int b0 = args.child_base[c], n = (c < 7 ? args.child_base[c + 1] : row_tiles) - b0;
            lo[c] = __builtin_amdgcn_readfirstlane(b0 + (int)((int64_t)n * xcd / 8));
            len[c] = __builtin_amdgcn_readfirstlane(b0 + (int)((int64_t)n * (xcd + 1) / 8)) - lo[c];
            n_mine += len[c];
        }
        first = 0;
        n_mine *= n_ct;
    } else {
        row_tiles = (int)((args.n_q + kTileRows - 1) / kTileRows);
        const int n_all = row_tiles * n_ct;
        first = xcd * (n_all >> 3) + min(xcd, n_all & 7);
        n_mine = (n_all >> 3) + (xcd < (n_all & 7) ? 1 : 0);
    }
    struct Tile {
        int lt, child, o0;  // list (row) tile, its child, first channel
    };
    // Tile u of this XCD (uniform).
    auto locate = [&](int u) {
        Tile t;
        if constexpr (kListed) {
            // children of equal rank j side by side, the longer lists' rest after
            int rem = u / n_ct, from = 0;
            t.lt = row_tiles, t.child = 0;
            for (int it = 0; it < 8; ++it) {
                int m = INT_MAX, cnt = 0;
#pragma unroll
                for (int c = 0; c < 8; ++c)
                    if (len[c] > from) {
                        ++cnt;
                        m = min(m, len[c]);
                    }
                if (cnt == 0) break;
                if (rem < (m - from) * cnt) {
                    const int j = from + rem / cnt;
                    int nth = rem % cnt;
#pragma unroll
                    for (int c = 0; c < 8; ++c)
                        if (len[c] > from && nth-- == 0) {
                            t.lt = lo[c] + j;
                            t.child = c;
                        }
                    break;
                }
                rem -= (m - from) * cnt;
                from = m;
            }
            t.o0 = t.child * args.child_ch + (u % n_ct) * 256;
        } else {
            t.lt = (first + u) / n_ct;
            t.child = 0;
            t.o0 = (first + u) % n_ct * 256;
        }
        return t;
    };
    const int u0 = blockIdx.x >> 3;
    if (u0 >= n_mine) return;
    Tile cur = locate(u0), nxt = cur;

    for (int i = tid; i < args.cout_g; i += 512) s_bias[i] = args.bias ? args.bias[i] : 0.f;
    if (kListed && tid < kTileRows) s_rows[0][tid] = args.perm[(int64_t)cur.lt * kTileRows + tid];

    const i32x4_rsrc a_rsrc = rsrc_words(args.input, (uint32_t)(args.n_q * (int64_t)cin * 2));
    const i32x4_rsrc w_rsrc = rsrc_words(args.weight, (uint32_t)((int64_t)args.cout_g * cin * 2));
    const i32x4_rsrc p_rsrc = rsrc_words(args.perm, kListed ? (uint32_t)row_tiles * (kTileRows * 4) : 0u);
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)s_buf;
    const uint32_t lds_rows = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) int32_t *)&s_rows[0][0];
    const uint32_t wave_kb = (uint32_t)__builtin_amdgcn_readfirstlane(1024 * wave);
    __syncthreads();

    // DMA sources of the tile being loaded: instruction h of this wave fills
    // rows (channels) 16 (wave + 8 h) .., lane L row L / 4, slot L % 4.
    uint32_t a_src[2], w_src[2];
    const uint32_t piece = (uint32_t)wslot<64>(lane >> 2, lane & 3) * 16u;
    auto sources = [&](const Tile &t, int parity) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int n = 16 * (wave + 8 * h) + (lane >> 2);
            int64_t row;
            if constexpr (kListed) {
                const int32_t p = s_rows[parity][n];
                row = p >= 0 && p < args.n_q ? p : -1;
            } else {
                row = (int64_t)t.lt * kTileRows + n;
                if (row >= args.n_q) row = -1;
            }
            a_src[h] = row >= 0 ? (uint32_t)(row * cin * 2) + piece : kOobOffset;
            w_src[h] = t.o0 + n < args.cout_g ? (uint32_t)((int64_t)(t.o0 + n) * cin * 2) + piece : kOobOffset;
        }
    };
    int l_u = u0, l_k = 0, l_buf = 0, l_par = 0;  // the next k-step to load
    auto dma = [&]() {
        const bool live = l_u < n_mine;
        const uint32_t step = (uint32_t)l_k * 64u, lds = lds0 + (uint32_t)l_buf * kStage + wave_kb;
#pragma unroll
        for (int h = 0; h < 2; ++h) lds_dma16(a_rsrc, live ? a_src[h] + step : kOobOffset, lds + 8192u * h);
#pragma unroll
        for (int h = 0; h < 2; ++h) lds_dma16(w_rsrc, live ? w_src[h] + step : kOobOffset, lds + 16384u + 8192u * h);
        l_buf = (l_buf + 1) & (kBuf - 1);
        if (++l_k == nk) {
            l_k = 0;
            l_u += per;
            l_par ^= 1;
            if (l_u < n_mine) sources(nxt, l_par);
        }
    };
    // Fragment offsets in a stage.  Block j's MFMA row m = 4 a + b is channel
    // 64 qc + 32 (j / 2) + 8 a + 4 (j % 2) + b.
    const int wch = 8 * (l16 >> 2) + (l16 & 3);
    int xoff = (128 * rh + l16) * 64 + wslot<64>(l16, q4) * 16;
    int woff0 = 16384 + (64 * qc + wch) * 64 + wslot<64>(wch, q4) * 16;
    int woff1 = 16384 + (64 * qc + wch + 4) * 64 + wslot<64>(wch + 4, q4) * 16;
    asm("" : "+v"(xoff));
    asm("" : "+v"(woff0));
    asm("" : "+v"(woff1));

    f32x4 acc[kI][4];
    auto clear = [&]() {
#pragma unroll
        for (int i = 0; i < kI; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    };
    clear();
    int buf = 0;
    auto step = [&]() {
        const unsigned char *base = s_buf + buf * kStage;
        uint4 x[kI], w[4];
#pragma unroll
        for (int i = 0; i < kI; ++i) x[i] = *reinterpret_cast<const uint4 *>(base + xoff + 1024 * i);
#pragma unroll
        for (int j = 0; j < 4; ++j)
            w[j] = *reinterpret_cast<const uint4 *>(base + ((j & 1) ? woff1 : woff0) + 2048 * (j >> 1));
        __builtin_amdgcn_sched_barrier(0);
        dma();
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int i = 0; i < kI; ++i) acc[i][j] = mfma_16x16x32<TA>(w[j], x[i], acc[i][j]);
        buf = (buf + 1) & (kBuf - 1);
    };

    // output rows (child rows when listed) x channels
    const int64_t out_rows = kListed ? args.scatter_n : args.n_q;
    const int pitch = kListed ? args.scatter_ch : (int)args.cout;
    const __amdgpu_buffer_rsrc_t o_rsrc = make_rsrc(args.out, (uint32_t)(out_rows * pitch * (int64_t)sizeof(TO)));
    const __amdgpu_buffer_rsrc_t r_rsrc =
        make_rsrc(args.residual, (uint32_t)(args.n_q * args.cout * (int64_t)sizeof(TO)));

    sources(cur, 0);
    for (int s = 0; s < kBuf - 1; ++s) dma();
    int par = 0;
    for (int u = u0; u < n_mine; u += per, par ^= 1, cur = nxt) {
        if (u + per < n_mine) nxt = locate(u + per);
        for (int k = 0; k < nk; ++k) {
            if (k < kBuf - 1 && u != u0)
                wait_vmcnt<2 * kPer + kStores>();
            else
                wait_vmcnt<2 * kPer>();
            __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
            __builtin_amdgcn_s_barrier();
            step();
            if (kListed && k == 0) {
                // the next tile's rows, read three steps before its first one
                // (nk >= 8: landed by then; last read a tile ago)
                lds_dma16(p_rsrc, (uint32_t)nxt.lt * (kTileRows * 4) + (uint32_t)lane * 16u,
                          lds_rows + (uint32_t)(par ^ 1) * (kTileRows * 4));
            }
        }
        // ---- epilogue: + bias -> SiLU -> + residual -> stores
        const int o0 = cur.o0 + 64 * qc + 8 * q4;  // this lane's channels: o0 + 32 jp + [0, 8)
        uint32_t dst[kI];
        if constexpr (kListed) {
            const int sub = o0 - cur.child * args.child_ch;
            int32_t cr[kI];
#pragma unroll
            for (int i = 0; i < kI; ++i) {
                const int32_t p = s_rows[par][128 * rh + 16 * i + l16];
                cr[i] = p >= 0 && p < args.n_q ? args.scatter_rows[(int64_t)p * 8 + cur.child] : -1;
            }
#pragma unroll
            for (int i = 0; i < kI; ++i)
                dst[i] = cr[i] >= 0 && cr[i] < args.scatter_n ? (uint32_t)(((int64_t)cr[i] * pitch + sub) * (int)sizeof(TO))
                                                             : kOobOffset;
        } else {
#pragma unroll
            for (int i = 0; i < kI; ++i) {
                const int64_t r = (int64_t)cur.lt * kTileRows + 128 * rh + 16 * i + l16;
                dst[i] = r < args.n_q ? (uint32_t)((r * pitch + o0) * (int)sizeof(TO)) : kOobOffset;
            }
        }
        constexpr int kRG = sizeof(TO) == 2 ? 4 : 2;  // row blocks whose residual is fetched together
#pragma unroll
        for (int ih = 0; ih < kI; ih += kRG) {
            uint4 rv[kRG][2][sizeof(TO) / 2];
            if (args.residual) {
#pragma unroll
                for (int ii = 0; ii < kRG; ++ii)
#pragma unroll
                    for (int jp = 0; jp < 2; ++jp)
#pragma unroll
                        for (int h = 0; h < (int)sizeof(TO) / 2; ++h)
                            rv[ii][jp][h] =
                                bload16(r_rsrc, dst[ih + ii] + (uint32_t)(32 * jp * (int)sizeof(TO) + 16 * h));
            }
#pragma unroll
            for (int ii = 0; ii < kRG; ++ii) {
#pragma unroll
                for (int jp = 0; jp < 2; ++jp) {
                    const bool ok = o0 + 32 * jp < args.cout_g;
                    const float4 *bp = reinterpret_cast<const float4 *>(s_bias + (ok ? o0 + 32 * jp : 0));
                    const float4 b0 = bp[0], b1 = bp[1];
                    const float bv[8] = {b0.x, b0.y, b0.z, b0.w, b1.x, b1.y, b1.z, b1.w};
                    float v[8];
#pragma unroll
                    for (int cc = 0; cc < 8; ++cc) v[cc] = acc[ih + ii][2 * jp + (cc >> 2)][cc & 3] + bv[cc];
                    if (args.silu) {
#pragma unroll
                        for (int cc = 0; cc < 8; ++cc) v[cc] = silu_f32(v[cc]);
                    }
                    if (args.residual) {
                        float r8[8];
                        typename Out8<TO>::V rr;
                        __builtin_memcpy(&rr, rv[ii][jp], sizeof(rr));
                        Out8<TO>::unpack(rr, r8);
#pragma unroll
                        for (int cc = 0; cc < 8; ++cc) v[cc] += r8[cc];
                    }
                    buf_store8<TO>(o_rsrc, ok ? dst[ih + ii] + (uint32_t)(32 * jp * (int)sizeof(TO)) : kOobOffset, v);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        clear();
        __builtin_amdgcn_sched_barrier(0);
    }
    wait_vmcnt<0>();
}

// Whether the persistent tile takes a dense linear (see above): whole 16-byte
// pieces, the bias in LDS, 32-bit offsets into the output, and enough tiles.
// The lines, measured in us against dense_gemm_kernel (bf16):
//  * 160 tiles: 12,000 rows 256 -> 1024 (188 tiles) 18.0 against 19.4, but
//    16,000 rows 512 -> 512 (126) 20.1 against 18.3; the child lists of 4,000
//    parents 256 -> 8 x 256 (about 63) 92 against 85;
//  * with more than 512 channels a second round of few tiles costs more than
//    it gives: 4,200 rows 1024 -> 4096 (272 tiles) 60 against 57, but 4,000
//    rows (256) 39 against 44 and 16,640 rows (1,040) 152 against 166;
//    of shorter rows such a round still gains (16,640 rows 256 -> 1024, 260
//    tiles: 27.0 against 28.8);
//  * columns at least 7/8 full: 66,000 rows 512 -> 640 (5/6) 66 against 66.
// cin: the ring's lead of three steps, and the row list read three steps
// before the next tile's first (nk >= 8).
template <typename TO>
bool dense_tile_takes(const ConvArgs &a, bool listed, int64_t row_tiles)
{
    const int64_t cols = listed ? a.child_ch : a.cout_g;
    const int64_t out = listed ? a.scatter_n * a.scatter_ch : a.n_q * a.cout;
    if (a.ln || a.vec_out != 8 || a.cout_g > kDenseBias || a.cin < (listed ? 256 : 128) ||
        (listed ? a.child_ch % 256 != 0 || a.residual != nullptr : a.scatter_rows != nullptr) ||
        out * (int64_t)sizeof(TO) > (int64_t)kOobOffset)
        return false;
    const int64_t n_ct = (cols + 255) / 256, tiles = row_tiles * n_ct;
    return cols * 8 >= n_ct * 256 * 7 && tiles >= 160 && (a.cin <= 512 || tiles <= 256 || tiles >= 384);
}

template <typename TA, typename TO, bool kListed>
int launch_dense_tile(const ConvArgs &a, int64_t row_tiles, hipStream_t s)
{
    const int64_t cols = kListed ? a.child_ch : a.cout_g;
    const int64_t tiles = row_tiles * ((cols + 255) / 256);
    if (tiles > INT32_MAX) return fail(SC_ERR_OVERFLOW, "dense linear grid overflow");
    const unsigned grid = (unsigned)std::min<int64_t>(256, (tiles + 7) / 8 * 8);  // one per CU
    dense_tile_kernel<TA, TO, kListed><<<grid, 512, 0, s>>>(a);
    SC_LAUNCH_CHECK("dense_tile_kernel launch");
    return SC_OK;
}
