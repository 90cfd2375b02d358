// f16 GEMM of few rows for gfx950: Y = epilogue(X[M][K] . W[N][K]^T), f16
// activations, weights f16 or dequantised to f16 in registers, for products
// whose 64-row tiles leave most of the chip idle (a streaming step, one
// utterance at a time).
//
// What bounds those is latency: a handful of workgroups each walk all of K
// with a barrier per 64 columns.  Here a tile is 16 TM rows x 32 columns, KG
// waves split its K, each streams its operands through a private LDS ring
// filled by DMA (whole 64- and 128-byte row pieces; loads straight into MFMA
// fragments touch 16 rows per instruction and were up to twice slower), with
// no barrier in the loop, and the partial tiles are summed through LDS in a
// fixed order (deterministic).  MI355X, q8_0, us before and after: M = 2,
// N = 512 K = 2048 9.8 -> 4.9, N = 2048 K = 512 6.4 -> 3.9; M = 125, N = 1024
// K = 1024 11.1 -> 4.4, K = 4096 12.3 -> 6.7, N = 4096 K = 1024 10.3 -> 6.9.
#include "gemm.hpp"
#include "gemm_common.hpp"

namespace pkx {

namespace {

// The 32 weight rows of a tile over one 64-column step, staged in LDS by DMA
// (BYTES, NI instructions of 1 KB), and a lane's operands of them: row lr of
// 16-row block j, columns A_STEP lg + A_HALF h + e of the step (lr = lane % 16,
// lg = lane / 16; the activations use the same columns, so the contraction is
// unchanged).  Scales go to registers.  The 16-byte chunks of a row are
// XOR-swizzled so that 16 rows read at one chunk spread over the LDS banks.
template <int WT> struct RowsW;

template <> struct RowsW<GT_F16> {
    static constexpr int A_STEP = 8, A_HALF = 32, NI = 4, BYTES = 4096, NS = 0;
    // instruction u: rows 8 u .. + 7, 128 bytes each
    __device__ __forceinline__ void issue(__amdgpu_buffer_rsrc_t rq, __amdgpu_buffer_rsrc_t, const GemmParams& p,
                                          uint8_t* lds, const int (&row0)[2], int, int lane, int st) {
        const int r = lane >> 3, c = (lane & 7) ^ r;
#pragma unroll
        for (int u = 0; u < 4; ++u)
            lds_dma16(rq, lds + 1024 * u, (uint32_t)((row0[u >> 1] + 8 * (u & 1) + r) * p.K + 64 * st + 8 * c) * 2u, 0);
    }
    __device__ __forceinline__ half8v get(const uint8_t* lds, int j, int h, int lr, int lg) const {
        return *(const half8v*)(lds + 2048 * j + 128 * lr + 16 * ((4 * h + lg) ^ (lr & 7)));
    }
};
template <> struct RowsW<GT_Q8_0> {
    static constexpr int A_STEP = 16, A_HALF = 8, NI = 2, BYTES = 2048, NS = 2;
    uint32_t d[2];
    // instruction j: the 16 rows of block j, 64 bytes each
    __device__ __forceinline__ void issue(__amdgpu_buffer_rsrc_t rq, __amdgpu_buffer_rsrc_t rs, const GemmParams& p,
                                          uint8_t* lds, const int (&row0)[2], int lg, int lane, int st) {
        const int slab = st * slab_rows(p), r = lane >> 2, c = (lane & 3) ^ ((r >> 2) & 3);
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            lds_dma16(rq, lds + 1024 * j, (uint32_t)(slab + row0[j] + r) * 64u + 16u * c, 0);
            d[j] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b16(rs, (slab + row0[j] + (lane & 15)) * 4 + (lg & 2), 0, 0);
        }
    }
    __device__ __forceinline__ half8v get(const uint8_t* lds, int j, int h, int lr, int lg) const {
        const int2v q = *(const int2v*)(lds + 1024 * j + 64 * lr + 16 * (lg ^ ((lr >> 2) & 3)) + 8 * h);
        const f16 dh = __builtin_bit_cast(f16, (uint16_t)d[j]);
        const half2v d2 = {dh, dh};
        half2v a, b, c, e;
        i8x4_to_f16((uint32_t)q[0], d2, a, b);
        i8x4_to_f16((uint32_t)q[1], d2, c, e);
        return half8v{a[0], a[1], b[0], b[1], c[0], c[1], e[0], e[1]};
    }
};
template <> struct RowsW<GT_Q4_K> {
    static constexpr int A_STEP = 8, A_HALF = 32, NI = 1, BYTES = 1024, NS = 2;
    int4v sm[2];   // {scale, min} of the step's two 32-column sub-blocks
    // one instruction: lanes 0 .. 31 the 16 rows of block 0, 32 bytes each, the others block 1
    __device__ __forceinline__ void issue(__amdgpu_buffer_rsrc_t rq, __amdgpu_buffer_rsrc_t rs, const GemmParams& p,
                                          uint8_t* lds, const int (&row0)[2], int, int lane, int st) {
        const int slab = st * slab_rows(p), r = (lane & 31) >> 1, c = (lane & 1) ^ ((r >> 3) & 1);
        lds_dma16(rq, lds, (uint32_t)(slab + (lane < 32 ? row0[0] : row0[1]) + r) * 32u + 16u * c, 0);
#pragma unroll
        for (int j = 0; j < 2; ++j)
            sm[j] = __builtin_amdgcn_raw_buffer_load_b128(rs, (slab + row0[j] + (lane & 15)) * 16, 0, 0);
    }
    __device__ __forceinline__ half8v get(const uint8_t* lds, int j, int h, int lr, int lg) const {
        const int2v q = *(const int2v*)(lds + 512 * j + 32 * lr + 16 * ((lg >> 1) ^ ((lr >> 3) & 1)) + 8 * (lg & 1));
        const float4v s = __builtin_bit_cast(float4v, sm[j]);
        const half2v m2 = {(f16)s[2 * h], (f16)s[2 * h]}, nm2 = {(f16)-s[2 * h + 1], (f16)-s[2 * h + 1]};
        half2v a, b, c, e;
        nib4_to_f16((uint32_t)q[0], h, m2, nm2, a, b);
        nib4_to_f16((uint32_t)q[1], h, m2, nm2, c, e);
        return half8v{a[0], a[1], b[0], b[1], c[0], c[1], e[0], e[1]};
    }
};

}  // namespace

// The weights are the MFMA's A operand, so a lane ends with 4 consecutive
// columns of one row for each of the tile's two 16-column blocks.  EPI_GLU: the
// blocks are the inputs of 16 output channels and their gates (pointwise_conv1
// rows are stored in alternating 32-row groups of inputs and gates).  Wave i
// finishes row block i: N % 32 == 0, so all of its columns exist.
template <int TM, int KG, int D, int WT, int EPI>
__global__ __launch_bounds__(64 * KG) void gemm_rows_kernel(GemmParams p) {
    static_assert(TM <= KG, "one finishing wave per row block");
    constexpr int BM = 16 * TM;
    constexpr bool GLU = EPI == EPI_GLU, FOLD = EPI == EPI_STORE || EPI == EPI_SILU || GLU;
    constexpr bool RES = EPI == EPI_RESID || EPI == EPI_RESID_LN;
    // per wave: D stages of {activation rows 16 TM x 128 bytes, weights}; then the partial tiles
    constexpr int STAGE = TM * 2048 + RowsW<WT>::BYTES, NI = 2 * TM + RowsW<WT>::NI + RowsW<WT>::NS;
    constexpr int RED = KG * TM * 2048, RING = KG * D * STAGE;
    static_assert(RING <= 150 * 1024 && (D - 1) * NI < 64, "LDS ring");
    __shared__ __attribute__((aligned(1024))) uint8_t smem[RING > RED ? RING : RED];
    __shared__ float2v rowtab[BM];   // folded LayerNorm: the rows' {mean, rstd}

    const int tid = threadIdx.x, lane = tid & 63;
    const int kg = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lr = lane & 15, lg = lane >> 4;
    const int nbm = cdiv_dev(p.M, BM), nbn = p.N / 32;
    int bm_, bn_;
    xcd_tile_2d(blockIdx.x, nbm, nbn, p.xcd_gm, bm_, bn_);
    const int m0 = bm_ * BM, n0 = bn_ * 32;

    // rows past M lie past the resource's end (zeros)
    const auto ra = make_rsrc((const f16*)p.A + (int64_t)m0 * p.lda, ((int64_t)(p.M - m0 - 1) * p.lda + p.K) * 2);
    const auto rq = make_rsrc(p.Wq, 0x7fffffff);   // every row of the tile exists; sizes are checked at launch
    const auto rs = make_rsrc(p.Ws, 0x7fffffff);
    int row0[2];   // first weight row of each 16-row block
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int c = n0 / 2;
        row0[j] = GLU ? 64 * (c >> 5) + (c & 31) + 32 * j : n0 + 16 * j;
    }
    const int nst = p.K / 64;
    const int s0 = nst * kg / KG, s1 = nst * (kg + 1) / KG;
    uint8_t* ring = smem + kg * D * STAGE;
    RowsW<WT> wreg[D];
    // steps past the group's range read its last one again (not used), so that
    // the number of loads in flight stays the same
    auto issue = [&](int d, int st) {
        st = max(min(st, s1 - 1), 0);
        uint8_t* lds = ring + d * STAGE;
        const int r = lane >> 3, c = (lane & 7) ^ r;   // 8 rows of 128 bytes an instruction
#pragma unroll
        for (int u = 0; u < 2 * TM; ++u)
            lds_dma16(ra, lds + 1024 * u, (uint32_t)((8 * u + r) * p.lda + 64 * st + 8 * c) * 2u, 0);
        wreg[d].issue(rq, rs, p, lds + TM * 2048, row0, lg, lane, st);
        __builtin_amdgcn_sched_barrier(0);
    };
    float4v acc[TM][2];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = float4v{0.f, 0.f, 0.f, 0.f};
    // the epilogue's operands, ahead of the DMAs (loads return in order): this lane's row and columns
    const bool fin = kg < TM;
    const int m = m0 + 16 * kg + lr;
    const bool live = fin && m < p.M;
    int col[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int c = n0 / 2 + 4 * lg;
        col[j] = GLU ? 64 * (c >> 5) + (c & 31) + 32 * j : n0 + 16 * j + 4 * lg;
    }
    const float4v zero = {0.f, 0.f, 0.f, 0.f};
    const bool fold = FOLD && p.fold_stats != nullptr;
    float4v bias[2] = {zero, zero}, c1[2] = {zero, zero}, res[2] = {zero, zero}, g[2] = {zero, zero};
    float4v rg[2] = {zero, zero}, rb[2] = {zero, zero}, st4[4] = {zero, zero, zero, zero};
    float2v rrow = {0.f, 0.f};
    if (fin) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            if (p.bias) bias[j] = *(const float4v*)(p.bias + col[j]);
            if (FOLD && fold) c1[j] = *(const float4v*)(p.fold_c1 + col[j]);
            if (RES && live) res[j] = *(const float4v*)((const float*)p.Y + (int64_t)m * p.ldy + col[j]);
            if constexpr (EPI == EPI_RESID_LN) {
                g[j] = *(const float4v*)(p.ln_g + col[j]);
                if (p.res_rows) {
                    rg[j] = *(const float4v*)(p.res_g + col[j]);
                    rb[j] = *(const float4v*)(p.res_b + col[j]);
                }
            }
        }
        if (EPI == EPI_RESID_LN && p.res_rows && live) rrow = ((const float2v*)p.res_rows)[m];
        // the row statistics of the block: four lanes a row, two 32-column groups a chunk
        if (FOLD && fold) {
            const int r = min(m0 + 16 * kg + (lane >> 2), p.M - 1), ch = p.fold_groups / 2;
            const float4v* s = (const float4v*)((const float2v*)p.fold_stats + (int64_t)r * p.fold_groups);
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if ((lane & 3) + 4 * i < ch) st4[i] = s[(lane & 3) + 4 * i];
        }
    }

    auto compute = [&](int d) {
        const uint8_t* lds = ring + d * STAGE;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int ch = (RowsW<WT>::A_STEP * lg + RowsW<WT>::A_HALF * h) / 8;   // activation chunk
            half8v af[TM];
#pragma unroll
            for (int i = 0; i < TM; ++i) af[i] = *(const half8v*)(lds + 2048 * i + 128 * lr + 16 * (ch ^ (lr & 7)));
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const half8v w = wreg[d].get(lds + TM * 2048, j, h, lr, lg);
#pragma unroll
                for (int i = 0; i < TM; ++i)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w, af[i], acc[i][j], 0, 0, 0);
            }
        }
    };
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int d = 0; d < D - 1; ++d) issue(d, s0 + d);
    for (int st = s0; st < s1; st += D) {
#pragma unroll
        for (int d = 0; d < D; ++d) {
            if (st + d >= s1) break;   // uniform over the wave
            issue((d + D - 1) % D, st + d + D - 1);
            wait_vmcnt<(D - 1) * NI>();
            compute(d);
            __builtin_amdgcn_s_waitcnt(0xc07f);   // lgkmcnt(0): the stage's reads are done before it is refilled
        }
    }
    wait_vmcnt<0>();

    if (FOLD && fold && fin) {
        // {mean, sum of squared deviations} of the row from its groups'
        const int ch = p.fold_groups / 2;
        float sum = 0.f, dev = 0.f, q = 0.f;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            sum += st4[i][0] + st4[i][2];
            dev += st4[i][1] + st4[i][3];
        }
        const float mean = group_sum(sum, 4) / (float)p.fold_groups;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if ((lane & 3) + 4 * i < ch) q += (st4[i][0] - mean) * (st4[i][0] - mean) + (st4[i][2] - mean) * (st4[i][2] - mean);
        const float d2 = group_sum(dev + 32.0f * q, 4);
        if ((lane & 3) == 0) rowtab[16 * kg + (lane >> 2)] = float2v{mean, rsqrtf(d2 / (32.0f * p.fold_groups) + p.fold_eps)};
    }
    __syncthreads();   // every wave is past its ring
    float4v* red = (float4v*)smem;   // [wave][row block][column block][lane]
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) red[((kg * TM + i) * 2 + j) * 64 + lane] = acc[i][j];
    __syncthreads();
    if (!fin) return;
    float4v v[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        v[j] = red[(kg * 2 + j) * 64 + lane];
#pragma unroll
        for (int i = 1; i < KG; ++i) v[j] += red[((i * TM + kg) * 2 + j) * 64 + lane];
    }
    if (FOLD && fold) {
        const float2v rt = rowtab[16 * kg + lr];
#pragma unroll
        for (int j = 0; j < 2; ++j) v[j] = rt.y * (v[j] - rt.x * c1[j]);
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) v[j] += bias[j];
    if constexpr (GLU) {
        const int c = n0 / 2 + 4 * lg;
        bool dead = false;
        if (p.valid && live) {
            const int b0 = m / p.T;
            dead = m - b0 * p.T >= p.valid[b0];
        }
        half4v o;
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = dead ? (f16)0.f : (f16)(v[0][e] * sigmoid_dev(v[1][e]));
        if (live) *(half4v*)((f16*)p.Y + (int64_t)m * p.ldy + c) = o;
        return;
    }
    if constexpr (EPI == EPI_SILU) {
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) v[j][e] = silu_dev(v[j][e]);
    } else {
#pragma unroll
        for (int j = 0; j < 2; ++j) v[j] *= p.alpha;
    }
    if constexpr (EPI == EPI_STORE || EPI == EPI_SILU) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const half4v h = {(f16)v[j][0], (f16)v[j][1], (f16)v[j][2], (f16)v[j][3]};
            if (live) *(half4v*)((f16*)p.Y + (int64_t)m * p.ldy + col[j]) = h;
        }
    } else {
        if constexpr (RES) {
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                float4v x = res[j];
                if (EPI == EPI_RESID_LN && p.res_rows) x = ((x - rrow.x) * rrow.y) * rg[j] + rb[j];
                v[j] = x + v[j];
            }
        }
#pragma unroll
        for (int j = 0; j < 2; ++j)
            if (live) *(float4v*)((float*)p.Y + (int64_t)m * p.ldy + col[j]) = v[j];
        if constexpr (EPI == EPI_RESID_LN) {
            // x * gamma, and the statistics of the row's 32 columns (8 here, 24 in the lanes 16, 32, 48 away)
            float sum = 0.f, dev = 0.f;
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const half4v h = {(f16)(v[j][0] * g[j][0]), (f16)(v[j][1] * g[j][1]), (f16)(v[j][2] * g[j][2]),
                                  (f16)(v[j][3] * g[j][3])};
                if (live) *(half4v*)((f16*)p.ln_h + (int64_t)m * p.N + col[j]) = h;
                sum += (v[j][0] + v[j][1]) + (v[j][2] + v[j][3]);
            }
            sum += __shfl_xor(sum, 16, 64);
            sum += __shfl_xor(sum, 32, 64);
            const float mean = sum * (1.0f / 32.0f);
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e) dev += (v[j][e] - mean) * (v[j][e] - mean);
            dev += __shfl_xor(dev, 16, 64);
            dev += __shfl_xor(dev, 32, 64);
            if (live && lg == 0) ((float2v*)p.ln_stats)[(int64_t)m * (p.N / 32) + n0 / 32] = float2v{mean, dev};
        }
    }
}

template <int TM, int KG, int D, int WT>
static void run_rows(int epi, const GemmParams& p, hipStream_t s) {
    GemmParams q = p;
    const int nbm = cdiv(p.M, 16 * TM), nbn = p.N / 32;
    // band split over the XCDs with the fewest L2-miss bytes
    q.xcd_gm = 1;
    double best = 1e300;
    const double wb = WT == GT_Q8_0 ? 34.0 / 32 : WT == GT_Q4_K ? 0.75 : 2.0;
    for (int gm : {1, 2, 4, 8}) {
        if (gm > nbm || 8 / gm > nbn) continue;
        const double cost = (8.0 / gm) * 2.0 * p.M + gm * wb * p.N;
        if (cost < best) {
            best = cost;
            q.xcd_gm = gm;
        }
    }
    const dim3 grid(nbm * nbn), block(64 * KG);
    switch (epi) {
    case EPI_STORE: launch((gemm_rows_kernel<TM, KG, D, WT, EPI_STORE>), grid, block, 0, s, q); break;
    case EPI_STORE_F32: launch((gemm_rows_kernel<TM, KG, D, WT, EPI_STORE_F32>), grid, block, 0, s, q); break;
    case EPI_SILU: launch((gemm_rows_kernel<TM, KG, D, WT, EPI_SILU>), grid, block, 0, s, q); break;
    case EPI_RESID: launch((gemm_rows_kernel<TM, KG, D, WT, EPI_RESID>), grid, block, 0, s, q); break;
    case EPI_GLU: launch((gemm_rows_kernel<TM, KG, D, WT, EPI_GLU>), grid, block, 0, s, q); break;
    default: launch((gemm_rows_kernel<TM, KG, D, WT, EPI_RESID_LN>), grid, block, 0, s, q); break;
    }
    PKX_LAUNCH_CHECK();
}
template <int WT>
static bool rows_shape(int epi, const GemmParams& p, hipStream_t s) {
    const int64_t nb = p.N / 32, cus = device_cu_count();
    const int64_t t1 = cdiv(p.M, 16) * nb, t2 = cdiv(p.M, 32) * nb, t4 = cdiv(p.M, 64) * nb;
    // Lines from a sweep on MI355X over M = 2 .. 1000 and the encoders' (N, K), us, this
    // kernel against the one the product took before:
    // one tile of 16 rows per CU (M = 125, N = 1024, K = 1024: 4.4 against 11.1)
    if (t1 <= cus) {
        run_rows<1, 8, 2, WT>(epi, p, s);
        return true;
    }
    // of 32 rows (M = 250, N = 1024: K = 1024 5.1 against 9.5; K = 4096 8.3 with eight K groups,
    // 8.7 with four, 12.8 before; f16 weights, twice the LDS, 8.0 and 7.4)
    if (t2 <= cus) {
        if (WT != GT_F16 && p.K >= 2048) run_rows<2, 8, 2, WT>(epi, p, s);
        else run_rows<2, 4, 2, WT>(epi, p, s);
        return true;
    }
    // of 64 rows (M = 500, N = 1024: K = 1024 6.8 against 9.5, K = 4096 12.1 against 16.8); quantised
    // residual products also with two per CU (M = 1000, N = 1024: 10.2 against 11.2, 20.4 against
    // 25.3; f16 weights 11.3 against 10.5)
    const bool resid = epi == EPI_RESID || epi == EPI_RESID_LN || epi == EPI_STORE_F32;
    if (t4 <= cus || (WT != GT_F16 && resid && p.M <= 1024 && t4 <= 2 * cus)) {
        run_rows<4, 4, 2, WT>(epi, p, s);
        return true;
    }
    // quantised: three 32-row tiles per CU (M = 250, N = 3072, K = 1024: 8.8 against 10.2; four,
    // N = 4096: 11.1 against 10.8; f16 weights at three, M = 749, N = 1024: 9.9 against 8.9), two where
    // K is below 512 (K = 256: M = 96, N = 4352 1.6 per CU, 10% faster, M = 640, N = 1024, 2.5, 5.7 against 5.3; GLU
    // gains at three too)
    const int64_t per_cu = p.K >= 512 || epi == EPI_GLU ? 3 : 2;
    if (WT != GT_F16 && t2 <= per_cu * cus) {
        run_rows<2, 4, 2, WT>(epi, p, s);
        return true;
    }
    return false;
}

static bool gemm_rows_supported(int wtype, int epi, const GemmParams& p) {
    if (wtype != GT_F16 && wtype != GT_Q8_0 && wtype != GT_Q4_K) return false;
    if (epi != EPI_STORE && epi != EPI_STORE_F32 && epi != EPI_SILU && epi != EPI_RESID && epi != EPI_GLU &&
        epi != EPI_RESID_LN)
        return false;
    if (p.N % 32 || p.K % 64 || p.ldy % 4 || (p.fold_stats && p.fold_groups != p.K / 32)) return false;
    // 16-byte accesses to every operand
    uintptr_t at = (uintptr_t)p.A | (uintptr_t)p.Wq | (uintptr_t)p.Ws | (uintptr_t)p.Y | (uintptr_t)p.bias |
                   (uintptr_t)p.fold_stats | (uintptr_t)p.fold_c1 | (uintptr_t)p.ln_g | (uintptr_t)p.ln_h |
                   (uintptr_t)p.res_g | (uintptr_t)p.res_b;
    if (at & 15) return false;
    // 32-bit offsets: the weights, and the rows of a tile
    const int64_t rows = p.ldw > 0 ? p.ldw : p.N;
    return rows * p.K * 2 < ((int64_t)1 << 31) && p.lda < (1 << 20);
}

bool launch_gemm_rows(int wtype, int epi, const GemmParams& p, hipStream_t s) {
    if (!gemm_rows_supported(wtype, epi, p)) return false;
    switch (wtype) {
    case GT_F16: return rows_shape<GT_F16>(epi, p, s);
    case GT_Q8_0: return rows_shape<GT_Q8_0>(epi, p, s);
    default: return rows_shape<GT_Q4_K>(epi, p, s);
    }
}

}  // namespace pkx
