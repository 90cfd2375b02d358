// f32 GEMM for gfx950: Y = epilogue(X[M][K] . W[N][K]^T), f32 weights, on
// v_mfma_f32_16x16x4_f32, for products with too few output tiles to fill the
// chip (an utterance at a time, a head over a batch).
//
// What bounds those is latency, not the matrix pipe: the barrier-per-slab
// kernel (gemm_f32_kernel in gemm.hip) walks K = 2048 in 64 dependent steps of
// ~0.4 us with 64 tiles for 256 CUs.  Here the waves of a workgroup split K,
// each with its own DMA ring and no barrier, and tiles shrink to 16 x 32.
// M = 125, N = 512 on MI355X: K = 2048 24.8 -> 9.0 us, K = 512 8.1 -> 5.0 us
// (the matrix pipe alone: 1.7 and 0.4 us).
#include "gemm.hpp"
#include "gemm_common.hpp"

namespace pkx {

// A workgroup of KG waves computes one tile of 16 TM x 16 TN, each wave over a
// contiguous 1/KG of K, the partial tiles summed through LDS in group order
// (deterministic).  Every wave streams its own
// operand rows, 32 K columns (whole 128-byte lines) a step, through a private
// D-stage LDS ring filled by DMA, so the loop has no barrier.  The weights are
// the MFMA's A operand, so a lane ends with 4 consecutive output columns of
// one row (16-byte stores).  glu: a wave's first TN / 2 column blocks are the
// inputs of 8 TN output channels and the others their gates (pointwise_conv1
// rows are stored in alternating 32-row groups of inputs and gates).
template <int TM, int TN, int KG, int D>
__global__ __launch_bounds__(64 * KG) void gemm_f32_ks_kernel(GemmParams p, int epi) {
    static_assert(TN % 2 == 0, "GLU pairs column blocks within a wave");
    constexpr int BM = 16 * TM, BN = 16 * TN;
    constexpr int NT = TM * TN;                   // 16 x 16 blocks of the tile
    constexpr int NI = 2 * (TM + TN);             // DMA instructions per step: 8 rows x 128 bytes each
    constexpr int STAGE = NI * 1024;
    constexpr int RED = KG * NT * 1024;
    constexpr int SMEM = KG * D * STAGE > RED ? KG * D * STAGE : RED;
    static_assert(SMEM <= 160 * 1024 && (D - 1) * NI < 64, "LDS ring");
    __shared__ __attribute__((aligned(1024))) uint8_t smem[SMEM];

    const int tid = threadIdx.x, lane = tid & 63;
    const int kg = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lr = lane & 15, lg = lane >> 4;
    const int nbm = cdiv_dev(p.M, BM), nbn = cdiv_dev(p.N, BN);
    int bm_, bn_;
    xcd_tile_2d(blockIdx.x, nbm, nbn, p.xcd_gm, bm_, bn_);
    const int m0 = bm_ * BM, n0 = bn_ * BN;
    const bool glu = epi == EPI_GLU;

    // rows past the edge and columns past K lie past the resources' ends (zeros)
    const int mb = min(m0, p.M - 1), nb = glu ? 64 * (n0 / 64) : min(n0, p.N - 1);   // GLU: N % 64 == 0
    const auto ra = make_rsrc((const float*)p.A + (int64_t)mb * p.lda, ((int64_t)(p.M - mb - 1) * p.lda + p.K) * 4);
    const auto rw = make_rsrc((const float*)p.Wq + (int64_t)nb * p.K, (int64_t)(p.N - nb) * p.K * 4);
    // DMA instruction u: rows 8 (u % 2) .. + 7 of 16-row block u / 2 (the TM
    // activation blocks, then the TN weight blocks); lane l brings the 16-byte
    // chunk (l % 8) ^ (l / 8) of row l / 8 (the swizzle keeps the reads below
    // free of bank conflicts)
    const int dr = lane >> 3, dc = (lane & 7) ^ dr;
    uint32_t src[NI];
#pragma unroll
    for (int u = 0; u < NI; ++u) {
        const int i = u / 2, r = 8 * (u & 1) + dr;
        if (i < TM) {
            const int64_t o = ((int64_t)(m0 - mb + 16 * i + r) * p.lda + 4 * dc) * 4;
            src[u] = o < (int64_t)OOB ? (uint32_t)o : OOB;
        } else {
            const int j = i - TM;
            const int c = n0 / 2 + 16 * (j % (TN / 2)) + r;
            const int n = glu ? 64 * (c >> 5) + (c & 31) + (j >= TN / 2 ? 32 : 0) : n0 + 16 * j + r;
            const int64_t o = ((int64_t)(n - nb) * p.K + 4 * dc) * 4;
            src[u] = n < p.N && o < (int64_t)OOB ? (uint32_t)o : OOB;
        }
    }
    const int nst = cdiv_dev(p.K, 32);
    const int s0 = nst * kg / KG, s1 = nst * (kg + 1) / KG;
    uint8_t* ring = smem + kg * D * STAGE;
    // one step's loads; past the group's range they read nothing, so that the
    // number in flight stays the same
    auto issue = [&](int d, int st) {
        const uint32_t ko = st < s1 && 32 * st + 4 * dc < p.K ? 128u * st : OOB;
#pragma unroll
        for (int u = 0; u < NI; ++u) lds_dma16(u / 2 < TM ? ra : rw, ring + d * STAGE + u * 1024, (src[u] | (ko & OOB)) + (ko & ~OOB), 0);
    };
    float4v acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = float4v{0.f, 0.f, 0.f, 0.f};
    auto compute = [&](int d) {
        const uint8_t* base = ring + d * STAGE + lr * 128;
        float4v f[TM + TN][2];
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int i = 0; i < TM + TN; ++i)
                f[i][c] = *(const float4v*)(base + 2048 * i + 16 * ((4 * c + lg) ^ (lr & 7)));
        // lane l holds k = 4 (l / 16) + e of the 16-column half for both operands
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int i = 0; i < TM; ++i)
#pragma unroll
                    for (int j = 0; j < TN; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(f[TM + j][c][e], f[i][c][e], acc[i][j], 0, 0, 0);
    };
#pragma unroll
    for (int d = 0; d < D - 1; ++d) issue(d, s0 + d);
    for (int st = s0, d = 0; st < s1; ++st) {
        // stage d - 1 was read in the last step (its reads were consumed by the MFMAs)
        issue(d == 0 ? D - 1 : d - 1, st + D - 1);
        wait_vmcnt<(D - 1) * NI>();
        compute(d);
        __builtin_amdgcn_s_waitcnt(0xc07f);   // lgkmcnt(0): this stage's reads are done before it is refilled
        d = d + 1 == D ? 0 : d + 1;
    }
    wait_vmcnt<0>();

    __syncthreads();
    float4v* red = (float4v*)smem;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) red[(kg * NT + i * TN + j) * 64 + lane] = acc[i][j];
    __syncthreads();
    auto sum = [&](int t) {   // block t of the tile, in group order
        float4v v = red[t * 64 + lane];
#pragma unroll
        for (int g = 1; g < KG; ++g) v += red[(g * NT + t) * 64 + lane];
        return v;
    };
    // The epilogue's arguments as values: read through p inside the branches
    // below, the compiler merges the branches' loads into one from a chosen
    // address, keeps a copy of the struct per thread for it, and finds that
    // copy through the dispatch packet in host memory (7 - 10 us per launch).
    const float alpha = p.alpha;
    const int* const valid = p.valid;
    const float *const bias = p.bias, *const bias2 = p.bias2;
    float* const Y = (float*)p.Y;
    const int64_t ldy = p.ldy;
    const int M = p.M, N = p.N, T = p.T, F = p.trF;
#pragma clang loop unroll(disable)
    for (int t = kg; t < NT; t += KG) {
        const int i = t / TN, j = t % TN;
        // lane: row m, columns n .. n + 3 (GLU: output channels n .. n + 3)
        const int m = m0 + 16 * i + lr;
        const int n = (glu ? n0 / 2 : n0) + 16 * j + 4 * lg;
        if (glu && j >= TN / 2) continue;
        if (m >= M || n >= (glu ? N / 2 : N)) continue;
        float4v v = sum(t);
        const int nv = min(4, (glu ? N / 2 : N) - n), na = glu ? 64 * (n >> 5) + (n & 31) : n;
        if (bias) {
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] += r < nv ? bias[na + r] : 0.f;
        }
        if (glu) {
            float4v g = sum(t + TN / 2);
            if (bias) {
#pragma unroll
                for (int r = 0; r < 4; ++r) g[r] += bias[na + 32 + r];
            }
            const bool dead = valid && m % T >= valid[m / T];
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] = dead ? 0.f : v[r] * sigmoid_dev(g[r]);
        } else if (epi == EPI_SILU) {
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] = silu_dev(v[r]);
        } else if (epi == EPI_STORE || epi == EPI_STORE_F32 || epi == EPI_RESID) {
            v *= alpha;
        } else {   // RELU, RELU_TR, RELU2_F32
            if (epi == EPI_RELU2_F32 && bias2) {
#pragma unroll
                for (int r = 0; r < 4; ++r) v[r] += r < nv ? bias2[n + r] : 0.f;
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] = v[r] > 0.f ? v[r] : 0.f;
        }
        if (epi == EPI_RELU_TR) {
            // rows are pixels (b, t, f), f fastest; store [b][t][c][f] (channel-major flatten)
            const int bt = m / F, f = m - bt * F;
            const bool dead = valid && bt % T >= valid[bt / T];
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (r < nv) Y[((int64_t)bt * N + n + r) * F + f] = dead ? 0.f : v[r];
            continue;
        }
        float* y = Y + (int64_t)m * ldy + n;
        if (nv == 4 && (ldy & 3) == 0 && ((uintptr_t)Y & 15) == 0) {
            *(float4v*)y = epi == EPI_RESID ? *(const float4v*)y + v : v;
        } else {
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (r < nv) y[r] = epi == EPI_RESID ? y[r] + v[r] : v[r];
        }
    }
}

template <int TM, int TN, int KG, int D>
static void run_f32_ks(int epi, const GemmParams& p, hipStream_t s) {
    GemmParams q = p;
    const int nbm = cdiv(p.M, 16 * TM), nbn = cdiv(p.N, 16 * TN);
    // band split over the XCDs with the fewest L2-miss bytes
    q.xcd_gm = 1;
    double best = 1e300;
    for (int gm : {1, 2, 4, 8}) {
        if (gm > nbm || 8 / gm > nbn) continue;
        const double cost = (8.0 / gm) * p.M + (double)gm * p.N;
        if (cost < best) {
            best = cost;
            q.xcd_gm = gm;
        }
    }
    launch((gemm_f32_ks_kernel<TM, TN, KG, D>), dim3(nbm * nbn), dim3(64 * KG), 0, s, q, epi);
    PKX_LAUNCH_CHECK();
}

// The lines below are from a sweep on MI355X over M = 12 .. 6000 and the
// (N, K) of the f32 products (us, this kernel's tile against the best shape of
// the barrier-per-slab kernel).
bool launch_gemm_f32_ks(int epi, const GemmParams& p, hipStream_t s) {
    if (epi == EPI_GLU_DW || epi == EPI_RESID_LN) return false;
    // the DMA's 16-byte pieces, and row offsets within a tile below 2 GB
    if (((uintptr_t)p.A | (uintptr_t)p.Wq) & 15 || p.lda % 4 || p.K > (1 << 20) || p.lda > (1 << 20)) return false;
    // short K leaves nothing to split: the other kernel is faster, but for GLU, which costs it 128-column
    // tiles (K = 128: M = 1000, N = 128 4.3 against 5.0, M = 2, N = 1025 3.9 against 4.4; GLU M = 125, N = 256 7.8
    // against 4.6)
    if (p.K < 256 && epi != EPI_GLU) return false;
    const int64_t t12 = (int64_t)cdiv(p.M, 16) * cdiv(p.N, 32), t22 = (int64_t)cdiv(p.M, 32) * cdiv(p.N, 32);
    const int cus = device_cu_count();
    if (t12 <= cus) {
        // one 16 x 32 tile per CU: eight K groups for long K (M = 125, N = 512: K = 2048
        // 9.0 with eight, 9.9 with four, 24.8 old; K = 512 5.0, 5.0, 8.1)
        if (p.K >= 1024) run_f32_ks<1, 2, 8, 2>(epi, p, s);
        else run_f32_ks<1, 2, 4, 2>(epi, p, s);
        return true;
    }
    // 32 x 32 tiles, two workgroups of four K groups per CU.  K >= 1024 pays up to
    // about eight tiles per CU (M = 2000: N = 512, K = 2048 46.1 against 57.3; N = 640,
    // K = 1024 33.4 against 35.9; N = 1025, K = 1024 59.0 against 61.7), K = 512 up to two
    // (M = 1000, N = 512 9.7 against 10.6; M = 375, N = 2048, three per CU: 14.5 against
    // 13.6), K = 256 not at all (M = 1250, N = 256: 7.4 against 6.5)
    if ((p.K >= 1024 && t22 <= 8 * cus + cus / 4) || (p.K >= 512 && t22 <= 2 * cus)) {
        run_f32_ks<2, 2, 4, 2>(epi, p, s);
        return true;
    }
    // GLU: the barrier-per-slab kernel needs 128-column tiles; single-wave 32 x 32 tiles with five
    // co-resident per CU beat them up to nine tiles per CU, about one round of its tiles (K = 512,
    // N = 1024: M = 1000 15.7 against 19.5, M = 2000 23.0 against 29.1, M = 2250 31.2 against 37.6; M = 2500,
    // 9.9 tiles, 41.6 against 37.8, M = 4000 51.7 against 47.0)
    if (epi == EPI_GLU && t22 <= 9 * cus) {
        run_f32_ks<2, 2, 1, 2>(epi, p, s);
        return true;
    }
    return false;
}

}  // namespace pkx
