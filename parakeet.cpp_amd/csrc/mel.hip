// Log-mel front end: pk::MelFrontend::compute (src/mel.cpp:99-185) on a batch
// of clips, stacked to T_max like build_mel_batch (src/model.cpp:114-146).
//
// The reference computes in f64 on the CPU: preemphasis, a radix-2 FFT whose
// twiddles advance by complex multiplication (src/fft.cpp:9-51), the power
// spectrum, the filterbank sum and the log; f32 only where it rounds (the
// windowed frame, the FFT output).  Every kernel here keeps those f32 rounding
// points, f64 between them, and contracts nothing by itself.
//
// mel_spec_kernel: each wave runs the reference's butterflies, in its order of
// operations and with its twiddle recurrence (a table built on the host), on one
// frame at a time in LDS (complex f64): per-frame results match the reference's up
// to the libm ulp of sqrt/pow/log.
// mel_spec512_kernel (n_fft 512, mag_power 2, a filterbank that fits its LDS):
// persistent workgroups over groups of four frames of a clip, a frame a wave.  The
// frame's 512 real samples are a 256-point complex FFT (x[2n] + i x[2n+1]) of four
// radix-4 stages, four values per lane in registers and one LDS exchange between
// stages, then split into the 257 bins; directly computed twiddles, fused complex
// multiplies, no sqrt or pow.  It differs from the reference's butterflies by f64
// ulps (windowed noise, rms error against 80 bits 2.7e-16 of the rms; theirs
// 4.0e-15), far below the f32 rounding of the bins, which they now and then move to
// the neighbouring f32 value.
// Both keep the frames' power spectra in LDS; the workgroup then computes the
// filterbank sums of its frames (one f64 chain per output, summed in bin order)
// and writes log-mel.
// mel_norm_kernel: one workgroup per (mel bin, clip): per-feature mean and
// unbiased std over the clip's first S/hop frames, normalisation, zeroing of
// the rest of the row up to T_max.
#pragma clang fp contract(off)

#include <algorithm>
#include <cmath>
#include <cstring>

#include "common.hpp"
#include "mel.hpp"

namespace pkx {

struct MelParams {
    const float* pcm;
    int64_t S_stride;
    const int* meta;           // samples of each clip, or null: in inl
    int inl[MEL_INLINE_CLIPS];
    const float* window;       // [n_fft]
    const float* fb;           // [n_mels][n_bins]
    const double* tw;          // [n_fft - 1][2]: stage of half-length h uses rows h-1 .. 2h-2
    const double* tw512;       // n_fft 512: [512][2] = exp(-2 pi i k / 512)
    const int4* span;          // [n_mels]: the filter's nonzero bins [x, y), packed offset z
    const float* fb_packed;    // the filters' values over their spans, back to back
    int fb_nnz;
    float* out;                // [B][n_mels][T_max]
    int T_max, n_fft, log2n, hop, n_mels, n_bins, per_feature;
    float preemph, mag_power, log_guard;
    __device__ __forceinline__ int samples(int b) const { return meta ? meta[b] : inl[b]; }
    // frames of an S-sample clip (MelFront::frames)
    __device__ __forceinline__ int frames(int S) const { return S <= 0 || S + 2 * (n_fft / 2) < n_fft ? 0 : 1 + (S + 2 * (n_fft / 2) - n_fft) / hop; }
};

// Filterbank + log (src/mel.cpp:82-89) of a workgroup's FB frames, one f64
// chain per output summed in bin order over the filter's nonzero span only:
// every other bin would add fb * power = +-0, which leaves the sum unchanged.
// Four bins' operands are read at a time (LDS latency is what bounds the
// chain).  Output (m, f) with f fastest.
// LDS: the filter values are in fbs.
template <int FB, bool LDS>
__device__ __forceinline__ void mel_bank(const MelParams& p, const double (*pw)[MEL_MAX_NFFT / 2 + 1], const float* fbs,
                                         const int4* spans, int b, int t0, int T) {
    const int tid = threadIdx.x, f = tid & (FB - 1), t = t0 + f;
    for (int m = tid / FB; m < p.n_mels; m += 256 / FB) {
        const int4 sp = spans[m];   // {first bin, end bin, packed offset, -}
        double acc = 0.0;
        auto run = [&](const float* w) {
            for (int k = sp.x; k < sp.y; k += 4) {
                float wv[4];
                double pv[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int kk = min(k + e, sp.y - 1);
                    wv[e] = w[kk - sp.x];
                    pv[e] = pw[f][kk];
                }
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (k + e < sp.y) acc += (double)wv[e] * pv[e];
            }
        };
        if constexpr (LDS) run(fbs + sp.z);
        else run(p.fb_packed + sp.z);
        if (t < T) p.out[((int64_t)b * p.n_mels + m) * p.T_max + t] = (float)log(acc + (double)p.log_guard);
    }
}

// The power of one bin from its f32-rounded value (src/mel.cpp:73-79, fft.cpp:70-71).
// pow(sqrt(x), 2) is x up to its own rounding: mag_power 2 takes x.
__device__ __forceinline__ double sq_abs(double re64, double im64) {
    const float re = (float)re64, im = (float)im64;
    return (double)re * re + (double)im * im;
}
__device__ __forceinline__ double mel_power(const MelParams& p, double re64, double im64) {
    const double sq = sq_abs(re64, im64);
    if (p.mag_power == 2.0f) return sq;
    const double mag = sqrt(sq);
    return p.mag_power == 1.0f ? mag : pow(mag, (double)p.mag_power);
}

struct Cplx {
    double x, y;
};
__device__ __forceinline__ Cplx operator+(Cplx a, Cplx b) { return {a.x + b.x, a.y + b.y}; }
__device__ __forceinline__ Cplx operator-(Cplx a, Cplx b) { return {a.x - b.x, a.y - b.y}; }
__device__ __forceinline__ Cplx cmul(Cplx a, Cplx b) {
    return {fma(a.x, b.x, -(a.y * b.y)), fma(a.x, b.y, a.y * b.x)};
}

// A workgroup takes groups of four frames, one a wave, gridDim.x apart in the
// order (clip, frame): its twiddles, window, filter spans and weights are loaded
// once, and the next group's samples are on their way while the current one
// computes.  What bounds it is VALU issue (about 700 instructions a wave and
// frame, most of them f64 at a quarter rate: half of the time) and the LDS
// exchanges' latency, four waves a SIMD.  16 x 10 s, 128 filters on MI355X:
// 39 us; the radix-2 butterflies through LDS with pow() 152; this FFT with one
// group of four frames a workgroup 50, of eight 60 (two waves a SIMD).
__global__ __launch_bounds__(256, 4) void mel_spec512_kernel(MelParams p, int groups, int n_groups) {
    constexpr int FB = 4;
    constexpr int LEN = 256 + 256 / 32;        // one pad per 32 values: the stage writes spread over the banks
    __shared__ double ex[4][2][LEN];           // per wave: re, im
    __shared__ double pws[2][FB][MEL_MAX_NFFT / 2 + 1];
    __shared__ int4 sps[MEL_SPAN_LDS];
    __shared__ float2v wins[256];
    __shared__ float fbs[MEL_FB_LDS];
    const int tid = threadIdx.x, j = tid & 63, w = tid >> 6;
    const double pre = (double)p.preemph;

    // samples q - 1, q, q + 1 of n = j + 64 r, q = 2n past the frame's start (groups: frame groups of a clip)
    // (inside: every sample of this wave's frame and the one before it exist)
    struct Group {
        int b, t0, S, T;
        bool inside;
    };
    float v[4][3];
    auto fetch = [&](int g) {
        Group u;
        u.b = g / groups;
        u.t0 = (g - u.b * groups) * FB;
        u.S = p.samples(u.b);
        u.T = p.frames(u.S);
        const float* x = p.pcm + (int64_t)u.b * p.S_stride;
        const int q0 = __builtin_amdgcn_readfirstlane((u.t0 + w) * p.hop - 256);
        u.inside = q0 > 0 && q0 + 512 <= u.S;
        if (u.inside) {
            x += q0 + 2 * j;
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int e = 0; e < 3; ++e) v[r][e] = x[128 * r + e - 1];
        } else {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int q = q0 + 2 * (j + 64 * r);
#pragma unroll
                for (int e = 0; e < 3; ++e)
                    v[r][e] = u.t0 + w < u.T && q + e - 1 >= 0 && q + e - 1 < u.S ? x[q + e - 1] : 0.0f;
            }
        }
        return u;
    };
    int g = blockIdx.x;
    Group cur = fetch(g);
    wins[tid] = *(const float2v*)(p.window + 2 * tid);
    // twiddles: stage s (butterfly span N = 4^s, s = 1..3) exp(-2 pi i r (j % N) / 4N), and the split's
    // exp(-2 pi i k / 512), k = j, j + 64
    auto tw = [&](int k) { return Cplx{p.tw512[2 * k], p.tw512[2 * k + 1]}; };
    Cplx ts[3][3], tk[2];
#pragma unroll
    for (int s = 0; s < 3; ++s)
#pragma unroll
        for (int r = 1; r < 4; ++r) ts[s][r - 1] = tw((r * (j & ((4 << (2 * s)) - 1)) * (32 >> (2 * s))) & 511);
    tk[0] = tw(j);
    tk[1] = tw(j + 64);
    for (int i = tid; i < p.n_mels; i += 256) sps[i] = p.span[i];
    for (int i = tid; i < p.fb_nnz; i += 256) fbs[i] = p.fb_packed[i];
    __syncthreads();

    double *er = ex[w][0], *ei = ex[w][1];
    auto at = [](int i) { return i + (i >> 5); };
    // the wave's LDS operations complete in order: these only keep the compiler's order
    auto fence = [] { __builtin_amdgcn_wave_barrier(); asm volatile("" ::: "memory"); };
    for (int buf = 0;; buf ^= 1) {
        // windowed samples 2n, 2n + 1 (src/mel.cpp:67-69)
        Cplx z[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int q = (cur.t0 + w) * p.hop + 2 * (j + 64 * r) - 256;
            const float2v wn = wins[j + 64 * r];
            float f[2];
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                double d = (double)v[r][e + 1];
                if (p.preemph > 0.0f && (cur.inside || (q + e > 0 && q + e < cur.S))) d = (double)v[r][e + 1] - pre * (double)v[r][e];
                f[e] = (float)(d * (double)wn[e]);
            }
            z[r] = {(double)f[0], (double)f[1]};
        }
        const Group now = cur;
        g += gridDim.x;
        if (g < n_groups) cur = fetch(g);
        if (now.t0 < now.T) {   // uniform over the workgroup
            // Stockham stages: lane j takes values j + 64 r, leaves (j / N) 4N + j % N + r N
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const int N = 1 << (2 * s);
                if (s > 0) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) z[r] = {er[at(j + 64 * r)], ei[at(j + 64 * r)]};
                    fence();
#pragma unroll
                    for (int r = 1; r < 4; ++r) z[r] = cmul(z[r], ts[s - 1][r - 1]);
                }
                const Cplx a = z[0] + z[2], c = z[0] - z[2], d = z[1] + z[3], e = z[1] - z[3];
                z[0] = a + d;
                z[2] = a - d;
                z[1] = {c.x + e.y, c.y - e.x};   // c - i e
                z[3] = {c.x - e.y, c.y + e.x};
                const int base = (j / N) * 4 * N + (j & (N - 1));
                if (s < 3) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        er[at(base + r * N)] = z[r].x;
                        ei[at(base + r * N)] = z[r].y;
                    }
                    fence();
                }
            }
            // bins k and 256 - k from Z[k] and Z[256 - k]: this lane has k = j, j + 64 (r = 0, 1)
            // and hands over 128 + j, 192 + j
#pragma unroll
            for (int r = 2; r < 4; ++r) {
                er[at(64 * r + j)] = z[r].x;
                ei[at(64 * r + j)] = z[r].y;
            }
            fence();
            double* P = pws[buf][w];
#pragma unroll
            for (int r = 0; r < 2; ++r) {
                const int k = j + 64 * r, kc = (256 - k) & 255;
                Cplx c = {er[at(kc)], ei[at(kc)]};
                if (k == 0) c = z[0];
                const Cplx e = {0.5 * (z[r].x + c.x), 0.5 * (z[r].y - c.y)};      // even samples' bin
                const Cplx o = {0.5 * (z[r].y + c.y), 0.5 * (c.x - z[r].x)};      // odd samples' bin
                const Cplx x = cmul(o, tk[r]);
                P[k] = sq_abs(e.x + x.x, e.y + x.y);
                P[256 - k] = sq_abs(e.x - x.x, x.y - e.y);
            }
            if (j == 0) P[128] = sq_abs(z[2].x, -z[2].y);
            fence();
        }
        // one barrier a group: the spectra alternate between two buffers, and every wave is past
        // the filterbank of the group before when it writes this one's successor
        __syncthreads();
        if (now.t0 < now.T) mel_bank<FB, true>(p, pws[buf], fbs, sps, now.b, now.t0, now.T);
        if (g >= n_groups) break;
    }
}

__global__ __launch_bounds__(256) void mel_spec_kernel(MelParams p) {
    constexpr int FB = MEL_FRAMES_PER_BLOCK, RPL = MEL_MAX_NFFT / 64;
    __shared__ double2 buf[4][MEL_MAX_NFFT];
    __shared__ double pw[FB][MEL_MAX_NFFT / 2 + 1];
    __shared__ double2 tws[MEL_MAX_NFFT];
    __shared__ float fbs[MEL_FB_LDS];
    const int b = blockIdx.y, t0 = blockIdx.x * FB;
    const int S = p.samples(b), T = p.frames(S);
    if (t0 >= T) return;                               // uniform over the workgroup
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int N = p.n_fft, pad = N / 2;
    const float* x = p.pcm + (int64_t)b * p.S_stride;
    const double pre = (double)p.preemph;

    // every frame's windowed samples (src/mel.cpp:67-69) are loaded up front,
    // one global-memory round trip for the workgroup; twiddles and the
    // filterbank's nonzero values go to LDS
    float fr[FB / 4][RPL];
#pragma unroll
    for (int r = 0; r < FB / 4; ++r) {
        const int t = t0 + 4 * r + w;
#pragma unroll
        for (int ii = 0; ii < RPL; ++ii) {
            const int i = lane + 64 * ii;
            const int q = t * p.hop + i - pad;         // sample index of padded[t*hop + i]
            double v = 0.0;
            if (i < N && t < T && q >= 0 && q < S) {
                v = (double)x[q];
                if (p.preemph > 0.0f && q > 0) v = (double)x[q] - pre * (double)x[q - 1];
            }
            fr[r][ii] = i < N ? (float)(v * (double)p.window[i]) : 0.0f;
        }
    }
    for (int i = tid; i < N - 1; i += 256) tws[i] = make_double2(p.tw[2 * i], p.tw[2 * i + 1]);
    if (p.fb_nnz <= MEL_FB_LDS)
        for (int i = tid; i < p.fb_nnz; i += 256) fbs[i] = p.fb_packed[i];

    for (int r = 0; r < FB / 4; ++r) {
        const int f = 4 * r + w;
        double2* B2 = buf[w];
        // the frame in bit-reversed order (src/fft.cpp:14-22)
#pragma unroll
        for (int ii = 0; ii < RPL; ++ii) {
            const int i = lane + 64 * ii;
            if (i < N) B2[(int)(__brev((unsigned)i) >> (32 - p.log2n))] = make_double2((double)fr[r][ii], 0.0);
        }
        __syncthreads();
        // butterfly stages (src/fft.cpp:25-50)
        for (int s = 0, h = 1; s < p.log2n; ++s, h <<= 1) {
            for (int bi = lane; bi < N / 2; bi += 64) {
                const int k = bi & (h - 1), u = ((bi >> s) << (s + 1)) + k, v = u + h;
                const double2 tw = tws[h - 1 + k];
                const double2 a = B2[u], c = B2[v];
                const double tr = tw.x * c.x - tw.y * c.y;
                const double ti = tw.x * c.y + tw.y * c.x;
                B2[v] = make_double2(a.x - tr, a.y - ti);
                B2[u] = make_double2(a.x + tr, a.y + ti);
            }
            __syncthreads();
        }
        for (int k = lane; k < p.n_bins; k += 64) pw[f][k] = mel_power(p, B2[k].x, B2[k].y);
        __syncthreads();
    }
    if (p.fb_nnz <= MEL_FB_LDS) mel_bank<FB, true>(p, pw, fbs, p.span, b, t0, T);
    else mel_bank<FB, false>(p, pw, fbs, p.span, b, t0, T);
}

__device__ __forceinline__ double block_sum_f64(double v, double* red) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    __syncthreads();
    if (lane == 0) red[w] = v;
    __syncthreads();
    return (red[0] + red[1]) + (red[2] + red[3]);
}

// Rows of up to 256 NV frames stay in registers between the passes (NV = 0:
// longer ones are read again): what bounds the kernel is the latency of its
// dependent passes over a row.
template <int NV>
__global__ __launch_bounds__(256) void mel_norm_kernel(MelParams p) {
    __shared__ double red[4];
    const int m = blockIdx.x, b = blockIdx.y;
    const int S = p.samples(b), T = p.frames(S);
    float* row = p.out + ((int64_t)b * p.n_mels + m) * p.T_max;
    int keep = T;
    if (p.per_feature && T > 0) {
        // src/mel.cpp:157-182: mean and unbiased std over the first S/hop frames
        const int valid = min(S / p.hop, T);
        float x[NV > 0 ? NV : 1];
        if constexpr (NV > 0) {
#pragma unroll
            for (int i = 0; i < NV; ++i) x[i] = threadIdx.x + 256 * i < (unsigned)valid ? row[threadIdx.x + 256 * i] : 0.0f;
        }
        // f(frame, value) over this thread's frames, in order
        auto each = [&](auto&& f) {
            if constexpr (NV > 0) {
#pragma unroll
                for (int i = 0; i < NV; ++i)
                    if (threadIdx.x + 256 * i < (unsigned)valid) f(threadIdx.x + 256 * i, x[i]);
            } else {
                for (int t = threadIdx.x; t < valid; t += 256) f(t, row[t]);
            }
        };
        double s = 0.0;
        each([&](int, float v) { s += (double)v; });
        const double mean = valid > 0 ? block_sum_f64(s, red) / (double)valid : 0.0;
        double q = 0.0;
        each([&](int, float v) {
            const double d = (double)v - mean;
            q += d * d;
        });
        const double ss = block_sum_f64(q, red);
        const double var = valid > 1 ? ss / (double)(valid - 1) : 0.0;
        const double sd = sqrt(var) + 1e-5;
        each([&](int t, float v) { row[t] = (float)(((double)v - mean) / sd); });
        keep = valid;
    }
    for (int t = keep + threadIdx.x; t < p.T_max; t += 256) row[t] = 0.0f;
}

MelFront::MelFront(const MelConfig& c, const float* window, int win_len, const float* fb) : cfg_(c) {
    require(c.n_fft >= 64 && c.n_fft <= MEL_MAX_NFFT && (c.n_fft & (c.n_fft - 1)) == 0,
            "mel: n_fft must be a power of two in [64, 512]");
    require(c.hop > 0 && c.n_mels > 0 && c.mag_power > 0.0f, "mel: hop, n_mels and mag_power must be positive");
    require(window && win_len > 0 && win_len <= c.n_fft, "mel: window of 1..n_fft values required");
    require(fb != nullptr, "mel: filterbank required");
    n_bins_ = c.n_fft / 2 + 1;
    log2n_ = 0;
    while ((1 << log2n_) < c.n_fft) ++log2n_;
    // window centre-padded to n_fft (src/mel.cpp:31-46)
    std::vector<float> wpad((size_t)c.n_fft, 0.0f);
    if (win_len == c.n_fft) {
        std::memcpy(wpad.data(), window, sizeof(float) * (size_t)c.n_fft);
    } else {
        const int left = (c.n_fft - win_len) / 2;
        for (int i = 0; i < win_len && left + i < c.n_fft; ++i)
            if (left + i >= 0) wpad[(size_t)(left + i)] = window[i];
    }
    // the twiddles each butterfly of src/fft.cpp:28-48 uses: w_0 = 1,
    // w_{k+1} = w_k * (cos a, sin a), a = -2 pi / len, same f64 operations
    std::vector<double> tw((size_t)(c.n_fft - 1) * 2);
    for (int len = 2; len <= c.n_fft; len <<= 1) {
        const double ang = -2.0 * M_PI / len, wr = std::cos(ang), wi = std::sin(ang);
        double cr = 1.0, ci = 0.0;
        for (int k = 0; k < len / 2; ++k) {
            tw[2 * (size_t)(len / 2 - 1 + k)] = cr;
            tw[2 * (size_t)(len / 2 - 1 + k) + 1] = ci;
            const double nr = cr * wr - ci * wi, ni = cr * wi + ci * wr;
            cr = nr;
            ci = ni;
        }
    }
    if (c.n_fft == 512) {
        std::vector<double> t5(2 * 512);
        for (int k = 0; k < 512; ++k) {
            const double a = -2.0 * M_PI * k / 512;
            t5[2 * (size_t)k] = std::cos(a);
            t5[2 * (size_t)k + 1] = std::sin(a);
        }
        PKX_HIP(hipMalloc(&d_tw512_, sizeof(double) * t5.size()));
        PKX_HIP(hipMemcpy(d_tw512_, t5.data(), sizeof(double) * t5.size(), hipMemcpyHostToDevice));
    }
    // each filter's nonzero span and its values packed back to back (the
    // kernel skips the exact zeros outside the span)
    std::vector<int4> span((size_t)c.n_mels);
    std::vector<float> packed;
    for (int m = 0; m < c.n_mels; ++m) {
        int lo = n_bins_, hi = 0;
        for (int k = 0; k < n_bins_; ++k)
            if (fb[(size_t)m * n_bins_ + k] != 0.0f) {
                lo = std::min(lo, k);
                hi = k + 1;
            }
        if (lo >= hi) lo = hi = 0;
        span[(size_t)m] = make_int4(lo, hi, (int)packed.size(), 0);
        for (int k = lo; k < hi; ++k) packed.push_back(fb[(size_t)m * n_bins_ + k]);
    }
    fb_nnz_ = (int)packed.size();
    PKX_HIP(hipMalloc(&d_span_, sizeof(int4) * span.size()));
    PKX_HIP(hipMemcpy(d_span_, span.data(), sizeof(int4) * span.size(), hipMemcpyHostToDevice));
    PKX_HIP(hipMalloc(&d_fbp_, sizeof(float) * std::max<size_t>(packed.size(), 1)));
    if (!packed.empty())
        PKX_HIP(hipMemcpy(d_fbp_, packed.data(), sizeof(float) * packed.size(), hipMemcpyHostToDevice));
    PKX_HIP(hipMalloc(&d_window_, sizeof(float) * (size_t)c.n_fft));
    PKX_HIP(hipMalloc(&d_fb_, sizeof(float) * (size_t)c.n_mels * n_bins_));
    PKX_HIP(hipMalloc(&d_tw_, sizeof(double) * tw.size()));
    PKX_HIP(hipMemcpy(d_window_, wpad.data(), sizeof(float) * wpad.size(), hipMemcpyHostToDevice));
    PKX_HIP(hipMemcpy(d_fb_, fb, sizeof(float) * (size_t)c.n_mels * n_bins_, hipMemcpyHostToDevice));
    PKX_HIP(hipMemcpy(d_tw_, tw.data(), sizeof(double) * tw.size(), hipMemcpyHostToDevice));
}

MelFront::~MelFront() {
    for (void* q : {(void*)d_window_, (void*)d_fb_, (void*)d_tw_, (void*)d_tw512_, (void*)d_meta_, d_span_, (void*)d_fbp_})
        if (q) (void)hipFree(q);
}

int MelFront::frames(int S) const {
    if (S <= 0) return 0;
    const int padded = S + 2 * (cfg_.n_fft / 2);
    return padded >= cfg_.n_fft ? 1 + (padded - cfg_.n_fft) / cfg_.hop : 0;
}

void MelFront::forward(const float* pcm, int B, int64_t S_stride, const int* n_samples, float* out, int T_max,
                       int* T_out, hipStream_t s) {
    require(B > 0 && T_max >= 0 && n_samples && T_out && out, "mel: bad batch arguments");
    require(B <= 65535, "mel: at most 65535 clips per call");
    meta_.assign(n_samples, n_samples + B);
    for (int b = 0; b < B; ++b) {
        require(n_samples[b] >= 0 && n_samples[b] <= S_stride, "mel: clip length outside [0, S_stride]");
        const int T = frames(n_samples[b]);
        require(T <= T_max, "mel: T_max smaller than a clip's frame count");
        T_out[b] = T;
    }
    require(pcm != nullptr || S_stride == 0 || *std::max_element(n_samples, n_samples + B) == 0,
            "mel: null pcm");
    if (T_max == 0) return;
    MelParams p{};
    p.pcm = pcm;
    p.S_stride = S_stride;
    if (B <= MEL_INLINE_CLIPS) {
        std::copy(meta_.begin(), meta_.end(), p.inl);   // the lengths travel with the kernel arguments
    } else {
        if (meta_cap_ < B) {
            if (d_meta_) PKX_HIP(hipFree(d_meta_));
            d_meta_ = nullptr;
            PKX_HIP(hipMalloc(&d_meta_, sizeof(int) * (size_t)B));
            meta_cap_ = B;
        }
        PKX_HIP(hipMemcpyAsync(d_meta_, meta_.data(), sizeof(int) * (size_t)B, hipMemcpyHostToDevice, s));
        p.meta = d_meta_;
    }
    p.window = d_window_;
    p.fb = d_fb_;
    p.tw = d_tw_;
    p.tw512 = d_tw512_;
    p.span = (const int4*)d_span_;
    p.fb_packed = d_fbp_;
    p.fb_nnz = fb_nnz_;
    p.out = out;
    p.T_max = T_max;
    p.n_fft = cfg_.n_fft;
    p.log2n = log2n_;
    p.hop = cfg_.hop;
    p.n_mels = cfg_.n_mels;
    p.n_bins = n_bins_;
    p.per_feature = cfg_.per_feature;
    p.preemph = cfg_.preemph;
    p.mag_power = cfg_.mag_power;
    p.log_guard = cfg_.log_guard;
    const int64_t n_groups = (int64_t)cdiv(T_max, 4) * B;
    if (cfg_.n_fft != 512 || cfg_.mag_power != 2.0f || fb_nnz_ > MEL_FB_LDS || cfg_.n_mels > MEL_SPAN_LDS ||
        n_groups >= ((int64_t)1 << 31) - (1 << 20)) {   // its group numbers are 32-bit
        launch(mel_spec_kernel, dim3(cdiv(T_max, MEL_FRAMES_PER_BLOCK), B), dim3(256), 0, s, p);
    } else {
        // four workgroups a CU (what their LDS and registers allow), each with its share of the groups
        launch(mel_spec512_kernel, dim3((unsigned)std::min<int64_t>(n_groups, 4 * device_cu_count())), dim3(256), 0, s, p,
               cdiv(T_max, 4), (int)n_groups);
    }
    PKX_LAUNCH_CHECK();
    const dim3 rows(cfg_.n_mels, B);
    if (T_max <= 1024) launch(mel_norm_kernel<4>, rows, dim3(256), 0, s, p);
    else if (T_max <= 4096) launch(mel_norm_kernel<16>, rows, dim3(256), 0, s, p);
    else launch(mel_norm_kernel<0>, rows, dim3(256), 0, s, p);
    PKX_LAUNCH_CHECK();
    // the host copy of meta_ is reused by the next call: finish the upload first
    PKX_HIP(hipStreamSynchronize(s));
}

}  // namespace pkx
