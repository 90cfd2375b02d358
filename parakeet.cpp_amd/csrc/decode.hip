// Greedy transducer decode on the device: transducer_greedy_batch
// (src/transducer_batch.cpp:24-213) with the prediction net of
// src/prediction.cpp:118-178 and the joint of src/joint.cpp:37-63,106-143.
//
// All B items advance in lockstep rounds; one round is L + 3 launches:
//   lstm layer l (dec_mm_kernel<MM_LSTM>): z = [x_l | h_l] . [W_ih | W_hh]^T
//       + (b_ih + b_hh) for the 4 gate rows of each hidden unit, then the
//       cell c' = s(f) c + s(i) tanh(g), h' = s(o) tanh(c') in the same kernel
//   joint (dec_mm_kernel<MM_JOINT>): f = ReLU(enc_proj[t_b] + W_pred g + b_pred)
//   logits (dec_mm_kernel<MM_PLAIN>): W_out f + b_out
//   greedy_rule_kernel: argmaxes, the TDT / RNNT rule of the per-item loops,
//       token records, state commit on emit.
// The products run on the f32 matrix pipe (16 rows x 16 items a workgroup, K
// split over eight waves; the quantisable joint projections are dequantised to
// f32 at load).  Every round recomputes the LSTM for all items: from an
// unchanged committed state it reproduces the same g bit for bit (the
// reference's g_valid cache skips that recomputation, with the same result).
// The host launches rounds in chunks and reads the active flags of one chunk
// while the next runs; rounds after the last item finished change nothing.
//
// Device state: X_l holds [x_l | committed h_l] for layer l (x_0 = embedding of
// the last token, zeros before the first emission; x_l = this round's
// h'_{l-1}), so a commit writes straight into the next round's input.  X_l, g
// and f are kept in the order the products read them (dec_at).
#include <algorithm>
#include <cmath>
#include <memory>
#include <mutex>
#include <vector>

#include "common.hpp"
#include "gemm.hpp"
#include "model.hpp"

namespace pkx {

struct DecState {
    int* t;          // current frame
    int* active;     // 1 while t < T
    int* sym;        // symbols emitted at the current frame
    int* count;      // tokens emitted
    int* overflow;   // a token did not fit in cap
    const int* T;    // frames per item
};

__device__ __forceinline__ float sigmoid_ref(float x) { return 1.0f / (1.0f + expf(-x)); }   // ggml_sigmoid

// Operand order of the decode products: 16-item blocks, within one the K columns
// in chunks of 16, a chunk as 64 lanes x 4 floats (lane = 16 (k % 16 / 4) +
// item % 16): the B fragments of four v_mfma_f32_16x16x4_f32, so a wave's load
// instruction is 1 KB contiguous.  The weights are packed the same way by
// 16-row tiles (pack_dec_weight).
__host__ __device__ __forceinline__ int64_t dec_at(int item, int k, int chunks) {
    return ((int64_t)(item >> 4) * chunks + (k >> 4)) * 256 + ((k >> 2) & 3) * 64 + (item & 15) * 4 + (k & 3);
}

enum { MM_LSTM = 0, MM_JOINT = 1, MM_PLAIN = 2 };

struct MmArgs {
    const float* x;   // [ceil(B / 16)][chunks][64][4] (dec_at)
    const float* W;   // [row tiles][chunks][64][4]
    const float* bias;
    int chunks, B;
    int block0;       // first 16-item block of the launch
    int n_out;        // MM_LSTM: hidden units H (tile row 4 u + g: gate g of unit 4 tile + u); else output rows
    float* y;         // MM_JOINT: dec_at order over y_chunks; MM_PLAIN: [B][n_out]
    int y_chunks;
    // MM_LSTM
    const float* c_in;
    float *out_h, *out_c, *x_next;   // x_next: dec_at order over next_chunks
    int next_chunks;
    // MM_JOINT
    const float* ep;
    int T_max;
};

// What bounds a round is latency: five dependent launches over 30 MB of weights
// that stay in the XCDs' L2s.  One workgroup per 16-row tile and 16-item block;
// a wave loads its share of K (up to MAXC chunks of weights and inputs, all in
// flight at once), runs four MFMAs a chunk, and wave 0 adds the eight partial
// tiles in a fixed order.  0.6B decoder, 16 items on MI355X, us per
// launch, against a kernel that kept its rows of W in registers and dotted them with
// the items staged through LDS: LSTM layer 12.9 -> 5.8, joint 8.5 -> 4.1, logits
// 11.0 -> 3.8 (an empty kernel's launch to launch is 2.5 to 3).
template <int MODE, int MAXC>
__global__ __launch_bounds__(512) void dec_mm_kernel(MmArgs a, DecState st) {
    __shared__ float4v red[8][64];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lr = lane & 15, lg = lane >> 4;
    const int tile = blockIdx.x, ib = a.block0 + blockIdx.y, b = 16 * ib + lr;
    const int c0 = a.chunks * w / 8, nc = a.chunks * (w + 1) / 8 - c0;   // <= MAXC
    const float4v* W = (const float4v*)a.W + ((int64_t)tile * a.chunks + c0) * 64 + lane;
    const float4v* x = (const float4v*)a.x + ((int64_t)ib * a.chunks + c0) * 64 + lane;
    const float4v zero = {0.f, 0.f, 0.f, 0.f};
    float4v wv[MAXC], xv[MAXC];
#pragma unroll
    for (int c = 0; c < MAXC; ++c) {
        xv[c] = c < nc ? x[64 * c] : zero;
        wv[c] = c < nc ? W[64 * c] : zero;
    }
    // the epilogue's operands: result rows 4 lg + r of the tile, item b
    const bool epi = w == 0 && b < a.B;
    const int row = 16 * tile + 4 * lg, u = 4 * tile + lg;
    float4v pb = zero, pe = zero;
    float pc = 0.f;
    if (epi) {
        if constexpr (MODE == MM_LSTM) {
#pragma unroll
            for (int g = 0; g < 4; ++g) pb[g] = a.bias[g * a.n_out + u];
            pc = a.c_in[(int64_t)b * a.n_out + u];
        } else {
#pragma unroll
            for (int r = 0; r < 4; ++r) pb[r] = row + r < a.n_out ? a.bias[row + r] : 0.f;
            if constexpr (MODE == MM_JOINT) {
                // inactive / boundary items read an edge frame (their logits are not used)
                const int t = max(0, min(st.t[b], st.T[b] - 1));
                if (row < a.n_out) pe = *(const float4v*)(a.ep + ((int64_t)b * a.T_max + t) * a.n_out + row);
            }
        }
    }
    float4v acc[4] = {zero, zero, zero, zero};   // four short chains: a smaller rounding error than one
#pragma unroll
    for (int c = 0; c < MAXC; ++c)
        if (c < nc) {   // uniform over the wave
#pragma unroll
            for (int e = 0; e < 4; ++e)
                acc[e] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[c][e], xv[c][e], acc[e], 0, 0, 0);
        }
    red[w][lane] = (acc[0] + acc[1]) + (acc[2] + acc[3]);
    __syncthreads();
    if (!epi) return;
    float4v z = ((red[0][lane] + red[1][lane]) + (red[2][lane] + red[3][lane])) +
                ((red[4][lane] + red[5][lane]) + (red[6][lane] + red[7][lane]));
    z += pb;
    if constexpr (MODE == MM_LSTM) {
        const int64_t i = (int64_t)b * a.n_out + u;
        const float c = sigmoid_ref(z[1]) * pc + sigmoid_ref(z[0]) * tanhf(z[2]);
        const float h = sigmoid_ref(z[3]) * tanhf(c);
        a.out_c[i] = c;
        a.out_h[i] = h;
        a.x_next[dec_at(b, u, a.next_chunks)] = h;
    } else if constexpr (MODE == MM_JOINT) {
        if (row >= a.n_out) return;   // n_out % 4 == 0
        z += pe;
#pragma unroll
        for (int r = 0; r < 4; ++r) z[r] = z[r] > 0.f ? z[r] : 0.f;
        *(float4v*)(a.y + dec_at(b, row, a.y_chunks)) = z;
    } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
            if (row + r < a.n_out) a.y[(int64_t)b * a.n_out + row + r] = z[r];
    }
}

__device__ __forceinline__ void argmax_first(float& v, int& k) {
    // wave-wide max with the lowest index among equal values (decode_common.hpp:5-9)
    for (int o = 32; o > 0; o >>= 1) {
        const float ov = __shfl_xor(v, o, 64);
        const int ok = __shfl_xor(k, o, 64);
        if (ov > v || (ov == v && ok < k)) {
            v = ov;
            k = ok;
        }
    }
}

struct RuleArgs {
    const float* logits;   // [B][Vp]
    int Vp, n_tok, n_dur, blank, max_symbols, cap, B, H, L;
    const int32_t* durations;
    const float* embed;    // [V1][H]
    float* X[4];           // per layer, dec_at order over xc chunks of [x | h]
    int xc;
    float* cc[4];          // committed c, [B][H]
    const float* oh[4];    // this round's h', [B][H]
    const float* oc[4];    // this round's c', [B][H]
    int32_t *ids, *frames, *spans;
    float* confs;
};

// One workgroup per item: the per-item rule of transducer_batch.cpp:128-205.
// Latency bound; 1024 threads, so that a thread's logits (9 of 8198) go out in
// one batch beside the state, both argmaxes share one barrier and the f64
// exponentials of the confidence are few per thread: 9.0 -> 6.3 us against 256
// threads and an argmax for each of tokens and durations (16 items, 1025 + 5).
constexpr int RULE_T = 1024;
__global__ __launch_bounds__(RULE_T) void greedy_rule_kernel(RuleArgs a, DecState st) {
    constexpr int NW = RULE_T / 64;
    __shared__ float rv[NW];
    __shared__ int rk[NW], rdk;
    __shared__ double rd[NW];
    const int b = blockIdx.x, tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    if (!st.active[b]) return;   // uniform over the workgroup
    // The item's state is read and written only by thread 0 of this workgroup:
    // its loads go out now, beside the logits', not after the commit stores.
    int t = 0, sym = 0, cnt = 0;
    if (tid == 0) {
        t = st.t[b];
        sym = st.sym[b];
        cnt = st.count[b];
    }
    // this step's (h', c') rows, loaded now and stored by the commit if the item
    // emits (L <= 4, H <= 1024: one value of each per thread and layer)
    float ph[4], pc[4];
#pragma unroll
    for (int l = 0; l < 4; ++l) {
        const bool ok = l < a.L && tid < a.H;
        ph[l] = ok ? a.oh[l][(int64_t)b * a.H + tid] : 0.f;
        pc[l] = ok ? a.oc[l][(int64_t)b * a.H + tid] : 0.f;
    }
    // argmax (first max) over the tokens: per thread, per wave, then over the waves
    const float* lz = a.logits + (int64_t)b * a.Vp;
    float v = -INFINITY;
    int k = 0x7fffffff;
    for (int i0 = tid; i0 < a.n_tok; i0 += 8 * RULE_T) {
        float x[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) x[j] = i0 + j * RULE_T < a.n_tok ? lz[i0 + j * RULE_T] : 0.f;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int i = i0 + j * RULE_T;
            if (i < a.n_tok && (x[j] > v || (x[j] == v && i < k))) {
                v = x[j];
                k = i;
            }
        }
    }
    argmax_first(v, k);
    if (lane == 0) {
        rv[w] = v;
        rk[w] = k;
    }
    if (w == NW - 1 && a.n_dur > 0) {   // the durations' argmax: the last wave's
        float dv = -INFINITY;
        int dk = 0x7fffffff;
        for (int i = lane; i < a.n_dur; i += 64) {
            const float x = lz[a.n_tok + i];
            if (x > dv || (x == dv && i < dk)) {
                dv = x;
                dk = i;
            }
        }
        argmax_first(dv, dk);
        if (lane == 0) rdk = a.durations[dk < a.n_dur ? dk : 0];
    }
    __syncthreads();
    v = rv[lane & (NW - 1)];
    k = rk[lane & (NW - 1)];
    argmax_first(v, k);
    if (k >= a.n_tok) k = 0;   // no value above -inf (NaN logits): index 0, as the scalar loop
    k = __builtin_amdgcn_readfirstlane(k);
    const bool emit = k != a.blank;
    double den = 0.0;
    if (emit) {
        // max_prob confidence of the emitted token (decode_common.hpp:12-20), f64
        for (int i = tid; i < a.n_tok; i += RULE_T) den += exp((double)lz[i] - (double)v);
        for (int o = 32; o > 0; o >>= 1) den += __shfl_xor(den, o, 64);
        if (lane == 0) rd[w] = den;
        // commit: the step's (h', c') become the item's state; the token's
        // embedding is the next step's layer-0 input
        if (tid < a.H) {
            a.X[0][dec_at(b, tid, a.xc)] = a.embed[(int64_t)k * a.H + tid];
#pragma unroll
            for (int l = 0; l < 4; ++l)
                if (l < a.L) {
                    a.X[l][dec_at(b, a.H + tid, a.xc)] = ph[l];
                    a.cc[l][(int64_t)b * a.H + tid] = pc[l];
                }
        }
        __syncthreads();
    }
    if (tid != 0) return;
    const int skip = a.n_dur > 0 ? rdk : 1;
    if (emit) {
        den = 0.0;
        for (int i = 0; i < NW; ++i) den += rd[i];
        const int n = cnt;
        if (n < a.cap) {
            const double p = 1.0 / den, N = (double)a.n_tok;   // exp(v - v) / den
            a.ids[(int64_t)b * a.cap + n] = k;
            a.frames[(int64_t)b * a.cap + n] = t;
            a.confs[(int64_t)b * a.cap + n] = (float)((N * p - 1.0) / (N - 1.0));
            a.spans[(int64_t)b * a.cap + n] = skip;
            st.count[b] = n + 1;
        } else {
            *st.overflow = 1;
        }
    }
    if (a.n_dur > 0) {
        // symbols_added += 1; t += skip; the frame is done unless skip == 0 and
        // symbols < max_symbols; a frame ended by max_symbols advances by 1
        sym += 1;
        t += skip;
        if (!(skip == 0 && sym < a.max_symbols)) {
            if (sym == a.max_symbols) t += 1;
            sym = 0;
        }
    } else if (!emit) {
        t += 1;   // RNNT blank: next frame
        sym = 0;
    } else if (++sym >= a.max_symbols) {
        t += 1;
        sym = 0;
    }
    st.t[b] = t;
    st.sym[b] = sym;
    st.active[b] = t < st.T[b] ? 1 : 0;
}

// Device and pinned host memory of the decode, kept between calls up to KEEP
// bytes (a larger call's memory is freed when it returns).  One call holds it
// at a time; a second one on the model meanwhile uses memory of its own.
struct DecodeWs {
    static constexpr size_t KEEP = (size_t)64 << 20;
    std::mutex mu;
    char *dev = nullptr, *host = nullptr;
    size_t dev_bytes = 0, host_bytes = 0;
    hipEvent_t ev[2] = {nullptr, nullptr};
    void grow(size_t nd, size_t nh) {
        if (nd > dev_bytes) {
            drop_dev();
            PKX_HIP(hipMalloc((void**)&dev, nd));
            dev_bytes = nd;
        }
        if (nh > host_bytes) {
            drop_host();
            PKX_HIP(hipHostMalloc((void**)&host, nh, hipHostMallocDefault));
            host_bytes = nh;
        }
        for (hipEvent_t& e : ev)
            if (!e) PKX_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    }
    void trim() {
        if (dev_bytes > KEEP) drop_dev();
        if (host_bytes > KEEP) drop_host();
    }
    void drop_dev() {
        if (dev) (void)hipFree(dev);
        dev = nullptr;
        dev_bytes = 0;
    }
    void drop_host() {
        if (host) (void)hipHostFree(host);
        host = nullptr;
        host_bytes = 0;
    }
    ~DecodeWs() {
        drop_dev();
        drop_host();
        for (hipEvent_t e : ev)
            if (e) (void)hipEventDestroy(e);
    }
};
std::shared_ptr<DecodeWs> make_decode_ws() { return std::make_shared<DecodeWs>(); }

namespace {
// Regions of one allocation, 256-byte aligned.
struct Carve {
    char* base = nullptr;
    size_t at = 0;
    template <typename T> T* get(size_t n) {
        T* p = (T*)(base + at);
        at += (n * sizeof(T) + 255) & ~(size_t)255;
        return p;
    }
};

// One workgroup per row tile and 16-item block, a launch per 65535 blocks (the grid's second dimension).
template <int MODE>
void launch_mm(MmArgs a, const DecState& st, int tiles, hipStream_t s) {
    const int blocks = cdiv(a.B, 16), per = cdiv(a.chunks, 8);   // chunks of a wave
    for (a.block0 = 0; a.block0 < blocks; a.block0 += 65535) {
        const dim3 grid(tiles, std::min(65535, blocks - a.block0));
        if (per <= 5) launch(dec_mm_kernel<MODE, 5>, grid, dim3(512), 0, s, a, st);
        else if (per <= 10) launch(dec_mm_kernel<MODE, 10>, grid, dim3(512), 0, s, a, st);
        else launch(dec_mm_kernel<MODE, 16>, grid, dim3(512), 0, s, a, st);
        PKX_LAUNCH_CHECK();
    }
}
}  // namespace

std::vector<float> pack_dec_weight(const std::vector<float>& w, int rows, int K, int H) {
    // H > 0: an LSTM's [4H][K], tile row 4 u + g = gate g of unit 4 tile + u
    const int tiles = cdiv(rows, 16), chunks = cdiv(K, 16);
    std::vector<float> out((size_t)tiles * chunks * 256, 0.f);
    for (int n = 0; n < rows; ++n) {
        const float* src = w.data() + (size_t)(H > 0 ? (n & 3) * H + (n >> 2) : n) * K;
        for (int k = 0; k < K; ++k) out[(size_t)dec_at(n, k, chunks)] = src[k];
    }
    return out;
}

void Model::transducer_greedy(const float* enc, int B, int T_max, const int* T_valid, const int32_t* durations,
                              int n_dur, int blank_id, int max_symbols, int cap, int32_t* ids, int32_t* frames,
                              float* conf, int32_t* span, int* counts, hipStream_t s) {
    require(finalized_ && has_decoder(), "model has no prediction network + joint");
    require(B >= 1 && T_max >= 1 && T_valid && counts && cap >= 1 && max_symbols >= 1, "decode: bad arguments");
    const int H = pred_.H, L = pred_.L, Hj = heads_.jenc.N, D = cfg_.d_model;
    const int Vp = heads_.jout.N;
    require(n_dur == heads_.n_dur, "decode: durations do not match the joint's duration outputs");
    const int n_tok = Vp - n_dur;
    require(blank_id >= 0 && blank_id < n_tok && blank_id < pred_.V1, "decode: blank_id outside the token range");
    require(n_tok <= pred_.V1, "decode: joint tokens exceed the embedding rows");
    require(H % 4 == 0 && Hj % 4 == 0, "decode: pred_hidden and joint_hidden must be multiples of 4");
    require(H <= 1024 && Hj <= 2048, "decode: pred_hidden above 1024 or joint_hidden above 2048");
    for (int b = 0; b < B; ++b) require(T_valid[b] >= 0 && T_valid[b] <= T_max, "decode: T_valid outside [0, T_max]");
    for (int i = 0; i < n_dur; ++i) require(durations && durations[i] >= 0, "decode: durations must be >= 0");

    const int B16 = cdiv(B, 16) * 16;
    const int xc = cdiv(2 * H, 16), gc = cdiv(H, 16), fc = cdiv(Hj, 16);   // 16-column chunks of the inputs
    float *ep, *X[4] = {}, *cc[4] = {}, *oh[4] = {}, *oc[4] = {}, *g, *f, *lg, *d_cf;
    int *ints;
    int32_t *d_dur, *d_ids, *d_fr, *d_sp;
    // ints: t [0, B), active [B, 2B), sym [2B, 3B), count [3B, 4B), T [5B, 6B), overflow 6B
    const size_t n_ints = (size_t)6 * B + 1;
    // the operands (zero beyond what is written), the cell states and the token records (their whole
    // [B][cap] is copied out, and an earlier call's records may lie here) start as zeros
    char* zero0 = nullptr;
    size_t zero_bytes = 0;
    auto carve = [&](char* base) {
        Carve m{base};
        ints = m.get<int>(n_ints);
        d_dur = m.get<int32_t>((size_t)std::max(n_dur, 1));
        const size_t z0 = m.at;
        for (int l = 0; l < L; ++l) {
            X[l] = m.get<float>((size_t)B16 * xc * 16);
            cc[l] = m.get<float>((size_t)B * H);
        }
        g = m.get<float>((size_t)B16 * gc * 16);
        f = m.get<float>((size_t)B16 * fc * 16);
        d_ids = m.get<int32_t>((size_t)B * cap);
        d_fr = m.get<int32_t>((size_t)B * cap);
        d_sp = m.get<int32_t>((size_t)B * cap);
        d_cf = m.get<float>((size_t)B * cap);
        zero0 = base + z0;
        zero_bytes = m.at - z0;
        for (int l = 0; l < L; ++l) {
            oh[l] = m.get<float>((size_t)B * H);
            oc[l] = m.get<float>((size_t)B * H);
        }
        lg = m.get<float>((size_t)B * Vp);
        ep = m.get<float>((size_t)B * T_max * Hj);
        return m.at;
    };
    DecodeWs own;
    std::unique_lock<std::mutex> lock(dec_ws_->mu, std::try_to_lock);
    DecodeWs& ws = lock.owns_lock() ? *dec_ws_ : own;
    struct Release {   // also when an error leaves: nothing of this call still runs on the memory
        DecodeWs& w;
        hipStream_t s;
        ~Release() {
            (void)hipStreamSynchronize(s);
            w.trim();
        }
    } release{ws, s};
    // host: the uploaded integers, then two copies of the active flags
    ws.grow(carve(nullptr), (n_ints + std::max(n_dur, 1) + 2 * (size_t)B) * sizeof(int));
    carve(ws.dev);
    int* h = (int*)ws.host;
    int* h_dur = h + n_ints;
    int* act[2] = {h_dur + std::max(n_dur, 1), h_dur + std::max(n_dur, 1) + B};
    std::fill(h, h + n_ints, 0);
    for (int b = 0; b < B; ++b) {
        h[(size_t)B + b] = T_valid[b] > 0 ? 1 : 0;   // active
        h[(size_t)5 * B + b] = T_valid[b];           // T
    }
    std::copy(durations, durations + n_dur, h_dur);
    PKX_HIP(hipMemcpyAsync(ints, h, sizeof(int) * n_ints, hipMemcpyHostToDevice, s));
    if (n_dur > 0) PKX_HIP(hipMemcpyAsync(d_dur, h_dur, sizeof(int32_t) * n_dur, hipMemcpyHostToDevice, s));
    PKX_HIP(hipMemsetAsync(zero0, 0, zero_bytes, s));   // SOS input, zero state, no records
    DecState st{ints, ints + B, ints + 2 * B, ints + 3 * B, ints + 6 * B, ints + 5 * B};

    // enc_proj over every frame of every item (joint.cpp:37-63)
    gemm(heads_.jenc, EPI_STORE_F32, enc, D, (int64_t)B * T_max, heads_.jenc_b, ep, Hj, 1.f, nullptr, 1, s,
         PREC_F32, -1);

    RuleArgs ra{};
    ra.logits = lg;
    ra.Vp = Vp;
    ra.n_tok = n_tok;
    ra.n_dur = n_dur;
    ra.blank = blank_id;
    ra.max_symbols = max_symbols;
    ra.cap = cap;
    ra.B = B;
    ra.H = H;
    ra.L = L;
    ra.xc = xc;
    ra.durations = d_dur;
    ra.embed = pred_.embed;
    for (int l = 0; l < L; ++l) {
        ra.X[l] = X[l];
        ra.cc[l] = cc[l];
        ra.oh[l] = oh[l];
        ra.oc[l] = oc[l];
    }
    ra.ids = d_ids;
    ra.frames = d_fr;
    ra.spans = d_sp;
    ra.confs = d_cf;

    auto round = [&]() {
        MmArgs a{};
        a.B = B;
        for (int l = 0; l < L; ++l) {
            a.x = X[l];
            a.chunks = xc;
            a.W = pred_.wpk[l];
            a.bias = pred_.bsum[l];
            a.n_out = H;
            a.c_in = cc[l];
            a.out_h = oh[l];
            a.out_c = oc[l];
            a.x_next = l + 1 < L ? X[l + 1] : g;
            a.next_chunks = l + 1 < L ? xc : gc;
            launch_mm<MM_LSTM>(a, st, H / 4, s);
        }
        a.x = g;
        a.chunks = gc;
        a.W = pred_.jpred;
        a.bias = heads_.jpred_b;
        a.n_out = Hj;
        a.y = f;
        a.y_chunks = fc;
        a.ep = ep;
        a.T_max = T_max;
        launch_mm<MM_JOINT>(a, st, cdiv(Hj, 16), s);
        a.x = f;
        a.chunks = fc;
        a.W = pred_.jout;
        a.bias = heads_.jout_b;
        a.n_out = Vp;
        a.y = lg;
        launch_mm<MM_PLAIN>(a, st, cdiv(Vp, 16), s);
        launch(greedy_rule_kernel, dim3(B), dim3(RULE_T), 0, s, ra, st);
        PKX_LAUNCH_CHECK();
    };

    // every round emits a token or advances a frame; at most max_symbols
    // tokens per frame: (max_symbols + 1) rounds per frame bound the loop.
    // Chunk i's flags are read while chunk i + 1 runs: no gap at a chunk's end, for
    // one chunk of rounds that change nothing (16 items of 125 frames, 0.6B decoder,
    // with the kernels above: 7.1 -> 3.6 ms a call).  Those rounds are a short call's
    // cost: with chunks of 8 one item of 12 frames took 522 us (497 with a wait after
    // each chunk and no look-ahead), with 4 453; 375 frames 10.1 and 10.2 ms.  Two
    // rounds no longer cover the host's launches (11.3).
    const int64_t max_rounds = (int64_t)T_max * (max_symbols + 1) + 1;
    constexpr int CHUNK = 4;
    int64_t rounds = 0;
    for (int i = 0;; ++i) {
        for (int r = 0; r < CHUNK; ++r) round();
        PKX_HIP(hipMemcpyAsync(act[i & 1], ints + B, sizeof(int) * B, hipMemcpyDeviceToHost, s));
        PKX_HIP(hipEventRecord(ws.ev[i & 1], s));
        if (i == 0) continue;
        rounds += CHUNK;   // those of chunk i - 1
        PKX_HIP(hipEventSynchronize(ws.ev[(i - 1) & 1]));
        const int* last = act[(i - 1) & 1];
        if (std::none_of(last, last + B, [](int v) { return v != 0; })) break;
        require(rounds <= max_rounds, "decode: round bound exceeded");
    }
    int ovf = 0;
    PKX_HIP(hipMemcpyAsync(counts, ints + 3 * B, sizeof(int) * B, hipMemcpyDeviceToHost, s));
    PKX_HIP(hipMemcpyAsync(&ovf, st.overflow, sizeof(int), hipMemcpyDeviceToHost, s));
    if (ids) PKX_HIP(hipMemcpyAsync(ids, d_ids, sizeof(int32_t) * B * cap, hipMemcpyDeviceToHost, s));
    if (frames) PKX_HIP(hipMemcpyAsync(frames, d_fr, sizeof(int32_t) * B * cap, hipMemcpyDeviceToHost, s));
    if (conf) PKX_HIP(hipMemcpyAsync(conf, d_cf, sizeof(float) * B * cap, hipMemcpyDeviceToHost, s));
    if (span) PKX_HIP(hipMemcpyAsync(span, d_sp, sizeof(int32_t) * B * cap, hipMemcpyDeviceToHost, s));
    PKX_HIP(hipStreamSynchronize(s));
    require(!ovf, "decode: more tokens than cap");
}

}  // namespace pkx
