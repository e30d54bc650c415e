// Learned warm start: an MLP (bus P, Q injections and PV setpoints -> |V|,
// theta) trained on the solver's own NR solutions, with hand-written
// training and inference kernels.  BF16 weights and activations, FP32
// accumulation on the matrix cores (v_mfma_f32_16x16x32_bf16), FP32 master
// weights updated by AdamW.  The NR solve that follows judges the
// prediction; flat start remains the fallback (batch.hip).
//
// No counterpart in the reference: it always starts from v_inicial /
// theta_inicial (CPU/estrutura/barra.cpp:20-25).

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <memory>
#include <string>
#include <vector>

#include "pf_internal.hpp"
#include "transfer.hpp"

typedef __bf16 bf16;
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

namespace pf {

enum { EPI_STORE = 0, EPI_BIAS = 1, EPI_BIAS_GELU = 2, EPI_DGELU = 3 };

__device__ __forceinline__ float gelu(float z) { return 0.5f * z * (1.0f + erff(z * 0.70710678118654752f)); }
__device__ __forceinline__ float gelu_grad(float z) {
    const float cdf = 0.5f * (1.0f + erff(z * 0.70710678118654752f));
    const float pdf = 0.39894228040143268f * expf(-0.5f * z * z);
    return cdf + z * pdf;
}

// Tile of TS x TS outputs, TK of the K dimension staged at a time: each
// thread then stages two 8-element vectors of either operand.
template <int TS> constexpr int kTileK = TS == 64 ? 64 : 128;

// The two vectors of 8 that a thread stages of an operand's tile (rows r0 ..
// of R, k0 .. of K).  KMAJOR: stored [R x K], vectors along k, one row's 16
// bytes each; else stored [K x R], vectors along the rows for two successive
// k, written to LDS as (k, k + 1) pairs.
template <int TS, bool KMAJOR>
struct TileStage {
    static constexpr int TK = kTileK<TS>, LD = TK + 8;   // +8: rows land on different banks
    bf16x8 v[2];
    int at[2];
    __device__ __forceinline__ void load(const bf16 *__restrict__ A, int ld, int r0, int R, int k0, int K, int t) {
        const bf16x8 zero8 = {};
#pragma unroll
        for (int u = 0; u < 2; u++) {
            int r, k;
            if (KMAJOR) {
                const int q = t + 256 * u;
                r = q / (TK / 8);
                k = q % (TK / 8) * 8;
            } else {
                r = t % (TS / 8) * 8;
                k = t / (TS / 8) * 2 + u;
            }
            at[u] = r * LD + k;
            const bool in = r0 + r < R && k0 + k < K;
            v[u] = in ? *reinterpret_cast<const bf16x8 *>(KMAJOR ? A + (size_t)(r0 + r) * ld + k0 + k
                                                                 : A + (size_t)(k0 + k) * ld + r0 + r)
                      : zero8;
        }
    }
    __device__ __forceinline__ void store(bf16 *s) const {
        if (KMAJOR) {
            *reinterpret_cast<bf16x8 *>(s + at[0]) = v[0];
            *reinterpret_cast<bf16x8 *>(s + at[1]) = v[1];
        } else {
#pragma unroll
            for (int i = 0; i < 8; i++) {
                bf16x2 p;
                p[0] = v[0][i];
                p[1] = v[1][i];
                *reinterpret_cast<bf16x2 *>(s + at[0] + i * LD) = p;
            }
        }
    }
};

// C[M x N] = op(A)[M x K] * op(B)[K x N], bf16 operands, fp32 accumulate.
//   TA = false: A row-major [M x K] (lda);  TA = true: A stored [K x M].
//   TB = false: B row-major [K x N] (ldb);  TB = true: B stored [N x K].
// Every dimension is a multiple of 8 (checked on the host), so 16-byte
// loads along the contiguous dimension never straddle the edge.
// 256 threads: 4 waves, each a quarter of the tile in MFMA 16x16x32 blocks
// (2 x 2 of them at TS = 64, one at 32).  At these sizes a workgroup waits
// for its loads, not for the matrix cores, so the next tile's vectors are in
// registers while this one's are multiplied, and products of few tiles take
// the small one (gemm()).  An output's sum runs through K in the same steps of
// 32 whatever the tile.  256 x 512 outputs, K = 2,832: 86 us with 64-wide
// tiles of 32 and no loads ahead, 20 now.
template <bool TA, bool TB, int EPI, int TS>
__global__ void __launch_bounds__(256) k_gemm(int M, int N, int K, const bf16 *__restrict__ A, int lda,
                                              const bf16 *__restrict__ B, int ldb, float *__restrict__ C,
                                              int ldc, bf16 *__restrict__ Cb, int ldcb,
                                              const float *__restrict__ bias, const float *__restrict__ Zs) {
    constexpr int TK = kTileK<TS>, LD = TK + 8, W = TS / 32;   // W x W blocks a wave
    __shared__ __align__(16) bf16 As[TS * LD];
    __shared__ __align__(16) bf16 Bs[TS * LD];
    const int t = threadIdx.x;
    const int m0 = blockIdx.y * TS, n0 = blockIdx.x * TS;
    const int w = t >> 6, l = t & 63;
    const int wm = (w >> 1) * (TS / 2), wn = (w & 1) * (TS / 2);
    f32x4 acc[W][W];
    for (int i = 0; i < W; i++)
        for (int j = 0; j < W; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    TileStage<TS, !TA> sa;
    TileStage<TS, TB> sb;
    sa.load(A, lda, m0, M, 0, K, t);
    sb.load(B, ldb, n0, N, 0, K, t);
    for (int k0 = 0; k0 < K; k0 += TK) {
        sa.store(As);
        sb.store(Bs);
        __syncthreads();
        if (k0 + TK < K) {
            sa.load(A, lda, m0, M, k0 + TK, K, t);
            sb.load(B, ldb, n0, N, k0 + TK, K, t);
        }
#pragma unroll
        for (int kk = 0; kk < TK; kk += 32) {
            bf16x8 a[W], b[W];
#pragma unroll
            for (int i = 0; i < W; i++)
                a[i] = *reinterpret_cast<const bf16x8 *>(&As[(wm + 16 * i + (l & 15)) * LD + kk + 8 * (l >> 4)]);
#pragma unroll
            for (int j = 0; j < W; j++)
                b[j] = *reinterpret_cast<const bf16x8 *>(&Bs[(wn + 16 * j + (l & 15)) * LD + kk + 8 * (l >> 4)]);
#pragma unroll
            for (int i = 0; i < W; i++)
#pragma unroll
                for (int j = 0; j < W; j++)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
        }
        __syncthreads();
    }
    // ---- epilogue: lane l owns rows 4*(l/16)+v, column l%16 of each 16x16 block
#pragma unroll
    for (int i = 0; i < W; i++)
#pragma unroll
        for (int j = 0; j < W; j++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int row = m0 + wm + 16 * i + 4 * (l >> 4) + v;
                const int col = n0 + wn + 16 * j + (l & 15);
                if (row >= M || col >= N) continue;
                float z = acc[i][j][v];
                const size_t o = (size_t)row * ldc + col;
                if (EPI == EPI_STORE) {
                    C[o] = z;
                } else if (EPI == EPI_BIAS) {
                    C[o] = z + bias[col];
                } else if (EPI == EPI_BIAS_GELU) {
                    z += bias[col];
                    C[o] = z;
                    Cb[(size_t)row * ldcb + col] = (bf16)gelu(z);
                } else {   // EPI_DGELU: z is dH, Zs the saved pre-activation
                    const float d = z * gelu_grad(Zs[o]);
                    C[o] = d;
                    Cb[(size_t)row * ldcb + col] = (bf16)d;
                }
            }
}

// rows idx[0 .. B) of X (idx null: rows 0 .. B), normalised
__global__ void k_norm_in(const float *X, const int *idx, int B, int n, const float *mean, const float *inv_std,
                          bf16 *Xn) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (size_t)B * n) return;
    const int r = (int)(i / n), c = (int)(i - (size_t)r * n);
    Xn[i] = (bf16)((X[(size_t)(idx ? idx[r] : r) * n + c] - mean[c]) * inv_std[c]);
}

// dY = 2 (Y - (T - mean)/std) / (B n), T's rows by idx as above; loss partial
// sums per block
__global__ void k_out_grad(const float *Y, const float *T, const int *idx, int B, int n, const float *mean,
                           const float *inv_std, float *dY, bf16 *dYb, float *loss_part) {
    __shared__ float red[256];
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    float e2 = 0.f;
    if (i < (size_t)B * n) {
        const int r = (int)(i / n), c = (int)(i - (size_t)r * n);
        const float d = Y[i] - (T[(size_t)(idx ? idx[r] : r) * n + c] - mean[c]) * inv_std[c];
        const float g = 2.f * d / ((float)B * (float)n);
        dY[i] = g;
        dYb[i] = (bf16)g;
        e2 = d * d;
    }
    red[threadIdx.x] = e2;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) loss_part[blockIdx.x] = red[0];
}

// column sums (bias gradient): db[c] = sum_r dZ[r, c], in row order (AdamW
// divides small gradients by their own size, so another order of the same
// sum shows in the weights).  A wave per 64 columns, a thread each, 64 rows in
// flight: the loads' latency, 60 us for 256 x 512 with a few in flight, is
// paid once per 64 rows, 4.6 us.
__global__ void __launch_bounds__(64) k_colsum(const float *dZ, int B, int n, float *db) {
    constexpr int U = 64;
    const int c = (int)blockIdx.x * 64 + (int)threadIdx.x;
    if (c >= n) return;
    float s = 0.f;
    int r = 0;
    for (; r + U <= B; r += U) {
        float v[U];
#pragma unroll
        for (int u = 0; u < U; u++) v[u] = (dZ + (size_t)(r + u) * n)[c];
#pragma unroll
        for (int u = 0; u < U; u++) s += v[u];
    }
    for (; r < B; r++) s += dZ[(size_t)r * n + c];
    db[c] = s;
}

// one AdamW update, and the bf16 copy of the parameters that the products read
__global__ void k_adamw(float *p, bf16 *pb, const float *g, float *m, float *v, size_t n, float lr, float b1, float b2,
                        float eps, float wd, float bc1, float bc2) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    const float mh = mi / bc1, vh = vi / bc2;
    const float pi = p[i] - lr * (mh / (sqrtf(vh) + eps) + wd * p[i]);
    p[i] = pi;
    pb[i] = (bf16)pi;
}

__global__ void k_to_bf16(const float *src, bf16 *dst, size_t n) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) dst[i] = (bf16)src[i];
}

__global__ void k_denorm(const float *Y, int B, int n, const float *mean, const float *std, float *out) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (size_t)B * n) return;
    const int c = (int)(i % n);
    out[i] = Y[i] * std[c] + mean[c];
}

}  // namespace pf

// ======================================================================= host
using namespace pf;

namespace {
#define MHIP(expr)                                                                 \
    do {                                                                           \
        hipError_t e_ = (expr);                                                    \
        if (e_ != hipSuccess) {                                                    \
            pf::set_last_error(std::string(#expr) + ": " + hipGetErrorString(e_));       \
            return PF_DEVICE_ERROR;                                                \
        }                                                                          \
    } while (0)
#define MCHK(expr)                  \
    do {                            \
        pf_status s_ = (expr);      \
        if (s_ != PF_OK) return s_; \
    } while (0)

// SplitMix64 for deterministic weight initialisation
inline unsigned long long sm64(unsigned long long &s) {
    s += 0x9E3779B97F4A7C15ull;
    unsigned long long z = s;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}
}  // namespace

struct pf_warmstart {
    int device = 0;
    int n_in = 0, n_out = 0, hidden = 0, n_layers = 0;   // n_layers = hidden layers + 1
    std::vector<int> K, N;                               // per layer
    std::vector<size_t> w_off, b_off;                    // into the parameter vector
    size_t n_params = 0;
    int step = 0;
    int Bcap = 0;
    int staged = 0;   // rows of features on the device for pf_warmstart_predict_into
    hipStream_t stream = nullptr;
    pf::PinnedSlots slots;
    std::vector<void *> allocs, ws_allocs;
    float *p = nullptr, *g = nullptr, *m = nullptr, *v = nullptr;
    bf16 *pb = nullptr;        // the parameters in bf16, laid out as p
    std::vector<bf16 *> Wb;    // its layers' weights
    float *fX = nullptr, *fT = nullptr;   // fit's resident rows and permutation, kept up to kFitKeep bytes
    int *fperm = nullptr;
    size_t fit_cap = 0;        // floats at fX (then fT)
    int perm_cap = 0;
    float *xm = nullptr, *xis = nullptr, *ym = nullptr, *yis = nullptr, *ys = nullptr;
    // workspace
    float *X = nullptr, *T = nullptr, *Yp = nullptr, *Yo = nullptr, *loss_part = nullptr;
    bf16 *Xn = nullptr;
    std::vector<float *> Z;    // per layer pre-activation / dZ fp32
    std::vector<bf16 *> H;     // per hidden layer activation
    float *dZf[2] = {nullptr, nullptr};
    bf16 *dZb[2] = {nullptr, nullptr};

    template <typename T_>
    pf_status alloc(T_ **q, size_t n, std::vector<void *> &lst) {
        void *r = nullptr;
        MHIP(hipMalloc(&r, sizeof(T_) * std::max<size_t>(n, 1)));
        lst.push_back(r);
        *q = (T_ *)r;
        return PF_OK;
    }
    ~pf_warmstart() {
        for (void *q : ws_allocs) (void)hipFree(q);
        for (void *q : allocs) (void)hipFree(q);
        (void)hipFree(fX);
        (void)hipFree(fperm);
        if (stream) (void)hipStreamDestroy(stream);
    }
    pf_status ensure(int B);
    pf_status sync_bf16();
    template <bool TA, bool TB, int EPI>
    pf_status gemm(int M_, int N_, int K_, const bf16 *A, int lda, const bf16 *B, int ldb, float *C, int ldc,
                   bf16 *Cb, int ldcb, const float *bias, const float *Zs);
    pf_status forward(int B, const float *rows, const int *idx);
    pf_status backward(int B, const float *targets, const int *idx, float *parts, double *loss);
    pf_status fit_room(int n);
};

pf_status pf_warmstart::ensure(int B) {
    if (B <= Bcap) return PF_OK;
    for (void *q : ws_allocs) MHIP(hipFree(q));
    ws_allocs.clear();
    staged = 0;   // the staged rows went with the old workspace
    Bcap = std::max(B, 64);
    const size_t b = Bcap;
    int maxN = std::max(n_out, hidden);
    MCHK(alloc(&X, b * n_in, ws_allocs));
    MCHK(alloc(&T, b * n_out, ws_allocs));
    MCHK(alloc(&Yp, b * n_out, ws_allocs));
    MCHK(alloc(&Yo, b * n_out, ws_allocs));
    MCHK(alloc(&loss_part, (b * n_out + 255) / 256, ws_allocs));
    MCHK(alloc(&Xn, b * n_in, ws_allocs));
    Z.assign(n_layers, nullptr);
    H.assign(n_layers, nullptr);
    for (int l = 0; l < n_layers; l++) {
        MCHK(alloc(&Z[l], b * N[l], ws_allocs));
        if (l < n_layers - 1) MCHK(alloc(&H[l], b * N[l], ws_allocs));
    }
    for (int i = 0; i < 2; i++) {
        MCHK(alloc(&dZf[i], b * maxN, ws_allocs));
        MCHK(alloc(&dZb[i], b * maxN, ws_allocs));
    }
    return PF_OK;
}

// Room for n rows of features and targets on the device: a small data set's
// stays with the network from one fit to the next.
constexpr size_t kFitKeep = 256u << 20;
pf_status pf_warmstart::fit_room(int n) {
    const size_t nx = (size_t)n * n_in, need = nx + (size_t)n * n_out;
    if (need > fit_cap) {
        MHIP(hipFree(fX));
        fX = nullptr;
        fit_cap = 0;
        MHIP(hipMalloc((void **)&fX, sizeof(float) * need));
        fit_cap = need;
    }
    fT = fX + nx;
    if (n > perm_cap) {
        MHIP(hipFree(fperm));
        fperm = nullptr;
        perm_cap = 0;
        MHIP(hipMalloc((void **)&fperm, sizeof(int) * n));
        perm_cap = n;
    }
    return PF_OK;
}

pf_status pf_warmstart::sync_bf16() {
    k_to_bf16<<<(unsigned)((n_params + 255) / 256), 256, 0, stream>>>(p, pb, n_params);
    MHIP(hipGetLastError());
    return PF_OK;
}

template <bool TA, bool TB, int EPI>
pf_status pf_warmstart::gemm(int M_, int N_, int K_, const bf16 *A, int lda, const bf16 *B, int ldb, float *C,
                             int ldc, bf16 *Cb, int ldcb, const float *bias, const float *Zs) {
    if (M_ % 8 || N_ % 8 || K_ % 8) return PF_INVALID_ARG;
    // 64-wide tiles where they give every CU one; else four times as many of 32
    // (256 x 1,888 outputs, K = 512, in 120 tiles of 64: 18 us; in 472 of 32: 7)
    const int wide = ((N_ + 63) / 64) * ((M_ + 63) / 64);
    if (wide >= 256) {
        dim3 grid((N_ + 63) / 64, (M_ + 63) / 64);
        k_gemm<TA, TB, EPI, 64><<<grid, 256, 0, stream>>>(M_, N_, K_, A, lda, B, ldb, C, ldc, Cb, ldcb, bias, Zs);
    } else {
        dim3 grid((N_ + 31) / 32, (M_ + 31) / 32);
        k_gemm<TA, TB, EPI, 32><<<grid, 256, 0, stream>>>(M_, N_, K_, A, lda, B, ldb, C, ldc, Cb, ldcb, bias, Zs);
    }
    MHIP(hipGetLastError());
    return PF_OK;
}

pf_status pf_warmstart::forward(int B, const float *rows, const int *idx) {
    size_t nx = (size_t)B * n_in;
    k_norm_in<<<(unsigned)((nx + 255) / 256), 256, 0, stream>>>(rows, idx, B, n_in, xm, xis, Xn);
    MHIP(hipGetLastError());
    const bf16 *in = Xn;
    for (int l = 0; l < n_layers; l++) {
        const float *bias = p + b_off[l];
        if (l < n_layers - 1) {
            MCHK((gemm<false, false, EPI_BIAS_GELU>(B, N[l], K[l], in, K[l], Wb[l], N[l], Z[l], N[l], H[l], N[l],
                                                    bias, nullptr)));
            in = H[l];
        } else {
            MCHK((gemm<false, false, EPI_BIAS>(B, N[l], K[l], in, K[l], Wb[l], N[l], Yp, N[l], nullptr, 0, bias,
                                               nullptr)));
        }
    }
    return PF_OK;
}

// loss partial sums go to parts; *loss (may be null) waits for them
pf_status pf_warmstart::backward(int B, const float *targets, const int *idx, float *parts_d, double *loss) {
    size_t ny = (size_t)B * n_out;
    unsigned nb = (unsigned)((ny + 255) / 256);
    int cur = 0;
    k_out_grad<<<nb, 256, 0, stream>>>(Yp, targets, idx, B, n_out, ym, yis, dZf[cur], dZb[cur], parts_d);
    MHIP(hipGetLastError());
    for (int l = n_layers - 1; l >= 0; l--) {
        const bf16 *hin = (l == 0) ? Xn : H[l - 1];
        // dW_l = H_{l-1}^T dZ_l : [K_l x N_l], reduction over the batch
        MCHK((gemm<true, false, EPI_STORE>(K[l], N[l], B, hin, K[l], dZb[cur], N[l], g + w_off[l], N[l], nullptr,
                                           0, nullptr, nullptr)));
        k_colsum<<<(N[l] + 63) / 64, 64, 0, stream>>>(dZf[cur], B, N[l], g + b_off[l]);
        MHIP(hipGetLastError());
        if (l > 0) {
            // dZ_{l-1} = (dZ_l W_l^T) * gelu'(Z_{l-1})
            MCHK((gemm<false, true, EPI_DGELU>(B, K[l], N[l], dZb[cur], N[l], Wb[l], N[l], dZf[cur ^ 1], K[l],
                                               dZb[cur ^ 1], K[l], nullptr, Z[l - 1])));
            cur ^= 1;
        }
    }
    if (loss) {
        std::vector<float> parts(nb);
        MHIP(hipMemcpyAsync(parts.data(), parts_d, sizeof(float) * nb, hipMemcpyDeviceToHost, stream));
        MHIP(hipStreamSynchronize(stream));
        double s = 0;
        for (float x : parts) s += x;
        *loss = s / ((double)B * n_out);
    }
    return PF_OK;
}

extern "C" {

pf_status pf_warmstart_create(int n_in, int n_out, int hidden, int n_hidden_layers, unsigned long long seed,
                              int device, pf_warmstart **out) {
    if (!out || n_in <= 0 || n_out <= 0 || hidden <= 0 || n_hidden_layers < 0 || n_in % 8 || n_out % 8 ||
        hidden % 8)
        return PF_INVALID_ARG;
    *out = nullptr;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || device < 0 || device >= ndev) return PF_DEVICE_ERROR;
    auto w = std::make_unique<pf_warmstart>();
    w->device = device;
    MHIP(hipSetDevice(device));
    MHIP(hipStreamCreateWithFlags(&w->stream, hipStreamNonBlocking));
    w->n_in = n_in;
    w->n_out = n_out;
    w->hidden = hidden;
    w->n_layers = n_hidden_layers + 1;
    size_t off = 0;
    for (int l = 0; l < w->n_layers; l++) {
        int k = (l == 0) ? n_in : hidden;
        int n = (l == w->n_layers - 1) ? n_out : hidden;
        w->K.push_back(k);
        w->N.push_back(n);
        w->w_off.push_back(off);
        off += (size_t)k * n;
        w->b_off.push_back(off);
        off += n;
    }
    w->n_params = off;
    // He-uniform initialisation (deterministic), zero biases
    std::vector<float> h(off, 0.f);
    unsigned long long s = seed;
    for (int l = 0; l < w->n_layers; l++) {
        const float a = std::sqrt(6.0f / (float)w->K[l]) * (l == w->n_layers - 1 ? 0.1f : 1.0f);
        for (size_t i = 0; i < (size_t)w->K[l] * w->N[l]; i++) {
            double u = (double)(sm64(s) >> 11) * (1.0 / 9007199254740992.0);
            h[w->w_off[l] + i] = (float)((2.0 * u - 1.0) * a);
        }
    }
    MCHK(w->alloc(&w->p, off, w->allocs));
    MCHK(w->alloc(&w->g, off, w->allocs));
    MCHK(w->alloc(&w->m, off, w->allocs));
    MCHK(w->alloc(&w->v, off, w->allocs));
    MCHK(w->alloc(&w->pb, off, w->allocs));
    MHIP(hipMemcpy(w->p, h.data(), sizeof(float) * off, hipMemcpyHostToDevice));
    MHIP(hipMemset(w->m, 0, sizeof(float) * off));
    MHIP(hipMemset(w->v, 0, sizeof(float) * off));
    MHIP(hipMemset(w->g, 0, sizeof(float) * off));
    w->Wb.resize(w->n_layers);
    for (int l = 0; l < w->n_layers; l++) w->Wb[l] = w->pb + w->w_off[l];   // 16-byte rows: every size is a multiple of 8
    MCHK(w->alloc(&w->xm, n_in, w->allocs));
    MCHK(w->alloc(&w->xis, n_in, w->allocs));
    MCHK(w->alloc(&w->ym, n_out, w->allocs));
    MCHK(w->alloc(&w->yis, n_out, w->allocs));
    MCHK(w->alloc(&w->ys, n_out, w->allocs));
    std::vector<float> zeros(std::max(n_in, n_out), 0.f), ones(std::max(n_in, n_out), 1.f);
    MHIP(hipMemcpy(w->xm, zeros.data(), 4 * n_in, hipMemcpyHostToDevice));
    MHIP(hipMemcpy(w->xis, ones.data(), 4 * n_in, hipMemcpyHostToDevice));
    MHIP(hipMemcpy(w->ym, zeros.data(), 4 * n_out, hipMemcpyHostToDevice));
    MHIP(hipMemcpy(w->yis, ones.data(), 4 * n_out, hipMemcpyHostToDevice));
    MHIP(hipMemcpy(w->ys, ones.data(), 4 * n_out, hipMemcpyHostToDevice));
    MCHK(w->sync_bf16());
    MHIP(hipStreamSynchronize(w->stream));
    *out = w.release();
    return PF_OK;
}

void pf_warmstart_destroy(pf_warmstart *w) {
    if (!w) return;
    (void)hipSetDevice(w->device);
    delete w;
}

pf_status pf_warmstart_info(pf_warmstart *w, size_t *n_params, int *n_layers) {
    if (!w) return PF_INVALID_ARG;
    if (n_params) *n_params = w->n_params;
    if (n_layers) *n_layers = w->n_layers;
    return PF_OK;
}

pf_status pf_warmstart_set_norm(pf_warmstart *w, const float *x_mean, const float *x_std, const float *y_mean,
                                const float *y_std) {
    if (!w || !x_mean || !x_std || !y_mean || !y_std) return PF_INVALID_ARG;
    MHIP(hipSetDevice(w->device));
    std::vector<float> xi(w->n_in), yi(w->n_out);
    for (int i = 0; i < w->n_in; i++) xi[i] = x_std[i] > 0 ? 1.0f / x_std[i] : 1.0f;
    for (int i = 0; i < w->n_out; i++) yi[i] = y_std[i] > 0 ? 1.0f / y_std[i] : 1.0f;
    std::vector<float> ysd(y_std, y_std + w->n_out);
    for (auto &x : ysd)
        if (!(x > 0)) x = 1.0f;
    MHIP(hipMemcpy(w->xm, x_mean, 4 * w->n_in, hipMemcpyHostToDevice));
    MHIP(hipMemcpy(w->xis, xi.data(), 4 * w->n_in, hipMemcpyHostToDevice));
    MHIP(hipMemcpy(w->ym, y_mean, 4 * w->n_out, hipMemcpyHostToDevice));
    MHIP(hipMemcpy(w->yis, yi.data(), 4 * w->n_out, hipMemcpyHostToDevice));
    MHIP(hipMemcpy(w->ys, ysd.data(), 4 * w->n_out, hipMemcpyHostToDevice));
    return PF_OK;
}

pf_status pf_warmstart_get_params(pf_warmstart *w, float *out) {
    if (!w || !out) return PF_INVALID_ARG;
    MHIP(hipSetDevice(w->device));
    const pf::CopyPiece all{out, w->p, sizeof(float) * w->n_params};
    MHIP(w->slots.fetch(&all, 1, w->stream));
    return PF_OK;
}

pf_status pf_warmstart_set_params(pf_warmstart *w, const float *in) {
    if (!w || !in) return PF_INVALID_ARG;
    MHIP(hipSetDevice(w->device));
    MHIP(hipMemcpy(w->p, in, sizeof(float) * w->n_params, hipMemcpyHostToDevice));
    MCHK(w->sync_bf16());
    MHIP(hipStreamSynchronize(w->stream));
    return PF_OK;
}

// forward + backward on one minibatch (raw inputs X [B x n_in], raw targets
// Y [B x n_out]); gradients (parameter layout) copied to grads if not NULL
pf_status pf_warmstart_grad(pf_warmstart *w, const float *X, const float *Y, int B, float *grads, double *loss) {
    if (!w || !X || !Y || B <= 0 || B % 8) return PF_INVALID_ARG;
    w->staged = 0;   // its rows replace the staged ones
    MHIP(hipSetDevice(w->device));
    MCHK(w->ensure(B));
    MHIP(hipMemcpyAsync(w->X, X, sizeof(float) * (size_t)B * w->n_in, hipMemcpyHostToDevice, w->stream));
    MHIP(hipMemcpyAsync(w->T, Y, sizeof(float) * (size_t)B * w->n_out, hipMemcpyHostToDevice, w->stream));
    MCHK(w->forward(B, w->X, nullptr));
    MCHK(w->backward(B, w->T, nullptr, w->loss_part, loss));
    if (grads) MHIP(hipMemcpyAsync(grads, w->g, sizeof(float) * w->n_params, hipMemcpyDeviceToHost, w->stream));
    MHIP(hipStreamSynchronize(w->stream));
    return PF_OK;
}

// AdamW training over a resident data set: X [n x n_in], Y [n x n_out] raw;
// `epochs` passes in minibatches of B rows (a permutation per epoch from
// `seed`); per-epoch mean loss written to epoch_loss (may be NULL)
pf_status pf_warmstart_fit(pf_warmstart *w, const float *X, const float *Y, int n, int epochs, int B, float lr,
                           float weight_decay, unsigned long long seed, double *epoch_loss) {
    if (!w || !X || !Y || n < B || B <= 0 || B % 8 || epochs <= 0) return PF_INVALID_ARG;
    w->staged = 0;   // staged rows do not outlive a fit, whose batch size may take their room
    MHIP(hipSetDevice(w->device));
    MCHK(w->ensure(B));
    MCHK(w->fit_room(n));
    float *dX = w->fX, *dY = w->fT;
    int *dperm = w->fperm;
    // every step's loss sums, read once an epoch
    const int nbat = n / B;
    const size_t nb = ((size_t)B * w->n_out + 255) / 256;
    std::vector<void *> tmp;
    float *parts = nullptr;
    std::vector<float> hp;
    if (epoch_loss) {
        MCHK(w->alloc(&parts, nb * nbat, tmp));
        hp.resize(nb * nbat);
    }
    pf_status st = PF_OK;
    auto ok = [&](hipError_t e) {
        if (e != hipSuccess && st == PF_OK) {
            pf::set_last_error(std::string("pf_warmstart_fit: ") + hipGetErrorString(e));
            st = PF_DEVICE_ERROR;
        }
    };
    const pf::CopyPiece rows[2] = {{(void *)X, dX, sizeof(float) * (size_t)n * w->n_in},
                                   {(void *)Y, dY, sizeof(float) * (size_t)n * w->n_out}};
    ok(w->slots.send(rows, 2, w->stream));
    std::vector<int> perm(n);
    for (int i = 0; i < n; i++) perm[i] = i;
    unsigned long long s = seed;
    for (int ep = 0; ep < epochs && st == PF_OK; ep++) {
        for (int i = n - 1; i > 0; i--) {
            int j = (int)(sm64(s) % (unsigned long long)(i + 1));
            std::swap(perm[i], perm[j]);
        }
        ok(hipMemcpyAsync(dperm, perm.data(), sizeof(int) * n, hipMemcpyHostToDevice, w->stream));
        ok(hipStreamSynchronize(w->stream));   // perm is shuffled again for the next epoch
        for (int bi = 0; bi < nbat && st == PF_OK; bi++) {
            const int *idx = dperm + (size_t)bi * B;
            st = w->forward(B, dX, idx);
            if (st == PF_OK) st = w->backward(B, dY, idx, parts ? parts + nb * bi : w->loss_part, nullptr);
            if (st != PF_OK) break;
            w->step++;
            const float b1 = 0.9f, b2 = 0.999f;
            const float bc1 = 1.0f - std::pow(b1, (float)w->step), bc2 = 1.0f - std::pow(b2, (float)w->step);
            k_adamw<<<(unsigned)((w->n_params + 255) / 256), 256, 0, w->stream>>>(w->p, w->pb, w->g, w->m, w->v,
                                                                                 w->n_params, lr, b1, b2, 1e-8f,
                                                                                 weight_decay, bc1, bc2);
            ok(hipGetLastError());
        }
        if (epoch_loss && st == PF_OK) {
            ok(hipMemcpyAsync(hp.data(), parts, sizeof(float) * hp.size(), hipMemcpyDeviceToHost, w->stream));
            ok(hipStreamSynchronize(w->stream));
            double acc = 0;
            for (int bi = 0; bi < nbat; bi++) {
                double l = 0;
                for (size_t i = 0; i < nb; i++) l += hp[nb * bi + i];
                acc += l / ((double)B * w->n_out);
            }
            epoch_loss[ep] = acc / nbat;
        }
    }
    ok(hipStreamSynchronize(w->stream));
    for (void *q : tmp) (void)hipFree(q);
    if (w->fit_cap * sizeof(float) > kFitKeep) {   // a large data set's room goes back
        (void)hipFree(w->fX);
        w->fX = w->fT = nullptr;
        w->fit_cap = 0;
    }
    return st;
}

// inference: X [B x n_in] raw -> Y [B x n_out] in target units
pf_status pf_warmstart_predict(pf_warmstart *w, const float *X, int B, float *Y) {
    if (!w || !X || !Y || B <= 0 || B % 8) return PF_INVALID_ARG;
    w->staged = 0;   // its rows replace the staged ones
    MHIP(hipSetDevice(w->device));
    MCHK(w->ensure(B));
    const pf::CopyPiece in{(void *)X, w->X, sizeof(float) * (size_t)B * w->n_in};
    MHIP(w->slots.send(&in, 1, w->stream));
    MCHK(w->forward(B, w->X, nullptr));
    size_t ny = (size_t)B * w->n_out;
    k_denorm<<<(unsigned)((ny + 255) / 256), 256, 0, w->stream>>>(w->Yp, B, w->n_out, w->ym, w->ys, w->Yo);
    MHIP(hipGetLastError());
    const pf::CopyPiece out{Y, w->Yo, sizeof(float) * ny};
    MHIP(w->slots.fetch(&out, 1, w->stream));
    return PF_OK;
}

pf_status pf_warmstart_stage(pf_warmstart *w, const float *X, int B) {
    if (!w || !X || B <= 0 || B % 8) return PF_INVALID_ARG;
    MHIP(hipSetDevice(w->device));
    MCHK(w->ensure(B));
    const pf::CopyPiece in{(void *)X, w->X, sizeof(float) * (size_t)B * w->n_in};
    MHIP(w->slots.send(&in, 1, w->stream));
    w->staged = B;
    return PF_OK;
}

pf_status pf_warmstart_predict_into(pf_warmstart *w, pf_batch *b, int v_col, int th_col) {
    if (!w || !b || w->staged <= 0) return PF_INVALID_ARG;
    MHIP(hipSetDevice(w->device));
    MCHK(w->forward(w->staged, w->X, nullptr));
    return batch_start_from_rows(b, w->device, w->staged, w->Yp, w->n_out, v_col, th_col, w->ym, w->ys,
                                 (void *)w->stream);
}

// one GEMM through the training kernel (tests): C = op(A) op(B), bf16 in, fp32 out
pf_status pf_warmstart_gemm_probe(pf_warmstart *w, int ta, int tb, int M, int N, int K, const float *A,
                                  const float *B, float *C) {
    if (!w || !A || !B || !C || M % 8 || N % 8 || K % 8) return PF_INVALID_ARG;
    MHIP(hipSetDevice(w->device));
    std::vector<void *> tmp;
    bf16 *dA, *dB;
    float *dC, *fA, *fB;
    MCHK(w->alloc(&fA, (size_t)M * K, tmp));
    MCHK(w->alloc(&fB, (size_t)K * N, tmp));
    MCHK(w->alloc(&dA, (size_t)M * K, tmp));
    MCHK(w->alloc(&dB, (size_t)K * N, tmp));
    MCHK(w->alloc(&dC, (size_t)M * N, tmp));
    pf_status st = PF_OK;
    (void)hipMemcpy(fA, A, 4 * (size_t)M * K, hipMemcpyHostToDevice);
    (void)hipMemcpy(fB, B, 4 * (size_t)K * N, hipMemcpyHostToDevice);
    k_to_bf16<<<(unsigned)(((size_t)M * K + 255) / 256), 256, 0, w->stream>>>(fA, dA, (size_t)M * K);
    k_to_bf16<<<(unsigned)(((size_t)K * N + 255) / 256), 256, 0, w->stream>>>(fB, dB, (size_t)K * N);
    const int lda = ta ? M : K, ldb = tb ? K : N;
    if (!ta && !tb) st = w->gemm<false, false, EPI_STORE>(M, N, K, dA, lda, dB, ldb, dC, N, nullptr, 0, nullptr, nullptr);
    else if (ta && !tb) st = w->gemm<true, false, EPI_STORE>(M, N, K, dA, lda, dB, ldb, dC, N, nullptr, 0, nullptr, nullptr);
    else if (!ta && tb) st = w->gemm<false, true, EPI_STORE>(M, N, K, dA, lda, dB, ldb, dC, N, nullptr, 0, nullptr, nullptr);
    else st = PF_INVALID_ARG;
    if (st == PF_OK && hipMemcpyAsync(C, dC, 4 * (size_t)M * N, hipMemcpyDeviceToHost, w->stream) != hipSuccess)
        st = PF_DEVICE_ERROR;
    (void)hipStreamSynchronize(w->stream);
    for (void *q : tmp) (void)hipFree(q);
    return st;
}

}  // extern "C"
