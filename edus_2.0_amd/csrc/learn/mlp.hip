// Per-k MLP kernels: BF16 GEMMs on the matrix cores (v_mfma_f32_16x16x16_bf16,
// FP32 accumulation) with fused bias / tanh / tanh-derivative epilogues, a
// split-K weight-gradient GEMM with a deterministic reduction, the MSE loss
// and Adam on FP32 master weights.
//
// Fragment layout of the 16x16x16 BF16 instruction (lane l, q = l / 16,
// i = l % 16): A row i, columns 4q .. 4q+3; B rows 4q .. 4q+3, column i; the
// FP32 result row 4q + v, column i in slot v.
#include <cmath>
#include <cstring>
#include <random>
#include <stdexcept>
#include <string>

#include "../engine/engine_internal.hpp"
#include "mlp.hpp"

#define HIP_CHECK EDUS_HIP_CHECK

namespace edus {

namespace {

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float flt4 __attribute__((ext_vector_type(4)));

constexpr int kTile = 64;   // rows and columns of C per work-group
constexpr int kKStep = 16;  // K per MFMA
constexpr int kStage = 64;  // K per pass through LDS
constexpr int kLd = kStage + 4;  // LDS row of an operand: 34 words, the fragment reads of 16 rows spread over the banks

struct GemmArgs {
    const uint16_t* A;
    long sam, sak;
    const uint16_t* B;
    long sbk, sbn;
    int M, N, K;
    int kchunk;        // K range per blockIdx.z (split-K)
    int ones_row;      // row of A that reads 1.0 (bias gradient), -1: none
    const float* bias;
    int act;           // 1: tanh
    float* C;          // FP32 out (split-K: partial [z][M][N])
    int ldc;
    uint16_t* Cb;      // BF16 out
    int ldcb;
    const uint16_t* mul;  // BF16 [M][ldm]: multiply by (1 - mul^2)
    int ldm;
};

// 4 consecutive BF16 values from p (8-byte aligned when VEC), those at index
// first + e < n
template <bool VEC>
__device__ inline ushort4 load4(const uint16_t* p, long first, long n)
{
    if (VEC && first + 4 <= n) return *reinterpret_cast<const ushort4*>(p);
    ushort4 v = make_ushort4(0, 0, 0, 0);
    if (first < n) v.x = p[0];
    if (first + 1 < n) v.y = p[1];
    if (first + 2 < n) v.z = p[2];
    if (first + 3 < n) v.w = p[3];
    return v;
}

// One operand's 64 x kStage tile in registers, then in LDS as s[row][k].
// KROW: k is the contiguous index in memory (a thread takes 16 k of one row);
// otherwise the rows are (a thread takes 8 rows at two adjacent k and writes
// pairs).  ones: a row that reads 1.0.
template <bool KROW, bool VEC>
struct Tile {
    ushort4 v[4];
    __device__ void load(const uint16_t* X, long sr, long sk, int r0, int rows, int k0, int ke, int ones)
    {
        const int t = threadIdx.x;
        if (KROW) {
            const int r = r0 + (t >> 2), k = k0 + (t & 3) * 16;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                v[e] = make_ushort4(0, 0, 0, 0);
                if (r < rows) v[e] = load4<VEC>(X + long(r) * sr + k + 4 * e, k + 4 * e, ke);
            }
        } else {
            const int r = r0 + (t & 7) * 8, k = k0 + (t >> 3) * 2;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int kk = k + (e >> 1), rr = r + (e & 1) * 4;
                v[e] = make_ushort4(0, 0, 0, 0);
                if (kk < ke) {
                    // the row of ones lies behind the operand's own rows
                    v[e] = load4<VEC>(X + long(kk) * sk + rr, rr, ones >= 0 ? ones : rows);
                    // (an index into v[e] at run time would put it in scratch memory)
                    if (ones >= 0) {
                        v[e].x = rr == ones ? 0x3f80 : v[e].x;
                        v[e].y = rr + 1 == ones ? 0x3f80 : v[e].y;
                        v[e].z = rr + 2 == ones ? 0x3f80 : v[e].z;
                        v[e].w = rr + 3 == ones ? 0x3f80 : v[e].w;
                    }
                }
            }
        }
    }
    __device__ void store(uint16_t (*s)[kLd]) const
    {
        const int t = threadIdx.x;
        if (KROW) {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                *reinterpret_cast<ushort4*>(&s[t >> 2][(t & 3) * 16 + 4 * e]) = v[e];
        } else {
            const int r = (t & 7) * 8, k = (t >> 3) * 2;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const ushort4 a = v[h], b = v[2 + h];
                const uint16_t x[4] = {a.x, a.y, a.z, a.w}, y[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    *reinterpret_cast<uint32_t*>(&s[r + 4 * h + e][k]) = uint32_t(x[e]) | (uint32_t(y[e]) << 16);
            }
        }
    }
};

// C = A B on 64 x 64 tiles, 16 rows of a tile per wave.  Both operands pass
// through LDS with k contiguous (whatever their order in memory), 64 k per
// barrier pair, the next 64 loaded into registers meanwhile; a fragment is one
// 8-byte read.  The products are summed over k in steps of 16 in ascending
// order, whatever the staging.  Bound by the latency of its few stages and, on
// small shapes, by the launch: 8192 rows, 256 x 256, 14 us; with one 2-byte element
// per load and read and 16 k per barrier it took 32 to 60.
template <bool AK, bool VEC>
__global__ void __launch_bounds__(256) gemm_bf16_kernel(GemmArgs g)
{
    __shared__ __align__(16) uint16_t sA[kTile][kLd];
    __shared__ __align__(16) uint16_t sB[kTile][kLd];
    const int m0 = blockIdx.x * kTile, n0 = blockIdx.y * kTile;
    const int kb = blockIdx.z * g.kchunk;
    const int ke = min(g.K, kb + g.kchunk);
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int i = lane & 15, q = lane >> 4;
    flt4 acc[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) acc[t] = flt4{0.f, 0.f, 0.f, 0.f};

    Tile<AK, VEC> ta;
    Tile<false, VEC> tb;
    ta.load(g.A, g.sam, g.sak, m0, g.M, kb, ke, g.ones_row);
    tb.load(g.B, g.sbn, g.sbk, n0, g.N, kb, ke, -1);
    for (int k0 = kb; k0 < ke; k0 += kStage) {
        ta.store(sA);
        tb.store(sB);
        __syncthreads();
        if (k0 + kStage < ke) {
            ta.load(g.A, g.sam, g.sak, m0, g.M, k0 + kStage, ke, g.ones_row);
            tb.load(g.B, g.sbn, g.sbk, n0, g.N, k0 + kStage, ke, -1);
        }
#pragma unroll
        for (int ks = 0; ks < kStage; ks += kKStep) {
            if (k0 + ks >= ke) break;
            const bf16x4 a = *reinterpret_cast<const bf16x4*>(&sA[16 * wave + i][ks + 4 * q]);
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const bf16x4 b = *reinterpret_cast<const bf16x4*>(&sB[16 * t + i][ks + 4 * q]);
                acc[t] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, acc[t], 0, 0, 0);
            }
        }
        __syncthreads();
    }

    float* C = g.C ? g.C + size_t(blockIdx.z) * g.M * g.N : nullptr;  // split-K partials
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int m = m0 + 16 * wave + 4 * q + v, n = n0 + 16 * t + i;
            if (m >= g.M || n >= g.N) continue;
            float x = acc[t][v];
            if (g.bias) x += g.bias[n];
            if (g.act) x = tanhf(x);
            if (g.mul) {
                const float h = bf2f(g.mul[size_t(m) * g.ldm + n]);
                x *= 1.0f - h * h;
            }
            if (C) C[size_t(m) * g.ldc + n] = x;
            if (g.Cb) g.Cb[size_t(m) * g.ldcb + n] = f2bf(x);
        }
}

// sum of split-K partials [nz][rows][N]: rows < nrw -> dW [rows][N], row nrw -> db
__global__ void reduce_partials_kernel(const float* __restrict__ part, int nz, int nrw, int N, float* __restrict__ dW,
                                       float* __restrict__ db)
{
    const int idx = blockIdx.x * blockDim.x + threadIdx.x;
    const int total = (nrw + 1) * N;
    if (idx >= total) return;
    float s = 0.f;
    for (int z = 0; z < nz; ++z) s += part[size_t(z) * total + idx];
    if (idx < nrw * N)
        dW[idx] = s;
    else
        db[idx - nrw * N] = s;
}

// dY = 2 (Y - T) / (M dout) as BF16, and per-block partial sums of (Y - T)^2
__global__ void mse_kernel(const float* __restrict__ Y, const float* __restrict__ T, long n, float scale,
                           uint16_t* __restrict__ dYb, float* __restrict__ part)
{
    __shared__ float sh[256];
    float acc = 0.f;
    for (long i = blockIdx.x * 256L + threadIdx.x; i < n; i += long(gridDim.x) * 256) {
        const float d = Y[i] - T[i];
        acc += d * d;
        dYb[i] = f2bf(2.0f * d * scale);
    }
    sh[threadIdx.x] = acc;
    __syncthreads();
    for (int st = 128; st > 0; st >>= 1) {
        if (threadIdx.x < st) sh[threadIdx.x] += sh[threadIdx.x + st];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = sh[0];
}

__global__ void sum_kernel(const float* __restrict__ part, int n, float scale, float* __restrict__ out)
{
    __shared__ float sh[256];
    float acc = 0.f;
    for (int i = threadIdx.x; i < n; i += 256) acc += part[i];
    sh[threadIdx.x] = acc;
    __syncthreads();
    for (int st = 128; st > 0; st >>= 1) {
        if (threadIdx.x < st) sh[threadIdx.x] += sh[threadIdx.x + st];
        __syncthreads();
    }
    if (threadIdx.x == 0) out[0] = sh[0] * scale;
}

__global__ void adam_kernel(float* __restrict__ P, const float* __restrict__ G, float* __restrict__ m,
                            float* __restrict__ v, long n, float lr, float b1, float b2, float eps, float c1, float c2)
{
    const long i = blockIdx.x * 256L + threadIdx.x;
    if (i >= n) return;
    const float g = G[i];
    const float mi = b1 * m[i] + (1.f - b1) * g;
    const float vi = b2 * v[i] + (1.f - b2) * g * g;
    m[i] = mi;
    v[i] = vi;
    P[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}

// W [rows][cols] FP32 -> BF16 W and its transpose
__global__ void to_bf16_kernel(const float* __restrict__ W, int rows, int cols, uint16_t* __restrict__ Wb,
                               uint16_t* __restrict__ WbT)
{
    const int idx = blockIdx.x * 256 + threadIdx.x;
    if (idx >= rows * cols) return;
    const int r = idx / cols, c = idx - r * cols;
    const uint16_t b = f2bf(W[idx]);
    Wb[idx] = b;
    WbT[size_t(c) * rows + r] = b;
}

// x rounded to BF16, four values per thread
__global__ void __launch_bounds__(256) round_bf16_kernel(const float* __restrict__ x, long n, uint16_t* __restrict__ b)
{
    const long i = (blockIdx.x * 256L + threadIdx.x) * 4;
    if (i + 4 <= n) {
        const float4 v = *reinterpret_cast<const float4*>(x + i);
        *reinterpret_cast<ushort4*>(b + i) = make_ushort4(f2bf(v.x), f2bf(v.y), f2bf(v.z), f2bf(v.w));
    } else {
        for (long e = i; e < n; ++e) b[e] = f2bf(x[e]);
    }
}

int cdiv(long a, long b) { return int((a + b - 1) / b); }

void launch_gemm(const GemmArgs& g, int nz, hipStream_t s)
{
    const dim3 grid(cdiv(g.M, kTile), cdiv(g.N, kTile), nz);
    // (a layer of one input has both strides 1: its weight gradient, with the row
    // of ones, is the form with contiguous rows)
    const bool ak = g.sak == 1 && g.ones_row < 0;
    if (g.sbn != 1 || (!ak && g.sam != 1))
        throw EngineError(EDUS_ERR_ARG, "GEMM operand order not supported");
    // 8-byte loads where every row starts on 8 bytes; kchunk is a multiple of 16
    const long ld = ak ? g.sam : g.sak;
    const bool vec = ld % 4 == 0 && g.sbk % 4 == 0 && reinterpret_cast<uintptr_t>(g.A) % 8 == 0 &&
                     reinterpret_cast<uintptr_t>(g.B) % 8 == 0;
    if (ak && vec)
        hipLaunchKernelGGL((gemm_bf16_kernel<true, true>), grid, dim3(256), 0, s, g);
    else if (ak)
        hipLaunchKernelGGL((gemm_bf16_kernel<true, false>), grid, dim3(256), 0, s, g);
    else if (vec)
        hipLaunchKernelGGL((gemm_bf16_kernel<false, true>), grid, dim3(256), 0, s, g);
    else
        hipLaunchKernelGGL((gemm_bf16_kernel<false, false>), grid, dim3(256), 0, s, g);
}

}  // namespace

void launch_gemm_bf16(const uint16_t* A, long sam, long sak, const uint16_t* B, long sbk, long sbn, int M, int N,
                      int K, const float* bias, int act, float* C, int ldc, uint16_t* Cb, int ldcb,
                      const uint16_t* mul, hipStream_t s)
{
    GemmArgs g{};
    g.A = A;
    g.sam = sam;
    g.sak = sak;
    g.B = B;
    g.sbk = sbk;
    g.sbn = sbn;
    g.M = M;
    g.N = N;
    g.K = K;
    g.kchunk = K;
    g.ones_row = -1;
    g.bias = bias;
    g.act = act;
    g.C = C;
    g.ldc = ldc;
    g.Cb = Cb;
    g.ldcb = ldcb;
    g.mul = mul;
    g.ldm = N;
    launch_gemm(g, 1, s);
}

void* Mlp::alloc(size_t bytes)
{
    void* p = nullptr;
    HIP_CHECK(hipMalloc(&p, bytes));
    owned.push_back(p);
    HIP_CHECK(hipMemsetAsync(p, 0, bytes, s));
    return p;
}

Mlp::Mlp(int din_, int dh_, int dout_, uint64_t seed, hipStream_t st) : din(din_), dh(dh_), dout(dout_), s(st)
{
    if (din < 1 || dh < 1 || dout < 1 || din > 4096 || dh > 4096 || dout > 4096)
        throw EngineError(EDUS_ERR_ARG, "MLP sizes must be in 1..4096");
    const int in[3] = {din, dh, dh}, out[3] = {dh, dh, dout};
    size_t o = 0;
    for (int l = 0; l < 3; ++l) {
        off_W[l] = o;
        o += size_t(in[l]) * out[l];
        off_b[l] = o;
        o += out[l];
    }
    nparam = o;
    P = static_cast<float*>(alloc(nparam * sizeof(float)));
    G = static_cast<float*>(alloc(nparam * sizeof(float)));
    Am = static_cast<float*>(alloc(nparam * sizeof(float)));
    Av = static_cast<float*>(alloc(nparam * sizeof(float)));
    for (int l = 0; l < 3; ++l) {
        Wb[l] = static_cast<uint16_t*>(alloc(size_t(in[l]) * out[l] * sizeof(uint16_t)));
        WbT[l] = static_cast<uint16_t*>(alloc(size_t(in[l]) * out[l] * sizeof(uint16_t)));
    }
    // Glorot-uniform weights, zero biases
    std::vector<float> h(nparam, 0.f);
    std::mt19937_64 rng(seed);
    for (int l = 0; l < 3; ++l) {
        const float a = std::sqrt(6.0f / float(in[l] + out[l]));
        std::uniform_real_distribution<float> u(-a, a);
        for (size_t k = 0; k < size_t(in[l]) * out[l]; ++k) h[off_W[l] + k] = u(rng);
    }
    set_params(h.data());
}

Mlp::~Mlp()
{
    (void)hipStreamSynchronize(s);
    for (void* p : owned) (void)hipFree(p);
    for (auto& b : io) (void)hipFree(b.p);
}

// Input buffer k of the calls on host arrays, at least `bytes` long: kept from
// call to call, replaced when a call needs more, released with the network.
void* Mlp::io_buffer(int k, size_t bytes)
{
    IoBuffer& b = io[k];
    if (bytes > b.bytes) {
        HIP_CHECK(hipStreamSynchronize(s));  // nothing queued reads the old one
        HIP_CHECK(hipFree(b.p));
        b.p = nullptr;
        b.bytes = 0;
        HIP_CHECK(hipMalloc(&b.p, bytes));
        b.bytes = bytes;
    }
    return b.p;
}

// n host values rounded to BF16 on the device, through a staging buffer of at
// most 16 MB (rounding 8192 x 148 values on one host core took 268 us, the
// copy of the FP32 values instead of the rounded ones takes 60 us more)
void Mlp::upload_bf16(const float* host, size_t n, uint16_t* dst)
{
    const size_t chunk = std::min<size_t>(n, size_t(4) << 20);
    float* st = static_cast<float*>(io_buffer(kIoStage, chunk * sizeof(float)));
    for (size_t o = 0; o < n; o += chunk) {
        const size_t m = std::min(chunk, n - o);
        HIP_CHECK(hipMemcpyAsync(st, host + o, m * sizeof(float), hipMemcpyHostToDevice, s));
        hipLaunchKernelGGL(round_bf16_kernel, dim3(cdiv(long(m), 1024)), dim3(256), 0, s, st, long(m), dst + o);
    }
}

void Mlp::set_params(const float* host)
{
    HIP_CHECK(hipMemcpyAsync(P, host, nparam * sizeof(float), hipMemcpyHostToDevice, s));
    HIP_CHECK(hipMemsetAsync(Am, 0, nparam * sizeof(float), s));
    HIP_CHECK(hipMemsetAsync(Av, 0, nparam * sizeof(float), s));
    adam_t = 0;
    refresh_bf16();
    HIP_CHECK(hipStreamSynchronize(s));
}

void Mlp::get_params(float* host) const
{
    HIP_CHECK(hipMemcpyAsync(host, P, nparam * sizeof(float), hipMemcpyDeviceToHost, s));
    HIP_CHECK(hipStreamSynchronize(s));
}

void Mlp::get_grads(float* host) const
{
    HIP_CHECK(hipMemcpyAsync(host, G, nparam * sizeof(float), hipMemcpyDeviceToHost, s));
    HIP_CHECK(hipStreamSynchronize(s));
}

void Mlp::refresh_bf16()
{
    const int in[3] = {din, dh, dh}, out[3] = {dh, dh, dout};
    for (int l = 0; l < 3; ++l)
        hipLaunchKernelGGL(to_bf16_kernel, dim3(cdiv(long(in[l]) * out[l], 256)), dim3(256), 0, s, P + off_W[l],
                           in[l], out[l], Wb[l], WbT[l]);
}

void Mlp::ensure_rows(int M)
{
    if (M <= cap_rows) return;
    H1 = static_cast<uint16_t*>(alloc(size_t(M) * dh * sizeof(uint16_t)));
    H2 = static_cast<uint16_t*>(alloc(size_t(M) * dh * sizeof(uint16_t)));
    dZ1 = static_cast<uint16_t*>(alloc(size_t(M) * dh * sizeof(uint16_t)));
    dZ2 = static_cast<uint16_t*>(alloc(size_t(M) * dh * sizeof(uint16_t)));
    dYb = static_cast<uint16_t*>(alloc(size_t(M) * dout * sizeof(uint16_t)));
    Ybuf = static_cast<float*>(alloc(size_t(M) * dout * sizeof(float)));
    cap_rows = M;
}

void Mlp::ensure_partial(size_t floats)
{
    if (floats <= partial_cap) return;
    partial = static_cast<float*>(alloc(floats * sizeof(float)));
    partial_cap = floats;
}

void Mlp::forward(const uint16_t* X, int M, float* Y, bool keep)
{
    if (M <= 0) return;
    ensure_rows(M);
    (void)keep;  // the activations always land in H1, H2
    launch_gemm_bf16(X, din, 1, Wb[0], dh, 1, M, dh, din, P + off_b[0], 1, nullptr, 0, H1, dh, nullptr, s);
    launch_gemm_bf16(H1, dh, 1, Wb[1], dh, 1, M, dh, dh, P + off_b[1], 1, nullptr, 0, H2, dh, nullptr, s);
    launch_gemm_bf16(H2, dh, 1, Wb[2], dout, 1, M, dout, dh, P + off_b[2], 0, Y ? Y : Ybuf, dout, nullptr, 0,
                     nullptr, s);
}

// dW [K][N] = A^T D over M rows, db [N] = column sums of D; A [M][lda], D [M][ldd]
void Mlp::weight_grad(const uint16_t* A, int lda, const uint16_t* D, int ldd, int M, int K, int N, float* dW,
                      float* db)
{
    // split-K: 256 rows per part, so that a few thousand rows fill the chip (8192
    // rows, 256 x 256 weights: 47 us in 8 parts of 1024 rows)
    const int nz = std::max(1, std::min(64, M / 256));
    const int kchunk = ((cdiv(M, nz) + kKStep - 1) / kKStep) * kKStep;
    const int nzz = cdiv(M, kchunk);
    ensure_partial(size_t(nzz) * (K + 1) * N);
    GemmArgs g{};
    g.A = A;
    g.sam = 1;
    g.sak = lda;
    g.B = D;
    g.sbk = ldd;
    g.sbn = 1;
    g.M = K + 1;  // the extra row reads ones: the bias gradient
    g.N = N;
    g.K = M;
    g.kchunk = kchunk;
    g.ones_row = K;
    g.C = partial;
    g.ldc = N;
    launch_gemm(g, nzz, s);
    hipLaunchKernelGGL(reduce_partials_kernel, dim3(cdiv(long(K + 1) * N, 256)), dim3(256), 0, s, partial, nzz, K, N,
                       dW, db);
}

void Mlp::backward(const uint16_t* X, const float* T, int M, float* loss_dev)
{
    if (M <= 0) return;
    ensure_rows(M);
    const long n = long(M) * dout;
    const int nblk = std::min(256, cdiv(n, 256));
    ensure_partial(size_t(nblk));
    hipLaunchKernelGGL(mse_kernel, dim3(nblk), dim3(256), 0, s, Ybuf, T, n, 1.0f / float(n), dYb, partial);
    if (loss_dev) hipLaunchKernelGGL(sum_kernel, dim3(1), dim3(256), 0, s, partial, nblk, 1.0f / float(n), loss_dev);
    // layer 3
    weight_grad(H2, dh, dYb, dout, M, dh, dout, G + off_W[2], G + off_b[2]);
    launch_gemm_bf16(dYb, dout, 1, WbT[2], dh, 1, M, dh, dout, nullptr, 0, nullptr, 0, dZ2, dh, H2, s);
    // layer 2
    weight_grad(H1, dh, dZ2, dh, M, dh, dh, G + off_W[1], G + off_b[1]);
    launch_gemm_bf16(dZ2, dh, 1, WbT[1], dh, 1, M, dh, dh, nullptr, 0, nullptr, 0, dZ1, dh, H1, s);
    // layer 1
    weight_grad(X, din, dZ1, dh, M, din, dh, G + off_W[0], G + off_b[0]);
}

void Mlp::adam_step(float lr, float beta1, float beta2, float eps)
{
    ++adam_t;
    const float c1 = 1.0f - std::pow(beta1, float(adam_t));
    const float c2 = 1.0f - std::pow(beta2, float(adam_t));
    hipLaunchKernelGGL(adam_kernel, dim3(cdiv(long(nparam), 256)), dim3(256), 0, s, P, G, Am, Av, long(nparam), lr,
                       beta1, beta2, eps, c1, c2);
    refresh_bf16();
}

}  // namespace edus
