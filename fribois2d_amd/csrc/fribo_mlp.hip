// Learned first iterate of the strong fluid-structure coupling loop: a small
// MLP (no counterpart in the reference, whose coupling is loose; the
// iterated coupling the reference prepares for is declarations.F90:250,
// 271-278) that maps the recent history of the body (displacement, velocity,
// loads) to the next step's loads.  The coupling iteration still decides the result:
// the network only proposes where it starts.
//
// Network: NI inputs -> H tanh -> H tanh -> NO linear outputs (H = 64), FP32
// parameters [W1 (H x NI, row-major), b1 (H), W2 (H x H), b2 (H), W3 (NO x H),
// b3 (NO)] at the C ABI.  On the device W1 and W2 are stored transposed (input
// by input, the 64 units side by side), so that every access of 64 lanes, one
// per unit, is one run; fribo_mlp_create and the read-backs convert.
//
// Training (FP32): the samples of a call go to the device once (sets of more
// than 64 MB in pieces); one step over a minibatch is two launches and no
// synchronisation:
//   k_mlp_step  workgroups of MLP_NS samples: both hidden layers, the outputs,
//               the back-propagated errors of the mean squared loss, and the
//               workgroup's part of the gradient, with the weights in LDS;
//   k_mlp_adam  one thread per parameter: the parts added in workgroup order
//               (deterministic) and the Adam update.
// A minibatch of 256 at NI = 45: 94 -> 16.7 us a step (65 us of the 94 one
// kernel that added 256 samples per parameter one after the other, the rest
// two pageable copies and a synchronisation).
// Inference (BF16): k_mlp_infer rounds inputs, weights and hidden
// activations to bfloat16 and accumulates in FP32.  Small sets are read from
// and written to pinned host memory by the kernel itself: one proposal 33 -> 21 us.
#include "fribo_internal.h"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <new>
#include <vector>

#define MLP_H 64
#define MLP_NS 8             // samples per workgroup, one per wave
#define MLP_NT (64 * MLP_NS) // threads per workgroup
#define MLP_PARTS 128        // most gradient parts of a minibatch
#define MLP_LDW (MLP_H + 1)  // LDS row pitch of W2: read along rows and columns

struct MlpDims {
    int ni, no;
    int w1, b1, w2, b2, w3, b3, np;   // parameter offsets and count
};

static MlpDims mlp_dims(int ni, int no)
{
    MlpDims d;
    d.ni = ni;
    d.no = no;
    d.w1 = 0;
    d.b1 = d.w1 + MLP_H * ni;
    d.w2 = d.b1 + MLP_H;
    d.b2 = d.w2 + MLP_H * MLP_H;
    d.w3 = d.b2 + MLP_H;
    d.b3 = d.w3 + no * MLP_H;
    d.np = d.b3 + no;
    return d;
}

// bfloat16 rounding (round to nearest even) of a finite float
__device__ inline float bf16r(float x)
{
    unsigned u = __float_as_uint(x);
    u = u + 0x7fffu + ((u >> 16) & 1u);
    return __uint_as_float(u & 0xffff0000u);
}

// Weights and samples of a workgroup in LDS (dynamic; floats).
struct MlpLds {
    float *w1, *b1, *w2, *b2, *w3, *b3, *x, *h1, *h2, *y, *d1, *d2;
};
__host__ __device__ inline size_t mlp_lds_floats(const MlpDims& d)
{
    return (size_t)MLP_H * d.ni + MLP_H + MLP_H * MLP_LDW + MLP_H + (size_t)d.no * MLP_H + 16 +
           (size_t)MLP_NS * d.ni + 4 * MLP_NS * MLP_H + MLP_NS * 16;
}
__device__ inline MlpLds mlp_lds(const MlpDims& d, float* l)
{
    MlpLds m;
    m.x = l;                       l += MLP_NS * d.ni;   // [ni][MLP_NS]: first, for 16-byte reads
    m.w1 = l;                      l += MLP_H * d.ni;    // [ni][H]
    m.b1 = l;                      l += MLP_H;
    m.w2 = l;                      l += MLP_H * MLP_LDW; // [H inputs][MLP_LDW]
    m.b2 = l;                      l += MLP_H;
    m.w3 = l;                      l += d.no * MLP_H;    // [no][H]
    m.b3 = l;                      l += 16;
    m.h1 = l;                      l += MLP_NS * MLP_H;  // [MLP_NS][H]
    m.h2 = l;                      l += MLP_NS * MLP_H;
    m.d1 = l;                      l += MLP_NS * MLP_H;
    m.d2 = l;                      l += MLP_NS * MLP_H;
    m.y = l;                                             // [MLP_NS][16]
    return m;
}

// Stages the parameters (rounded to bfloat16 for inference); every array of
// the device layout but b3 starts and ends on 16 bytes.
template <bool BF16>
__device__ inline void mlp_stage(const MlpDims& d, const float* __restrict__ p, const MlpLds& m)
{
    const int t = threadIdx.x;
    auto r4 = [](float4 v) {
        return BF16 ? make_float4(bf16r(v.x), bf16r(v.y), bf16r(v.z), bf16r(v.w)) : v;
    };
    const float4* const w1 = (const float4*)(p + d.w1);
    const float4* const w2 = (const float4*)(p + d.w2);
    const float4* const w3 = (const float4*)(p + d.w3);
#pragma unroll 4
    for (int q = t; q < MLP_H / 4 * d.ni; q += MLP_NT) ((float4*)m.w1)[q] = r4(w1[q]);
#pragma unroll
    for (int q = t; q < MLP_H * MLP_H / 4; q += MLP_NT) {
        const float4 v = r4(w2[q]);
        float* const o = m.w2 + (q >> 4) * MLP_LDW + 4 * (q & 15);
        o[0] = v.x;
        o[1] = v.y;
        o[2] = v.z;
        o[3] = v.w;
    }
    if (t < MLP_H / 4 * d.no) ((float4*)m.w3)[t] = r4(w3[t]);
    if (t < MLP_H) {
        m.b1[t] = BF16 ? bf16r(p[d.b1 + t]) : p[d.b1 + t];
        m.b2[t] = BF16 ? bf16r(p[d.b2 + t]) : p[d.b2 + t];
    }
    if (t < d.no) m.b3[t] = BF16 ? bf16r(p[d.b3 + t]) : p[d.b3 + t];
}

// Inputs of the samples [b0, b0 + MLP_NS) below B, zeros past them; wave g
// takes sample g.
template <bool BF16>
__device__ inline void mlp_inputs(const MlpDims& d, const float* __restrict__ X, int b0, int B, const MlpLds& m)
{
    const int s = threadIdx.x >> 6;
    for (int i = threadIdx.x & 63; i < d.ni; i += 64) {
        const float x = b0 + s < B ? X[(size_t)(b0 + s) * d.ni + i] : 0.0f;
        m.x[i * MLP_NS + s] = BF16 ? bf16r(x) : x;
    }
}

// Both hidden layers and the outputs (m.y) of the staged samples: wave g
// takes sample g, lane u unit u; sums in input order from the bias on.
template <bool BF16>
__device__ inline void mlp_forward(const MlpDims& d, const MlpLds& m)
{
    const int t = threadIdx.x, u = t & 63, s = t >> 6;
    float a = m.b1[u];
#pragma unroll 8
    for (int i = 0; i < d.ni; ++i) a = fmaf(m.w1[i * MLP_H + u], m.x[i * MLP_NS + s], a);
    a = tanhf(a);
    m.h1[s * MLP_H + u] = BF16 ? bf16r(a) : a;
    __syncthreads();
    a = m.b2[u];
#pragma unroll 16
    for (int i = 0; i < MLP_H; ++i) a = fmaf(m.w2[i * MLP_LDW + u], m.h1[s * MLP_H + i], a);
    a = tanhf(a);
    m.h2[s * MLP_H + u] = BF16 ? bf16r(a) : a;
    __syncthreads();
    if (u < d.no) {
        float y = m.b3[u];
#pragma unroll 16
        for (int i = 0; i < MLP_H; ++i) y = fmaf(m.w3[u * MLP_H + i], m.h2[s * MLP_H + i], y);
        m.y[s * 16 + u] = y;
    }
    __syncthreads();
}

// Forward and backward of a minibatch of B samples, loss
// L = (1 / (B NO)) sum (Y - T)^2: workgroup g takes the groups of MLP_NS
// samples g, g + parts, ... and leaves its part of the gradient (device
// layout) in G + g * np; Y (optional) receives the outputs.
__global__ __launch_bounds__(MLP_NT) void k_mlp_step(MlpDims d, const float* __restrict__ p, int B,
                                                     const float* __restrict__ X, const float* __restrict__ T,
                                                     float* __restrict__ G, float* __restrict__ Y)
{
    extern __shared__ __attribute__((aligned(16))) float lds[];
    const MlpLds m = mlp_lds(d, lds);
    const int u = threadIdx.x & 63, g = threadIdx.x >> 6;
    const float sc = 2.0f / (float)(B * d.no);
    float* const part = G + (size_t)blockIdx.x * d.np;
    mlp_stage<false>(d, p, m);
    for (int b0 = blockIdx.x * MLP_NS; b0 < B; b0 += gridDim.x * MLP_NS) {
        const bool first = b0 == (int)blockIdx.x * MLP_NS;
        const int b = b0 + g;   // the wave's sample
        mlp_inputs<false>(d, X, b0, B, m);
        const float tgt = u < d.no && b < B ? T[(size_t)b * d.no + u] : 0.0f;
        __syncthreads();
        mlp_forward<false>(d, m);
        // output errors in place of the outputs
        if (u < d.no) {
            const float y = m.y[g * 16 + u];
            if (b < B && Y) Y[(size_t)b * d.no + u] = y;
            m.y[g * 16 + u] = b < B ? sc * (y - tgt) : 0.0f;
        }
        __syncthreads();
        float a = 0.0f;
        for (int o = 0; o < d.no; ++o) a = fmaf(m.w3[o * MLP_H + u], m.y[g * 16 + o], a);
        float h = m.h2[g * MLP_H + u];
        m.d2[g * MLP_H + u] = a * (1.0f - h * h);
        __syncthreads();
        a = 0.0f;
        // unit o's weight of input u
#pragma unroll 16
        for (int o = 0; o < MLP_H; ++o) a = fmaf(m.w2[u * MLP_LDW + o], m.d2[g * MLP_H + o], a);
        h = m.h1[g * MLP_H + u];
        m.d1[g * MLP_H + u] = a * (1.0f - h * h);
        __syncthreads();
        // gradient parts: lane u, wave g takes every MLP_NS-th input
        float e1[MLP_NS], e2[MLP_NS];
#pragma unroll
        for (int s = 0; s < MLP_NS; ++s) {
            e1[s] = m.d1[s * MLP_H + u];
            e2[s] = m.d2[s * MLP_H + u];
        }
        auto put = [&](int q, float v) { part[q] = first ? v : part[q] + v; };
#pragma unroll 4
        for (int i = g; i < d.ni; i += MLP_NS) {
            float v = 0.0f;
#pragma unroll
            for (int s = 0; s < MLP_NS; ++s) v = fmaf(e1[s], m.x[i * MLP_NS + s], v);
            put(d.w1 + i * MLP_H + u, v);
        }
#pragma unroll
        for (int i = g; i < MLP_H; i += MLP_NS) {
            float v = 0.0f;
#pragma unroll
            for (int s = 0; s < MLP_NS; ++s) v = fmaf(e2[s], m.h1[s * MLP_H + i], v);
            put(d.w2 + i * MLP_H + u, v);
        }
        for (int o = g; o < d.no; o += MLP_NS) {
            float v = 0.0f;
#pragma unroll
            for (int s = 0; s < MLP_NS; ++s) v = fmaf(m.y[s * 16 + o], m.h2[s * MLP_H + u], v);
            put(d.w3 + o * MLP_H + u, v);
        }
        if (g == 0) {
            float v1 = 0.0f, v2 = 0.0f;
#pragma unroll
            for (int s = 0; s < MLP_NS; ++s) {
                v1 += e1[s];
                v2 += e2[s];
            }
            put(d.b1 + u, v1);
            put(d.b2 + u, v2);
            if (u < d.no) {
                float v3 = 0.0f;
#pragma unroll
                for (int s = 0; s < MLP_NS; ++s) v3 += m.y[s * 16 + u];
                put(d.b3 + u, v3);
            }
        }
        __syncthreads();
    }
}

// Gradient of every parameter (the parts in workgroup order) and, when
// lr > 0, the Adam step t (c1, c2: bias corrections); grad (optional)
// receives the gradient.
__global__ __launch_bounds__(256) void k_mlp_adam(int np, float* __restrict__ p, float* __restrict__ m1,
                                                  float* __restrict__ m2, int parts, const float* __restrict__ G,
                                                  float lr, float c1, float c2, float* __restrict__ grad)
{
    const int q = blockIdx.x * 256 + threadIdx.x;
    if (q >= np) return;
    float g = 0.0f;
    const float a1 = m1[q], a2 = m2[q], pq = p[q];
#pragma unroll 16
    for (int w = 0; w < parts; ++w) g += G[(size_t)w * np + q];
    if (grad) grad[q] = g;
    if (lr <= 0.0f) return;
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    const float a = b1 * a1 + (1.0f - b1) * g;
    const float v = b2 * a2 + (1.0f - b2) * g * g;
    m1[q] = a;
    m2[q] = v;
    p[q] = pq - lr * (a * c1) / (sqrtf(v * c2) + eps);
}

// BF16 inference of n samples (products of two bfloat16 values are exact in
// FP32, so the fused accumulation rounds as a separate one does).
__global__ __launch_bounds__(MLP_NT) void k_mlp_infer(MlpDims d, const float* __restrict__ p, int n,
                                                      const float* __restrict__ X, float* __restrict__ Y)
{
    extern __shared__ __attribute__((aligned(16))) float lds[];
    const MlpLds m = mlp_lds(d, lds);
    const int u = threadIdx.x & 63, b = blockIdx.x * MLP_NS + (threadIdx.x >> 6);
    mlp_inputs<true>(d, X, blockIdx.x * MLP_NS, n, m);
    mlp_stage<true>(d, p, m);
    __syncthreads();
    mlp_forward<true>(d, m);
    if (u < d.no && b < n) Y[(size_t)b * d.no + u] = m.y[(threadIdx.x >> 6) * 16 + u];
}

// ---------------------------------------------------------------------------
// C ABI
struct fribo_mlp_ctx {
    MlpDims d;
    hipStream_t st = nullptr;
    float *p = nullptr, *m1 = nullptr, *m2 = nullptr, *g = nullptr;   // one allocation, device layout
    float* work = nullptr;       // device work space of `cap` floats
    size_t cap = 0;
    float* pin = nullptr;        // pinned host memory: MLP_PIN floats and the staged parameters
    long step = 0;               // Adam steps taken
};
typedef fribo_mlp_ctx* fribo_mlp;

// Floats of pinned memory a network keeps (64 KB): the largest set whose
// inputs and outputs the inference kernel reads and writes on the host.
#define MLP_PIN 16384

// Most floats of a training set (inputs and targets, 64 MB) that are copied to
// the device at once and kept there with the network; a larger set goes in
// pieces, again in every epoch.
#define MLP_SET ((size_t)16 << 20)

static int mlp_reserve(fribo_mlp m, size_t floats)
{
    if (floats <= m->cap) return 0;
    if (m->work) hipFree(m->work);
    m->work = nullptr;
    m->cap = 0;
    if (hipMalloc(&m->work, floats * sizeof(float)) != hipSuccess) return FRIBO_E_HIP;
    m->cap = floats;
    return 0;
}

// Device layout <-> C ABI layout of parameters and gradients.
static void mlp_layout(const MlpDims& d, const float* src, float* dst, bool to_device)
{
    auto turn = [&](int o, int ncol) {   // H x ncol rows at the ABI, ncol x H on the device
        for (int u = 0; u < MLP_H; ++u)
            for (int i = 0; i < ncol; ++i) {
                const int a = o + u * ncol + i, b = o + i * MLP_H + u;
                if (to_device) dst[b] = src[a];
                else dst[a] = src[b];
            }
    };
    turn(d.w1, d.ni);
    std::copy(src + d.b1, src + d.w2, dst + d.b1);
    turn(d.w2, MLP_H);
    std::copy(src + d.b2, src + d.np, dst + d.b2);
}

// Network with ni inputs (<= 256) and no outputs (<= 16); parameters from
// init (np floats, as fribo_mlp_size reports) or, when init is NULL,
// Glorot-uniform weights from the seed and zero biases.
extern "C" int fribo_mlp_create(int32_t ni, int32_t no, const float* init, uint64_t seed, fribo_mlp* out)
{
    if (!out || ni < 1 || ni > 256 || no < 1 || no > 16) return FRIBO_E_ARG;
    fribo_mlp m = new fribo_mlp_ctx();
    m->d = mlp_dims(ni, no);
    const MlpDims& d = m->d;
    std::vector<float> p0(d.np, 0.0f);
    if (init) {
        std::copy(init, init + d.np, p0.begin());
    } else {
        uint64_t s = seed ? seed : 0x9e3779b97f4a7c15ull;
        auto uni = [&s]() {   // splitmix64 -> [-1, 1)
            uint64_t z = (s += 0x9e3779b97f4a7c15ull);
            z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
            z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
            z = z ^ (z >> 31);
            return (float)((double)(z >> 11) * (2.0 / 9007199254740992.0) - 1.0);
        };
        const float a1 = std::sqrt(6.0f / (ni + MLP_H)), a2 = std::sqrt(6.0f / (2 * MLP_H)),
                    a3 = std::sqrt(6.0f / (MLP_H + no));
        for (int q = d.w1; q < d.b1; ++q) p0[q] = a1 * uni();
        for (int q = d.w2; q < d.b2; ++q) p0[q] = a2 * uni();
        for (int q = d.w3; q < d.b3; ++q) p0[q] = a3 * uni();
    }
    // parameters, both moments (zero) and the gradient in one allocation; the
    // upload is staged past the pinned memory of the inference and not waited for
    const size_t nb = (size_t)d.np * sizeof(float);
    if (hipStreamCreate(&m->st) != hipSuccess || hipMalloc(&m->p, 4 * nb) != hipSuccess ||
        hipHostMalloc((void**)&m->pin, MLP_PIN * sizeof(float) + nb, hipHostMallocDefault) != hipSuccess ||
        (mlp_layout(d, p0.data(), m->pin + MLP_PIN, true), false) ||
        hipMemcpyAsync(m->p, m->pin + MLP_PIN, nb, hipMemcpyHostToDevice, m->st) != hipSuccess ||
        hipMemsetAsync(m->p + d.np, 0, 2 * nb, m->st) != hipSuccess) {
        if (m->p) hipFree(m->p);
        if (m->pin) hipHostFree(m->pin);
        if (m->st) hipStreamDestroy(m->st);
        delete m;
        return FRIBO_E_HIP;
    }
    m->m1 = m->p + d.np;
    m->m2 = m->m1 + d.np;
    m->g = m->m2 + d.np;
    *out = m;
    return 0;
}

extern "C" int fribo_mlp_destroy(fribo_mlp m)
{
    if (!m) return FRIBO_E_ARG;
    hipStreamSynchronize(m->st);
    if (m->work) hipFree(m->work);
    hipFree(m->p);
    hipHostFree(m->pin);
    hipStreamDestroy(m->st);
    delete m;
    return 0;
}

extern "C" int fribo_mlp_size(fribo_mlp m)
{
    return m ? m->d.np : -1;
}

// A device array of np floats in the ABI's layout.
static int mlp_fetch(fribo_mlp m, const float* dev, float* out)
{
    std::vector<float> v(m->d.np);
    if (hipMemcpyAsync(v.data(), dev, v.size() * sizeof(float), hipMemcpyDeviceToHost, m->st) != hipSuccess ||
        hipStreamSynchronize(m->st) != hipSuccess)
        return FRIBO_E_HIP;
    mlp_layout(m->d, v.data(), out, false);
    return 0;
}

extern "C" int fribo_mlp_get_params(fribo_mlp m, float* out)
{
    if (!m || !out) return FRIBO_E_ARG;
    return mlp_fetch(m, m->p, out);
}

// Passes over n samples (X n x ni, T n x no, row-major) in minibatches of
// `batch`, `epochs` times: forward, backward and, with lr > 0, one Adam step
// per minibatch.  grad (optional, np floats) receives the last minibatch's
// gradient of the mean squared loss, loss (optional) its value.
static int mlp_run(fribo_mlp m, int n, const float* X, const float* T, int epochs, int batch, float lr, float* grad,
                   float* loss)
{
    const MlpDims& d = m->d;
    batch = std::min(batch, n);
    const int most = std::min((batch + MLP_NS - 1) / MLP_NS, MLP_PARTS);
    // the samples on the device at a time: all of them, or as many whole
    // minibatches as MLP_SET floats hold (one at least)
    const size_t per = (size_t)d.ni + d.no;
    int win = n;
    if (per * n > MLP_SET) win = std::max(1, (int)std::min<size_t>(MLP_SET / per, n) / batch) * batch;
    win = std::min(win, n);
    const size_t nx = (size_t)win * d.ni, nt = (size_t)win * d.no, ny = loss ? (size_t)batch * d.no : 0;
    if (mlp_reserve(m, nx + nt + ny + (size_t)most * d.np)) return FRIBO_E_HIP;
    float *dX = m->work, *dT = dX + nx, *dY = dT + nt, *dG = dY + ny;
    const size_t lds = mlp_lds_floats(d) * sizeof(float);
    int b = 0, s = 0, w0 = -1;   // w0: first sample on the device
    for (int e = 0; e < epochs; ++e)
        for (s = 0; s < n; s += batch) {
            b = std::min(batch, n - s);
            if (w0 < 0 || s < w0 || s - w0 >= win) {
                w0 = s;
                const size_t c = std::min(win, n - s);
                if (hipMemcpyAsync(dX, X + (size_t)s * d.ni, c * d.ni * sizeof(float), hipMemcpyHostToDevice, m->st) !=
                        hipSuccess ||
                    hipMemcpyAsync(dT, T + (size_t)s * d.no, c * d.no * sizeof(float), hipMemcpyHostToDevice, m->st) !=
                        hipSuccess)
                    return FRIBO_E_HIP;
            }
            const size_t o = s - w0;
            const bool last = e == epochs - 1 && s + batch >= n;
            const int parts = std::min((b + MLP_NS - 1) / MLP_NS, MLP_PARTS);
            hipLaunchKernelGGL(k_mlp_step, dim3(parts), dim3(MLP_NT), lds, m->st, d, (const float*)m->p, b,
                               (const float*)dX + o * d.ni, (const float*)dT + o * d.no, dG,
                               last && loss ? dY : (float*)nullptr);
            float c1 = 1.0f, c2 = 1.0f;
            if (lr > 0.0f) {
                ++m->step;
                c1 = 1.0f / (1.0f - std::pow(0.9f, (float)m->step));
                c2 = 1.0f / (1.0f - std::pow(0.999f, (float)m->step));
            }
            hipLaunchKernelGGL(k_mlp_adam, dim3((d.np + 255) / 256), dim3(256), 0, m->st, d.np, m->p, m->m1, m->m2,
                               parts, (const float*)dG, lr, c1, c2, grad && last ? m->g : (float*)nullptr);
            if (last) break;
        }
    if (hipGetLastError() != hipSuccess) return FRIBO_E_HIP;
    std::vector<float> y;
    if (loss) {
        y.resize((size_t)b * d.no);
        if (hipMemcpyAsync(y.data(), dY, y.size() * sizeof(float), hipMemcpyDeviceToHost, m->st) != hipSuccess)
            return FRIBO_E_HIP;
    }
    if (hipStreamSynchronize(m->st) != hipSuccess) return FRIBO_E_HIP;
    if (grad) {
        const int rc = mlp_fetch(m, m->g, grad);
        if (rc) return rc;
    }
    if (loss) {
        double v = 0.0;
        for (size_t i = 0; i < y.size(); ++i) {
            const double e = (double)y[i] - (double)T[(size_t)s * d.no + i];
            v += e * e;
        }
        *loss = (float)(v / (double)y.size());
    }
    return 0;
}

// Gradient of the mean squared loss over the n samples (no update).
extern "C" int fribo_mlp_grad(fribo_mlp m, int32_t n, const float* X, const float* T, float* grad, float* loss)
{
    if (!m || n < 1 || !X || !T) return FRIBO_E_ARG;
    return mlp_run(m, n, X, T, 1, n, 0.0f, grad, loss);
}

// Adam training: epochs passes over the n samples in minibatches of
// `batch` samples (in order; the caller shuffles), learning rate lr.
// loss (optional) gets the mean squared loss of the last minibatch.
extern "C" int fribo_mlp_train(fribo_mlp m, int32_t n, const float* X, const float* T, int32_t epochs,
                               int32_t batch, float lr, float* loss)
{
    if (!m || n < 1 || epochs < 1 || batch < 1 || !(lr > 0.0f) || !X || !T) return FRIBO_E_ARG;
    return mlp_run(m, n, X, T, epochs, batch, lr, nullptr, loss);
}

// Inference in BF16 (FP32 accumulation) of n samples: Y = net(X).
extern "C" int fribo_mlp_predict(fribo_mlp m, int32_t n, const float* X, float* Y)
{
    if (!m || n < 1 || !X || !Y) return FRIBO_E_ARG;
    const MlpDims& d = m->d;
    const size_t nx = (size_t)n * d.ni, ny = (size_t)n * d.no;
    const size_t lds = mlp_lds_floats(d) * sizeof(float);
    const dim3 g((n + MLP_NS - 1) / MLP_NS);
    if (nx + ny <= MLP_PIN) {
        // the kernel reads and writes the pinned memory itself: no copies
        memcpy(m->pin, X, nx * sizeof(float));
        hipLaunchKernelGGL(k_mlp_infer, g, dim3(MLP_NT), lds, m->st, d, (const float*)m->p, n, (const float*)m->pin,
                           m->pin + nx);
        if (hipGetLastError() != hipSuccess || hipStreamSynchronize(m->st) != hipSuccess) return FRIBO_E_HIP;
        memcpy(Y, m->pin + nx, ny * sizeof(float));
        return 0;
    }
    if (mlp_reserve(m, nx + ny)) return FRIBO_E_HIP;
    if (hipMemcpyAsync(m->work, X, nx * sizeof(float), hipMemcpyHostToDevice, m->st) != hipSuccess) return FRIBO_E_HIP;
    hipLaunchKernelGGL(k_mlp_infer, g, dim3(MLP_NT), lds, m->st, d, (const float*)m->p, n, (const float*)m->work,
                       m->work + nx);
    if (hipGetLastError() != hipSuccess) return FRIBO_E_HIP;
    if (hipMemcpyAsync(Y, m->work + nx, ny * sizeof(float), hipMemcpyDeviceToHost, m->st) != hipSuccess ||
        hipStreamSynchronize(m->st) != hipSuccess)
        return FRIBO_E_HIP;
    return 0;
}
