// dmx_mlp.hip -- training of the learned slope limiter on the GPU:
// forward and backward passes of the 40-64-64-8 GELU network (float32),
// mean-squared-error loss, Adam, and on-device minibatch sampling from a
// resident data set (two kernels a step); plus a self-test of the bf16 MFMA lane layout that the
// inference kernel of the step relies on.
#include <hip/hip_runtime.h>

#include <stdint.h>
#include <string.h>

#include <algorithm>

#include "dmx.h"
#include "dmx_engine.h"
#include "dmx_mlp.h"

namespace dmx {
namespace mlp {

// minibatch of rows drawn from n rows with a counter-based hash (splitmix64
// finaliser of seed + draw number)
__device__ __forceinline__ unsigned long long mix64(unsigned long long z)
{
    z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ULL;
    z = (z ^ (z >> 27)) * 0x94d049bb133111ebULL;
    return z ^ (z >> 31);
}

// ---------------------------------------------------------------------------
// Forward and backward pass in one kernel.  A block takes tiles of TS rows
// (tile blockIdx.x, + gridDim.x, ...) through the three layers with the
// weights and every activation in LDS, and adds the tiles' parameter
// gradients in registers; its sums go to part[block][NPARAM] and k_reduce
// adds the blocks'.  With a launch per layer and pass the activations went
// through HBM, and the weight gradients (one block per output column, a
// reduction per weight) took most of a step: 0.90 ms a step of 4096 rows in
// 11 launches, now 0.03 ms in 2.
//
// TS = 16 gives a batch of 4096 256 blocks, one per CU; larger batches give
// a block several tiles.  W2 rows are padded to 65 words, so that the
// backward pass reads its columns without bank conflicts.
// ---------------------------------------------------------------------------
constexpr int TS = 16, MAXBLK = 256, LW2S = NH + 1;

struct TrainLds {
    float w1[NIN * NH], w2[NH * LW2S], w3[NH * NOUT];
    float b1[NH], b2[NH], b3[NOUT];
    float x[NIN][TS], t[NOUT][TS];               // rows of the tile, transposed
    float h1[NH][TS], d1[NH][TS];                // gelu(a1), gelu'(a1); then d1 holds dL/da1
    float h2[NH][TS], d2[NH][TS];
    float g3[NOUT][TS];                          // dL/dy
    double loss[TS * NOUT];
    long long row[TS];
};

// X, T: data (rows drawn by the hash of key when ndata > 0, else row s of the
// batch is row s); n rows in the batch; y: outputs (may be null); part: block
// gradients (null: forward only); lpart: block sums of 0.5 (y - T)^2 / n, in
// float64 from the single terms on
__global__ __launch_bounds__(256) void k_fwd_bwd(const float* __restrict__ X, const float* __restrict__ T, long long ndata,
                                                 int n, unsigned long long key, const float* __restrict__ th,
                                                 float* __restrict__ y, float* __restrict__ part,
                                                 double* __restrict__ lpart)
{
    __shared__ TrainLds L;
    const int tid = threadIdx.x;
    for (int i = tid; i < NIN * NH; i += 256) L.w1[i] = th[OFF_W1 + i];
    for (int i = tid; i < NH * NH; i += 256) L.w2[(i / NH) * LW2S + i % NH] = th[OFF_W2 + i];
    for (int i = tid; i < NH * NOUT; i += 256) L.w3[i] = th[OFF_W3 + i];
    if (tid < NH) {
        L.b1[tid] = th[OFF_B1 + tid];
        L.b2[tid] = th[OFF_B2 + tid];
    }
    if (tid < NOUT) L.b3[tid] = th[OFF_B3 + tid];
    // thread (o, q): column o of a layer, rows 4 q .. 4 q + 3 of the tile (and
    // quarter q of a weight matrix's rows)
    const int o = tid & 63, q = tid >> 6, s0 = 4 * q;
    float gw1[NIN / 4] = {}, gw2[NH / 4] = {}, gw3[2] = {}, gb = 0.0f;
    double lsum = 0.0;   // float64: a block of a large batch adds hundreds of tiles' terms
    const float rows = (float)n;
    const int ntile = (n + TS - 1) / TS;
    for (int tile = blockIdx.x; tile < ntile; tile += gridDim.x) {
        const int base = tile * TS;
        __syncthreads();   // the previous tile's reads are done, the weights are there
        if (tid < TS) {
            const unsigned long long b = (unsigned long long)(base + tid);
            L.row[tid] = ndata > 0 ? (long long)(mix64(key + b * 0x9e3779b97f4a7c15ULL) % (unsigned long long)ndata)
                                   : (long long)b;
        }
        __syncthreads();
        for (int e = tid; e < TS * NIN; e += 256) {
            const int s = e / NIN, i = e - s * NIN;
            L.x[i][s] = base + s < n ? X[L.row[s] * NIN + i] : 0.0f;
        }
        if (T && tid < TS * NOUT) {
            const int s = tid / NOUT, i = tid % NOUT;
            L.t[i][s] = base + s < n ? T[L.row[s] * NOUT + i] : 0.0f;
        }
        __syncthreads();
        {
            float a[4];
            for (int r = 0; r < 4; r++) a[r] = L.b1[o];
#pragma unroll 8
            for (int i = 0; i < NIN; i++) {
                const float w = L.w1[i * NH + o];
                for (int r = 0; r < 4; r++) a[r] += L.x[i][s0 + r] * w;
            }
            for (int r = 0; r < 4; r++) gelu_both(a[r], L.h1[o][s0 + r], L.d1[o][s0 + r]);
        }
        __syncthreads();
        {
            float a[4];
            for (int r = 0; r < 4; r++) a[r] = L.b2[o];
#pragma unroll 8
            for (int i = 0; i < NH; i++) {
                const float w = L.w2[i * LW2S + o];
                for (int r = 0; r < 4; r++) a[r] += L.h1[i][s0 + r] * w;
            }
            for (int r = 0; r < 4; r++) gelu_both(a[r], L.h2[o][s0 + r], L.d2[o][s0 + r]);
        }
        __syncthreads();
        if (tid < TS * NOUT) {
            const int s = tid / NOUT, c = tid % NOUT;
            float a = L.b3[c];
#pragma unroll 8
            for (int i = 0; i < NH; i++) a += L.h2[i][s] * L.w3[i * NOUT + c];
            const bool on = base + s < n;
            if (y && on) y[(long long)(base + s) * NOUT + c] = a;
            const float r = T && on ? a - L.t[c][s] : 0.0f;
            L.g3[c][s] = r / rows;
            lsum += 0.5f * r * r / rows;
        }
        __syncthreads();
        if (!part) continue;
        // layer 3: weight and input gradients
        for (int m = 0; m < 2; m++) {
            const int e = tid + 256 * m, i = e / NOUT, c = e % NOUT;
            for (int s = 0; s < TS; s++) gw3[m] += L.h2[i][s] * L.g3[c][s];
        }
        {
            float a[4] = {};
#pragma unroll
            for (int c = 0; c < NOUT; c++)
                for (int r = 0; r < 4; r++) a[r] += L.g3[c][s0 + r] * L.w3[o * NOUT + c];
            for (int r = 0; r < 4; r++) L.d2[o][s0 + r] *= a[r];
        }
        __syncthreads();
        // layer 2
#pragma unroll 4
        for (int s = 0; s < TS; s++) {
            const float g = L.d2[o][s];
            for (int m = 0; m < NH / 4; m++) gw2[m] += L.h1[q * (NH / 4) + m][s] * g;
        }
        {
            float a[4] = {};
#pragma unroll 8
            for (int c = 0; c < NH; c++) {
                const float w = L.w2[o * LW2S + c];
                for (int r = 0; r < 4; r++) a[r] += L.d2[c][s0 + r] * w;
            }
            for (int r = 0; r < 4; r++) L.d1[o][s0 + r] *= a[r];
        }
        __syncthreads();
        // layer 1, and the biases: b1 (q = 0), b2 (q = 1), b3 (q = 2, o < 8)
#pragma unroll 4
        for (int s = 0; s < TS; s++) {
            const float g = L.d1[o][s];
            for (int m = 0; m < NIN / 4; m++) gw1[m] += L.x[q * (NIN / 4) + m][s] * g;
        }
        if (q < 2 || (q == 2 && o < NOUT)) {
            const float* d = q == 0 ? L.d1[o] : (q == 1 ? L.d2[o] : L.g3[o]);
            for (int s = 0; s < TS; s++) gb += d[s];
        }
    }
    if (lpart) {
        if (tid < TS * NOUT) L.loss[tid] = lsum;
        __syncthreads();
        for (int w = TS * NOUT / 2; w > 0; w >>= 1) {
            if (tid < w) L.loss[tid] += L.loss[tid + w];
            __syncthreads();
        }
        if (tid == 0) lpart[blockIdx.x] = L.loss[0];
    }
    if (!part) return;
    float* P = part + (long long)blockIdx.x * NPARAM;
    for (int m = 0; m < NIN / 4; m++) P[OFF_W1 + (q * (NIN / 4) + m) * NH + o] = gw1[m];
    for (int m = 0; m < NH / 4; m++) P[OFF_W2 + (q * (NH / 4) + m) * NH + o] = gw2[m];
    for (int m = 0; m < 2; m++) P[OFF_W3 + tid + 256 * m] = gw3[m];
    if (q == 0) P[OFF_B1 + o] = gb;
    if (q == 1) P[OFF_B2 + o] = gb;
    if (q == 2 && o < NOUT) P[OFF_B3 + o] = gb;
}

// gradient = sum of the blocks' (64 parameters per block, a sixteenth of the
// blocks per wave), and with lr > 0 the Adam update (Kingma and Ba 2015) with
// the bias-corrected step size; block 0 adds the blocks' losses in float64
constexpr int RW = 16;
__global__ __launch_bounds__(64 * RW) void k_reduce(const float* __restrict__ part, const double* __restrict__ lpart,
                                                    int nblk, float* __restrict__ gr, float* __restrict__ loss,
                                                    float* __restrict__ th, float* __restrict__ m,
                                                    float* __restrict__ v, float lr, float b1, float b2, float eps,
                                                    float c1, float c2)
{
    __shared__ float red[RW][64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int t = blockIdx.x * 64 + lane;
    float a = 0.0f;
    if (t < NPARAM)
#pragma unroll 4
        for (int b = w; b < nblk; b += RW) a += part[(long long)b * NPARAM + t];
    red[w][lane] = a;
    __syncthreads();
    if (w == 0 && t < NPARAM) {
        float g = red[0][lane];
        for (int r = 1; r < RW; r++) g += red[r][lane];
        gr[t] = g;
        if (lr > 0.0f) {
            float mm = b1 * m[t] + (1.0f - b1) * g;
            float vv = b2 * v[t] + (1.0f - b2) * g * g;
            m[t] = mm;
            v[t] = vv;
            th[t] -= lr * (mm / c1) / (sqrtf(vv / c2) + eps);
        }
    }
    if (blockIdx.x == 0 && w == 1) {
        double l = 0.0;
        for (int b = lane; b < nblk; b += 64) l += lpart[b];
        for (int off = 32; off > 0; off >>= 1) l += __shfl_xor(l, off, 64);
        if (lane == 0) *loss = (float)l;
    }
}

// D = A B for A[i][k] = (i + 2k mod 7) / 8, B[k][j] = (3k + j mod 5) / 4 - 0.5
// (exact in bf16), through the MFMA lane layout of dmx_mlp.h
__global__ void k_mfma_selftest(float* out)
{
    const int l = threadIdx.x;
    bf16x8 a, b;
    for (int e = 0; e < 8; e++) {
        int k = 8 * (l / 16) + e;
        a[e] = (__bf16)(float((l % 16 + 2 * k) % 7) / 8.0f);
        b[e] = (__bf16)(float((3 * k + l % 16) % 5) / 4.0f - 0.5f);
    }
    f32x4 c = {0.0f, 0.0f, 0.0f, 0.0f};
    c = mfma16x16x32(a, b, c);
    for (int r = 0; r < 4; r++) out[(4 * (l / 16) + r) * 16 + (l % 16)] = c[r];
}

} // namespace mlp
} // namespace dmx

using namespace dmx::mlp;

struct dmx_mlp {
    int cap = 0;
    float* th = nullptr;     // parameters
    float* gr = nullptr;     // gradient
    float* m = nullptr;
    float* v = nullptr;
    float* ws = nullptr;     // workspace
    float* X = nullptr;      // resident data set
    float* T = nullptr;
    long long ndata = 0;
    long long adam_t = 0;
    hipStream_t stream = nullptr;
    // workspace views: a batch from the host and its outputs, the blocks'
    // gradients and losses, the losses of up to LCAP steps
    float *xb, *tb, *y, *part, *loss;
    double* lpart;
};

#define MCHK(x)                                                                           \
    do {                                                                                  \
        hipError_t e_ = (x);                                                              \
        if (e_ != hipSuccess) {                                                           \
            dmx::set_error("%s:%d %s: %s", __FILE__, __LINE__, #x, hipGetErrorString(e_)); \
            return DMX_E_HIP;                                                             \
        }                                                                                 \
    } while (0)

static int cdivi(long long a, int b) { return (int)((a + b - 1) / b); }
constexpr int LCAP = 4096;

static int blocks_of(int n) { return std::min(MAXBLK, cdivi(n, TS)); }

// loss and gradient of n rows (X, T, ndata, key as k_fwd_bwd), the loss left
// in *loss on the device; with lr > 0 an Adam step
static int gradient(dmx_mlp* m, const float* X, const float* T, long long ndata, int n, unsigned long long key,
                    float* loss, float lr, float b1, float b2, float eps, float c1, float c2)
{
    const int nb = blocks_of(n);
    hipLaunchKernelGGL(k_fwd_bwd, dim3(nb), dim3(256), 0, m->stream, X, T, ndata, n, key, (const float*)m->th,
                       (float*)nullptr, m->part, m->lpart);
    hipLaunchKernelGGL(k_reduce, dim3(cdivi(NPARAM, 64)), dim3(64 * RW), 0, m->stream, (const float*)m->part,
                       (const double*)m->lpart, nb, m->gr, loss, m->th, m->m, m->v, lr, b1, b2, eps, c1, c2);
    MCHK(hipGetLastError());
    return DMX_OK;
}

extern "C" {

int dmx_mlp_create(int32_t max_batch, dmx_mlp** out)
{
    if (!out || max_batch < 1 || max_batch > (1 << 22)) {
        dmx::set_error("dmx_mlp_create: max_batch must be in [1, 4194304]");
        return DMX_E_PARAM;
    }
    *out = nullptr;
    dmx_mlp* m = new dmx_mlp();
    m->cap = max_batch;
    size_t cap = (size_t)max_batch;
    size_t wsz = cap * (NIN + NOUT + NOUT) + (size_t)MAXBLK * (NPARAM + 2) + LCAP;
    if (hipStreamCreate(&m->stream) != hipSuccess || hipMalloc(&m->th, sizeof(float) * NPARAM) != hipSuccess ||
        hipMalloc(&m->gr, sizeof(float) * NPARAM) != hipSuccess || hipMalloc(&m->m, sizeof(float) * NPARAM) != hipSuccess ||
        hipMalloc(&m->v, sizeof(float) * NPARAM) != hipSuccess || hipMalloc(&m->ws, sizeof(float) * wsz) != hipSuccess) {
        dmx::set_error("dmx_mlp_create: device allocation failed");
        dmx_mlp_destroy(m);
        return DMX_E_NOMEM;
    }
    float* p = m->ws;
    m->xb = p; p += cap * NIN;
    m->tb = p; p += cap * NOUT;
    m->y = p; p += cap * NOUT;
    m->part = p; p += (size_t)MAXBLK * NPARAM;
    static_assert((NIN + NOUT + NOUT) % 2 == 0 && NPARAM % 2 == 0, "float64 alignment of lpart");
    m->lpart = (double*)p; p += 2 * MAXBLK;
    m->loss = p;
    hipMemsetAsync(m->th, 0, sizeof(float) * NPARAM, m->stream);
    hipMemsetAsync(m->m, 0, sizeof(float) * NPARAM, m->stream);
    hipMemsetAsync(m->v, 0, sizeof(float) * NPARAM, m->stream);
    if (hipStreamSynchronize(m->stream) != hipSuccess) {
        dmx::set_error("dmx_mlp_create: initialisation failed");
        dmx_mlp_destroy(m);
        return DMX_E_HIP;
    }
    *out = m;
    return DMX_OK;
}

void dmx_mlp_destroy(dmx_mlp* m)
{
    if (!m) return;
    if (m->stream) hipStreamSynchronize(m->stream);
    float* bufs[] = {m->th, m->gr, m->m, m->v, m->ws, m->X, m->T};
    for (float* b : bufs)
        if (b) hipFree(b);
    if (m->stream) hipStreamDestroy(m->stream);
    delete m;
}

int dmx_mlp_set_params(dmx_mlp* m, const float* theta, int32_t n)
{
    if (!m || !theta || n != NPARAM) { dmx::set_error("dmx_mlp_set_params: need %d parameters", NPARAM); return DMX_E_PARAM; }
    MCHK(hipMemcpy(m->th, theta, sizeof(float) * NPARAM, hipMemcpyHostToDevice));
    MCHK(hipMemset(m->m, 0, sizeof(float) * NPARAM));
    MCHK(hipMemset(m->v, 0, sizeof(float) * NPARAM));
    m->adam_t = 0;
    return DMX_OK;
}

int dmx_mlp_get_params(dmx_mlp* m, float* theta, int32_t n)
{
    if (!m || !theta || n != NPARAM) { dmx::set_error("dmx_mlp_get_params: need %d parameters", NPARAM); return DMX_E_PARAM; }
    MCHK(hipStreamSynchronize(m->stream));
    MCHK(hipMemcpy(theta, m->th, sizeof(float) * NPARAM, hipMemcpyDeviceToHost));
    return DMX_OK;
}

int dmx_mlp_forward(dmx_mlp* m, const float* X, int32_t n, float* Y)
{
    if (!m || !X || !Y || n < 1 || n > m->cap) { dmx::set_error("dmx_mlp_forward: bad arguments"); return DMX_E_PARAM; }
    MCHK(hipMemcpyAsync(m->xb, X, sizeof(float) * (size_t)n * NIN, hipMemcpyHostToDevice, m->stream));
    hipLaunchKernelGGL(k_fwd_bwd, dim3(blocks_of(n)), dim3(256), 0, m->stream, (const float*)m->xb,
                       (const float*)nullptr, 0LL, n, 0ULL, (const float*)m->th, m->y, (float*)nullptr,
                       (double*)nullptr);
    MCHK(hipGetLastError());
    MCHK(hipMemcpyAsync(Y, m->y, sizeof(float) * (size_t)n * NOUT, hipMemcpyDeviceToHost, m->stream));
    MCHK(hipStreamSynchronize(m->stream));
    return DMX_OK;
}

int dmx_mlp_loss_grad(dmx_mlp* m, const float* X, const float* T, int32_t n, float* loss, float* grad)
{
    if (!m || !X || !T || !loss || !grad || n < 1 || n > m->cap) {
        dmx::set_error("dmx_mlp_loss_grad: bad arguments");
        return DMX_E_PARAM;
    }
    MCHK(hipMemcpyAsync(m->xb, X, sizeof(float) * (size_t)n * NIN, hipMemcpyHostToDevice, m->stream));
    MCHK(hipMemcpyAsync(m->tb, T, sizeof(float) * (size_t)n * NOUT, hipMemcpyHostToDevice, m->stream));
    int rc = gradient(m, m->xb, m->tb, 0, n, 0, m->loss, 0.0f, 0.0f, 0.0f, 0.0f, 1.0f, 1.0f);
    if (rc) return rc;
    MCHK(hipMemcpyAsync(loss, m->loss, sizeof(float), hipMemcpyDeviceToHost, m->stream));
    MCHK(hipStreamSynchronize(m->stream));
    MCHK(hipMemcpy(grad, m->gr, sizeof(float) * NPARAM, hipMemcpyDeviceToHost));
    return DMX_OK;
}

int dmx_mlp_load_data(dmx_mlp* m, const float* X, const float* T, int64_t n)
{
    if (!m || !X || !T || n < 1) { dmx::set_error("dmx_mlp_load_data: bad arguments"); return DMX_E_PARAM; }
    if (m->X) hipFree(m->X);
    if (m->T) hipFree(m->T);
    m->X = m->T = nullptr;
    m->ndata = 0;
    if (hipMalloc(&m->X, sizeof(float) * (size_t)n * NIN) != hipSuccess ||
        hipMalloc(&m->T, sizeof(float) * (size_t)n * NOUT) != hipSuccess) {
        dmx::set_error("dmx_mlp_load_data: device allocation failed");
        return DMX_E_NOMEM;
    }
    MCHK(hipMemcpy(m->X, X, sizeof(float) * (size_t)n * NIN, hipMemcpyHostToDevice));
    MCHK(hipMemcpy(m->T, T, sizeof(float) * (size_t)n * NOUT, hipMemcpyHostToDevice));
    m->ndata = n;
    return DMX_OK;
}

int dmx_mlp_train(dmx_mlp* m, int32_t steps, int32_t batch, float lr, uint64_t seed, float* losses)
{
    if (!m || steps < 0 || batch < 1 || batch > m->cap || !(lr > 0.0f)) {
        dmx::set_error("dmx_mlp_train: bad arguments");
        return DMX_E_PARAM;
    }
    if (!m->ndata) { dmx::set_error("dmx_mlp_train: no data loaded"); return DMX_E_STATE; }
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    for (int s0 = 0; s0 < steps; s0 += LCAP) {
        const int ns = std::min(LCAP, steps - s0);
        for (int s = 0; s < ns; s++) {
            unsigned long long key = seed * 0x632be59bd9b4e019ULL + (unsigned long long)(m->adam_t + 1) * 0x9e3779b97f4a7c15ULL;
            m->adam_t++;
            float c1 = 1.0f - powf(b1, (float)m->adam_t), c2 = 1.0f - powf(b2, (float)m->adam_t);
            int rc = gradient(m, m->X, m->T, m->ndata, batch, key, m->loss + s, lr, b1, b2, eps, c1, c2);
            if (rc) return rc;
        }
        if (losses) {
            // the losses of these steps, read back once
            MCHK(hipMemcpyAsync(losses + s0, m->loss, sizeof(float) * ns, hipMemcpyDeviceToHost, m->stream));
            MCHK(hipStreamSynchronize(m->stream));
        }
    }
    MCHK(hipStreamSynchronize(m->stream));
    return DMX_OK;
}

int dmx_mfma_selftest(float* out)
{
    if (!out) { dmx::set_error("null out"); return DMX_E_PARAM; }
    float* d = nullptr;
    MCHK(hipMalloc(&d, sizeof(float) * 256));
    hipLaunchKernelGGL(k_mfma_selftest, dim3(1), dim3(64), 0, 0, d);
    hipError_t e = hipGetLastError();
    if (e == hipSuccess) e = hipMemcpy(out, d, sizeof(float) * 256, hipMemcpyDeviceToHost);
    hipFree(d);
    if (e != hipSuccess) { dmx::set_error("mfma selftest: %s", hipGetErrorString(e)); return DMX_E_HIP; }
    return DMX_OK;
}

} // extern "C"
