// Training and standalone inference of the learned rate-and-state Newton
// guess (network and numerics in eqd_mlp.h), and the C entry points
// eqd_mlp_forward / eqd_mlp_grad / eqd_mlp_train of include/eqdyna_amd.h.
//
// One training step over a batch: mlp_grad_kernel (four waves per 64 samples:
// forward, mean-squared-error loss, backward; per-workgroup partial gradients
// written once, no atomics) and mlp_adam_kernel (sums the partials in
// workgroup order, so training is deterministic, then Adam on float32 master
// weights and the bfloat16 copies and transposes for the next forward pass).
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>
#include <string.h>

#include <mutex>
#include <vector>

#include "../../include/eqdyna_amd.h"

#include "eqd_mlp.h"

namespace eqd {

// Device buffers of one network: float32 master parameters and the bfloat16
// operands derived from them.
struct MlpBuffers {
    float *p = nullptr;       // [kMlpNParams]
    __bf16 *wb = nullptr;     // w1 [64][16], w2, w3, w2t, w3t [64][64]
    float *w4r = nullptr;     // [64]
    MlpNet net() const
    {
        MlpNet M;
        M.w1 = wb;
        M.w2 = wb + 64 * 16;
        M.w3 = M.w2 + 4096;
        M.w2t = M.w3 + 4096;
        M.w3t = M.w2t + 4096;
        M.b1 = p + kOffB1;
        M.b2 = p + kOffB2;
        M.b3 = p + kOffB3;
        M.w4r = w4r;
        M.b4 = p + kOffB4;
        M.norm = p + kOffNorm;
        return M;
    }
};

// trainable parameter j, rounded to b, to its places among the forward and
// backward passes' operands (biases are read from the master parameters)
__device__ __forceinline__ void put_operand(int j, __bf16 b, __bf16 *wb, float *w4r)
{
    __bf16 *w1 = wb, *w2 = wb + 64 * 16, *w3 = w2 + 4096, *w2t = w3 + 4096, *w3t = w2t + 4096;
    if (j < kOffB1) {
        w1[j / kMlpIn * kMlpK1 + j % kMlpIn] = b;
    } else if (j >= kOffW2 && j < kOffB2) {
        const int i = j - kOffW2;
        w2[i] = b;
        w2t[(i & 63) * 64 + (i >> 6)] = b;
    } else if (j >= kOffW3 && j < kOffB3) {
        const int i = j - kOffW3;
        w3[i] = b;
        w3t[(i & 63) * 64 + (i >> 6)] = b;
    } else if (j >= kOffW4 && j < kOffB4) {
        w4r[j - kOffW4] = from_bf16(b);
    }
}

__global__ void __launch_bounds__(256) mlp_prepare_kernel(const float *p, __bf16 *wb, float *w4r)
{
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j < kMlpNTrain) put_operand(j, to_bf16(p[j]), wb, w4r);
    // layer 1's K is padded from 6 to 16 with zeros
    if (j < 64 * kMlpK1 && j % kMlpK1 >= kMlpIn) wb[j] = to_bf16(0.0f);
}

constexpr int kPrepareGrid = (kMlpNTrain + 255) / 256, kAdamGrid = (kMlpNTrain + 63) / 64;

// Standalone inference: one wave per 64 samples, X[n][6] raw inputs, out = r.
__global__ void __launch_bounds__(64) mlp_forward_kernel(MlpNet M, const float *X, int64_t n, float *out)
{
    __shared__ __attribute__((aligned(16))) __bf16 buf0[64 * kLd0];
    __shared__ __attribute__((aligned(16))) __bf16 buf[64 * kLd];
    const int64_t s = (int64_t)blockIdx.x * 64 + threadIdx.x;
    float x[kMlpIn];
    for (int k = 0; k < kMlpIn; k++) x[k] = s < n ? X[s * kMlpIn + k] : M.norm[k];
    const float y = mlp_wave_forward(M, x, buf0, buf);
    if (s < n) out[s] = y * M.norm[2 * kMlpIn + 1] + M.norm[2 * kMlpIn];
}

// Sample of batch position j: an affine permutation of 0..n-1 (mult coprime
// to n; n, mult, add < 2^31 keep the product in 64 bits).
__device__ __forceinline__ int64_t perm(int64_t j, int64_t n, uint64_t mult, uint64_t add)
{
    return (int64_t)(((uint64_t)j * mult + add) % (uint64_t)n);
}

// One 32 x 32 tile (mt, nt) of a 64 x 64 product, by one wave: A is 64 x K
// row-major in LDS, bw the wave's B operands (rows nt * 32 + r of W), K in
// steps of 16 in the order wave_mm takes them.
template <int kSteps>
__device__ __forceinline__ f32x16 tile_mm(const __bf16 *A, int lda, int mt, const bf16x8 *bw)
{
    const int l = threadIdx.x & 63, r = l & 31, h = l >> 5;
    f32x16 acc;
#pragma unroll
    for (int i = 0; i < 16; i++) acc[i] = 0.0f;
#pragma unroll
    for (int s = 0; s < kSteps; s++) {
        const bf16x8 a = *(const bf16x8 *)(A + (mt * 32 + r) * lda + s * 16 + 8 * h);
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, bw[s], acc, 0, 0, 0);
    }
    return acc;
}

// this wave's B operands of a weight matrix (or LDS tile) W with row stride ldw
template <int kSteps>
__device__ __forceinline__ void tile_b(const __bf16 *W, int ldw, int nt, bf16x8 *bw)
{
    const int l = threadIdx.x & 63, r = l & 31, h = l >> 5;
#pragma unroll
    for (int s = 0; s < kSteps; s++) bw[s] = *(const bf16x8 *)(W + (nt * 32 + r) * ldw + s * 16 + 8 * h);
}

// Forward + backward of one workgroup over batch positions
// [b0 + 64*blockIdx.x, +64) of a batch of nb samples; writes this workgroup's
// partial gradient (kMlpNTrain floats) and partial squared-error sum.
//
// Bound by latency: a batch of 4096 is 64 workgroups on 256 CUs, so what
// counts is the length of one workgroup's chain.  Four waves share the 64
// samples, each with one 32 x 32 tile of every product: a lane then has 16
// GELUs (two erf and an exp each) per layer instead of the 64 of one wave
// doing all four tiles, the weights' operands are loaded once, at the start,
// beside the samples, the activations' transposes are written by the same
// epilogue, and gelu' stays in the registers of the tile that needs it.  Every
// sum keeps its order (products over K in steps of 16, samples in ascending
// order), so gradients and trained weights are bit for bit those of one wave
// per workgroup.  Batch of 4096: 52 -> 18.8 us a launch.
__global__ void __launch_bounds__(256) mlp_grad_kernel(MlpNet M, const float *X, const float *logv, int64_t n,
                                                       int64_t b0, int64_t nb, uint64_t mult, uint64_t add,
                                                       float *partial, float *partial_loss)
{
    __shared__ __attribute__((aligned(16))) __bf16 a0[64 * kLd0];
    __shared__ __attribute__((aligned(16))) __bf16 a1[64 * kLd], a2[64 * kLd], a3[64 * kLd];
    __shared__ __attribute__((aligned(16))) __bf16 a1t[64 * kLd], a2t[64 * kLd];
    __shared__ __attribute__((aligned(16))) __bf16 dz[64 * kLd], dzt[64 * kLd];
    __shared__ float gz[64 * 64];  // dz in float, for the sums over samples
    __shared__ float dyv[64], red[64];
    const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
    const int mt = w >> 1, nt = w & 1;
    const int n0 = acc_col(nt);  // this lane's column of the wave's tile
    // the products' weight operands, in flight while the samples arrive
    bf16x8 w1[1], w2[4], w3[4], w3t[4], w2t[4];
    tile_b<1>(M.w1, kMlpK1, nt, w1);
    tile_b<4>(M.w2, 64, nt, w2);
    tile_b<4>(M.w3, 64, nt, w3);
    tile_b<4>(M.w3t, 64, nt, w3t);
    tile_b<4>(M.w2t, 64, nt, w2t);
    const float bias1 = M.b1[n0], bias2 = M.b2[n0], bias3 = M.b3[n0], w4n = M.w4r[n0];
    const int64_t jb = (int64_t)blockIdx.x * 64 + l;  // position within the batch
    const bool valid = jb < nb;
    float target = 0.0f;
    if (w == 0) {
        const int64_t s = valid ? perm(b0 + jb, n, mult, add) : 0;
        float x[kMlpIn];
        for (int k = 0; k < kMlpIn; k++) x[k] = valid ? X[s * kMlpIn + k] : M.norm[k];
        if (valid) target = logv[s];
        write_input_row(M, x, a0);
    }
    // forward, keeping activations, their transposes and gelu'(z)
    f32x16 acc;
    float g1[16], g2[16], g3[16];
    auto layer = [&](float bias, __bf16 *out, __bf16 *outt, float *g) {
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const int m = acc_row(mt, i);
            const float z = acc[i] + bias;
            const __bf16 v = to_bf16(gelu(z));
            out[m * kLd + n0] = v;
            if (outt) outt[n0 * kLd + m] = v;
            g[i] = gelu_grad(z);
        }
        __syncthreads();
    };
    __syncthreads();
    acc = tile_mm<1>(a0, kLd0, mt, w1);
    layer(bias1, a1, a1t, g1);
    acc = tile_mm<4>(a1, kLd, mt, w2);
    layer(bias2, a2, a2t, g2);
    acc = tile_mm<4>(a2, kLd, mt, w3);
    layer(bias3, a3, nullptr, g3);
    if (w == 0) {
        float y = M.b4[0];
#pragma unroll 16
        for (int i = 0; i < 64; i++) y = y + from_bf16(a3[l * kLd + i]) * M.w4r[i];
        const float t = valid ? (target - M.norm[2 * kMlpIn]) / M.norm[2 * kMlpIn + 1] : y;
        const float r = y - t;
        dyv[l] = valid ? 2.0f * r / (float)nb : 0.0f;
        red[l] = valid ? r * r : 0.0f;
    }
    __syncthreads();
    float *P = partial + (int64_t)blockIdx.x * kMlpNTrain;
    // dz of a layer from v (this lane's tile values): float for the sums,
    // bfloat16 and its transpose for the products
    auto put_dz = [&](const float *v, bool operands) {
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const int m = acc_row(mt, i);
            gz[m * 64 + n0] = v[i];
            if (operands) {
                const __bf16 b = to_bf16(v[i]);
                dz[m * kLd + n0] = b;
                dzt[n0 * kLd + m] = b;
            }
        }
        __syncthreads();
    };
    // lane l's column sum of gz over the samples
    auto column = [&]() {
        float sb = 0.0f;
#pragma unroll 16
        for (int m = 0; m < 64; m++) sb = sb + gz[m * 64 + l];
        return sb;
    };
    auto put_tile = [&](int off) {
#pragma unroll
        for (int i = 0; i < 16; i++) P[off + acc_row(mt, i) * 64 + n0] = acc[i];
    };
    float v[16];
    // dz3 = dy * w4 * gelu'(z3)
#pragma unroll
    for (int i = 0; i < 16; i++) v[i] = dyv[acc_row(mt, i)] * w4n * g3[i];
    put_dz(v, true);
    // dz2 = (dz3 W3) * gelu'(z2), grad W3 = dz3^T a2, and the sums over samples
    acc = tile_mm<4>(dz, kLd, mt, w3t);
#pragma unroll
    for (int i = 0; i < 16; i++) v[i] = acc[i] * g2[i];
    bf16x8 at[4];
    tile_b<4>(a2t, kLd, nt, at);
    acc = tile_mm<4>(dzt, kLd, mt, at);
    put_tile(kOffW3);
    if (w == 0) P[kOffB3 + l] = column();
    if (w == 1) {
        float gw = 0.0f;
#pragma unroll 16
        for (int m = 0; m < 64; m++) gw = gw + dyv[m] * from_bf16(a3[m * kLd + l]);
        P[kOffW4 + l] = gw;
    }
    if (w == 2 && l < 2) {
        const float *src = l == 0 ? red : dyv;
        float s = 0.0f;
#pragma unroll 16
        for (int m = 0; m < 64; m++) s = s + src[m];
        if (l == 0) partial_loss[blockIdx.x] = s;
        else P[kOffB4] = s;
    }
    __syncthreads();
    put_dz(v, true);
    // dz1 = (dz2 W2) * gelu'(z1), grad W2 = dz2^T a1
    acc = tile_mm<4>(dz, kLd, mt, w2t);
#pragma unroll
    for (int i = 0; i < 16; i++) v[i] = acc[i] * g1[i];
    tile_b<4>(a1t, kLd, nt, at);
    acc = tile_mm<4>(dzt, kLd, mt, at);
    put_tile(kOffW2);
    if (w == 0) P[kOffB2 + l] = column();
    __syncthreads();
    put_dz(v, false);
    // grad b1 and grad W1 = dz1^T a0 (K = 6): lane l owns output l, the waves
    // take its seven sums in turn
    for (int k = w; k < kMlpIn + 1; k += 4) {
        if (k == kMlpIn) {
            P[kOffB1 + l] = column();
        } else {
            float gw = 0.0f;
#pragma unroll 16
            for (int m = 0; m < 64; m++) gw = gw + gz[m * 64 + l] * from_bf16(a0[m * kLd0 + k]);
            P[kOffW1 + l * kMlpIn + k] = gw;
        }
    }
}

// Sum of the partial gradients in workgroup order; with grad null an Adam step
// (step number t >= 1) on the master parameters, and each changed parameter's
// bfloat16 operands for the next forward pass (as mlp_prepare_kernel writes
// them), else the sum goes to grad.
//
// One thread per parameter, a wave per workgroup so that the 139 waves spread
// over the CUs; the partials of a parameter are loaded sixteen at a time ahead
// of the additions, which keep workgroup order.  Loaded one by one, with the
// operands written by a launch of their own, 64 workgroups took 19.4 + 4.7 us,
// now 5.1; 64 batches of 4096 with both kernels changed 5.14 -> 1.86 ms.
__global__ void __launch_bounds__(64) mlp_adam_kernel(float *p, float *mom, float *vel, const float *partial, int nwg,
                                                      const float *partial_loss, float *loss_acc, float lr,
                                                      float beta1, float beta2, float eps, int t, float *grad,
                                                      __bf16 *wb, float *w4r)
{
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    constexpr int kAhead = 16;
    auto sum = [&](const float *q, int64_t stride) {
        float s = 0.0f;
        int w = 0;
        for (; w + kAhead <= nwg; w += kAhead) {
            float x[kAhead];
#pragma unroll
            for (int i = 0; i < kAhead; i++) x[i] = q[(int64_t)(w + i) * stride];
#pragma unroll
            for (int i = 0; i < kAhead; i++) s = s + x[i];
        }
        for (; w < nwg; w++) s = s + q[(int64_t)w * stride];
        return s;
    };
    // the loss by a thread that has no parameter
    if (j == kMlpNTrain && loss_acc) loss_acc[0] = loss_acc[0] + sum(partial_loss, 1);
    if (j >= kMlpNTrain) return;
    const float g = sum(partial + j, kMlpNTrain);
    if (grad) {
        grad[j] = g;
        return;
    }
    const float m = beta1 * mom[j] + (1.0f - beta1) * g;
    const float v = beta2 * vel[j] + (1.0f - beta2) * g * g;
    mom[j] = m;
    vel[j] = v;
    const float mh = m / (1.0f - powf(beta1, (float)t));
    const float vh = v / (1.0f - powf(beta2, (float)t));
    const float x = p[j] - lr * mh / (sqrtf(vh) + eps);
    p[j] = x;
    put_operand(j, to_bf16(x), wb, w4r);
}
static_assert(kMlpNTrain % 64 != 0, "the last workgroup of mlp_adam_kernel has a thread for the loss");

hipError_t launch_mlp_prepare(const float *p, __bf16 *wb, float *w4r, hipStream_t s)
{
    mlp_prepare_kernel<<<kPrepareGrid, 256, 0, s>>>(p, wb, w4r);
    return hipGetLastError();
}

}  // namespace eqd

using namespace eqd;

namespace {

struct DevMem {
    std::vector<void *> ptrs;
    ~DevMem()
    {
        for (void *q : ptrs) (void)hipFree(q);
    }
    template <typename T>
    T *alloc(size_t count)
    {
        void *q = nullptr;
        if (hipMalloc(&q, count * sizeof(T) + 16) != hipSuccess) return nullptr;
        ptrs.push_back(q);
        return (T *)q;
    }
};

int prepare(MlpBuffers &B, hipStream_t s)
{
    mlp_prepare_kernel<<<kPrepareGrid, 256, 0, s>>>(B.p, B.wb, B.w4r);
    return hipGetLastError() == hipSuccess ? EQD_OK : EQD_EHIP;
}

bool alloc_net(DevMem &D, MlpBuffers &B)
{
    B.p = D.alloc<float>(kMlpNParams);
    B.wb = D.alloc<__bf16>(64 * 16 + 4 * 4096);
    B.w4r = D.alloc<float>(64);
    return B.p && B.wb && B.w4r;
}

// ---------------- scratch of the allocation-free entry point
// The network's prepared operands (bf16 weights w1, w2, w3 and their
// transposes, and w4 as float) of eqd_mlp_forward_noalloc live in this
// file-scope device array: kNoAllocScratch bytes per device, held until the
// process ends.  Host code never uses its name as an address: the device
// address comes from hipGetSymbolAddress, looked up once per device.
constexpr size_t kWbCount = 64 * 16 + 4 * 4096;                       // bf16 values
constexpr size_t kW4rOffset = (kWbCount * sizeof(__bf16) + 255) / 256 * 256;  // bytes
constexpr size_t kNoAllocScratch = kW4rOffset + 64 * sizeof(float);
static_assert(kNoAllocScratch == EQD_MLP_NOALLOC_SCRATCH_BYTES, "scratch size and header disagree");
static __device__ __align__(256) unsigned char scratch[kNoAllocScratch];

constexpr int kMaxDevices = 64;
void *g_scratch_ptr[kMaxDevices] = {};
std::mutex g_scratch_mu;

// device address of this device's scratch array (device current), or null
void *scratch_on(int device)
{
    if (device < 0 || device >= kMaxDevices) return nullptr;
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch_ptr[device]) {
        void *ptr = nullptr;
        if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)) != hipSuccess) return nullptr;
        g_scratch_ptr[device] = ptr;
    }
    return g_scratch_ptr[device];
}

int check_params(const float *params)
{
    const float *nrm = params + kOffNorm;
    for (int k = 0; k < kMlpNParams; k++)
        if (!(params[k] == params[k])) return EQD_EINVAL;
    if (nrm[2 * kMlpIn + 1] == 0.0f) return EQD_EINVAL;
    return EQD_OK;
}

}  // namespace

extern "C" {

int eqd_mlp_forward(const float *params, const float *X, int64_t n, float *r_out, int32_t device)
{
    if (!params || (n > 0 && (!X || !r_out)) || n < 0) return EQD_EINVAL;
    if (check_params(params) != EQD_OK) return EQD_EINVAL;
    if (n == 0) return EQD_OK;
    if (hipSetDevice(device) != hipSuccess) return EQD_EHIP;
    DevMem D;
    MlpBuffers B;
    if (!alloc_net(D, B)) return EQD_EOOM;
    float *dX = D.alloc<float>((size_t)n * kMlpIn), *dy = D.alloc<float>((size_t)n);
    if (!dX || !dy) return EQD_EOOM;
    if (hipMemcpy(B.p, params, kMlpNParams * sizeof(float), hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(dX, X, (size_t)n * kMlpIn * sizeof(float), hipMemcpyHostToDevice) != hipSuccess)
        return EQD_EHIP;
    if (prepare(B, 0)) return EQD_EHIP;
    mlp_forward_kernel<<<(unsigned)((n + 63) / 64), 64>>>(B.net(), dX, n, dy);
    if (hipGetLastError() != hipSuccess) return EQD_EHIP;
    if (hipMemcpy(r_out, dy, (size_t)n * sizeof(float), hipMemcpyDeviceToHost) != hipSuccess) return EQD_EHIP;
    return EQD_OK;
}

int eqd_mlp_forward_noalloc(const float *params, const float *X, int64_t n, float *r_out, int32_t device,
                            void *stream)
{
    if (!params || (n > 0 && (!X || !r_out)) || n < 0) return EQD_EINVAL;
    if (n > (int64_t)0xFFFFFFFF * 64) return EQD_EINVAL;  // one launch covers at most 2^32 - 1 waves
    if (n == 0) return EQD_OK;
    if (hipSetDevice(device) != hipSuccess) return EQD_EHIP;
    unsigned char *sc = (unsigned char *)scratch_on(device);
    if (!sc) return EQD_EHIP;
    MlpBuffers B;
    B.p = const_cast<float *>(params);
    B.wb = (__bf16 *)sc;
    B.w4r = (float *)(sc + kW4rOffset);
    const hipStream_t st = (hipStream_t)stream;
    mlp_prepare_kernel<<<kPrepareGrid, 256, 0, st>>>(B.p, B.wb, B.w4r);
    mlp_forward_kernel<<<(unsigned)((n + 63) / 64), 64, 0, st>>>(B.net(), X, n, r_out);
    return hipGetLastError() == hipSuccess ? EQD_OK : EQD_EHIP;
}

int eqd_mlp_grad(const float *params, const float *X, const float *logv, int64_t n, float *grad_out,
                 float *loss_out, int32_t device)
{
    if (!params || !X || !logv || !grad_out || n <= 0 || n > (int64_t)1 << 24) return EQD_EINVAL;
    if (check_params(params) != EQD_OK) return EQD_EINVAL;
    if (hipSetDevice(device) != hipSuccess) return EQD_EHIP;
    DevMem D;
    MlpBuffers B;
    if (!alloc_net(D, B)) return EQD_EOOM;
    const int nwg = (int)((n + 63) / 64);
    float *dX = D.alloc<float>((size_t)n * kMlpIn), *dl = D.alloc<float>((size_t)n);
    float *part = D.alloc<float>((size_t)nwg * kMlpNTrain), *pl = D.alloc<float>(nwg), *la = D.alloc<float>(1);
    float *g = D.alloc<float>(kMlpNTrain);
    if (!dX || !dl || !part || !pl || !la || !g) return EQD_EOOM;
    if (hipMemcpy(B.p, params, kMlpNParams * sizeof(float), hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(dX, X, (size_t)n * kMlpIn * sizeof(float), hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(dl, logv, (size_t)n * sizeof(float), hipMemcpyHostToDevice) != hipSuccess ||
        hipMemset(la, 0, sizeof(float)) != hipSuccess)
        return EQD_EHIP;
    if (prepare(B, 0)) return EQD_EHIP;
    mlp_grad_kernel<<<nwg, 256>>>(B.net(), dX, dl, n, 0, n, 1, 0, part, pl);
    mlp_adam_kernel<<<kAdamGrid, 64>>>(B.p, nullptr, nullptr, part, nwg, pl, la, 0.0f, 0.0f, 0.0f, 0.0f, 1, g, B.wb,
                                       B.w4r);
    if (hipGetLastError() != hipSuccess) return EQD_EHIP;
    float ls = 0.0f;
    if (hipMemcpy(grad_out, g, kMlpNTrain * sizeof(float), hipMemcpyDeviceToHost) != hipSuccess ||
        hipMemcpy(&ls, la, sizeof(float), hipMemcpyDeviceToHost) != hipSuccess)
        return EQD_EHIP;
    if (loss_out) *loss_out = ls / (float)n;
    return EQD_OK;
}

static uint64_t gcd64(uint64_t a, uint64_t b)
{
    while (b) {
        const uint64_t t = a % b;
        a = b;
        b = t;
    }
    return a;
}

static uint64_t splitmix(uint64_t &s)
{
    uint64_t z = (s += 0x9E3779B97F4A7C15ull);
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

int eqd_mlp_train(const float *X, const float *logv, int64_t n, const eqd_mlp_train_opts *o, float *params,
                  float *epoch_loss)
{
    if (!X || !logv || !o || !params || n <= 0 || n >= ((int64_t)1 << 31) || o->epochs <= 0 || o->batch <= 0 ||
        o->batch > (1 << 20) || !(o->lr > 0.0f))
        return EQD_EINVAL;
    if (check_params(params) != EQD_OK) return EQD_EINVAL;
    if (hipSetDevice(o->device) != hipSuccess) return EQD_EHIP;
    DevMem D;
    MlpBuffers B;
    if (!alloc_net(D, B)) return EQD_EOOM;
    const int64_t bs = o->batch < n ? o->batch : n;
    const int nwg = (int)((bs + 63) / 64);
    float *dX = D.alloc<float>((size_t)n * kMlpIn), *dl = D.alloc<float>((size_t)n);
    float *part = D.alloc<float>((size_t)nwg * kMlpNTrain), *pl = D.alloc<float>(nwg);
    float *mom = D.alloc<float>(kMlpNTrain), *vel = D.alloc<float>(kMlpNTrain), *la = D.alloc<float>(o->epochs);
    if (!dX || !dl || !part || !pl || !mom || !vel || !la) return EQD_EOOM;
    if (hipMemcpy(B.p, params, kMlpNParams * sizeof(float), hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(dX, X, (size_t)n * kMlpIn * sizeof(float), hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(dl, logv, (size_t)n * sizeof(float), hipMemcpyHostToDevice) != hipSuccess ||
        hipMemset(mom, 0, kMlpNTrain * sizeof(float)) != hipSuccess ||
        hipMemset(vel, 0, kMlpNTrain * sizeof(float)) != hipSuccess ||
        hipMemset(la, 0, o->epochs * sizeof(float)) != hipSuccess)
        return EQD_EHIP;
    if (prepare(B, 0)) return EQD_EHIP;
    uint64_t rs = o->seed;
    int t = 0;
    const int64_t nbatch = n / bs;  // full batches per epoch
    for (int e = 0; e < o->epochs; e++) {
        uint64_t mult;
        do {
            mult = splitmix(rs) % (uint64_t)n;
        } while (mult == 0 || gcd64(mult, (uint64_t)n) != 1);
        const uint64_t add = splitmix(rs) % (uint64_t)n;
        for (int64_t b = 0; b < nbatch; b++) {
            t++;
            mlp_grad_kernel<<<nwg, 256>>>(B.net(), dX, dl, n, b * bs, bs, mult, add, part, pl);
            mlp_adam_kernel<<<kAdamGrid, 64>>>(B.p, mom, vel, part, nwg, pl, la + e, o->lr, o->beta1, o->beta2, o->eps,
                                               t, nullptr, B.wb, B.w4r);
        }
        if (hipGetLastError() != hipSuccess) return EQD_EHIP;
    }
    if (hipDeviceSynchronize() != hipSuccess) return EQD_EHIP;
    if (hipMemcpy(params, B.p, kMlpNTrain * sizeof(float), hipMemcpyDeviceToHost) != hipSuccess) return EQD_EHIP;
    if (epoch_loss) {
        std::vector<float> h(o->epochs);
        if (hipMemcpy(h.data(), la, o->epochs * sizeof(float), hipMemcpyDeviceToHost) != hipSuccess) return EQD_EHIP;
        for (int e = 0; e < o->epochs; e++) epoch_loss[e] = h[e] / (float)(nbatch * bs);
    }
    return EQD_OK;
}

}  // extern "C"
