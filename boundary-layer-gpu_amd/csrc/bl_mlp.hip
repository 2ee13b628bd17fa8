// Learned subgrid closure: training on the device (no counterpart in the
// reference solver, which only has the dynamic Smagorinsky model).
//
// Network: 10 -> 64 -> 64 -> 64 -> 1 with SiLU, predicting the dimensionless
// eddy viscosity c = nu_t / (Delta^2 |S|) from the normalised velocity-
// gradient tensor and the wall distance.  FP32 master parameters, Adam; one
// kernel does the forward and backward passes and the weight gradients of a
// batch in FP32 on the matrix cores, with per-block partial gradients that the
// update kernel adds in a fixed order (deterministic).  A BF16 copy of the
// weights feeds the MFMA inference kernel (bl_closure.hip).
//
// Dataset rows (kRow floats): 10 features, target c, weight, Delta^2 |S|,
// then S_ij and tau_ij (6 + 6, the a-priori checks).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <string>
#include <type_traits>
#include <vector>

#include "../../include/blgpu.h"
#include "bl_mlp.hpp"

namespace blgpu {

namespace {

constexpr int kH = kMlpHidden, kIn = kMlpIn;
// parameter offsets (W1[64][10], b1, W2[64][64], b2, W3[64][64], b3, W4[64], b4)
constexpr int oW1 = 0, ob1 = oW1 + kH * kIn, oW2 = ob1 + kH, ob2 = oW2 + kH * kH, oW3 = ob2 + kH,
              ob3 = oW3 + kH * kH, oW4 = ob3 + kH, ob4 = oW4 + kH;
static_assert(ob4 + 1 == kMlpParams, "parameter layout");

__device__ __forceinline__ unsigned long long mix64(unsigned long long z) {
    z += 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

// sum and count of the positive row weights, per block (fixed order)
__global__ __launch_bounds__(256) void k_wsum(const float *__restrict__ rows, long long n, double *__restrict__ part) {
    __shared__ double sh[2][4];
    double s = 0.0, c = 0.0;
    for (long long r = (long long)blockIdx.x * 256 + threadIdx.x; r < n; r += (long long)gridDim.x * 256) {
        const float w = rows[r * kMlpRow + kIn + 1];
        if (w > 0.f) {
            s += w;
            c += 1.0;
        }
    }
    for (int o = 32; o > 0; o >>= 1) {
        s += __shfl_down(s, o);
        c += __shfl_down(c, o);
    }
    if ((threadIdx.x & 63) == 0) {
        sh[0][threadIdx.x >> 6] = s;
        sh[1][threadIdx.x >> 6] = c;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        part[2 * blockIdx.x] = (sh[0][0] + sh[0][1]) + (sh[0][2] + sh[0][3]);
        part[2 * blockIdx.x + 1] = (sh[1][0] + sh[1][1]) + (sh[1][2] + sh[1][3]);
    }
}

// ------------------------------------------------------------------------
// Forward, backward and weight gradients of a batch, loss = (1/B) sum w (y-t)^2.
// A block of eight waves takes tiles of kTs = 128 samples, 16 per wave, and
// keeps everything of a tile on the chip.  Every product runs on
// v_mfma_f32_16x16x4_f32 (lane l holds A[l%16][l/16], B[l/16][l%16] and
// D[4 (l/16) + r][l%16], r < 4):
//   layers   D = W h, columns = the wave's samples.  Accumulator register
//            (t, r) of a lane is feature 16 t + 4 (l/16) + r of sample l%16;
//            taking the features in that order along K, it is the next layer's
//            B operand as it stands, and A is four consecutive weights of a
//            row, so activations never leave the registers
//   backward the same with A = W^T, read from the same copy of W
//   dW       = dz h^T over the 128 samples: dz and h pass through LDS
//            ([feature][sample]), each wave owns two 16 x 16 tiles of dW2 and
//            dW3 and half of one of dW1
// Bias and output-layer gradients are sums over lanes, kept per lane until
// the end.  The row strides (68, 132) put the 16 rows of an operand read on
// different banks.  Bound: 3.5 GFLOP at batch 65536 are 22 us of FP32 matrix
// time, plus the SiLU evaluations between the products; measured 65 us, and
// 11 us for the update.  The form before it (one sample per lane on the vector
// units, activations and deltas through memory, seven launches) took 0.99 ms a
// step.
// ------------------------------------------------------------------------
typedef float f32x4 __attribute__((ext_vector_type(4)));
constexpr int kTs = 128, kTWaves = 8;          // samples and waves per block
constexpr int kWs = 68, kW1s = 13, kSs = 132;  // LDS row strides: W2 and W3, W1, sample rows

__device__ __forceinline__ f32x4 mfma32(float a, float b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// where the batch comes from: rows drawn by the counter hash of (seed, step,
// slot) from the dataset (rows set), or the arrays X[f][b], t, w
struct BatchSrc {
    const float *rows;
    long long n;
    unsigned long long seed;
    long long step;
    float wscale;
    const float *X, *t, *w;
};

struct TrainLds {
    float w2[kH * kWs], w3[kH * kWs], w1[kH * kW1s];
    float b1[kH], b2[kH], b3[kH], w4[kH];
};
struct GradLds {
    float x[16 * kSs], h1[kH * kSs], h2[kH * kSs], d[kH * kSs];
};

// GRAD: write the block's partial gradients (part[block][kMlpParams]) and loss
// sum; otherwise only y[b]
template <bool GRAD>
__global__ __launch_bounds__(64 * kTWaves) void k_batch(const float *__restrict__ theta, BatchSrc src, int B,
                                                        float *__restrict__ y, float *__restrict__ part,
                                                        double *__restrict__ loss) {
    __shared__ TrainLds L;
    __shared__ typename std::conditional<GRAD, GradLds, int>::type G_;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, l16 = lane & 15, q4 = lane >> 4;
    for (int q = tid; q < kH * kH; q += 64 * kTWaves) {
        L.w2[(q >> 6) * kWs + (q & 63)] = theta[oW2 + q];
        L.w3[(q >> 6) * kWs + (q & 63)] = theta[oW3 + q];
    }
    for (int q = tid; q < kH * 12; q += 64 * kTWaves) {
        const int o = q / 12, i = q - o * 12;
        L.w1[o * kW1s + i] = i < kIn ? theta[oW1 + o * kIn + i] : 0.f;
    }
    if (tid < kH) {
        L.b1[tid] = theta[ob1 + tid];
        L.b2[tid] = theta[ob2 + tid];
        L.b3[tid] = theta[ob3 + tid];
        L.w4[tid] = theta[oW4 + tid];
    }
    if constexpr (GRAD)
        for (int q = tid; q < 4 * kSs; q += 64 * kTWaves) G_.x[12 * kSs + q] = 0.f;  // features 12..15 do not exist
    const float b4 = theta[ob4];
    __syncthreads();
    // per lane: bias and output-layer gradients of its features and samples
    f32x4 g4[4], gb1[4], gb2[4], gb3[4], gw2[2], gw3[2], gw1;
    float gb4 = 0.f;
    double sq = 0.0;
#pragma unroll
    for (int t = 0; t < 4; ++t) g4[t] = gb1[t] = gb2[t] = gb3[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    gw2[0] = gw2[1] = gw3[0] = gw3[1] = gw1 = f32x4{0.f, 0.f, 0.f, 0.f};
    // dW tiles of this wave: rows 16 rt.., columns 16 (ct + c)..; dW1: rows
    // 16 (wave % 4).. over half of the samples
    const int rt = wave >> 1, ct = 2 * (wave & 1);
    auto layer = [&](const float *W, const float *bias, const f32x4 h[4], f32x4 z[4]) {
#pragma unroll
        for (int o = 0; o < 4; ++o) z[o] = *reinterpret_cast<const f32x4 *>(bias + 16 * o + 4 * q4);
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int o = 0; o < 4; ++o) {
                const f32x4 w = *reinterpret_cast<const f32x4 *>(W + (16 * o + l16) * kWs + 16 * t + 4 * q4);
#pragma unroll
                for (int r = 0; r < 4; ++r) z[o] = mfma32(w[r], h[t][r], z[o]);
            }
    };
    // z -> SiLU(z) in place, and its derivative
    auto act = [&](f32x4 z[4], f32x4 ds[4]) {
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float v = z[t][r], s = 1.f / (1.f + expf(-v));
                if constexpr (GRAD) ds[t][r] = s * (1.f + v * (1.f - s));
                z[t][r] = v / (1.f + expf(-v));
            }
    };
    const int ntile = (B + kTs - 1) / kTs;
    for (int tile = blockIdx.x; tile < ntile; tile += gridDim.x) {
        const int col = 16 * wave + l16, b = tile * kTs + col;
        const bool live = b < B;
        const int bc = live ? b : B - 1;
        float x[3], tgt, w;
        if (src.rows) {
            const unsigned long long h =
                mix64(src.seed ^ mix64((unsigned long long)src.step * 0x100000001B3ull + (unsigned long long)bc));
            const float *row = src.rows + (long long)(h % (unsigned long long)src.n) * kMlpRow;
#pragma unroll
            for (int ks = 0; ks < 3; ++ks) x[ks] = 4 * ks + q4 < kIn ? row[4 * ks + q4] : 0.f;
            tgt = row[kIn];
            w = row[kIn + 1] * src.wscale;
        } else {
#pragma unroll
            for (int ks = 0; ks < 3; ++ks) x[ks] = 4 * ks + q4 < kIn ? src.X[(long long)(4 * ks + q4) * B + bc] : 0.f;
            tgt = GRAD ? src.t[bc] : 0.f;
            w = GRAD ? src.w[bc] : 0.f;
        }
        if (!live) w = 0.f;
        f32x4 h[4], z[4], ds1[4], ds2[4], ds3[4];
#pragma unroll
        for (int o = 0; o < 4; ++o) {
            z[o] = *reinterpret_cast<const f32x4 *>(L.b1 + 16 * o + 4 * q4);
#pragma unroll
            for (int ks = 0; ks < 3; ++ks) z[o] = mfma32(L.w1[(16 * o + l16) * kW1s + 4 * ks + q4], x[ks], z[o]);
        }
        act(z, ds1);
        auto put = [&](float *dst, const f32x4 v[4]) {
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int r = 0; r < 4; ++r) dst[(16 * t + 4 * q4 + r) * kSs + col] = v[t][r];
        };
        if constexpr (GRAD) {
#pragma unroll
            for (int ks = 0; ks < 3; ++ks) G_.x[(4 * ks + q4) * kSs + col] = x[ks];
            put(G_.h1, z);
        }
        layer(L.w2, L.b2, z, h);
        act(h, ds2);
        if constexpr (GRAD) put(G_.h2, h);
        layer(L.w3, L.b3, h, z);
        act(z, ds3);
        float yv = 0.f;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const f32x4 w4 = *reinterpret_cast<const f32x4 *>(L.w4 + 16 * t + 4 * q4);
#pragma unroll
            for (int r = 0; r < 4; ++r) yv += w4[r] * z[t][r];
        }
        yv += __shfl_xor(yv, 16);
        yv += __shfl_xor(yv, 32);
        yv += b4;
        if constexpr (!GRAD) {
            if (live && q4 == 0) y[b] = yv;
        } else {
            const float e = yv - tgt;
            const float dy = 2.f * w * e / (float)B;
            if (q4 == 0) {
                sq += (double)(w * e * e);
                gb4 += dy;
            }
            f32x4 dz[4];
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const f32x4 w4 = *reinterpret_cast<const f32x4 *>(L.w4 + 16 * t + 4 * q4);
                g4[t] += dy * z[t];
                dz[t] = dy * w4 * ds3[t];
                gb3[t] += dz[t];
            }
            // dz of a layer from that of the layer above: W^T dz, times the derivative
            auto back = [&](const float *W, const f32x4 ds[4]) {
                f32x4 a[4];
#pragma unroll
                for (int o = 0; o < 4; ++o) a[o] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int t = 0; t < 4; ++t)
#pragma unroll
                    for (int r = 0; r < 4; ++r)
#pragma unroll
                        for (int o = 0; o < 4; ++o)
                            a[o] = mfma32(W[(16 * t + 4 * q4 + r) * kWs + 16 * o + l16], dz[t][r], a[o]);
#pragma unroll
                for (int o = 0; o < 4; ++o) dz[o] = a[o] * ds[o];
            };
            // dW tiles of this wave over the block's samples
            auto wgrad = [&](const float *hs, f32x4 g[2]) {
#pragma unroll
                for (int k = 0; k < kTs / 16; ++k) {
                    const f32x4 a = *reinterpret_cast<const f32x4 *>(G_.d + (16 * rt + l16) * kSs + 16 * k + 4 * q4);
#pragma unroll
                    for (int c = 0; c < 2; ++c) {
                        const f32x4 v =
                            *reinterpret_cast<const f32x4 *>(hs + (16 * (ct + c) + l16) * kSs + 16 * k + 4 * q4);
#pragma unroll
                        for (int r = 0; r < 4; ++r) g[c] = mfma32(a[r], v[r], g[c]);
                    }
                }
            };
            put(G_.d, dz);
            __syncthreads();
            wgrad(G_.h2, gw3);
            back(L.w3, ds2);
#pragma unroll
            for (int t = 0; t < 4; ++t) gb2[t] += dz[t];
            __syncthreads();  // the deltas of layer 3 are read
            put(G_.d, dz);
            __syncthreads();
            wgrad(G_.h1, gw2);
            back(L.w2, ds1);
#pragma unroll
            for (int t = 0; t < 4; ++t) gb1[t] += dz[t];
            __syncthreads();
            put(G_.d, dz);
            __syncthreads();
            {
                const int k0 = (wave >> 2) * (kTs / 32);
#pragma unroll
                for (int k = k0; k < k0 + kTs / 32; ++k) {
                    const f32x4 a =
                        *reinterpret_cast<const f32x4 *>(G_.d + (16 * (wave & 3) + l16) * kSs + 16 * k + 4 * q4);
                    const f32x4 v = *reinterpret_cast<const f32x4 *>(G_.x + l16 * kSs + 16 * k + 4 * q4);
#pragma unroll
                    for (int r = 0; r < 4; ++r) gw1 = mfma32(a[r], v[r], gw1);
                }
            }
            __syncthreads();  // before the next tile's x, h and deltas
        }
    }
    if constexpr (GRAD) {
        float *P = part + (long long)blockIdx.x * kMlpParams;
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int e = (16 * rt + 4 * q4 + r) * kH + 16 * (ct + c) + l16;
                P[oW2 + e] = gw2[c][r];
                P[oW3 + e] = gw3[c][r];
            }
        // sums over the 16 lanes of a feature, then over the waves
        auto sum16 = [&](float v) {
#pragma unroll
            for (int o = 1; o < 16; o <<= 1) v += __shfl_xor(v, o);
            return v;
        };
        float *sr = G_.h1;                                 // [wave][4][kH], then gb4
        float *s1 = G_.h2;                                 // the second half of dW1
        double *sd = reinterpret_cast<double *>(G_.d);     // [wave]
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int f = 16 * t + 4 * q4 + r;
                const float a = sum16(gb1[t][r]), c = sum16(gb2[t][r]), e = sum16(gb3[t][r]), g = sum16(g4[t][r]);
                if (l16 == 0) {
                    sr[(wave * 4 + 0) * kH + f] = a;
                    sr[(wave * 4 + 1) * kH + f] = c;
                    sr[(wave * 4 + 2) * kH + f] = e;
                    sr[(wave * 4 + 3) * kH + f] = g;
                }
            }
        gb4 = sum16(gb4);  // lanes 0..15 hold the samples
#pragma unroll
        for (int o = 1; o < 16; o <<= 1) sq += __shfl_xor(sq, o);
        if (lane == 0) {
            sr[kTWaves * 4 * kH + wave] = gb4;
            sd[wave] = sq;
        }
        if (wave >= 4)
#pragma unroll
            for (int r = 0; r < 4; ++r) s1[((wave - 4) * 4 + r) * 64 + lane] = gw1[r];
        __syncthreads();
        if (wave < 4 && l16 < kIn)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                P[oW1 + (16 * wave + 4 * q4 + r) * kIn + l16] = gw1[r] + s1[(wave * 4 + r) * 64 + lane];
        if (tid < 4 * kH) {
            const int c = tid >> 6, f = tid & 63;
            float a = 0.f;
#pragma unroll
            for (int v = 0; v < kTWaves; ++v) a += sr[(v * 4 + c) * kH + f];
            P[(c == 0 ? ob1 : (c == 1 ? ob2 : (c == 2 ? ob3 : oW4))) + f] = a;
        }
        if (tid == 4 * kH) {
            float a = 0.f;
            double l = 0.0;
            for (int v = 0; v < kTWaves; ++v) {
                a += sr[kTWaves * 4 * kH + v];
                l += sd[v];
            }
            P[ob4] = a;
            loss[blockIdx.x] = l;
        }
    }
}

// g = the sum of the nb block partials, added in double in a fixed order:
// eight groups of blocks, then the groups.  32 parameters per block, so that
// the rows are read as 128-byte segments; one more block adds the loss sums
// into lossf[0].  adam: also the update.
__global__ __launch_bounds__(256) void k_update(const float *__restrict__ part, const double *__restrict__ loss, int nb,
                                                float *__restrict__ g, float *__restrict__ theta,
                                                float *__restrict__ m, float *__restrict__ v, int adam, float lr,
                                                float c1, float c2, float *__restrict__ lossf) {
    __shared__ double sh[8][32];
    if (blockIdx.x == gridDim.x - 1) {
        double *t = &sh[0][0], l = 0.0;
        for (int q = threadIdx.x; q < nb; q += 256) l += loss[q];
        t[threadIdx.x] = l;
        __syncthreads();
        for (int st = 128; st > 0; st >>= 1) {
            if ((int)threadIdx.x < st) t[threadIdx.x] += t[threadIdx.x + st];
            __syncthreads();
        }
        if (threadIdx.x == 0) lossf[0] = (float)t[0];
        return;
    }
    const int f = threadIdx.x & 31, s = threadIdx.x >> 5, p = blockIdx.x * 32 + f;
    double a = 0.0;
    if (p < kMlpParams)
        for (int q = s; q < nb; q += 8) a += (double)part[(long long)q * kMlpParams + p];
    sh[s][f] = a;
    __syncthreads();
    if (s == 0 && p < kMlpParams) {
        double t = 0.0;
#pragma unroll
        for (int q = 0; q < 8; ++q) t += sh[q][f];
        const float gp = (float)t;
        g[p] = gp;
        if (adam) {
            const float mp = 0.9f * m[p] + 0.1f * gp;
            const float vp = 0.999f * v[p] + 0.001f * gp * gp;
            m[p] = mp;
            v[p] = vp;
            theta[p] -= lr * (mp / c1) / (sqrtf(vp / c2) + 1e-8f);
        }
    }
}

void check() {
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        last_error() = std::string("kernel launch: ") + hipGetErrorString(e);
        throw DeviceError();
    }
}

template <class T>
T *alloc(size_t n) {
    void *p = nullptr;
    if (hipMalloc(&p, std::max<size_t>(n, 1) * sizeof(T)) != hipSuccess) {
        last_error() = "out of device memory (learned closure, " + std::to_string(n * sizeof(T)) + " bytes)";
        throw std::bad_alloc();
    }
    return static_cast<T *>(p);
}

}  // namespace

void mlp_init(Mlp &m, long long capacity, int batch_max) {
    m.cap = capacity;
    m.n = 0;
    m.bmax = batch_max;
    BL_HIP(hipStreamCreate(&m.stream));
    m.rows = alloc<float>((size_t)capacity * kMlpRow);
    m.theta = alloc<float>(kMlpParams);
    m.adam_m = alloc<float>(kMlpParams);
    m.adam_v = alloc<float>(kMlpParams);
    m.g = alloc<float>(kMlpParams);
    int dev = 0, ncu = 0;
    BL_HIP(hipGetDevice(&dev));
    BL_HIP(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev));
    // one resident block per compute unit (its LDS), each looping over tiles
    m.nblk = std::max(1, std::min(ncu, (batch_max + kTs - 1) / kTs));
    m.part = alloc<float>((size_t)m.nblk * kMlpParams);
    m.loss = alloc<double>(m.nblk);
    m.Xb = alloc<float>((size_t)kIn * batch_max);
    m.tb = alloc<float>(batch_max);
    m.wb = alloc<float>(batch_max);
    m.y = alloc<float>(batch_max);
    m.scal = alloc<float>(16);
    BL_HIP(hipMemsetAsync(m.theta, 0, kMlpParams * sizeof(float), m.stream));
    BL_HIP(hipMemsetAsync(m.adam_m, 0, kMlpParams * sizeof(float), m.stream));
    BL_HIP(hipMemsetAsync(m.adam_v, 0, kMlpParams * sizeof(float), m.stream));
    m.step = 0;
}

void mlp_free(Mlp &m) {
    for (void *p : {(void *)m.rows, (void *)m.theta, (void *)m.adam_m, (void *)m.adam_v, (void *)m.g, (void *)m.part,
                    (void *)m.loss, (void *)m.Xb, (void *)m.tb, (void *)m.wb, (void *)m.y, (void *)m.scal,
                    (void *)m.hist})
        if (p) (void)hipFree(p);
    if (m.stream) {
        (void)hipStreamSynchronize(m.stream);
        (void)hipStreamDestroy(m.stream);
    }
}

namespace {
void launch_grad(Mlp &m, const BatchSrc &src, int B, bool adam, float lr, float c1, float c2, float *loss) {
    const int nb = std::min(m.nblk, (B + kTs - 1) / kTs);
    hipLaunchKernelGGL(k_batch<true>, dim3(nb), dim3(64 * kTWaves), 0, m.stream, m.theta, src, B, (float *)nullptr,
                       m.part, m.loss);
    check();
    hipLaunchKernelGGL(k_update, dim3((kMlpParams + 31) / 32 + 1), dim3(256), 0, m.stream, m.part, m.loss, nb, m.g, m.theta,
                       m.adam_m, m.adam_v, adam ? 1 : 0, lr, c1, c2, loss);
    check();
}
}  // namespace

// the batch in Xb/tb/wb: forward into y, or the gradient into g and the batch
// loss sum into scal[0]
void mlp_fwd_bwd(Mlp &m, int B, bool backward) {
    BatchSrc src{};
    src.X = m.Xb;
    src.t = m.tb;
    src.w = m.wb;
    if (backward) {
        launch_grad(m, src, B, false, 0.f, 1.f, 1.f, m.scal);
        return;
    }
    hipLaunchKernelGGL(k_batch<false>, dim3((B + kTs - 1) / kTs), dim3(64 * kTWaves), 0, m.stream, m.theta, src, B, m.y,
                       (float *)nullptr, (double *)nullptr);
    check();
}

void mlp_load_batch(Mlp &m, const float *x, const float *t, int n) {
    // host rows x[n][10] -> feature-major Xb; targets; unit weights
    std::vector<float> xb((size_t)kIn * n), w((size_t)n, 1.f), tt((size_t)n, 0.f);
    for (int b = 0; b < n; ++b)
        for (int f = 0; f < kIn; ++f) xb[(size_t)f * n + b] = x[(size_t)b * kIn + f];
    if (t) std::memcpy(tt.data(), t, sizeof(float) * n);
    BL_HIP(hipMemcpyAsync(m.Xb, xb.data(), xb.size() * sizeof(float), hipMemcpyHostToDevice, m.stream));
    BL_HIP(hipMemcpyAsync(m.tb, tt.data(), tt.size() * sizeof(float), hipMemcpyHostToDevice, m.stream));
    BL_HIP(hipMemcpyAsync(m.wb, w.data(), w.size() * sizeof(float), hipMemcpyHostToDevice, m.stream));
    BL_HIP(hipStreamSynchronize(m.stream));
}

void mlp_train(Mlp &m, int steps, int B, float lr, unsigned long long seed, float *loss_hist) {
    if (m.n < 1) {
        last_error() = "bl_mlp_train: the dataset is empty";
        throw ArgError();
    }
    if (B < 1 || B > m.bmax) {
        last_error() = "bl_mlp_train: batch must be in [1, batch_max]";
        throw ArgError();
    }
    const dim3 blk(256);
    // weights rescaled to mean 1 over the weighted rows of the dataset (the
    // partial sums go through the gradient buffer, which each step rewrites)
    constexpr int kWBlk = 128;
    static_assert(2 * kWBlk * sizeof(double) <= kMlpParams * sizeof(float), "partials fit in g");
    double *wpart = reinterpret_cast<double *>(m.g);
    hipLaunchKernelGGL(k_wsum, dim3(kWBlk), blk, 0, m.stream, m.rows, m.n, wpart);
    check();
    double hp[2 * kWBlk];
    BL_HIP(hipMemcpyAsync(hp, wpart, sizeof(hp), hipMemcpyDeviceToHost, m.stream));
    BL_HIP(hipStreamSynchronize(m.stream));
    double wsum = 0.0, wcnt = 0.0;
    for (int q = 0; q < kWBlk; ++q) {
        wsum += hp[2 * q];
        wcnt += hp[2 * q + 1];
    }
    if (!(wsum > 0.0)) {
        last_error() = "bl_mlp_train: the dataset has no row with a positive weight";
        throw ArgError();
    }
    const float wscale = (float)(wcnt / wsum);
    // the steps' loss sums stay on the device and cross to the host once
    if (loss_hist && m.nhist < steps) {
        if (m.hist) BL_HIP(hipFree(m.hist));
        m.hist = nullptr;
        m.nhist = 0;
        m.hist = alloc<float>(steps);
        m.nhist = steps;
    }
    BatchSrc src{};
    src.rows = m.rows;
    src.n = m.n;
    src.seed = seed;
    src.wscale = wscale;
    for (int s = 0; s < steps; ++s) {
        src.step = m.step;
        m.step += 1;
        const float c1 = 1.f - powf(0.9f, (float)m.step), c2 = 1.f - powf(0.999f, (float)m.step);
        launch_grad(m, src, B, true, lr, c1, c2, loss_hist ? m.hist + s : m.scal);
    }
    if (loss_hist && steps > 0)
        BL_HIP(hipMemcpyAsync(loss_hist, m.hist, sizeof(float) * steps, hipMemcpyDeviceToHost, m.stream));
    BL_HIP(hipStreamSynchronize(m.stream));
    if (loss_hist)
        for (int s = 0; s < steps; ++s) loss_hist[s] /= (float)B;
}

}  // namespace blgpu

// ------------------------------------------------------------------------
// C ABI
// ------------------------------------------------------------------------
using namespace blgpu;

namespace {
template <class F>
int mlp_guarded(F &&fn) {
    try {
        fn();
        return BL_OK;
    } catch (const ArgError &) {
        return BL_EINVAL;
    } catch (const DeviceError &) {
        return BL_EDEVICE;
    } catch (const std::bad_alloc &) {
        if (last_error().empty()) last_error() = "out of memory";
        return BL_ENOMEM;
    } catch (...) {
        last_error() = "unexpected exception";
        return BL_EDEVICE;
    }
}
Mlp &MM(bl_mlp *m) {
    if (!m) {
        last_error() = "null closure handle";
        throw ArgError();
    }
    return *m;
}
void need(bool ok, const char *msg) {
    if (!ok) {
        last_error() = msg;
        throw ArgError();
    }
}
}  // namespace

extern "C" {

int bl_mlp_create(long long capacity, int batch_max, bl_mlp **out) {
    last_error().clear();
    if (!out || capacity < 1 || batch_max < 1) {
        last_error() = "bl_mlp_create: need capacity >= 1, batch_max >= 1 and an output pointer";
        return BL_EINVAL;
    }
    *out = nullptr;
    bl_mlp *m = new (std::nothrow) bl_mlp();
    if (!m) return BL_ENOMEM;
    std::memset(static_cast<Mlp *>(m), 0, sizeof(Mlp));
    const int rc = mlp_guarded([&] { mlp_init(*m, capacity, batch_max); });
    if (rc != BL_OK) {
        mlp_free(*m);
        delete m;
        return rc;
    }
    *out = m;
    return BL_OK;
}

void bl_mlp_destroy(bl_mlp *m) {
    if (!m) return;
    mlp_free(*m);
    delete m;
}

int bl_mlp_set_params(bl_mlp *mm, const float *theta) {
    return mlp_guarded([&] {
        Mlp &m = MM(mm);
        need(theta != nullptr, "bl_mlp_set_params: null parameters");
        BL_HIP(hipMemcpyAsync(m.theta, theta, kMlpParams * sizeof(float), hipMemcpyHostToDevice, m.stream));
        BL_HIP(hipMemsetAsync(m.adam_m, 0, kMlpParams * sizeof(float), m.stream));
        BL_HIP(hipMemsetAsync(m.adam_v, 0, kMlpParams * sizeof(float), m.stream));
        BL_HIP(hipStreamSynchronize(m.stream));
        m.step = 0;
    });
}

int bl_mlp_get_params(bl_mlp *mm, float *theta) {
    return mlp_guarded([&] {
        Mlp &m = MM(mm);
        need(theta != nullptr, "bl_mlp_get_params: null output");
        BL_HIP(hipMemcpyAsync(theta, m.theta, kMlpParams * sizeof(float), hipMemcpyDeviceToHost, m.stream));
        BL_HIP(hipStreamSynchronize(m.stream));
    });
}

int bl_mlp_forward(bl_mlp *mm, const float *x, int n, float *y) {
    return mlp_guarded([&] {
        Mlp &m = MM(mm);
        need(x && y && n >= 1 && n <= m.bmax, "bl_mlp_forward: need 1 <= n <= batch_max and buffers");
        mlp_load_batch(m, x, nullptr, n);
        mlp_fwd_bwd(m, n, false);
        BL_HIP(hipMemcpyAsync(y, m.y, sizeof(float) * n, hipMemcpyDeviceToHost, m.stream));
        BL_HIP(hipStreamSynchronize(m.stream));
    });
}

int bl_mlp_gradient(bl_mlp *mm, const float *x, const float *t, int n, float *g, float *loss) {
    return mlp_guarded([&] {
        Mlp &m = MM(mm);
        need(x && t && g && n >= 1 && n <= m.bmax, "bl_mlp_gradient: need 1 <= n <= batch_max and buffers");
        mlp_load_batch(m, x, t, n);
        mlp_fwd_bwd(m, n, true);
        BL_HIP(hipMemcpyAsync(g, m.g, sizeof(float) * kMlpParams, hipMemcpyDeviceToHost, m.stream));
        float l = 0.f;
        BL_HIP(hipMemcpyAsync(&l, m.scal, sizeof(float), hipMemcpyDeviceToHost, m.stream));
        BL_HIP(hipStreamSynchronize(m.stream));
        if (loss) *loss = l / (float)n;
    });
}

int bl_mlp_add_rows(bl_mlp *mm, const float *rows, long long n) {
    return mlp_guarded([&] {
        Mlp &m = MM(mm);
        need(rows && n >= 0, "bl_mlp_add_rows: null rows");
        need(m.n + n <= m.cap, "bl_mlp_add_rows: dataset capacity exceeded");
        BL_HIP(hipMemcpyAsync(m.rows + m.n * kMlpRow, rows, sizeof(float) * kMlpRow * n, hipMemcpyHostToDevice,
                              m.stream));
        BL_HIP(hipStreamSynchronize(m.stream));
        m.n += n;
    });
}

int bl_mlp_get_rows(bl_mlp *mm, long long first, long long n, float *rows) {
    return mlp_guarded([&] {
        Mlp &m = MM(mm);
        need(rows && first >= 0 && n >= 0 && first + n <= m.n, "bl_mlp_get_rows: range outside the dataset");
        BL_HIP(hipMemcpyAsync(rows, m.rows + first * kMlpRow, sizeof(float) * kMlpRow * n, hipMemcpyDeviceToHost,
                              m.stream));
        BL_HIP(hipStreamSynchronize(m.stream));
    });
}

int bl_mlp_count(bl_mlp *mm, long long *n) {
    return mlp_guarded([&] {
        need(n != nullptr, "bl_mlp_count: null output");
        *n = MM(mm).n;
    });
}

int bl_mlp_clear(bl_mlp *mm) {
    return mlp_guarded([&] { MM(mm).n = 0; });
}

int bl_mlp_train(bl_mlp *mm, int steps, int batch, float lr, unsigned long long seed, float *loss_hist) {
    return mlp_guarded([&] {
        Mlp &m = MM(mm);
        need(steps >= 0 && lr > 0.f, "bl_mlp_train: need steps >= 0 and lr > 0");
        mlp_train(m, steps, batch, lr, seed, loss_hist);
    });
}

}  // extern "C"
