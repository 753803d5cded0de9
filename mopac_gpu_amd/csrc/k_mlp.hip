// Small MLP for the learned starting density: BF16 weights and layer inputs,
// FP32 accumulation, tanh hidden activations, linear output.  Forward,
// backward (mean-squared error), and Adam, all on the device.
//
// Layer l: Z = bf16(X_l) * bf16(W_l) + b_l (FP32), X_{l+1} = tanh(Z) (hidden),
// Y = Z (last).  Master weights stay FP32; the BF16 copies are refreshed after
// every optimizer step.  Backward treats the BF16 rounding of activations as
// the identity (straight-through), the usual mixed-precision convention.
//
// Every product runs on the BF16 matrix cores.  The forward operands are BF16
// already.  The backward's FP32 operand dZ goes in as three BF16 parts that
// add up to it exactly (8 significand bits each, by truncation), the leading
// part and the two others summed separately in FP32, so no bit of it is lost.
#include <vector>

#include "common.h"

namespace mhip {
namespace {

__device__ __forceinline__ unsigned short f2bf(float x) {
  // round to nearest even
  unsigned u = __float_as_uint(x);
  if ((u & 0x7f800000u) == 0x7f800000u) return (unsigned short)(u >> 16);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (unsigned short)(u >> 16);
}

// x = p[0] + p[1] + p[2] in BF16, exactly (down to the smallest normal
// numbers); an infinity or NaN stays in p[0]
__device__ __forceinline__ void split3(float x, unsigned short p[3]) {
  const unsigned u = __float_as_uint(x);
  p[0] = (unsigned short)(u >> 16);
  if ((u & 0x7f800000u) == 0x7f800000u) {
    p[1] = p[2] = 0;
    return;
  }
  const float r1 = x - __uint_as_float(u & 0xffff0000u);
  const unsigned u1 = __float_as_uint(r1);
  p[1] = (unsigned short)(u1 >> 16);
  p[2] = (unsigned short)(__float_as_uint(r1 - __uint_as_float(u1 & 0xffff0000u)) >> 16);
}

typedef __bf16 bf8_t __attribute__((ext_vector_type(8)));
typedef float f4_t __attribute__((ext_vector_type(4)));

// v_mfma_f32_16x16x32_bf16: lane l gives A[l % 16][8 (l / 16) ..+7] and
// B[8 (l / 16) ..+7][l % 16] and holds D[4 (l / 16) + t][l % 16].
__device__ __forceinline__ f4_t mma(bf8_t a, bf8_t b, f4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

constexpr int MLP_NT = 256;
constexpr int MLP_BN = 256;  // output columns per workgroup: 64 per wave

// C[M x N] = A[M x K] * B (+ epilogue), A row-major FP32, B given as BF16 rows
// per output column, Kp long (K padded to 32 with zeros).  A tile of A is
// converted once into LDS (PARTS = 1: rounded to BF16; 3: split exactly), B
// is read from L2 in the operand layout.  One workgroup has BM rows and up to
// 256 columns, so A is read from memory once.
//   forward  (PARTS 1): C = act(A B + bias), act 1 = tanh
//   backward (PARTS 3): C = A B (1 - act_in^2), act_in the tanh outputs
// Bound by the FP32 activations it reads and writes: 28 us a layer on average
// for 30000 rows of 168-256-256-256-16 (61 MB through memory for a 256 x 256
// layer); FP32 vector tiles of 32x32, with a conversion pass before each
// product, took 140 us.
template <int BM, int PARTS>
__global__ __launch_bounds__(MLP_NT) void k_layer(int M, int N, int K, int Kp, const float* __restrict__ A,
                                                  const unsigned short* __restrict__ B,
                                                  const float* __restrict__ bias, int act,
                                                  const float* __restrict__ act_in, float* __restrict__ C) {
  constexpr int KC = PARTS == 1 ? 256 : 128, LD = KC + 8;
  __shared__ __align__(16) unsigned short as[PARTS][BM][LD];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int li = lane & 15, lg = lane >> 4;
  const int m0 = blockIdx.x * BM, n0 = blockIdx.y * MLP_BN + 64 * w;
  const bool vec = (K & 3) == 0 && (reinterpret_cast<uintptr_t>(A) & 15) == 0;
  f4_t big[BM / 16][4], corr[BM / 16][4];
#pragma unroll
  for (int i = 0; i < BM / 16; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) big[i][j] = corr[i][j] = f4_t{0.f, 0.f, 0.f, 0.f};
  for (int kc = 0; kc < Kp; kc += KC) {
    const int kk = min(KC, Kp - kc), quads = BM * (kk >> 2);
    if (kc) __syncthreads();
    constexpr int QPT = BM * KC / 4 / MLP_NT;
    float4 v[QPT];
#pragma unroll
    for (int q = 0; q < QPT; ++q) {
      const int idx = tid + MLP_NT * q;
      v[q] = make_float4(0.f, 0.f, 0.f, 0.f);
      if (idx < quads) {
        const int r = m0 + idx / (kk >> 2), k = kc + 4 * (idx % (kk >> 2));
        if (r < M) {
          const float* src = A + (size_t)r * K + k;
          if (vec) {
            if (k < K) v[q] = *reinterpret_cast<const float4*>(src);
          } else {
            if (k < K) v[q].x = src[0];
            if (k + 1 < K) v[q].y = src[1];
            if (k + 2 < K) v[q].z = src[2];
            if (k + 3 < K) v[q].w = src[3];
          }
        }
      }
    }
#pragma unroll
    for (int q = 0; q < QPT; ++q) {
      const int idx = tid + MLP_NT * q;
      if (idx >= quads) continue;
      const int r = idx / (kk >> 2), k = 4 * (idx % (kk >> 2));
      const float x[4] = {v[q].x, v[q].y, v[q].z, v[q].w};
      unsigned short p[4][3];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        if constexpr (PARTS == 1) p[t][0] = f2bf(x[t]);
        else split3(x[t], p[t]);
      }
#pragma unroll
      for (int pl = 0; pl < PARTS; ++pl)
        *reinterpret_cast<ushort4*>(&as[pl][r][k]) = make_ushort4(p[0][pl], p[1][pl], p[2][pl], p[3][pl]);
    }
    __syncthreads();
    if (n0 >= N) continue;
    for (int k = 0; k < kk; k += 32) {
      bf8_t b[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int n = n0 + 16 * j + li;
        b[j] = n < N ? *reinterpret_cast<const bf8_t*>(B + (size_t)n * Kp + kc + k + 8 * lg) : bf8_t{};
      }
#pragma unroll
      for (int i = 0; i < BM / 16; ++i) {
        bf8_t a[PARTS];
#pragma unroll
        for (int pl = 0; pl < PARTS; ++pl)
          a[pl] = *reinterpret_cast<const bf8_t*>(&as[pl][16 * i + li][k + 8 * lg]);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          if constexpr (PARTS == 3) {
            corr[i][j] = mma(a[2], b[j], corr[i][j]);
            corr[i][j] = mma(a[1], b[j], corr[i][j]);
          }
          big[i][j] = mma(a[0], b[j], big[i][j]);
        }
      }
    }
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int n = n0 + 16 * j + li;
    if (n >= N) continue;
    const float bn = bias ? bias[n] : 0.f;
#pragma unroll
    for (int i = 0; i < BM / 16; ++i)
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int r = m0 + 16 * i + 4 * lg + t;
        if (r >= M) continue;
        const size_t at = (size_t)r * N + n;
        if constexpr (PARTS == 1) {
          const float z = big[i][j][t] + bn;
          C[at] = act == 1 ? tanhf(z) : z;
        } else {
          const float x = act_in[at];
          C[at] = (big[i][j][t] + corr[i][j][t]) * (1.f - x * x);
        }
      }
  }
}

// One layer of the network, in the flat parameter vector and in the padded
// BF16 copies: wt has out rows of inp (in padded to 32), wp in rows of outp.
struct LayerDev {
  int in, out, inp, outp;
  long long woff, boff, wt, wp;
  long long pre;  // sum of the widths before the layer's input
  int tile0;      // first 64x64 tile of the layer in k_dw's grid
};

__device__ __forceinline__ const LayerDev& layer_of_tile(const LayerDev* __restrict__ L, int nl, int tile) {
  int l = 0;
  while (l + 1 < nl && tile >= L[l + 1].tile0) ++l;
  return L[l];
}

// Every layer's dW = bf16(X)^T dZ and db = column sums of dZ, in one launch:
// a workgroup has a 64x64 tile of one layer's dW and a slice of the batch
// (blockIdx.y), whose part goes to part[slice] in the parameter layout.  X
// and dZ are transposed on their way into LDS (a thread packs eight batch
// rows of one column into 16 bytes), dZ in its three exact parts.
// The matrix of a layer alone fills a few dozen workgroups, each over the
// whole batch (171 us a layer at a batch of 2048, and 364 us for the column
// sums of one thread per column); the slices fill the chip: 13 us for the
// four layers of 96-256-256-256-16.
__global__ __launch_bounds__(MLP_NT) void k_dw(int nl, const LayerDev* __restrict__ L, int batch, int rows,
                                               const float* __restrict__ acts, const float* __restrict__ dz,
                                               long long np, float* __restrict__ part) {
  constexpr int LD = 40;
  __shared__ __align__(16) unsigned short xs[64][LD], zs[3][64][LD];
  __shared__ float red[4][64];
  const LayerDev& y = layer_of_tile(L, nl, blockIdx.x);
  const int tile = blockIdx.x - y.tile0, nj = (y.out + 63) / 64;
  const int i0 = 64 * (tile / nj), j0 = 64 * (tile % nj);
  const int in = y.in, out = y.out;
  const float* X = acts + (size_t)batch * y.pre;
  const float* Z = dz + (size_t)batch * (y.pre + in);
  const int b0 = blockIdx.y * rows, b1 = min(batch, b0 + rows);
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int li = lane & 15, lg = lane >> 4;
  const int wm = 32 * (w >> 1), wn = 32 * (w & 1);
  const bool xi = i0 + lane < in, zj = j0 + lane < out;
  f4_t big[2][2], corr[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) big[i][j] = corr[i][j] = f4_t{0.f, 0.f, 0.f, 0.f};
  float sum = 0.f, xv[8], zv[8];
  auto load = [&](int b) {
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      const int row = b + 8 * w + r;
      xv[r] = xi && row < b1 ? X[(size_t)row * in + i0 + lane] : 0.f;
      zv[r] = zj && row < b1 ? Z[(size_t)row * out + j0 + lane] : 0.f;
    }
  };
  load(b0);
  for (int b = b0; b < b1; b += 32) {
    {
      union { unsigned short h[8]; uint4 q; } x, z[3];
#pragma unroll
      for (int r = 0; r < 8; ++r) {
        x.h[r] = f2bf(xv[r]);
        unsigned short p[3];
        split3(zv[r], p);
        z[0].h[r] = p[0];
        z[1].h[r] = p[1];
        z[2].h[r] = p[2];
        sum += zv[r];
      }
      *reinterpret_cast<uint4*>(&xs[lane][8 * w]) = x.q;
#pragma unroll
      for (int pl = 0; pl < 3; ++pl) *reinterpret_cast<uint4*>(&zs[pl][lane][8 * w]) = z[pl].q;
    }
    __syncthreads();
    if (b + 32 < b1) load(b + 32);
    bf8_t a[2], bz[2][3];
#pragma unroll
    for (int i = 0; i < 2; ++i) a[i] = *reinterpret_cast<const bf8_t*>(&xs[wm + 16 * i + li][8 * lg]);
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int pl = 0; pl < 3; ++pl)
        bz[j][pl] = *reinterpret_cast<const bf8_t*>(&zs[pl][wn + 16 * j + li][8 * lg]);
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        corr[i][j] = mma(a[i], bz[j][2], corr[i][j]);
        corr[i][j] = mma(a[i], bz[j][1], corr[i][j]);
        big[i][j] = mma(a[i], bz[j][0], big[i][j]);
      }
    __syncthreads();
  }
  float* o = part + (size_t)blockIdx.y * np;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int r = i0 + wm + 16 * i + 4 * lg + t, c = j0 + wn + 16 * j + li;
        if (r < in && c < out) o[y.woff + (long long)r * out + c] = big[i][j][t] + corr[i][j][t];
      }
  if (i0 == 0) {
    red[w][lane] = sum;
    __syncthreads();
    if (w == 0 && zj) o[y.boff + j0 + lane] = red[0][lane] + red[1][lane] + red[2][lane] + red[3][lane];
  }
}

// grad = sum of the batch slices' parts, in slice order; the first workgroup
// also sums the loss's parts
__global__ __launch_bounds__(256) void k_grad_sum(long long np, int slices, const float* __restrict__ part,
                                                  float* __restrict__ grad, int nloss,
                                                  const float* __restrict__ lpart, float scale,
                                                  float* __restrict__ loss) {
  const long long i = blockIdx.x * 256LL + threadIdx.x;
  if (i < np) {
    float s = 0.f;
    for (int k = 0; k < slices; ++k) s += part[(size_t)k * np + i];
    grad[i] = s;
  }
  if (blockIdx.x == 0 && threadIdx.x < 64) {
    double s = 0.0;
    for (int k = threadIdx.x; k < nloss; k += 64) s += lpart[k];
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    if (threadIdx.x == 0) *loss = (float)(s * scale);
  }
}

// both BF16 copies of every weight
__global__ __launch_bounds__(256) void k_refresh(int nl, const LayerDev* __restrict__ L,
                                                 const float* __restrict__ w, unsigned short* __restrict__ bf) {
  const LayerDev y = L[blockIdx.y];
  const long long len = (long long)y.in * y.out;
  for (long long i = blockIdx.x * 256LL + threadIdx.x; i < len; i += (long long)gridDim.x * 256) {
    const int r = (int)(i / y.out), c = (int)(i % y.out);
    const unsigned short h = f2bf(w[y.woff + i]);
    bf[y.wt + (long long)c * y.inp + r] = h;
    bf[y.wp + (long long)r * y.outp + c] = h;
  }
}

__global__ void k_zero_u16(long long n, unsigned short* __restrict__ p) {
  for (long long i = blockIdx.x * 256LL + threadIdx.x; i < n; i += (long long)gridDim.x * 256) p[i] = 0;
}

// dY = (Y - T) * 2 / (B * nout); partial loss sums per block
__global__ __launch_bounds__(256) void k_mse(long long n, float scale, const float* __restrict__ y,
                                             const float* __restrict__ t, float* __restrict__ dy,
                                             float* __restrict__ part) {
  __shared__ float red[256];
  float s = 0.f;
  for (long long i = blockIdx.x * 256LL + threadIdx.x; i < n; i += (long long)gridDim.x * 256) {
    const float d = y[i] - t[i];
    s += d * d;
    dy[i] = 2.f * d * scale;
  }
  red[threadIdx.x] = s;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

__global__ void k_adam(long long n, float* __restrict__ w, const float* __restrict__ g,
                       float* __restrict__ m, float* __restrict__ v, float lr, float b1, float b2,
                       float c1, float c2, float eps) {
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n;
       i += (long long)gridDim.x * blockDim.x) {
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    w[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
  }
}

inline int cdiv(long long a, long long b) { return (int)((a + b - 1) / b); }

}  // namespace
}  // namespace mhip

using namespace mhip;

struct mhip_mlp {
  int nl = 0;
  std::vector<int> dims;
  std::vector<LayerDev> lay;
  int ntiles = 0;  // 64x64 tiles of all weight matrices
  size_t np = 0;
  hipStream_t s = nullptr;
  DevBuf w32, wbf, grad, m, v, layers;
  DevBuf acts;   // X_0..X_nl (FP32) for the current batch
  DevBuf dz;     // the gradients by the layers' outputs, laid out as acts
  DevBuf gpart;  // the batch slices' parts of the gradient
  DevBuf tgt, part, loss;
  int batch_cap = 0;
  long long step = 0;
};

namespace {

void mlp_ensure_batch(mhip_mlp* q, int batch) {
  if (batch <= q->batch_cap) return;
  size_t tot = 0;
  for (int l = 0; l <= q->nl; ++l) tot += (size_t)batch * q->dims[l];
  q->acts.ensure(sizeof(float) * tot);
  q->tgt.ensure(sizeof(float) * (size_t)batch * q->dims[q->nl]);
  q->part.ensure(sizeof(float) * 1024);
  q->loss.ensure(sizeof(float) * 4);
  q->batch_cap = batch;
}

float* act_ptr(mhip_mlp* q, int batch, int l) {
  size_t off = 0;
  for (int i = 0; i < l; ++i) off += (size_t)batch * q->dims[i];
  return q->acts.as<float>() + off;
}

void refresh_bf16(mhip_mlp* q) {
  hipLaunchKernelGGL(k_refresh, dim3(128, q->nl), dim3(256), 0, q->s, q->nl, q->layers.as<LayerDev>(),
                     q->w32.as<float>(), q->wbf.as<unsigned short>());
  MHIP_LAUNCH_CHECK();
}

// rows per workgroup: 32 where that fills the chip twice over, else 16
template <int PARTS>
void layer(mhip_mlp* q, int M, int N, int K, int Kp, const float* A, const unsigned short* B, const float* bias,
           int act, const float* act_in, float* C) {
  const int ny = cdiv(N, MLP_BN);
  if (cdiv(M, 32) * ny >= 512)
    hipLaunchKernelGGL((k_layer<32, PARTS>), dim3(cdiv(M, 32), ny), dim3(MLP_NT), 0, q->s, M, N, K, Kp, A, B, bias,
                       act, act_in, C);
  else
    hipLaunchKernelGGL((k_layer<16, PARTS>), dim3(cdiv(M, 16), ny), dim3(MLP_NT), 0, q->s, M, N, K, Kp, A, B, bias,
                       act, act_in, C);
  MHIP_LAUNCH_CHECK();
}

void forward(mhip_mlp* q, int batch) {
  for (int l = 0; l < q->nl; ++l) {
    const LayerDev& y = q->lay[l];
    layer<1>(q, batch, y.out, y.in, y.inp, act_ptr(q, batch, l), q->wbf.as<unsigned short>() + y.wt,
             q->w32.as<float>() + y.boff, (l + 1 < q->nl) ? 1 : 0, nullptr, act_ptr(q, batch, l + 1));
  }
}

// gradients of the mean squared error into q->grad; loss on the device
void backward(mhip_mlp* q, int batch) {
  const int nout = q->dims[q->nl];
  const long long ny = (long long)batch * nout;
  size_t tot = 0;
  for (int l = 0; l <= q->nl; ++l) tot += (size_t)batch * q->dims[l];
  // slices of whole 32-row steps: enough of them to fill the chip, each at
  // least 128 rows, at most 16 (each one writes and reads a gradient)
  const int slices = std::max(1, std::min(16, batch / 128)), rows = cdiv(cdiv(batch, slices), 32) * 32;
  const int nslice = cdiv(batch, rows);
  q->dz.ensure(sizeof(float) * tot);
  q->gpart.ensure(sizeof(float) * q->np * nslice);
  float* dz = q->dz.as<float>();
  auto dz_of = [&](int l) { return dz + (act_ptr(q, batch, l) - q->acts.as<float>()); };
  const int pb = std::min(1024, cdiv(ny, 256));
  hipLaunchKernelGGL(k_mse, dim3(pb), dim3(256), 0, q->s, ny, 1.f / (float)ny, act_ptr(q, batch, q->nl),
                     q->tgt.as<float>(), dz_of(q->nl), q->part.as<float>());
  MHIP_LAUNCH_CHECK();
  // dZ of a layer's input: dZ W^T through that input's tanh
  for (int l = q->nl - 1; l > 0; --l) {
    const LayerDev& y = q->lay[l];
    layer<3>(q, batch, y.in, y.out, y.outp, dz_of(l + 1), q->wbf.as<unsigned short>() + y.wp, nullptr, 0,
             act_ptr(q, batch, l), dz_of(l));
  }
  hipLaunchKernelGGL(k_dw, dim3(q->ntiles, nslice), dim3(MLP_NT), 0, q->s, q->nl, q->layers.as<LayerDev>(), batch,
                     rows, q->acts.as<float>(), dz, (long long)q->np, q->gpart.as<float>());
  MHIP_LAUNCH_CHECK();
  hipLaunchKernelGGL(k_grad_sum, dim3(cdiv(q->np, 256)), dim3(256), 0, q->s, (long long)q->np, nslice,
                     q->gpart.as<float>(), q->grad.as<float>(), pb, q->part.as<float>(), 1.f / (float)ny,
                     q->loss.as<float>());
  MHIP_LAUNCH_CHECK();
}

template <class F>
int guard(F&& fn) {
  try {
    fn();
    return 0;
  } catch (const HipError& e) {
    set_error(e.msg);
    return 1;
  }
}

}  // namespace

// Device-resident forward pass for callers in other files (the learned
// guess): they write the batch into mlp_input, then mlp_forward_resident
// runs the network on the network's own stream, waits for it and returns the
// device pointer of the outputs (batch x dims[nl], row-major).
namespace mhip {
float* mlp_input(mhip_mlp* q, int batch) {
  mlp_ensure_batch(q, batch);
  return act_ptr(q, batch, 0);
}
const float* mlp_forward_resident(mhip_mlp* q, int batch) {
  forward(q, batch);
  MHIP_CHECK(hipStreamSynchronize(q->s));
  return act_ptr(q, batch, q->nl);
}
int mlp_layers(const mhip_mlp* q) { return q->nl; }
int mlp_dim(const mhip_mlp* q, int l) { return q->dims[l]; }
}  // namespace mhip

extern "C" {

int mhip_mlp_create(int nlayers, const int* dims, mhip_mlp** out) {
  return guard([&] {
    MHIP_REQUIRE(nlayers > 0 && dims && out, "mhip_mlp_create: bad arguments");
    auto* q = new mhip_mlp();
    q->nl = nlayers;
    q->dims.assign(dims, dims + nlayers + 1);
    long long off = 0, bf = 0, pre = 0;
    for (int l = 0; l < nlayers; ++l) {
      LayerDev y{};
      y.in = dims[l];
      y.out = dims[l + 1];
      y.inp = cdiv(y.in, 32) * 32;
      y.outp = cdiv(y.out, 32) * 32;
      y.woff = off;
      off += (long long)y.in * y.out;
      y.boff = off;
      off += y.out;
      y.wt = bf;
      bf += (long long)y.out * y.inp;
      y.wp = bf;
      bf += (long long)y.in * y.outp;
      y.pre = pre;
      pre += y.in;
      y.tile0 = q->ntiles;
      q->ntiles += cdiv(y.in, 64) * cdiv(y.out, 64);
      q->lay.push_back(y);
    }
    q->np = (size_t)off;
    MHIP_CHECK(hipStreamCreateWithFlags(&q->s, hipStreamNonBlocking));
    q->layers.ensure(sizeof(LayerDev) * nlayers);
    MHIP_CHECK(hipMemcpyAsync(q->layers.ptr, q->lay.data(), sizeof(LayerDev) * nlayers, hipMemcpyHostToDevice, q->s));
    q->w32.ensure(sizeof(float) * off);
    // the padding stays zero: refreshes write the weights only
    q->wbf.ensure(sizeof(unsigned short) * bf);
    hipLaunchKernelGGL(k_zero_u16, dim3(256), dim3(256), 0, q->s, bf, q->wbf.as<unsigned short>());
    MHIP_LAUNCH_CHECK();
    q->grad.ensure(sizeof(float) * off);
    q->m.ensure(sizeof(float) * off);
    q->v.ensure(sizeof(float) * off);
    MHIP_CHECK(hipMemsetAsync(q->m.ptr, 0, sizeof(float) * off, q->s));
    MHIP_CHECK(hipMemsetAsync(q->v.ptr, 0, sizeof(float) * off, q->s));
    MHIP_CHECK(hipStreamSynchronize(q->s));
    *out = q;
  });
}

void mhip_mlp_destroy(mhip_mlp* q) {
  if (!q) return;
  (void)hipStreamSynchronize(q->s);
  for (DevBuf* b : {&q->w32, &q->wbf, &q->grad, &q->m, &q->v, &q->layers, &q->acts, &q->dz, &q->gpart, &q->tgt,
                    &q->part, &q->loss})
    b->release();
  (void)hipStreamDestroy(q->s);
  delete q;
}

int mhip_mlp_set_params(mhip_mlp* q, const float* params) {
  return guard([&] {
    MHIP_CHECK(hipMemcpyAsync(q->w32.ptr, params, sizeof(float) * q->np, hipMemcpyHostToDevice, q->s));
    refresh_bf16(q);
    MHIP_CHECK(hipMemsetAsync(q->m.ptr, 0, sizeof(float) * q->np, q->s));
    MHIP_CHECK(hipMemsetAsync(q->v.ptr, 0, sizeof(float) * q->np, q->s));
    q->step = 0;
    MHIP_CHECK(hipStreamSynchronize(q->s));
  });
}

int mhip_mlp_get_params(mhip_mlp* q, float* params) {
  return guard([&] {
    MHIP_CHECK(hipMemcpyAsync(params, q->w32.ptr, sizeof(float) * q->np, hipMemcpyDeviceToHost, q->s));
    MHIP_CHECK(hipStreamSynchronize(q->s));
  });
}

int mhip_mlp_forward(mhip_mlp* q, int batch, const float* x, float* y) {
  return guard([&] {
    MHIP_REQUIRE(batch > 0, "mhip_mlp_forward: empty batch");
    mlp_ensure_batch(q, batch);
    MHIP_CHECK(hipMemcpyAsync(act_ptr(q, batch, 0), x, sizeof(float) * (size_t)batch * q->dims[0],
                              hipMemcpyHostToDevice, q->s));
    forward(q, batch);
    MHIP_CHECK(hipMemcpyAsync(y, act_ptr(q, batch, q->nl), sizeof(float) * (size_t)batch * q->dims[q->nl],
                              hipMemcpyDeviceToHost, q->s));
    MHIP_CHECK(hipStreamSynchronize(q->s));
  });
}

int mhip_mlp_gradients(mhip_mlp* q, int batch, const float* x, const float* t, float* grad,
                       float* loss) {
  return guard([&] {
    MHIP_REQUIRE(batch > 0, "mhip_mlp_gradients: empty batch");
    mlp_ensure_batch(q, batch);
    MHIP_CHECK(hipMemcpyAsync(act_ptr(q, batch, 0), x, sizeof(float) * (size_t)batch * q->dims[0],
                              hipMemcpyHostToDevice, q->s));
    MHIP_CHECK(hipMemcpyAsync(q->tgt.ptr, t, sizeof(float) * (size_t)batch * q->dims[q->nl],
                              hipMemcpyHostToDevice, q->s));
    forward(q, batch);
    backward(q, batch);
    MHIP_CHECK(hipMemcpyAsync(grad, q->grad.ptr, sizeof(float) * q->np, hipMemcpyDeviceToHost, q->s));
    MHIP_CHECK(hipMemcpyAsync(loss, q->loss.ptr, sizeof(float), hipMemcpyDeviceToHost, q->s));
    MHIP_CHECK(hipStreamSynchronize(q->s));
  });
}

int mhip_mlp_train_step(mhip_mlp* q, int batch, const float* x, const float* t, float lr,
                        float* loss) {
  return guard([&] {
    MHIP_REQUIRE(batch > 0, "mhip_mlp_train_step: empty batch");
    mlp_ensure_batch(q, batch);
    MHIP_CHECK(hipMemcpyAsync(act_ptr(q, batch, 0), x, sizeof(float) * (size_t)batch * q->dims[0],
                              hipMemcpyHostToDevice, q->s));
    MHIP_CHECK(hipMemcpyAsync(q->tgt.ptr, t, sizeof(float) * (size_t)batch * q->dims[q->nl],
                              hipMemcpyHostToDevice, q->s));
    forward(q, batch);
    backward(q, batch);
    q->step += 1;
    const float b1 = 0.9f, b2 = 0.999f;
    const float c1 = 1.f - std::pow(b1, (float)q->step), c2 = 1.f - std::pow(b2, (float)q->step);
    hipLaunchKernelGGL(k_adam, dim3(std::min(4096, cdiv(q->np, 256))), dim3(256), 0, q->s,
                       (long long)q->np, q->w32.as<float>(), q->grad.as<float>(), q->m.as<float>(),
                       q->v.as<float>(), lr, b1, b2, c1, c2, 1e-8f);
    MHIP_LAUNCH_CHECK();
    refresh_bf16(q);
    if (loss) {
      MHIP_CHECK(hipMemcpyAsync(loss, q->loss.ptr, sizeof(float), hipMemcpyDeviceToHost, q->s));
    }
    MHIP_CHECK(hipStreamSynchronize(q->s));
  });
}

}  // extern "C"
