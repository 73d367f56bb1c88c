// mlp.hip -- the learned band: per-gap features, a 272-256-128-1 MLP with
// bf16 weights and fp32 accumulation (forward, backward, Adam), and the band
// prediction that feeds the banded DP.  No counterpart in the reference,
// whose NWSmall always fills the whole matrix.
//
// Numerics (the CPU oracle restates exactly these roundings):
//   x_bf = bf16(x); W_bf = bf16(W) for W1, W2, w3 (master weights fp32)
//   h1 = bf16(relu(x_bf W1_bf^T + b1)); h2 = bf16(relu(h1 W2_bf^T + b2))
//   y  = h2 . w3_bf + b3                                   (fp32)
//   loss = sum (y - t)^2 / (2B);  g = bf16((y - t) / B)
//   dz2 = bf16(g w3_bf) where h2 > 0, else 0;  dw3 = g^T h2;  db3 = sum g
//   dW2 = dz2^T h1;  db2 = colsum dz2
//   dz1 = bf16(dz2 W2_bf) where h1 > 0, else 0
//   dW1 = dz1^T x_bf;  db1 = colsum dz1
// bf16 rounding is round-to-nearest-even; products of two bf16 values are
// exact in fp32; every sum accumulates in fp32.
#include "mh_internal.hpp"
#include <algorithm>
#include <cmath>
#include <cstring>
#include <random>

namespace mh {
namespace {

constexpr int NIN = MH_MLP_IN, NH1 = MH_MLP_H1, NH2 = MH_MLP_H2;
// flat parameter layout (fp32): W1 [NH1][NIN], b1, W2 [NH2][NH1], b2, w3 [NH2], b3
constexpr int OFF_W1 = 0;
constexpr int OFF_B1 = OFF_W1 + NH1 * NIN;
constexpr int OFF_W2 = OFF_B1 + NH1;
constexpr int OFF_B2 = OFF_W2 + NH2 * NH1;
constexpr int OFF_W3 = OFF_B2 + NH2;
constexpr int OFF_B3 = OFF_W3 + NH2;
constexpr int NPARAM = OFF_B3 + 1;
static_assert(NPARAM == MH_MLP_NPARAMS, "parameter count");
// bf16 copies: W1, W2, w3 back to back
constexpr int BOFF_W1 = 0, BOFF_W2 = NH1 * NIN, BOFF_W3 = BOFF_W2 + NH2 * NH1, NBF = BOFF_W3 + NH2;

__host__ __device__ inline uint16_t to_bf16(float f)
{
    uint32_t u;
    std::memcpy(&u, &f, 4);
    u += 0x7FFFu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}

__host__ __device__ inline float from_bf16(uint16_t h)
{
    const uint32_t u = (uint32_t)h << 16;
    float f;
    std::memcpy(&f, &u, 4);
    return f;
}

// ---- features ----------------------------------------------------------------
//
// Per job (A of length la, B of length lb):
//   f[0] = log2(la)/16, f[1] = log2(lb)/16, f[2] = log2(1 + |la - lb|)/16
//   f[3] = sum_k |cA[k] - cB[k]| / max(1, nA + nB)       (4-mer L1 distance)
//   f[4 + k] = clamp((cA[k] - cB[k]) * 512 / max(512, nA + nB), -8, 8) / 8
//   f[260 + 6*side + s], s = 0..5: flank seed density at scale w = 16 << s:
//       the fraction of the 8-mers of A starting at distance p < w from the
//       gap's left (side 0) or right (side 1) end that occur in B within 8
//       positions of the corner-to-corner line (B start floor(p*lb/la) from
//       the same end, +-8); 0 when no 8-mer fits.
// cA, cB are 4-mer counts (codes 0..3 packed 2 bits per letter, first letter
// high), nA = max(0, la - 3), nB likewise.

struct FeatJob {
    uint64_t a_off, b_off;
    uint32_t la, lb;
};

__device__ inline uint32_t pack8(const uint8_t *s)
{
    uint32_t v = 0;
#pragma unroll
    for (int q = 0; q < 8; ++q) v = (v << 2) | (s[q] & 3u);
    return v;
}

__global__ __launch_bounds__(256) void features_kernel(const uint8_t *__restrict__ A, const uint8_t *__restrict__ B,
                                                       const mh_dp_job *__restrict__ jobs, uint64_t njobs,
                                                       float *__restrict__ feat)
{
    __shared__ int ha[256], hb[256];
    __shared__ int hits[2][6], valid[2][6];
    __shared__ int l1part[256];
    const int t = threadIdx.x;
    const uint64_t jx = blockIdx.x;
    if (jx >= njobs) return;
    const mh_dp_job jb = jobs[jx];
    const int la = (int)jb.a_len, lb = (int)jb.b_len;
    const uint8_t *a = A + jb.a_off, *b = B + jb.b_off;
    ha[t] = 0;
    hb[t] = 0;
    if (t < 12) {
        hits[t / 6][t % 6] = 0;
        valid[t / 6][t % 6] = 0;
    }
    __syncthreads();
    for (int p = t; p + 4 <= la; p += 256)
        atomicAdd(&ha[((a[p] & 3) << 6) | ((a[p + 1] & 3) << 4) | ((a[p + 2] & 3) << 2) | (a[p + 3] & 3)], 1);
    for (int p = t; p + 4 <= lb; p += 256)
        atomicAdd(&hb[((b[p] & 3) << 6) | ((b[p + 1] & 3) << 4) | ((b[p + 2] & 3) << 2) | (b[p + 3] & 3)], 1);
    // flank densities: thread t takes p = t and t + 256 on both sides
    if (la >= 8 && lb >= 8) {
        for (int side = 0; side < 2; ++side) {
            for (int p = t; p < 512; p += 256) {
                if (p + 8 > la) continue;
                const uint32_t a8 = pack8(side == 0 ? a + p : a + (la - 8 - p));
                const int64_t qc = ((int64_t)p * lb) / la;
                bool hit = false;
                for (int64_t q = qc - 8; q <= qc + 8; ++q) {
                    if (q < 0 || q + 8 > lb) continue;
                    const uint32_t b8 = pack8(side == 0 ? b + q : b + (lb - 8 - q));
                    hit |= (b8 == a8);
                }
#pragma unroll
                for (int s = 0; s < 6; ++s)
                    if (p < (16 << s)) {
                        atomicAdd(&valid[side][s], 1);
                        if (hit) atomicAdd(&hits[side][s], 1);
                    }
            }
        }
    }
    __syncthreads();
    const int na = la >= 3 ? la - 3 : 0, nb = lb >= 3 ? lb - 3 : 0;
    const int diff = ha[t] - hb[t];
    l1part[t] = diff < 0 ? -diff : diff;
    __syncthreads();
    for (int off = 128; off > 0; off >>= 1) {
        if (t < off) l1part[t] += l1part[t + off];
        __syncthreads();
    }
    float *f = feat + jx * (uint64_t)NIN;
    const int tot = na + nb;
    float r = (float)diff * 512.0f / (float)(tot > 512 ? tot : 512);
    r = r < -8.0f ? -8.0f : (r > 8.0f ? 8.0f : r);
    f[4 + t] = r / 8.0f;
    if (t == 0) {
        f[0] = log2f((float)la) / 16.0f;
        f[1] = log2f((float)lb) / 16.0f;
        f[2] = log2f(1.0f + (float)(la > lb ? la - lb : lb - la)) / 16.0f;
        f[3] = (float)l1part[0] / (float)(tot > 1 ? tot : 1);
    }
    if (t < 12) {
        const int side = t / 6, s = t % 6;
        const int v = valid[side][s];
        f[260 + t] = v ? (float)hits[side][s] / (float)v : 0.0f;
    }
}

// ---- GEMM on MFMA ---------------------------------------------------------
//
// C[M x N] = A[M x K] . B[K x N], bf16 operands (fp32 sources are rounded on
// load), fp32 accumulation with v_mfma_f32_16x16x16bf16, k ascending.  A
// workgroup of 4 waves computes a 64x64 tile, each wave a 32x32 quarter as 2x2
// MFMA blocks; K advances 32 at a time through LDS, the next step's loads
// issued before the current step's MFMAs.  An operand is laid out with either
// its k or its other index contiguous (KC); a thread loads 8 consecutive
// elements of that index at once, so a wavefront reads whole lines either way.
// idx gathers rows of the memory layout (a batch of examples).  gridDim.z > 1
// splits K: split z covers k in [z * kchunk, (z + 1) * kchunk) and writes its
// own fp32 partial of EPI_F32 (summed by grad_reduce_kernel, z ascending).
//
// These products are small (rows x 272 x 256), so the kernel is bound by load
// latency and by the workgroups in flight, not by MFMA.  One element a load
// and no split of K, a 4,096-row batch's products took 1,121 us a pass (the
// weight gradients' K is the row count: 8 and 20 workgroups); 8 elements a
// load and K split at 128 rows they take 74 us.

struct Operand {
    const void *p;
    int64_t ld;             // elements from one index of the outer (memory row) dimension to the next
    const uint32_t *idx;
};

enum { EPI_F32 = 0, EPI_BIAS_RELU_BF16 = 1, EPI_MASK_BF16 = 2 };

struct Epilogue {
    int mode;
    const float *bias;      // per column (EPI_BIAS_RELU_BF16)
    float *c32;             // EPI_F32; split z at c32 + z * zstride
    int64_t zstride;
    uint16_t *cbf;          // bf16 outputs
    int64_t ldc;
    const uint16_t *mask;   // EPI_MASK_BF16: keep where mask > 0
    int64_t ldm;
};

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int GT = 64, GK = 32, GKP = GK + 4;   // tile, k step, padded LDS row

// eight consecutive floats at any float address, eight bf16 at any bf16 address
struct __attribute__((packed, aligned(4))) F8 { float v[8]; };
struct __attribute__((packed, aligned(2))) H8 { uint16_t v[8]; };

// Elements (outer, inner .. inner + 7) of an operand, as bf16; zeros past the bounds.
template <bool F32>
__device__ __forceinline__ void load8(const Operand &o, int outer, int n_outer, int inner, int n_inner, uint16_t *v)
{
#pragma unroll
    for (int q = 0; q < 8; ++q) v[q] = 0;
    if (outer >= n_outer || inner >= n_inner) return;
    const int64_t row = o.idx ? (int64_t)o.idx[outer] : (int64_t)outer;
    const int64_t at = row * o.ld + inner;
    if (inner + 8 <= n_inner) {
        if constexpr (F32) {
            const F8 x = *reinterpret_cast<const F8 *>(static_cast<const float *>(o.p) + at);
#pragma unroll
            for (int q = 0; q < 8; ++q) v[q] = to_bf16(x.v[q]);
        } else {
            const H8 x = *reinterpret_cast<const H8 *>(static_cast<const uint16_t *>(o.p) + at);
#pragma unroll
            for (int q = 0; q < 8; ++q) v[q] = x.v[q];
        }
    } else {
        for (int q = 0; q < 8 && inner + q < n_inner; ++q) {
            if constexpr (F32) v[q] = to_bf16(static_cast<const float *>(o.p)[at + q]);
            else v[q] = static_cast<const uint16_t *>(o.p)[at + q];
        }
    }
}

// KC: k contiguous, memory row = m (or n); else m (or n) contiguous, memory row = k.
// The thread's 8 elements of the 64 x 32 tile at (x0, k0); nx, k1 the bounds.
template <bool KC, bool F32>
__device__ __forceinline__ void tile_load(const Operand &o, int t, int x0, int nx, int k0, int k1, uint16_t *v)
{
    if constexpr (KC) load8<F32>(o, x0 + (t >> 2), nx, k0 + (t & 3) * 8, k1, v);
    else load8<F32>(o, k0 + (t >> 3), k1, x0 + (t & 7) * 8, nx, v);
}

template <bool KC> __device__ __forceinline__ void tile_store(uint16_t (*s)[GKP], int t, const uint16_t *v)
{
    if constexpr (KC) {
#pragma unroll
        for (int q = 0; q < 8; ++q) s[t >> 2][(t & 3) * 8 + q] = v[q];
    } else {
#pragma unroll
        for (int q = 0; q < 8; ++q) s[(t & 7) * 8 + q][t >> 3] = v[q];
    }
}

template <bool AKC, bool AF32, bool BKC, bool BF32>
__global__ __launch_bounds__(256) void gemm_kernel(int M, int N, int K, int kchunk, Operand A, Operand Bo, Epilogue E)
{
    __shared__ uint16_t As[GT][GKP];   // [m][k]
    __shared__ uint16_t Bs[GT][GKP];   // [n][k]
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
    const int m0 = blockIdx.x * GT, n0 = blockIdx.y * GT;
    const int kb = blockIdx.z * kchunk, ke = min(K, kb + kchunk);
    const int wm = (wv >> 1) * 32, wn = (wv & 1) * 32;
    f32x4 acc[2][2];
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y) acc[x][y] = f32x4{0.f, 0.f, 0.f, 0.f};
    uint16_t va[8], vb[8];
    tile_load<AKC, AF32>(A, t, m0, M, kb, ke, va);
    tile_load<BKC, BF32>(Bo, t, n0, N, kb, ke, vb);
    for (int k0 = kb; k0 < ke; k0 += GK) {
        tile_store<AKC>(As, t, va);
        tile_store<BKC>(Bs, t, vb);
        __syncthreads();
        if (k0 + GK < ke) {
            tile_load<AKC, AF32>(A, t, m0, M, k0 + GK, ke, va);
            tile_load<BKC, BF32>(Bo, t, n0, N, k0 + GK, ke, vb);
        }
        const int li = lane & 15;
#pragma unroll
        for (int kk = 0; kk < GK; kk += 16) {
            const int lk = kk + (lane >> 4) * 4;
            bf16x4 av[2], bv[2];
#pragma unroll
            for (int x = 0; x < 2; ++x) {
                const uint16_t *pa = &As[wm + 16 * x + li][lk];
                const uint16_t *pb = &Bs[wn + 16 * x + li][lk];
                av[x] = bf16x4{(short)pa[0], (short)pa[1], (short)pa[2], (short)pa[3]};
                bv[x] = bf16x4{(short)pb[0], (short)pb[1], (short)pb[2], (short)pb[3]};
            }
#pragma unroll
            for (int x = 0; x < 2; ++x)
#pragma unroll
                for (int y = 0; y < 2; ++y)
                    acc[x][y] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(av[x], bv[y], acc[x][y], 0, 0, 0);
        }
        __syncthreads();
    }
    // D[i][j] of a 16x16 block: lane holds column j = lane%16, rows 4*(lane/16) + 0..3
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int gm = m0 + wm + 16 * x + 4 * (lane >> 4) + q;
                const int gn = n0 + wn + 16 * y + (lane & 15);
                if (gm >= M || gn >= N) continue;
                const float v = acc[x][y][q];
                const int64_t o = (int64_t)gm * E.ldc + gn;
                if (E.mode == EPI_F32) {
                    E.c32[(int64_t)blockIdx.z * E.zstride + o] = v;
                } else if (E.mode == EPI_BIAS_RELU_BF16) {
                    const float z = v + E.bias[gn];
                    E.cbf[o] = to_bf16(z > 0.f ? z : 0.f);
                } else {
                    const uint16_t mk = E.mask[(int64_t)gm * E.ldm + gn];
                    const bool pos = mk != 0 && !(mk & 0x8000u);
                    E.cbf[o] = pos ? to_bf16(v) : (uint16_t)0;
                }
            }
}

// y[b] = b3 + sum_k h2[b][k] * w3[k]  (fp32, k ascending)
__global__ void head_kernel(const uint16_t *__restrict__ h2, int n, const uint16_t *__restrict__ w3bf,
                            const float *__restrict__ b3, float *__restrict__ y)
{
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= n) return;
    float s = 0.f;
    for (int k = 0; k < NH2; ++k) s += from_bf16(h2[(int64_t)r * NH2 + k]) * from_bf16(w3bf[k]);
    y[r] = s + b3[0];
}

// one workgroup: g = bf16((y - t)/n), loss = sum (y - t)^2 / (2n)
__global__ __launch_bounds__(256) void loss_kernel(const float *__restrict__ y, const float *__restrict__ target,
                                                   const uint32_t *__restrict__ idx, int n,
                                                   uint16_t *__restrict__ g, float *__restrict__ loss)
{
    __shared__ float part[256];
    const int t = threadIdx.x;
    float s = 0.f;
    for (int r = t; r < n; r += 256) {
        const float d = y[r] - target[idx ? idx[r] : (uint32_t)r];
        g[r] = to_bf16(d / (float)n);
        s += d * d;
    }
    part[t] = s;
    __syncthreads();
    for (int off = 128; off > 0; off >>= 1) {
        if (t < off) part[t] += part[t + off];
        __syncthreads();
    }
    if (t == 0) loss[0] = part[0] / (2.0f * (float)n);
}

// dz2[b][k] = bf16(g[b] * w3[k]) where h2 > 0
__global__ void head_back_kernel(const uint16_t *__restrict__ g, const uint16_t *__restrict__ h2, int n,
                                 const uint16_t *__restrict__ w3bf, uint16_t *__restrict__ dz2)
{
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= (int64_t)n * NH2) return;
    const int r = (int)(e / NH2), k = (int)(e % NH2);
    const uint16_t h = h2[e];
    const bool pos = h != 0 && !(h & 0x8000u);
    dz2[e] = pos ? to_bf16(from_bf16(g[r]) * from_bf16(w3bf[k])) : (uint16_t)0;
}

// The column sums of the backward pass over the rows of split z = blockIdx.x
// (kchunk rows), fp32, rows ascending: db1 = colsum dz1, db2 = colsum dz2, dw3
// = g^T h2, db3 = sum g, into the split's partial gradient.  One thread a
// column walking every row took 3,034 us for 4,096 rows (three launches of one
// or two workgroups, a chain of dependent loads); a split's 128 rows, 8 loads
// in flight, take 9 us.
__global__ __launch_bounds__(256) void colsums_kernel(const uint16_t *__restrict__ dz1, const uint16_t *__restrict__ dz2,
                                                      const uint16_t *__restrict__ h2, const uint16_t *__restrict__ gy,
                                                      int rows, int kchunk, float *__restrict__ part)
{
    static_assert(NH1 == 256 && NH2 == 128, "a thread a column of dz1; dz2 and h2 half the workgroup each");
    const int t = threadIdx.x;
    const int lo = blockIdx.x * kchunk, hi = min(rows, lo + kchunk);
    float *out = part + (int64_t)blockIdx.x * NPARAM;
    const bool head = t >= NH2;
    const int c = head ? t - NH2 : t;
    const uint16_t *v2 = head ? h2 : dz2;
    float s1 = 0.f, s2 = 0.f, s3 = 0.f;
#pragma unroll 8
    for (int r = lo; r < hi; ++r) {
        const float g = from_bf16(gy[r]);
        const float x = from_bf16(v2[(int64_t)r * NH2 + c]);
        s1 += from_bf16(dz1[(int64_t)r * NH1 + t]);
        s2 += head ? x * g : x;
        s3 += g;
    }
    out[OFF_B1 + t] = s1;
    out[(head ? OFF_W3 : OFF_B2) + c] = s2;
    if (t == 0) out[OFF_B3] = s3;
}

// g = the sum of the splits' partial gradients, splits ascending
__global__ void grad_reduce_kernel(const float *__restrict__ part, int nsplit, float *__restrict__ g)
{
    const int x = blockIdx.x * blockDim.x + threadIdx.x;
    if (x >= NPARAM) return;
    float s = 0.f;
#pragma unroll 8
    for (int z = 0; z < nsplit; ++z) s += part[(int64_t)z * NPARAM + x];
    g[x] = s;
}

// Adam on the fp32 master weights, then the bf16 copies
__global__ void adam_kernel(float *__restrict__ p, float *__restrict__ m, float *__restrict__ v,
                            const float *__restrict__ g, uint16_t *__restrict__ wbf, float lr, float b1, float b2,
                            float c1, float c2, float eps, float wd)
{
    const int x = blockIdx.x * blockDim.x + threadIdx.x;
    if (x >= NPARAM) return;
    const float gx = g[x];
    const float mx = b1 * m[x] + (1.f - b1) * gx;
    const float vx = b2 * v[x] + (1.f - b2) * gx * gx;
    m[x] = mx;
    v[x] = vx;
    float px = p[x];
    px -= lr * ((mx / c1) / (sqrtf(vx / c2) + eps) + wd * px);
    p[x] = px;
    int bx = -1;
    if (x < OFF_B1) bx = BOFF_W1 + x;
    else if (x >= OFF_W2 && x < OFF_B2) bx = BOFF_W2 + (x - OFF_W2);
    else if (x >= OFF_W3 && x < OFF_B3) bx = BOFF_W3 + (x - OFF_W3);
    if (bx >= 0) wbf[bx] = to_bf16(px);
}

__global__ void refresh_bf16_kernel(const float *__restrict__ p, uint16_t *__restrict__ wbf)
{
    const int x = blockIdx.x * blockDim.x + threadIdx.x;
    if (x >= NBF) return;
    int px;
    if (x < BOFF_W2) px = OFF_W1 + x;
    else if (x < BOFF_W3) px = OFF_W2 + (x - BOFF_W2);
    else px = OFF_W3 + (x - BOFF_W3);
    wbf[x] = to_bf16(p[px]);
}

// band = max(min_band, ceil(2^(y + delta)))
__global__ void band_kernel(const float *__restrict__ y, uint64_t n, float delta, uint32_t min_band,
                            uint32_t *__restrict__ band)
{
    const uint64_t x = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (x >= n) return;
    float e = y[x] + delta;
    e = e > 30.f ? 30.f : e;
    const uint32_t w = (uint32_t)ceilf(exp2f(e));
    band[x] = w > min_band ? w : min_band;
}

}  // namespace
}  // namespace mh

using namespace mh;

struct mh_mlp {
    mh_context *ctx = nullptr;
    DevBuf p, m, v, g, wbf;
    DevBuf h1, h2, y, gy, dz1, dz2, loss, idx;
    DevBuf part;          // partial gradients, one a split of the batch's rows
    uint64_t cap = 0;     // batch rows the activation buffers hold
    uint64_t step = 0;
    uint64_t seed = 0;
};

namespace {

int mlp_reserve(mh_mlp *n, uint64_t rows)
{
    if (rows <= n->cap) return MH_OK;
    int rc;
    if ((rc = n->h1.ensure(rows * NH1 * 2 + 64)) != MH_OK) return rc;
    if ((rc = n->h2.ensure(rows * NH2 * 2 + 64)) != MH_OK) return rc;
    if ((rc = n->y.ensure(rows * 4 + 64)) != MH_OK) return rc;
    if ((rc = n->gy.ensure(rows * 2 + 64)) != MH_OK) return rc;
    if ((rc = n->dz1.ensure(rows * NH1 * 2 + 64)) != MH_OK) return rc;
    if ((rc = n->dz2.ensure(rows * NH2 * 2 + 64)) != MH_OK) return rc;
    n->cap = rows;
    return MH_OK;
}

// Rows of a split of the weight gradients' K (= the batch's rows): 128, so that
// a 2,048-row training batch gives dW1 320 workgroups and dW2 128, and at most
// 64 splits (65,536 rows: 1,024 rows each).
int grad_kchunk(int rows)
{
    const int per = (rows + 63) / 64;
    return std::max(128, (per + GK - 1) / GK * GK);
}

template <bool AKC, bool AF32, bool BKC, bool BF32>
void launch_gemm(hipStream_t st, int M, int N, int K, int kchunk, const Operand &A, const Operand &B, const Epilogue &E)
{
    hipLaunchKernelGGL((gemm_kernel<AKC, AF32, BKC, BF32>),
                       dim3((M + GT - 1) / GT, (N + GT - 1) / GT, (K + kchunk - 1) / kchunk), dim3(256), 0, st, M, N, K,
                       kchunk, A, B, E);
}

// forward over `rows` examples (features x rows, or x[idx[r]]): h1, h2, y
void mlp_forward_rows(mh_mlp *n, const float *x, const uint32_t *idx, int rows)
{
    hipStream_t st = n->ctx->stream;
    const float *p = n->p.as<float>();
    const uint16_t *wbf = n->wbf.as<uint16_t>();
    Operand X{x, NIN, idx};
    Operand W1t{wbf + BOFF_W1, NIN, nullptr};          // (k = in, n = out) at W1[out][in]
    Epilogue e1{EPI_BIAS_RELU_BF16, p + OFF_B1, nullptr, 0, n->h1.as<uint16_t>(), NH1, nullptr, 0};
    launch_gemm<true, true, true, false>(st, rows, NH1, NIN, NIN, X, W1t, e1);
    Operand H1{n->h1.as<uint16_t>(), NH1, nullptr};
    Operand W2t{wbf + BOFF_W2, NH1, nullptr};
    Epilogue e2{EPI_BIAS_RELU_BF16, p + OFF_B2, nullptr, 0, n->h2.as<uint16_t>(), NH2, nullptr, 0};
    launch_gemm<true, false, true, false>(st, rows, NH2, NH1, NH1, H1, W2t, e2);
    hipLaunchKernelGGL(head_kernel, dim3((rows + 255) / 256), dim3(256), 0, st, n->h2.as<uint16_t>(), rows,
                       wbf + BOFF_W3, p + OFF_B3, n->y.as<float>());
}

// loss and gradients of one batch into n->g (fp32, flat parameter layout)
int mlp_backward_rows(mh_mlp *n, const float *x, const float *target, const uint32_t *idx, int rows)
{
    hipStream_t st = n->ctx->stream;
    const uint16_t *wbf = n->wbf.as<uint16_t>();
    uint16_t *gy = n->gy.as<uint16_t>(), *h1 = n->h1.as<uint16_t>(), *h2 = n->h2.as<uint16_t>();
    uint16_t *dz1 = n->dz1.as<uint16_t>(), *dz2 = n->dz2.as<uint16_t>();
    const int kc = grad_kchunk(rows), ns = (rows + kc - 1) / kc;
    int rc;
    if ((rc = n->part.ensure((size_t)ns * NPARAM * 4 + 64)) != MH_OK) return rc;
    float *part = n->part.as<float>();
    hipLaunchKernelGGL(loss_kernel, dim3(1), dim3(256), 0, st, n->y.as<float>(), target, idx, rows, gy,
                       n->loss.as<float>());
    hipLaunchKernelGGL(head_back_kernel, dim3((unsigned)(((int64_t)rows * NH2 + 255) / 256)), dim3(256), 0, st, gy,
                       h2, rows, wbf + BOFF_W3, dz2);
    // layer 2: dW2 = dz2^T h1 (M = NH2, N = NH1, K = rows), dz1
    {
        Operand A{dz2, NH2, nullptr};             // (m = out2, k = row) at dz2[row][out2]
        Operand B{h1, NH1, nullptr};              // (k = row, n = in2) at h1[row][in2]
        Epilogue e{EPI_F32, nullptr, part + OFF_W2, NPARAM, nullptr, NH1, nullptr, 0};
        launch_gemm<false, false, false, false>(st, NH2, NH1, rows, kc, A, B, e);
    }
    {
        Operand A{dz2, NH2, nullptr};             // (m = row, k = out2)
        Operand B{wbf + BOFF_W2, NH1, nullptr};   // (k = out2, n = in2) at W2[out2][in2]
        Epilogue e{EPI_MASK_BF16, nullptr, nullptr, 0, dz1, NH1, h1, NH1};
        launch_gemm<true, false, false, false>(st, rows, NH1, NH2, NH2, A, B, e);
    }
    // layer 1: dW1 = dz1^T x (M = NH1, N = NIN, K = rows)
    {
        Operand A{dz1, NH1, nullptr};
        Operand B{x, NIN, idx};                   // (k = row, n = feature) at x[idx[row]][feature]
        Epilogue e{EPI_F32, nullptr, part + OFF_W1, NPARAM, nullptr, NIN, nullptr, 0};
        launch_gemm<false, false, false, true>(st, NH1, NIN, rows, kc, A, B, e);
    }
    // biases and the head: dw3 = g^T h2, db3 = sum g
    hipLaunchKernelGGL(colsums_kernel, dim3(ns), dim3(256), 0, st, dz1, dz2, h2, gy, rows, kc, part);
    hipLaunchKernelGGL(grad_reduce_kernel, dim3((NPARAM + 255) / 256), dim3(256), 0, st, part, ns, n->g.as<float>());
    return MH_OK;
}

}  // namespace

extern "C" {

int mh_gap_features_device(mh_context *ctx, const uint8_t *d_a, const uint8_t *d_b, const mh_dp_job *jobs,
                           uint64_t njobs, float *d_feat)
{
    MH_CHECK(ctx, MH_ERR_INVALID, "null context");
    if (njobs == 0) return MH_OK;
    MH_CHECK(jobs && d_a && d_b && d_feat, MH_ERR_INVALID, "null argument");
    MH_CHECK(njobs < (1ull << 31), MH_ERR_INVALID, "too many jobs in one call");
    MH_HIP(hipSetDevice(ctx->device));
    int rc;
    if ((rc = ctx->ml_jobs.ensure(njobs * sizeof(mh_dp_job) + 64)) != MH_OK) return rc;
    MH_HIP(hipMemcpyAsync(ctx->ml_jobs.ptr, jobs, njobs * sizeof(mh_dp_job), hipMemcpyHostToDevice, ctx->stream));
    {
        TimedLaunch tl(ctx, "band_features");
        hipLaunchKernelGGL(features_kernel, dim3((unsigned)njobs), dim3(256), 0, ctx->stream, d_a, d_b,
                           ctx->ml_jobs.as<mh_dp_job>(), njobs, d_feat);
        MH_HIP(hipGetLastError());
    }
    MH_HIP(hipStreamSynchronize(ctx->stream));
    return MH_OK;
}

int mh_mlp_create(mh_context *ctx, uint64_t seed, mh_mlp **out)
{
    MH_CHECK(ctx && out, MH_ERR_INVALID, "null argument");
    MH_HIP(hipSetDevice(ctx->device));
    mh_mlp *n = new mh_mlp();
    n->ctx = ctx;
    n->seed = seed;
    int rc;
    if ((rc = n->p.ensure(NPARAM * 4 + 64)) != MH_OK || (rc = n->m.ensure(NPARAM * 4 + 64)) != MH_OK ||
        (rc = n->v.ensure(NPARAM * 4 + 64)) != MH_OK || (rc = n->g.ensure(NPARAM * 4 + 64)) != MH_OK ||
        (rc = n->wbf.ensure(NBF * 2 + 64)) != MH_OK || (rc = n->loss.ensure(64)) != MH_OK) {
        delete n;
        return rc;
    }
    // He-uniform weights, zero biases (mt19937_64 from the seed)
    std::vector<float> h(NPARAM, 0.f);
    std::mt19937_64 rng(seed);
    auto fill = [&](int off, int fan_out, int fan_in) {
        const float lim = std::sqrt(6.0f / (float)fan_in);
        std::uniform_real_distribution<float> u(-lim, lim);
        for (int x = 0; x < fan_out * fan_in; ++x) h[off + x] = u(rng);
    };
    fill(OFF_W1, NH1, NIN);
    fill(OFF_W2, NH2, NH1);
    fill(OFF_W3, 1, NH2);
    *out = n;
    return mh_mlp_set_params(ctx, n, h.data());
}

void mh_mlp_free(mh_mlp *n)
{
    delete n;
}

int mh_mlp_set_params(mh_context *ctx, mh_mlp *n, const float *params)
{
    MH_CHECK(ctx && n && params, MH_ERR_INVALID, "null argument");
    MH_HIP(hipSetDevice(ctx->device));
    MH_HIP(hipMemcpyAsync(n->p.ptr, params, NPARAM * 4, hipMemcpyHostToDevice, ctx->stream));
    MH_HIP(hipMemsetAsync(n->m.ptr, 0, NPARAM * 4, ctx->stream));
    MH_HIP(hipMemsetAsync(n->v.ptr, 0, NPARAM * 4, ctx->stream));
    hipLaunchKernelGGL(refresh_bf16_kernel, dim3((NBF + 255) / 256), dim3(256), 0, ctx->stream, n->p.as<float>(),
                       n->wbf.as<uint16_t>());
    MH_HIP(hipGetLastError());
    MH_HIP(hipStreamSynchronize(ctx->stream));
    n->step = 0;
    return MH_OK;
}

int mh_mlp_get_params(mh_context *ctx, const mh_mlp *n, float *params)
{
    MH_CHECK(ctx && n && params, MH_ERR_INVALID, "null argument");
    MH_HIP(hipSetDevice(ctx->device));
    MH_HIP(hipMemcpyAsync(params, n->p.ptr, NPARAM * 4, hipMemcpyDeviceToHost, ctx->stream));
    MH_HIP(hipStreamSynchronize(ctx->stream));
    return MH_OK;
}

int mh_mlp_forward(mh_context *ctx, mh_mlp *n, const float *d_x, uint64_t rows, float *d_y)
{
    MH_CHECK(ctx && n, MH_ERR_INVALID, "null argument");
    if (rows == 0) return MH_OK;
    MH_CHECK(d_x && d_y, MH_ERR_INVALID, "null argument");
    MH_HIP(hipSetDevice(ctx->device));
    const uint64_t chunk = 65536;
    int rc;
    if ((rc = mlp_reserve(n, std::min<uint64_t>(rows, chunk))) != MH_OK) return rc;
    TimedLaunch tl(ctx, "band_mlp_forward");
    for (uint64_t r0 = 0; r0 < rows; r0 += chunk) {
        const int nr = (int)std::min<uint64_t>(chunk, rows - r0);
        mlp_forward_rows(n, d_x + r0 * NIN, nullptr, nr);
        MH_HIP(hipMemcpyAsync(d_y + r0, n->y.ptr, (size_t)nr * 4, hipMemcpyDeviceToDevice, ctx->stream));
    }
    MH_HIP(hipGetLastError());
    return MH_OK;
}

int mh_mlp_grad(mh_context *ctx, mh_mlp *n, const float *d_x, const float *d_t, uint64_t rows, float *grads,
                float *loss)
{
    MH_CHECK(ctx && n && d_x && d_t && grads, MH_ERR_INVALID, "null argument");
    MH_CHECK(rows > 0 && rows <= 65536, MH_ERR_INVALID, "gradient batch must hold 1..65536 rows");
    MH_HIP(hipSetDevice(ctx->device));
    int rc;
    if ((rc = mlp_reserve(n, rows)) != MH_OK) return rc;
    mlp_forward_rows(n, d_x, nullptr, (int)rows);
    if ((rc = mlp_backward_rows(n, d_x, d_t, nullptr, (int)rows)) != MH_OK) return rc;
    MH_HIP(hipGetLastError());
    MH_HIP(hipMemcpyAsync(grads, n->g.ptr, NPARAM * 4, hipMemcpyDeviceToHost, ctx->stream));
    float l = 0.f;
    MH_HIP(hipMemcpyAsync(&l, n->loss.ptr, 4, hipMemcpyDeviceToHost, ctx->stream));
    MH_HIP(hipStreamSynchronize(ctx->stream));
    if (loss) *loss = l;
    return MH_OK;
}

int mh_mlp_train(mh_context *ctx, mh_mlp *n, const float *d_x, const float *d_t, uint64_t rows,
                 const mh_mlp_train_opts *opt, float *epoch_loss)
{
    MH_CHECK(ctx && n && d_x && d_t && opt, MH_ERR_INVALID, "null argument");
    MH_CHECK(rows > 0 && rows < (1ull << 32), MH_ERR_INVALID, "training set must hold 1..2^32-1 rows");
    MH_CHECK(opt->batch > 0 && opt->batch <= 65536 && opt->epochs > 0, MH_ERR_INVALID, "bad batch or epochs");
    MH_HIP(hipSetDevice(ctx->device));
    int rc;
    const uint32_t bs = opt->batch;
    if ((rc = mlp_reserve(n, bs)) != MH_OK) return rc;
    if ((rc = n->idx.ensure(rows * 4 + 64)) != MH_OK) return rc;
    std::vector<uint32_t> perm(rows);
    for (uint64_t r = 0; r < rows; ++r) perm[r] = (uint32_t)r;
    std::mt19937_64 rng(opt->seed);
    DevBuf lossbuf;
    const uint64_t nb = rows / bs;   // full batches only
    MH_CHECK(nb > 0, MH_ERR_INVALID, "training set smaller than one batch");
    if ((rc = lossbuf.ensure(nb * 4 + 64)) != MH_OK) return rc;
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    TimedLaunch tl(ctx, "band_mlp_train");
    for (uint32_t ep = 0; ep < opt->epochs; ++ep) {
        std::shuffle(perm.begin(), perm.end(), rng);
        MH_HIP(hipMemcpyAsync(n->idx.ptr, perm.data(), rows * 4, hipMemcpyHostToDevice, ctx->stream));
        for (uint64_t bi = 0; bi < nb; ++bi) {
            const uint32_t *idx = n->idx.as<uint32_t>() + bi * bs;
            mlp_forward_rows(n, d_x, idx, (int)bs);
            if ((rc = mlp_backward_rows(n, d_x, d_t, idx, (int)bs)) != MH_OK) return rc;
            ++n->step;
            // cosine decay of the learning rate over the run
            const double prog = ((double)ep * nb + bi) / ((double)opt->epochs * nb);
            const float lr = (float)(opt->lr * 0.5 * (1.0 + std::cos(3.14159265358979 * prog)));
            const float c1 = 1.f - std::pow(b1, (float)n->step), c2 = 1.f - std::pow(b2, (float)n->step);
            hipLaunchKernelGGL(adam_kernel, dim3((NPARAM + 255) / 256), dim3(256), 0, ctx->stream,
                               n->p.as<float>(), n->m.as<float>(), n->v.as<float>(), n->g.as<float>(),
                               n->wbf.as<uint16_t>(), lr, b1, b2, c1, c2, eps, opt->weight_decay);
            MH_HIP(hipMemcpyAsync(lossbuf.as<float>() + bi, n->loss.ptr, 4, hipMemcpyDeviceToDevice, ctx->stream));
        }
        MH_HIP(hipGetLastError());
        if (epoch_loss) {
            std::vector<float> l(nb);
            MH_HIP(hipMemcpyAsync(l.data(), lossbuf.ptr, nb * 4, hipMemcpyDeviceToHost, ctx->stream));
            MH_HIP(hipStreamSynchronize(ctx->stream));
            double s = 0;
            for (float v : l) s += v;
            epoch_loss[ep] = (float)(s / nb);
        }
    }
    MH_HIP(hipStreamSynchronize(ctx->stream));
    return MH_OK;
}

int mh_band_predict(mh_context *ctx, mh_mlp *n, const float *d_feat, uint64_t rows, float delta,
                    uint32_t min_band, uint32_t *bands)
{
    MH_CHECK(ctx && n, MH_ERR_INVALID, "null argument");
    if (rows == 0) return MH_OK;
    MH_CHECK(d_feat && bands, MH_ERR_INVALID, "null argument");
    int rc;
    if ((rc = ctx->ml_y.ensure(rows * 8 + 64)) != MH_OK) return rc;
    float *y = ctx->ml_y.as<float>();
    uint32_t *b = reinterpret_cast<uint32_t *>(y + rows);
    if ((rc = mh_mlp_forward(ctx, n, d_feat, rows, y)) != MH_OK) return rc;
    hipLaunchKernelGGL(band_kernel, dim3((unsigned)((rows + 255) / 256)), dim3(256), 0, ctx->stream, y, rows, delta,
                       min_band, b);
    MH_HIP(hipGetLastError());
    MH_HIP(hipMemcpyAsync(bands, b, rows * 4, hipMemcpyDeviceToHost, ctx->stream));
    MH_HIP(hipStreamSynchronize(ctx->stream));
    return MH_OK;
}

}  // extern "C"
