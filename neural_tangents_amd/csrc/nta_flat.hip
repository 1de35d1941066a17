// Fully-connected networks on flat inputs: Dense [+ activation] stages on
// [N, D] rows, i.e. 1x1 states.  The input covariance is a plain Gram matrix
// and everything after it is pointwise in the pair, so one launch computes a
// tile of the Gram on FP32 MFMA and runs the whole network in its epilogue.
//
// nta_flat_tables runs the same products on the diagonal blocks and leaves
// every activation's normalisers q.  Both sum over D in the same order --
// four partial sums over the 16-wide chunks c = 0, 1, 2, 3 mod 4, added
// pairwise -- so that the Gram entry of a row with an equal row is its q bit
// for bit, and the activation's q1 q2 - c^2 is exactly 0 there.
#include "nta_common.h"

namespace nta {

constexpr int kFlatMaxStages = 48;    // the stage table travels in kernargs

typedef float f32x16 __attribute__((ext_vector_type(16)));

struct FlatStage {
  int conv, act;          // act: 0 none, else NTA_RELU | NTA_ACT_*
  float w, b, k1, k0;
};
struct FlatPlan {
  int nstage, n1, n2, nimg, D, sym, ntk;
  float inv_d;
  double a, b, c, d, e;
  FlatStage s[kFlatMaxStages];
};

__device__ __forceinline__ const float* flat_row(const FlatPlan& P,
                                                 const float* x1,
                                                 const float* x2, int i) {
  return i < P.n1 ? x1 + (long long)i * P.D
                  : x2 + (long long)(i - P.n1) * P.D;
}

constexpr int kFlatK = 64;                  // columns staged at a time
constexpr int kFlatPitch = kFlatK + 4;      // LDS row pitch (floats)

__device__ __forceinline__ f32x16 zero16() {
  f32x16 v;
#pragma unroll
  for (int r = 0; r < 16; ++r) v[r] = 0.0f;
  return v;
}

// The next kFlatK columns of 64 T rows, on their way from memory to LDS
// through registers: 16 lanes read 256 contiguous bytes of a row.
template <int T, bool VEC>
struct FlatStager {
  static constexpr int ROWS = 64 * T, NV = ROWS * 16 / 256;
  static constexpr int PF = T == 1 ? 2 : 1;      // blocks in flight
  const float* row[NV];
  float4 v[PF][NV];
  template <typename RowPtr>
  __device__ __forceinline__ void init(RowPtr ptr) {
#pragma unroll
    for (int q = 0; q < NV; ++q) row[q] = ptr((threadIdx.x >> 4) + 16 * q);
  }
  __device__ __forceinline__ void load(int p, int k0, int D) {
    const int k = k0 + 4 * (threadIdx.x & 15);
#pragma unroll
    for (int q = 0; q < NV; ++q) {
      v[p][q] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      if constexpr (VEC) {
        if (k < D) v[p][q] = *reinterpret_cast<const float4*>(row[q] + k);
      } else {
        if (k < D) v[p][q].x = row[q][k];
        if (k + 1 < D) v[p][q].y = row[q][k + 1];
        if (k + 2 < D) v[p][q].z = row[q][k + 2];
        if (k + 3 < D) v[p][q].w = row[q][k + 3];
      }
    }
  }
  __device__ __forceinline__ void store(int p, float* __restrict__ buf) const {
#pragma unroll
    for (int q = 0; q < NV; ++q)
      *reinterpret_cast<float4*>(buf +
                                 ((threadIdx.x >> 4) + 16 * q) * kFlatPitch +
                                 4 * (threadIdx.x & 15)) = v[p][q];
  }
};

// acc += chunk ch (16 columns) of the staged rows a and b of this lane: the
// lane halves hold columns 0-7 and 8-15, eight 32x32x2 products take one of
// each.
__device__ __forceinline__ void flat_mul(const float* __restrict__ buf,
                                         int ra, int rb, int ch, int half,
                                         f32x16& acc) {
  const float* pa = buf + ra * kFlatPitch + 16 * ch + 8 * half;
  const float* pb = buf + rb * kFlatPitch + 16 * ch + 8 * half;
  const float4 a0 = *reinterpret_cast<const float4*>(pa);
  const float4 a1 = *reinterpret_cast<const float4*>(pa + 4);
  const float4 b0 = *reinterpret_cast<const float4*>(pb);
  const float4 b1 = *reinterpret_cast<const float4*>(pb + 4);
  const float a[8] = {a0.x, a0.y, a0.z, a0.w, a1.x, a1.y, a1.z, a1.w};
  const float b[8] = {b0.x, b0.y, b0.z, b0.w, b1.x, b1.y, b1.z, b1.w};
#pragma unroll
  for (int q = 0; q < 8; ++q)
    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[q], b[q], acc, 0, 0, 0);
}

// Runs body(buffer) on every staged block of kFlatK columns; two buffers of
// 64 T rows, the next block's loads in flight during the current one.
template <int T, bool VEC, typename RowPtr, typename Body>
__device__ __forceinline__ void flat_sweep(int D, float* __restrict__ bufs,
                                           RowPtr ptr, Body body) {
  constexpr int BUF = 64 * T * kFlatPitch;
  using St = FlatStager<T, VEC>;
  St st;
  st.init(ptr);
#pragma unroll
  for (int p = 0; p < St::PF; ++p) st.load(p, p * kFlatK, D);
  // two buffers: the one written now was last read before the previous
  // barrier
  for (int k0 = 0; k0 < D; k0 += 2 * kFlatK) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int k = k0 + h * kFlatK, p = h % St::PF;
      if (k < D) {
        float* buf = bufs + h * BUF;
        st.store(p, buf);
        st.load(p, k + St::PF * kFlatK, D);
        __syncthreads();
        body(buf);
      }
    }
  }
  __syncthreads();
}

// 32x32 block of the Gram by the four waves of a workgroup, wave w the
// chunks c = w mod 4; the sum of the parts lands in tile[32][33].  bufs:
// staging space (2 x 64 rows), reused for the parts.
template <bool VEC, typename RowPtr>
__device__ __forceinline__ void flat_block32(int D, RowPtr ptr,
                                             float* __restrict__ bufs,
                                             float* __restrict__ tile) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int col = lane & 31, half = lane >> 5;
  f32x16 acc = zero16();
  flat_sweep<1, VEC>(D, bufs, ptr, [&](const float* buf) {
    flat_mul(buf, col, 32 + col, wave, half, acc);
  });
  float* part = bufs;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int m = 8 * (r >> 2) + 4 * half + (r & 3);
    part[(wave * 32 + m) * 33 + col] = acc[r];
  }
  __syncthreads();
  for (int q = threadIdx.x; q < 1024; q += 256) {
    const int o = (q >> 5) * 33 + (q & 31);
    constexpr int W = 32 * 33;
    tile[o] = (part[o] + part[W + o]) + (part[2 * W + o] + part[3 * W + o]);
  }
  __syncthreads();
}

// Normalisers of every stage ([stage][image]) and the self covariances.
template <bool VEC>
__global__ __launch_bounds__(256) void k_flat_tables(
    FlatPlan P, const float* __restrict__ x1, const float* __restrict__ x2,
    float* __restrict__ q, float* __restrict__ cov) {
  __shared__ __align__(16) float bufs[2 * 64 * kFlatPitch];
  float* tile = bufs + 4 * 32 * 33;
  const int i0 = blockIdx.x * 32;
  const int col = threadIdx.x & 31;
  const int i = i0 + col < P.nimg ? i0 + col : P.nimg - 1;
  flat_block32<VEC>(
      P.D,
      [&](int r) {
        r &= 31;
        return flat_row(P, x1, x2, i0 + r < P.nimg ? i0 + r : P.nimg - 1);
      },
      bufs, tile);
  if (threadIdx.x >= 32 || i0 + col >= P.nimg) return;
  float n = tile[col * 33 + col] * P.inv_d;
  for (int s = 0; s < P.nstage; ++s) {
    const FlatStage S = P.s[s];
    if (S.conv) n = fmaf(S.w, n, S.b);
    if (S.act) {
      q[(long long)s * P.nimg + i] = n;
      float ds;
      n = act_map(S.act, n, n, n, S.k1, S.k0, &ds);
    }
  }
  if (cov) cov[i] = (float)(P.a * n + P.b);
}

// relu_map for many elements: with s^2 = q1 q2 - c^2 (one rounding, exactly 0
// for equal rows) and h = sqrt(q1 q2), 1 - |rho| = s^2 / (h (h + |c|)) has no
// cancellation, so theta = sqrt(1 - |rho|) P(|rho|) is accurate up to
// |rho| = 1 with one reciprocal and two square roots (about 30 instructions
// against 110 for atan2f and the IEEE square root).  a, b: (q, sqrt q).  Its
// hardware root and reciprocal take no subnormal s^2 or h^2: flat_plain.
__device__ __forceinline__ float flat_relu(float c, float2 a, float2 b,
                                           float k1, float k0, float* ds) {
  const float d = fmaxf(prod_minus_sq(a.x, b.x, c), 0.0f);
  const float h = a.y * b.y;
  const float g = h * (h + fabsf(c));
  // q1 q2 = 0: theta = pi / 2
  const float u = g > 0.0f ? fminf(d * __builtin_amdgcn_rcpf(g), 1.0f) : 1.0f;
  const float th = acos_pos(1.0f - u, u);
  const float pm = 0.5f * kPi + copysignf(0.5f * kPi - th, c);
  *ds = fmaf(k1 * kInv2Pi, pm, k0);
  return fmaf(k1 * kInv2Pi, fmaf(pm, c, fsqrt(d)), k0 * c);
}

// Is a normaliser where flat_relu's products stay normal numbers (or 0, which
// it treats apart)?  Otherwise a tile takes relu_map.
__device__ __forceinline__ bool flat_plain(float q) {
  return !(q > 0.0f && q < 0x1p-40f) && !(q > 0x1p40f);
}

// The network on E elements per thread.  qa(s, e), qb(s, e): normalisers
// (q, sqrt q).  plain: flat_plain of all of them.
template <int E, typename QA, typename QB>
__device__ __forceinline__ void flat_chain(const FlatPlan& P, bool plain,
                                           float (&n)[E], float (&t)[E],
                                           QA qa, QB qb) {
#pragma unroll
  for (int e = 0; e < E; ++e) {
    n[e] *= P.inv_d;
    t[e] = 0.0f;
  }
  for (int s = 0; s < P.nstage; ++s) {
    const FlatStage S = P.s[s];
    if (S.conv) {
#pragma unroll
      for (int e = 0; e < E; ++e) {
        n[e] = fmaf(S.w, n[e], S.b);
        t[e] = fmaf(S.w, t[e], n[e]);
      }
    }
    if (S.act == NTA_RELU && plain) {
#pragma unroll
      for (int e = 0; e < E; ++e) {
        float ds;
        n[e] = flat_relu(n[e], qa(s, e), qb(s, e), S.k1, S.k0, &ds);
        t[e] *= ds;
      }
    } else if (S.act) {
#pragma unroll
      for (int e = 0; e < E; ++e) {
        float ds;
        n[e] = act_map(S.act, n[e], qa(s, e).x, qb(s, e).x, S.k1, S.k0, &ds);
        t[e] *= ds;
      }
    }
  }
}

// T = 1: a 32x32 tile, the four waves split D.  T = 2: a 64x64 tile, a wave
// per 32x32 quadrant with the four partial sums in registers.  Bound: FP32
// MFMA and, for few stages of D, the latency of a stage.  1,000 rows of 784
// with themselves, 3 ReLU layers: 25 us (and 8 us for the normalisers), where
// one thread per pair took 2.92 ms for the Gram, 0.29 ms for the rows' own
// products and 0.06 ms for the layers; 4,000 rows: 0.27 ms.
template <int T, bool VEC>
__global__ __launch_bounds__(256) void k_flat_pairs(
    FlatPlan P, const float* __restrict__ x1, const float* __restrict__ x2,
    const float* __restrict__ q, float* __restrict__ out_n,
    float* __restrict__ out_t, long long ld) {
  constexpr int B = 32 * T, LP = B + 1;
  __shared__ __align__(16) float bufs[2 * 64 * T * kFlatPitch];
  // after the product: n and t of the tile (T = 1: flat_block32's parts
  // first, below tile)
  float* part = bufs;
  float* tile = bufs + 4 * 32 * 33;
  static_assert(T == 2 || 4 * 32 * 33 + B * LP <= 2 * 64 * kFlatPitch, "");
  static_assert(T == 1 || B * LP <= 4 * 32 * 33, "");
  const int cols = P.sym ? P.n1 : P.n2;
  const int tj = (cols + B - 1) / B;
  const int bi = blockIdx.x / tj, bj = blockIdx.x - bi * tj;
  if (P.sym && bj < bi) return;        // mirrored from the upper triangle
  const int i0 = bi * B, j0 = bj * B;
  const int joff = P.sym ? 0 : P.n1;   // image index of column 0
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int col = lane & 31, half = lane >> 5;
  auto img_i = [&](int r) { return i0 + r < P.n1 ? i0 + r : P.n1 - 1; };
  auto img_j = [&](int c) {
    return joff + (j0 + c < cols ? j0 + c : cols - 1);
  };
  // The normalisers of the tile's rows and columns, in flight beside the
  // product: qs[stage][row | B + column].
  extern __shared__ float2 qs[];
  __shared__ int odd;
  if (threadIdx.x == 0) odd = 0;
  __syncthreads();
  for (int k = threadIdx.x; k < P.nstage * 2 * B; k += 256) {
    const int s = k / (2 * B), o = k - s * (2 * B);
    if (P.s[s].act) {
      const float v =
          q[(long long)s * P.nimg + (o < B ? img_i(o) : img_j(o - B))];
      qs[k] = make_float2(v, fsqrt(fmaxf(v, 0.0f)));
      if (!flat_plain(v)) odd = 1;
    }
  }
  // staged rows: the tile's rows, then its columns
  auto row_ptr = [&](int r) {
    return flat_row(P, x1, x2, r < B ? img_i(r) : img_j(r - B));
  };
  // element (r, c) of the tile -> tile (n) and part (t)
  if constexpr (T == 1) {
    flat_block32<VEC>(P.D, row_ptr, bufs, tile);
    float n[4], t[4];
    const int c = threadIdx.x & 31, r0 = threadIdx.x >> 5;
#pragma unroll
    for (int e = 0; e < 4; ++e) n[e] = tile[(r0 + 8 * e) * LP + c];
    flat_chain<4>(
        P, odd == 0, n, t,
        [&](int s, int e) { return qs[s * 2 * B + r0 + 8 * e]; },
        [&](int s, int) { return qs[s * 2 * B + B + c]; });
    __syncthreads();
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      tile[(r0 + 8 * e) * LP + c] = n[e];
      part[(r0 + 8 * e) * LP + c] = t[e];
    }
  } else {
    const int wi = 32 * (wave >> 1), wj = 32 * (wave & 1);
    f32x16 acc[4] = {zero16(), zero16(), zero16(), zero16()};
    flat_sweep<2, VEC>(P.D, bufs, row_ptr, [&](const float* buf) {
#pragma unroll
      for (int ch = 0; ch < 4; ++ch)
        flat_mul(buf, wi + col, B + wj + col, ch, half, acc[ch]);
    });
    float n[16], t[16];
#pragma unroll
    for (int r = 0; r < 16; ++r)
      n[r] = (acc[0][r] + acc[1][r]) + (acc[2][r] + acc[3][r]);
    auto row = [&](int r) { return wi + 8 * (r >> 2) + 4 * half + (r & 3); };
    flat_chain<16>(
        P, odd == 0, n, t,
        [&](int s, int r) { return qs[s * 2 * B + row(r)]; },
        [&](int s, int) { return qs[s * 2 * B + B + wj + col]; });
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      tile[row(r) * LP + wj + col] = n[r];
      part[row(r) * LP + wj + col] = t[r];
    }
  }
  __syncthreads();
  // Rows of the tile, and for the upper triangle its columns as the rows of
  // the mirror image.
  auto put = [&](long long r, long long c, float n, float t) {
    out_n[r * ld + c] = (float)(P.a * n + P.b);
    if (P.ntk) out_t[r * ld + c] = (float)(P.c * n + P.d * t + P.e);
  };
  const bool diag = P.sym && bi == bj;
  for (int k = threadIdx.x; k < B * B; k += 256) {
    const int r = k / B, c = k - r * B;
    if (i0 + r < P.n1 && j0 + c < cols) {
      const bool lower = diag && c < r;     // exactly symmetric
      const int o = lower ? c * LP + r : r * LP + c;
      put(i0 + r, j0 + c, tile[o], part[o]);
    }
    if (P.sym && !diag && i0 + c < P.n1 && j0 + r < cols)
      put(j0 + r, i0 + c, tile[c * LP + r], part[c * LP + r]);
  }
}

static int flat_plan(const char* who, FlatPlan& P, const float* x1,
                     const float* x2, int n1, int n2, int D, int nstage,
                     const int* desc, const float* wb) {
  if (n1 < 0 || n2 < 0 || D <= 0 || nstage <= 0 || nstage > kFlatMaxStages ||
      !desc || !wb)
    return set_error(NTA_EINVAL, "%s: bad n1=%d n2=%d D=%d nstage=%d (<= %d)",
                     who, n1, n2, D, nstage, kFlatMaxStages);
  if ((n1 > 0 && !x1) || (n2 > 0 && !x2))
    return set_error(NTA_EINVAL, "%s: null pointer", who);
  P = FlatPlan();
  P.nstage = nstage;
  P.n1 = n1;
  P.n2 = n2;
  P.nimg = n1 + n2;
  P.D = D;
  P.inv_d = 1.0f / (float)D;
  for (int s = 0; s < nstage; ++s) {
    FlatStage& S = P.s[s];
    S.conv = (desc[s] & NTA_CONV) ? 1 : 0;
    S.act = (desc[s] & NTA_RELU)
                ? desc[s] & (NTA_RELU | NTA_ACT_ERF | NTA_ACT_GELU)
                : 0;
    S.w = wb[4 * s];
    S.b = wb[4 * s + 1];
    S.k1 = wb[4 * s + 2];
    S.k0 = wb[4 * s + 3];
  }
  return NTA_OK;
}

static bool flat_vec(const float* x1, const float* x2, int D) {
  return D % 4 == 0 && (reinterpret_cast<uintptr_t>(x1) & 15) == 0 &&
         (reinterpret_cast<uintptr_t>(x2) & 15) == 0;
}

}  // namespace nta

using namespace nta;

extern "C" int nta_flat_tables(const float* x1, const float* x2, int n1,
                               int n2, int D, int nstage,
                               const int* stage_flags, const float* stage_wb,
                               double a, double b, float* q, float* cov,
                               void* stream) {
  FlatPlan P;
  int rc = flat_plan("nta_flat_tables", P, x1, x2, n1, n2, D, nstage,
                     stage_flags, stage_wb);
  if (rc) return rc;
  if (P.nimg == 0) return NTA_OK;
  if (!q) return set_error(NTA_EINVAL, "nta_flat_tables: null pointer");
  P.a = a;
  P.b = b;
  const dim3 grid((P.nimg + 31) / 32);
  if (flat_vec(x1, x2, D))
    hipLaunchKernelGGL(k_flat_tables<true>, grid, dim3(256), 0,
                       (hipStream_t)stream, P, x1, x2, q, cov);
  else
    hipLaunchKernelGGL(k_flat_tables<false>, grid, dim3(256), 0,
                       (hipStream_t)stream, P, x1, x2, q, cov);
  return check_launch("nta_flat_tables");
}

extern "C" int nta_flat_pairs(const float* x1, const float* x2, int n1,
                              int n2, int D, int nstage,
                              const int* stage_flags, const float* stage_wb,
                              const float* q, int flags, double a, double b,
                              double c, double d, double e, float* out_nngp,
                              float* out_ntk, long long ld, void* stream) {
  FlatPlan P;
  int rc = flat_plan("nta_flat_pairs", P, x1, x2, n1, n2, D, nstage,
                     stage_flags, stage_wb);
  if (rc) return rc;
  P.sym = (flags & NTA_TORUS_UPPER) ? 1 : 0;
  P.ntk = (flags & NTA_NTK) ? 1 : 0;
  const int cols = P.sym ? n1 : n2;
  if (n1 == 0 || cols == 0) return NTA_OK;
  if (!q || !out_nngp || (P.ntk && !out_ntk))
    return set_error(NTA_EINVAL, "nta_flat_pairs: null pointer");
  if (ld < cols)
    return set_error(NTA_EINVAL, "nta_flat_pairs: ld=%lld < %d", ld, cols);
  P.a = a;
  P.b = b;
  P.c = c;
  P.d = d;
  P.e = e;
  auto tiles = [&](int B) {
    return (long long)((n1 + B - 1) / B) * ((cols + B - 1) / B);
  };
  // 64x64 tiles read half the rows per product; 32x32 ones put four times as
  // many waves on a small matrix.  Below two 64x64 tiles per compute unit the
  // last round of them costs more than that: 1,000 rows with themselves (136
  // tiles of 64) 25 us with 32x32 tiles.
  const bool big = tiles(64) / (P.sym ? 2 : 1) >= 512;
  const long long nb = tiles(big ? 64 : 32);
  if (nb > 0x7fffffffLL)
    return set_error(NTA_EINVAL, "nta_flat_pairs: %d x %d is too large", n1,
                     cols);
  const bool vec = flat_vec(x1, x2, D);
  const dim3 grid((unsigned)nb);
  const hipStream_t st = (hipStream_t)stream;
  const size_t lds = (size_t)nstage * 2 * (big ? 64 : 32) * sizeof(float2);
#define NTA_FLAT_GO(T_, V_)                                               \
  hipLaunchKernelGGL((k_flat_pairs<T_, V_>), grid, dim3(256), lds, st, P, \
                     x1, x2, q, out_nngp, out_ntk, ld)
  if (big) {
    if (vec) NTA_FLAT_GO(2, true);
    else NTA_FLAT_GO(2, false);
  } else {
    if (vec) NTA_FLAT_GO(1, true);
    else NTA_FLAT_GO(1, false);
  }
#undef NTA_FLAT_GO
  return check_launch("nta_flat_pairs");
}
