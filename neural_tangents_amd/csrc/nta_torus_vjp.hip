// Host side of the register-resident adjoints (nta_torus_vjp.h): launch
// shapes, the sums over partner images and the C entry points.
#include <algorithm>

#include "nta_torus_vjp.h"

namespace nta {

// acc[image * pitch + q] += the image's shares of the pairs [p0, p0 + np), in
// the order of the pairs, FP64 within a call.  A thread per (image, q < Ks).
__global__ __launch_bounds__(256) void k_torus_vjp_sum(
    TorusArgs A, int nsplit, int Ks, const float* __restrict__ part,
    int pitch, float* __restrict__ acc) {
  const long long total = (long long)A.nimg * Ks;
  const long long x = blockIdx.x * 256LL + threadIdx.x;
  if (x >= total) return;
  const int m = (int)(x / Ks), q = (int)(x - (long long)m * Ks);
  double v = 0.0;
  auto add = [&](long long p, int side) {
    const float* src = part + (p - A.p0) * nsplit * (2LL * Ks) + side * Ks + q;
    for (int s = 0; s < nsplit; ++s) v += (double)src[s * (2LL * Ks)];
  };
  const long long lo = A.p0, hi = A.p0 + A.np;
  bool any = false;
  // partners at p = first + a step, the pairs of this call
  auto run = [&](long long first, long long step, long long count, int side) {
    long long a = first >= lo ? 0 : (lo - first + step - 1) / step;
    long long b = first >= hi ? 0 : (hi - first + step - 1) / step;
    if (b > count) b = count;
    if (a < b) any = true;
#pragma unroll 4
    for (; a < b; ++a) add(first + a * step, side);
  };
  if (A.mode == 2) {
    run(m, 1, 1, 0);
    run(m, 1, 1, 1);
  } else if (A.mode == 1) {
    const long long n = A.n1;
    run(m * n - (long long)m * (m - 1) / 2, 1, n - m, 0);
    for (int i = 0; i <= m; ++i) {
      const long long p = i * n - (long long)i * (i - 1) / 2 + (m - i);
      if (p >= lo && p < hi) {
        any = true;
        add(p, 1);
      }
    }
  } else if (m < A.n1) {
    run((long long)m * A.n2, 1, A.n2, 0);
  } else {
    run(m - A.n1, A.n2, A.n1, 1);
  }
  if (any) acc[(long long)m * pitch + q] += (float)v;
}

// acc[t] += sum over the workgroups of wbp[.][t], t < 2 L, in a fixed order.
__global__ __launch_bounds__(256) void k_torus_vjp_wb(
    const double* __restrict__ wbp, long long parts, int L2,
    double* __restrict__ acc) {
  __shared__ double red[256];
  const int t = blockIdx.x;
  double v = 0.0;
#pragma unroll 4
  for (long long q = threadIdx.x; q < parts; q += 256) v += wbp[q * L2 + t];
  red[threadIdx.x] = v;
  __syncthreads();
  for (int h = 128; h > 0; h >>= 1) {
    if ((int)threadIdx.x < h) red[threadIdx.x] += red[threadIdx.x + h];
    __syncthreads();
  }
  if (threadIdx.x == 0) acc[t] += red[0];
}

static bool vjp_ok(int side, int C, int L) {
  const bool img = C > 0;
  if (L < 1 || L > 3 || C < 0 || C > 3) return false;
  if (img ? !(side == 8 || side == 16 || side == 32)
          : !(side == 2 || side == 4 || side == 8 || side == 16))
    return false;
  return vjp_fits(side, img, L) && !(img && side == 32 && L > 2);
}

// Slices and workgroups of a call; band: pooled diagonals with a cotangent.
static void vjp_shape(VjpArgs& V, int side, long long np, int band) {
  V.d0 = V.e0 = 0;
  V.nd = V.ne = side;
  V.bo = band;
  const int reach = 2 * band + 1;
  if (band >= 0 && 2 * reach + 1 < side) {
    V.d0 = V.e0 = -reach;
    V.nd = V.ne = 2 * reach + 1;
  }
  V.nE = V.nsplit = V.xE = V.xsplit = 1;
  if (side != 32) return;
  if (V.ne < side) {
    V.nsplit = (V.ne + 7) / 8;
    V.xsplit = (V.ne + 3) / 4;
    return;
  }
  // Four e a wave; one or two where that fills idle compute units (a
  // workgroup's own cost is worth about eight slices of its waves).  The
  // pixels' workgroups have half the waves and two share a compute unit.
  const int cu = torus_units();
  long long best = -1;
  for (int ns = 1; ns <= 4; ns *= 2) {
    const long long cost = ((np * ns + cu - 1) / cu) * (128 / ns + 8);
    if (best < 0 || cost < best) {
      best = cost;
      V.nsplit = ns;
      V.nE = 4 / ns;
    }
  }
  best = -1;
  for (int ns = 1; ns <= 8; ns *= 2) {
    const long long cost =
        ((np * ns + 2 * cu - 1) / (2 * cu)) * (256 / ns + 16);
    if (best < 0 || cost < best) {
      best = cost;
      V.xsplit = ns;
      V.xE = 8 / ns;
    }
  }
}

// Workspace: wbp, part, then for images xpart and G.
static long long vjp_floats(const VjpArgs& V, int side, int C, int L) {
  const long long S2 = (long long)side * side;
  return V.nsplit * (4LL * L + 2 * L * S2) +
         (C ? V.xsplit * 2 * C * S2 + (long long)V.ne * V.nd * S2 : 0);
}

}  // namespace nta

using namespace nta;

extern "C" int nta_torus_vjp_supported(int side, int C, int L) {
  return vjp_ok(side, C, L);
}

extern "C" long long nta_torus_vjp_work_bytes(int side, int C, int L,
                                              long long np, int band) {
  if (!vjp_ok(side, C, L) || np < 0) return 0;
  VjpArgs V = VjpArgs();
  vjp_shape(V, side, np, band);
  return 4 * np * vjp_floats(V, side, C, L);
}

extern "C" int nta_torus_vjp(const float* x1, const float* x2, int n1, int n2,
                             long long p0, long long np, const float* in_nngp,
                             const float* in_ntk, int side, int C, int L,
                             const double* wb, int flags, int band,
                             const float* tables, const float* g_nngp,
                             const float* g_ntk, int uniform, float* gin_nngp,
                             float* gin_ntk, float* acc, double* wb_acc,
                             void* work, long long work_bytes, void* stream) {
  TorusArgs A;
  TorusGeom g, go;
  int act;
  const bool img = in_nngp == nullptr;
  const bool ntk = flags & NTA_NTK;
  const bool self = flags & NTA_TORUS_SELF;
  if (!vjp_ok(side, img ? C : 0, L) || (flags & NTA_CONV_CIRCULAR))
    return set_error(NTA_EUNSUPPORTED, "nta_torus_vjp: side=%d C=%d L=%d "
                     "flags=%d", side, C, L, flags);
  int rc = torus_fill("nta_torus_vjp", A, g, side, side, C, img, L, wb, flags,
                      &act);
  if (rc) return rc;
  if (act != kActRelu && act != kActAb)
    return set_error(NTA_EUNSUPPORTED, "nta_torus_vjp: flags=%d", flags);
  rc = torus_set_pairs("nta_torus_vjp", A, n1, n2, flags, p0, np);
  if (rc) return rc;
  if (self && ntk)
    return set_error(NTA_EINVAL, "nta_torus_vjp: ntk of a self chain");
  if (np == 0) return NTA_OK;
  if (!tables || !acc || !wb_acc || !work || (!self && !g_nngp) ||
      (ntk && !g_ntk) ||
      (img ? ((n1 > 0 && !x1) || (n2 > 0 && !x2))
           : (!gin_nngp || (ntk && (!in_ntk || !gin_ntk)))))
    return set_error(NTA_EINVAL, "nta_torus_vjp: null pointer");
  VjpArgs V = VjpArgs();
  vjp_shape(V, side, np, self && !uniform ? band : -1);
  const int S2 = side * side, pitch = (L + (img ? C : 0)) * S2;
  if (work_bytes < 4 * np * vjp_floats(V, side, img ? C : 0, L))
    return set_error(NTA_EINVAL, "nta_torus_vjp: work of %lld bytes",
                     work_bytes);
  if (np * V.xsplit > 0x3fffffffLL ||
      ((long long)A.nimg * pitch + 255) / 256 > 0x3fffffffLL)
    return set_error(NTA_EINVAL, "nta_torus_vjp: too many pairs (%lld)", np);
  V.uniform = uniform ? 1 : 0;
  if (!uniform && g_nngp &&
      (!torus_geom(side / 2, side / 2, 0, go) || go.P != side / 2))
    return set_error(NTA_EUNSUPPORTED, "nta_torus_vjp: pooled side %d",
                     side / 2);
  V.osc = (float)(A.out_scale * (uniform ? 1.0 : 1.0 / 16.0));
  const float2* tab = reinterpret_cast<const float2*>(tables);
  const hipStream_t st = (hipStream_t)stream;
  auto launch = [&](const float* seed) {
    const long long parts = np * V.nsplit;
    double* wbp = reinterpret_cast<double*>(work);
    float* part = reinterpret_cast<float*>(wbp + parts * 2 * L);
    float* xpart = part + parts * 2 * L * S2;
    float* G = xpart + np * V.xsplit * 2 * C * S2;
    int r = img ? vjp_images(side, L, ntk, A, V, x1, x2, tab, g_nngp, g_ntk,
                             seed, G, part, wbp, xpart, st)
                : vjp_state(side, L, ntk, A, V, tab, in_nngp, in_ntk, g_nngp,
                            g_ntk, seed, gin_nngp, gin_ntk, part, wbp, st);
    if (r) return r;
    auto sums = [&](const float* src, int nsplit, int Ks, float* dst) {
      hipLaunchKernelGGL(
          k_torus_vjp_sum,
          dim3((unsigned)(((long long)A.nimg * Ks + 255) / 256)), dim3(256), 0,
          st, A, nsplit, Ks, src, pitch, dst);
    };
    sums(part, V.nsplit, L * S2, acc);
    if (img) sums(xpart, V.xsplit, C * S2, acc + L * S2);
    hipLaunchKernelGGL(k_torus_vjp_wb, dim3(2 * L), dim3(256), 0, st, wbp,
                       parts, 2 * L, wb_acc);
    return check_launch("nta_torus_vjp");
  };
  if (!self) return launch(nullptr);
  // Self chains: the normalisers are the values on slice (0, 0), so their
  // cotangents, which the other slices of the same image add to, enter there,
  // last.
  if (g_nngp) {
    V.skip00 = 1;
    rc = launch(nullptr);
    if (rc) return rc;
    V.skip00 = 0;
  }
  V.seeded = 1;
  V.d0 = V.e0 = 0;
  V.nd = V.ne = V.nE = V.nsplit = V.xE = V.xsplit = 1;
  return launch(acc);
}
