// Host side of the register-resident chains (nta_torus.h): geometry, launch
// shapes, the readout of the partial sums and the C entry points.
#include <algorithm>
#include <atomic>

#include "nta_torus.h"

namespace nta {

template <int ACT>
int torus_pool_act(int lw, bool ntk, bool img, const TorusArgs& A,
                   const float* x1, const float* x2, const float2* tab,
                   const float* in_n, const float* in_t, float* out_n,
                   float* out_t, hipStream_t st);
template <int ACT>
int torus_gap_act(int lw, bool ntk, bool img, const TorusArgs& A,
                  const float* x1, const float* x2, const float2* tab,
                  const float* in_n, const float* in_t, double2* partial,
                  hipStream_t st);
template <int ACT>
int torus_tables_act(int lw, bool img, const TorusArgs& A, const float* x1,
                     const float* x2, const float* state, float2* tab,
                     double cov_a, double cov_b, float* cov, hipStream_t st);
template <int ACT>
int torus_diag_act(int lw, bool big, bool ntk, const TorusArgs& A,
                   const float* x1, const float* x2, const float2* tab,
                   double inv, const double* h, float* out_n, float* out_t,
                   long long ld, hipStream_t st);

// Even periods, so that a diagonal's parity survives the wrap; CIRCULAR
// needs the periods to be the sizes (and whole half waves of rows).
bool torus_geom(int H, int W, int circ, TorusGeom& g, bool diag) {
  if (H < 1 || W < 1 || H > 32 || W > 32) return false;
  const int m = std::max(H, W);
  g.lw = m > 16 ? 32 : (m > 8 || diag ? 16 : 8);
  g.P = H + (H & 1);
  g.Q = W + (W & 1);
  if (circ && (g.P != H || g.Q != W || (g.lw == 32 && H % 4 != 0)))
    return false;
  g.RP = g.lw == 32 ? ((g.P / 2 + 1) & ~1) : g.P;
  g.PR = g.lw == 32 ? 2 * g.RP : g.RP;
  g.TR = g.P + g.PR;
  return true;
}

// One wave per pair adds the chunks' sums in a fixed order and applies the
// readout's affine map; mode 1 (upper triangle) writes both halves.
__global__ __launch_bounds__(256) void k_torus_readout(
    TorusArgs A, const double2* __restrict__ partial, double inv, double a,
    double b, double c, double d, double e, int ntk,
    float* __restrict__ out_n, float* __restrict__ out_t, long long ld) {
  const long long pl = (long long)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (pl >= A.np) return;
  const int lane = threadIdx.x & 63;
  double sn = 0.0, st = 0.0;
  for (int k = lane; k < A.nchunk; k += 64) {
    const double2 v = partial[pl * A.nchunk + k];
    sn += v.x;
    st += v.y;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    sn += __shfl_xor(sn, o);
    st += __shfl_xor(st, o);
  }
  if (lane) return;
  const double m = sn * inv, mt = st * inv;
  const float vn = (float)(a * m + b);
  const float vt = (float)(c * m + d * mt + e);
  const PairIdx q = torus_pair(A, A.p0 + pl);
  if (A.mode == 2) {
    out_n[q.oi] = vn;
    return;
  }
  out_n[q.oi * ld + q.oj] = vn;
  if (ntk) out_t[q.oi * ld + q.oj] = vt;
  if (A.mode == 1) {
    out_n[q.oj * ld + q.oi] = vn;
    if (ntk) out_t[q.oj * ld + q.oi] = vt;
  }
}

// Compute units of the current device (workgroups of a launch are balanced
// over them).
int torus_units() {
  static std::atomic<int> cus[16];        // several threads may ask first
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 16) return 256;
  int v = cus[dev].load(std::memory_order_relaxed);
  if (v == 0) {
    if (hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount,
                              dev) != hipSuccess || v <= 0)
      v = 256;
    cus[dev].store(v, std::memory_order_relaxed);
  }
  return v;
}

// Fills the geometry and the layers' constants; *act receives the kernel's
// activation.
int torus_fill(const char* who, TorusArgs& A, TorusGeom& g, int H, int W,
               int C, bool img, int L, const double* wb, int flags,
               int* act) {
  // (flags & NTA_TORUS_DIAG: the layout of nta_torus_diag)
  A = TorusArgs();
  const int circ = (flags & NTA_CONV_CIRCULAR) ? 1 : 0;
  if (H <= 0 || W <= 0 || L <= 0 || (img && C <= 0) || !wb)
    return set_error(NTA_EINVAL, "%s: bad H=%d W=%d C=%d L=%d", who, H, W, C,
                     L);
  if (!torus_geom(H, W, circ, g, flags & NTA_TORUS_DIAG) ||
      L > kTorusMaxL || (img ? C > 4 : g.lw == 32))
    return set_error(NTA_EUNSUPPORTED, "%s: H=%d W=%d C=%d L=%d flags=%d",
                     who, H, W, C, L, flags);
  A.L = L;
  A.H = H;
  A.W = W;
  A.C = img ? C : 1;
  A.P = g.P;
  A.Q = g.Q;
  A.RP = g.RP;
  A.PR = g.PR;
  A.TR = g.TR;
  A.TS = g.TR * g.lw + 2;
  A.circ = circ;
  A.band = -1;
  *act = (flags & NTA_ACT_ERF) ? kActErf
                               : ((flags & NTA_ACT_GELU) ? kActGelu
                                                         : kActRelu);
  // The layers' constants in FP64, rounded once each; a weight's rounding
  // error (up to 3e-8, the same for every pair) is made up for in the next
  // layer's weight and in the readout's factor.  The kernels' pi is the FP32
  // one (2.8e-8 too large), so 2 pi is twice that: at correlation 1 the map
  // and its derivative are then exact.
  constexpr double k2Pi = 2.0 * (double)kPi;
  double scale = img ? 1.0 / (double)C : 1.0;
  for (int l = 0; l < L; ++l) {
    const double k1 = wb[4 * l + 2], k0 = wb[4 * l + 3];
    const double w = wb[4 * l] * scale / 9.0;
    A.w[l] = (float)w;
    A.b[l] = (float)wb[4 * l + 1];
    scale = A.w[l] != 0.0f ? w / (double)A.w[l] : 1.0;
    if (*act == kActRelu || *act == kActAb) {
      if (!(k1 > 0.0))
        return set_error(NTA_EUNSUPPORTED, "%s: linear activation", who);
      A.k[l] = (float)(k2Pi * k0 / k1);
      if (k1 != 1.0 || k0 != 0.0) *act = kActAb;
      scale *= k1 / k2Pi;
    } else {
      const double k = *act == kActErf ? k1 * (2.0 / 3.14159265358979323846)
                                       : k1;
      A.k[l] = (float)k;
      A.k2[l] = (float)k0;
      scale = *act == kActErf && k0 == 0.0 && A.k[l] != 0.0f
                  ? k / (double)A.k[l] : 1.0;
    }
  }
  A.out_scale = scale;
  // as torus_map: the size with a correlation-form instance
  A.exact = !(*act == kActRelu && !circ && H == 32 && W == 32 &&
              !(flags & (NTA_TORUS_DIAG | NTA_TORUS_EXACT)));
  return NTA_OK;
}

int torus_set_pairs(const char* who, TorusArgs& A, int n1, int n2, int flags,
                    long long p0, long long np) {
  A.n1 = n1;
  A.n2 = n2;
  A.nimg = n1 + n2;
  A.p0 = p0;
  A.np = np;
  long long all;
  if (flags & NTA_TORUS_SELF) {
    A.mode = 2;
    all = (long long)n1 + n2;
  } else if (flags & NTA_TORUS_UPPER) {
    A.mode = 1;
    all = (long long)n1 * (n1 + 1) / 2;
  } else {
    A.mode = 0;
    all = (long long)n1 * n2;
  }
  if (n1 < 0 || n2 < 0 || p0 < 0 || np < 0 || p0 + np > all)
    return set_error(NTA_EINVAL, "%s: pairs [%lld, %lld) of n1=%d n2=%d", who,
                     p0, p0 + np, n1, n2);
  return NTA_OK;
}

// Workgroups of k_torus_pool.  A pooled diagonal costs two d, the prologue
// about one, and so does the d before a share's first diagonal.
// Rounds of whole pairs over the compute units, then what is left in equal
// shares of a pair, as many as make the last rounds shortest (whole calls:
// 1,650 pairs of 32x32, Myrtle-10, 4.81 -> 4.59 ms; 2,628 pairs, Myrtle-5,
// 5.40 -> 5.10 ms, then 4.51 and 5.01 without the repeated d; the 20 self
// chains of 10 x 10 images, a workgroup for each of 7 diagonals: 49 -> 25 us).
static void choose_split(TorusArgs& A, long long blocks, long long room) {
  const long long rounds = blocks / room;
  long long best = -1;
  for (long long r = rounds; r >= 0 && r >= rounds - 1; --r) {
    const long long rest = blocks - r * room;
    for (int ns = 1; ns <= A.units; ++ns) {
      const int nD = (A.units + ns - 1) / ns;
      const int shares = (A.units + nD - 1) / nD;
      const int one = 2 * nD + (nD == A.units ? 1 : 2);
      const long long cost = r * (2 * A.units + 1) +
                             ((rest * shares + room - 1) / room) * one;
      if (best < 0 || cost < best) {
        best = cost;
        A.full = r * room;
        A.nD = nD;
        A.nsplit = shares;
      }
    }
  }
}

// Slices (groups of them) a wave of k_torus_gap takes: enough waves to fill
// the chip several times over, few enough that a slice's setup and the
// partial sums stay small.
static void choose_chunks(TorusArgs& A, const TorusGeom& g) {
  if (g.lw == 32) {
    // k_torus_gap32: a workgroup of 16 waves, one per compute unit, takes 16
    // slices a pass
    A.ns = A.P * A.Q;
    const int passes = (A.ns + 15) / 16;
    const long long room = torus_units();
    long long best = -1;
    for (int m = 1;; m *= 2) {
      if (m > passes) m = passes;
      const int nc = (passes + m - 1) / m;
      const long long cost =
          ((A.np * nc + room - 1) / room) * (16LL * m + 1);
      if (best < 0 || cost < best) {
        best = cost;
        A.cs = 16 * m;
        A.nchunk = nc;
      }
      if (m >= passes) break;
    }
    return;
  }
  const int spw = 64 / g.lw;
  A.ns = A.P * ((A.Q + spw - 1) / spw);
  const long long room = 16LL * torus_units();   // waves in flight
  long long best = -1;
  for (int cs = 1;; cs *= 2) {
    if (cs > A.ns) cs = A.ns;
    const int nc = (A.ns + cs - 1) / cs;
    const long long jobs = A.np * nc;
    // rounds of waves x slices of a wave, in quarters of a slice's time
    const long long cost = (4 * cs + 1) * ((jobs + room - 1) / room);
    if (best < 0 || cost < best) {
      best = cost;
      A.cs = cs;
      A.nchunk = nc;
    }
    if (cs >= A.ns) break;
  }
}

}  // namespace nta

using namespace nta;

extern "C" int nta_torus_supported(int H, int W, int C, int L, int pool,
                                   int flags) {
  TorusGeom g;
  if (!torus_geom(H, W, flags & NTA_CONV_CIRCULAR, g,
                  flags & NTA_TORUS_DIAG))
    return 0;
  if (L < 1 || L > kTorusMaxL || C < 0 || C > 4) return 0;
  if (C == 0 && g.lw == 32) return 0;
  if (pool && (H < 2 || W < 2 || torus_pool_lds(g.lw, g.Q, g.PR, g.TR, L, C > 0) >
                                160 * 1024))
    return 0;
  return 1;
}

extern "C" long long nta_torus_table_floats(int H, int W, int flags) {
  TorusGeom g;
  return torus_geom(H, W, 0, g, flags & NTA_TORUS_DIAG) ? 2LL * (g.TR * g.lw + 2)
                                                        : 0;
}

extern "C" long long nta_torus_state_floats(int H, int W) {
  TorusGeom g;
  return torus_geom(H, W, 0, g) ? (long long)g.P * g.Q * H * W : 0;
}

extern "C" long long nta_torus_gap_work_bytes(int H, int W, long long np) {
  TorusGeom g;
  if (!torus_geom(H, W, 0, g) || np < 0) return 0;
  TorusArgs A = TorusArgs();
  A.P = g.P;
  A.Q = g.Q;
  A.np = np;
  choose_chunks(A, g);
  return 16 * np * A.nchunk;
}

extern "C" int nta_torus_tables(const float* x1, const float* x2, int n1,
                                int n2, const float* state, int H, int W,
                                int C, int L, const double* wb, int flags,
                                float* tables, double cov_a, double cov_b,
                                float* cov, void* stream) {
  TorusArgs A;
  TorusGeom g;
  int act;
  const bool img = state == nullptr;
  int rc = torus_fill("nta_torus_tables", A, g, H, W, C, img, L, wb, flags, &act);
  if (rc) return rc;
  rc = torus_set_pairs("nta_torus_tables", A, n1, n2, NTA_TORUS_SELF, 0,
                 (long long)n1 + n2);
  if (rc) return rc;
  if (A.nimg == 0) return NTA_OK;
  if (!tables || (img && ((n1 > 0 && !x1) || (n2 > 0 && !x2))))
    return set_error(NTA_EINVAL, "nta_torus_tables: null pointer");
  float2* tab = reinterpret_cast<float2*>(tables);
  const hipStream_t st = (hipStream_t)stream;
  switch (act) {
    case kActRelu: return torus_tables_act<kActRelu>(g.lw, img, A, x1, x2,
                                                     state, tab, cov_a, cov_b,
                                                     cov, st);
    case kActAb: return torus_tables_act<kActAb>(g.lw, img, A, x1, x2, state,
                                                 tab, cov_a, cov_b, cov, st);
    case kActErf: return torus_tables_act<kActErf>(g.lw, img, A, x1, x2,
                                                   state, tab, cov_a, cov_b,
                                                   cov, st);
  }
  return torus_tables_act<kActGelu>(g.lw, img, A, x1, x2, state, tab, cov_a,
                                    cov_b, cov, st);
}

extern "C" int nta_torus_pool(const float* x1, const float* x2, int n1,
                              int n2, long long p0, long long np,
                              const float* in_nngp, const float* in_ntk,
                              int H, int W, int C, int L, const double* wb,
                              int flags, int band, const float* tables,
                              float* out_nngp, float* out_ntk,
                              void* stream) {
  TorusArgs A;
  TorusGeom g, go;
  int act;
  const bool img = in_nngp == nullptr;
  const bool ntk = flags & NTA_NTK;
  int rc = torus_fill("nta_torus_pool", A, g, H, W, C, img, L, wb, flags, &act);
  if (rc) return rc;
  rc = torus_set_pairs("nta_torus_pool", A, n1, n2, flags, p0, np);
  if (rc) return rc;
  if (H < 2 || W < 2 || !torus_geom(H / 2, W / 2, 0, go))
    return set_error(NTA_EINVAL, "nta_torus_pool: %dx%d does not pool", H, W);
  if (np == 0) return NTA_OK;
  if (!tables || !out_nngp || (ntk && !out_ntk) ||
      (img ? ((n1 > 0 && !x1) || (n2 > 0 && !x2)) : (ntk && !in_ntk)))
    return set_error(NTA_EINVAL, "nta_torus_pool: null pointer");
  A.Ho = H / 2;
  A.Wo = W / 2;
  A.Pn = go.P;
  A.Qn = go.Q;
  A.out_scale *= 1.0 / 16.0;
  const int Ph = A.P / 2;
  const size_t lds = torus_pool_lds(g.lw, g.Q, g.PR, g.TR, L, img);
  const long long per_cu =
      g.lw == 32 ? 1 : std::max<long long>(1, std::min<long long>(
                           4, (160 * 1024) / (long long)lds));
  const long long room = per_cu * torus_units();
  const long long blocks = g.lw == 8 ? (np + 3) / 4 : np;
  A.units = Ph;
  if (band >= 0 && 2 * band + 1 < Ph) {
    // self chains: a workgroup a diagonal (D = 0 has to begin one)
    A.band = band;
    A.D0 = -band;
    A.units = 2 * band + 1;
    A.nD = 1;
    A.nsplit = A.units;
  } else {
    choose_split(A, blocks, room);
  }
  const long long nblk = A.full + (blocks - A.full) * A.nsplit;
  if (nblk > 0x7fffffffLL)
    return set_error(NTA_EINVAL, "nta_torus_pool: too many pairs (%lld)", np);
  const float2* tab = reinterpret_cast<const float2*>(tables);
  const hipStream_t st = (hipStream_t)stream;
  switch (act) {
    case kActRelu: return torus_pool_act<kActRelu>(
        g.lw, ntk, img, A, x1, x2, tab, in_nngp, in_ntk, out_nngp, out_ntk,
        st);
    case kActAb: return torus_pool_act<kActAb>(
        g.lw, ntk, img, A, x1, x2, tab, in_nngp, in_ntk, out_nngp, out_ntk,
        st);
    case kActErf: return torus_pool_act<kActErf>(
        g.lw, ntk, img, A, x1, x2, tab, in_nngp, in_ntk, out_nngp, out_ntk,
        st);
  }
  return torus_pool_act<kActGelu>(g.lw, ntk, img, A, x1, x2, tab, in_nngp,
                                  in_ntk, out_nngp, out_ntk, st);
}

extern "C" int nta_torus_gap(const float* x1, const float* x2, int n1, int n2,
                             long long p0, long long np, const float* in_nngp,
                             const float* in_ntk, int H, int W, int C, int L,
                             const double* wb, int flags, int crop_h,
                             int crop_w, const float* tables, double a,
                             double b, double c, double d, double e,
                             float* out_nngp, float* out_ntk, long long ld,
                             void* work, long long work_bytes, void* stream) {
  TorusArgs A;
  TorusGeom g;
  int act;
  const bool img = in_nngp == nullptr;
  const bool ntk = (flags & NTA_NTK) && !(flags & NTA_TORUS_SELF);
  int rc = torus_fill("nta_torus_gap", A, g, H, W, C, img, L, wb,
                      flags | NTA_TORUS_EXACT, &act);
  if (rc) return rc;
  rc = torus_set_pairs("nta_torus_gap", A, n1, n2, flags, p0, np);
  if (rc) return rc;
  if (crop_h < 1 || crop_h > H || crop_w < 1 || crop_w > W)
    return set_error(NTA_EINVAL, "nta_torus_gap: crop %dx%d of %dx%d", crop_h,
                     crop_w, H, W);
  if (np == 0) return NTA_OK;
  A.Hc = crop_h;
  A.Wc = crop_w;
  choose_chunks(A, g);
  if (!tables || !out_nngp || (ntk && !out_ntk) || !work ||
      (img ? ((n1 > 0 && !x1) || (n2 > 0 && !x2)) : (ntk && !in_ntk)))
    return set_error(NTA_EINVAL, "nta_torus_gap: null pointer");
  if (work_bytes < 16 * np * A.nchunk)
    return set_error(NTA_EINVAL, "nta_torus_gap: work of %lld bytes",
                     work_bytes);
  if (np * A.nchunk > 0x7ffffff0LL)
    return set_error(NTA_EINVAL, "nta_torus_gap: too many pairs (%lld)", np);
  const int cols = A.mode == 1 ? n1 : n2;
  if (A.mode != 2 && ld < cols)
    return set_error(NTA_EINVAL, "nta_torus_gap: ld=%lld < %d", ld, cols);
  const float2* tab = reinterpret_cast<const float2*>(tables);
  double2* part = reinterpret_cast<double2*>(work);
  const hipStream_t st = (hipStream_t)stream;
  switch (act) {
    case kActRelu:
      rc = torus_gap_act<kActRelu>(g.lw, ntk, img, A, x1, x2, tab, in_nngp,
                                   in_ntk, part, st);
      break;
    case kActAb:
      rc = torus_gap_act<kActAb>(g.lw, ntk, img, A, x1, x2, tab, in_nngp,
                                 in_ntk, part, st);
      break;
    case kActErf:
      rc = torus_gap_act<kActErf>(g.lw, ntk, img, A, x1, x2, tab, in_nngp,
                                  in_ntk, part, st);
      break;
    default:
      rc = torus_gap_act<kActGelu>(g.lw, ntk, img, A, x1, x2, tab, in_nngp,
                                   in_ntk, part, st);
  }
  if (rc) return rc;
  const double area = (double)crop_h * crop_w;
  hipLaunchKernelGGL(k_torus_readout, dim3((unsigned)((np + 3) / 4)),
                     dim3(256), 0, st, A, part,
                     A.out_scale / (area * area), a, b, c, d, e,
                     (int)ntk, out_nngp, out_ntk, ld);
  return check_launch("nta_torus_gap");
}

extern "C" int nta_torus_diag(const float* x1, const float* x2, int n1,
                              int n2, int H, int W, int C, int L,
                              const double* wb, int flags,
                              const float* tables, double a, double b,
                              double c, double d, double e, float* out_nngp,
                              float* out_ntk, long long ld, void* stream) {
  TorusArgs A;
  TorusGeom g;
  int act;
  const bool ntk = flags & NTA_NTK;
  int rc = torus_fill("nta_torus_diag", A, g, H, W, C, true, L, wb,
                flags | NTA_TORUS_DIAG, &act);
  if (rc) return rc;
  const bool upper = flags & NTA_TORUS_UPPER;
  rc = torus_set_pairs("nta_torus_diag", A, n1, n2, flags & NTA_TORUS_UPPER, 0, 0);
  if (rc) return rc;
  const int cols = upper ? n1 : n2;
  if (n1 == 0 || cols == 0) return NTA_OK;
  if (!x1 || (!upper && !x2) || !tables || !out_nngp || (ntk && !out_ntk))
    return set_error(NTA_EINVAL, "nta_torus_diag: null pointer");
  if (ld < cols)
    return set_error(NTA_EINVAL, "nta_torus_diag: ld=%lld < %d", ld, cols);
  const double inv = A.out_scale / ((double)H * W);
  const double head[5] = {a, b, c, d, e};
  // Workgroups of 16 waves share more of the tables; of 4 while those would
  // leave compute units idle.
  const int spw = g.lw == 32 ? 1 : 4;
  const long long pairs = (long long)n1 * cols / (upper ? 2 : 1);
  const bool big = pairs >= 16LL * spw * torus_units();
  const float2* tab = reinterpret_cast<const float2*>(tables);
  const hipStream_t st = (hipStream_t)stream;
  switch (act) {
    case kActRelu: return torus_diag_act<kActRelu>(
        g.lw, big, ntk, A, x1, x2, tab, inv, head, out_nngp, out_ntk, ld, st);
    case kActAb: return torus_diag_act<kActAb>(
        g.lw, big, ntk, A, x1, x2, tab, inv, head, out_nngp, out_ntk, ld, st);
    case kActErf: return torus_diag_act<kActErf>(
        g.lw, big, ntk, A, x1, x2, tab, inv, head, out_nngp, out_ntk, ld, st);
  }
  return torus_diag_act<kActGelu>(g.lw, big, ntk, A, x1, x2, tab, inv, head,
                                  out_nngp, out_ntk, ld, st);
}
