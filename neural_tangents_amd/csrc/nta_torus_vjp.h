// Adjoint of a register-resident segment (nta_torus.h): L x [Conv 3x3, ABRelu]
// between pools, for the ReLU family on square power-of-two sides.
//
// A slice's layers are run forward again from its input (pixels or the state
// before the segment), the pre-activations of all but the last layer parked in
// LDS, and the cotangents taken back through them in the same registers: the
// stencil is its own adjoint.  With the values scaled as in torus_act
// (v = (pi - theta + k) c + s, t' = t (pi - theta + k), c = y + b with
// y = w stencil(v_in), t = u + c with u = w stencil(t_in)) a layer's cotangents
// (gn, gt) of (v, t') become
//   gc  = gn pk + gt t / s,  gt <- gt pk,  gct = gc + gt      (pk = pi - theta + k)
//   q_i += f / (2 q_i),  q_j += f / (2 q_j),  f = gn s - gt t c / s
//   w d/dw += gct y + gt u,  d/db += gct
// and the next cotangents are w stencil(gct), w stencil(gt).  Terms in 1 / s
// vanish at s = 0, which is taken where both arguments are the same position
// of the same image.
#pragma once

#include "nta_torus.h"

namespace nta {

struct VjpArgs {
  int uniform;            // g_n, g_t: one value per pair (the mean's)
  int bo;                 // pooled diagonals with a cotangent (-1: all)
  int skip00, seeded;
  int d0, nd, e0, ne;     // slices: d0 <= d < d0 + nd, likewise e (mod P, Q)
  int nE, nsplit;         // e of a wave one after the other; workgroups a pair
  int xE, xsplit;         // the same of k_torus_pixels
  float osc;
};

struct VjpAngle {
  float s, rs, pk;        // s, 1 / s (0 at s = 0), pi - theta + k
};

// keep = 0: the same position of the same image (s = 0).
__device__ __forceinline__ VjpAngle vjp_angle(float c, float2 qa, float2 qb,
                                              float k, float keep) {
  VjpAngle r;
  const float rh = qa.y * qb.y;
  const float rho = c * rh;
  const float a = fminf(fabsf(rho), 1.0f);
  // s^2; one reciprocal root for s and 1 / s
  const float d = prod_minus_sq(qa.x, qb.x, c) * keep;
  r.rs = d > 1.2e-38f ? __builtin_amdgcn_rsqf(d) : 0.0f;
  r.s = d * r.rs;
  float h = fmaf(-(r.s * rh), acos_over_sin<9>(a), 0.5f * kPi);
  h = rh > 0.0f ? h : 0.0f;             // no variance: theta = pi / 2
  r.pk = (0.5f * kPi + copysignf(h, rho)) + k;
  return r;
}

// x <- w9 stencil(x), in place.  em[r] = 0 where row r is cut from the row
// before.
template <int LW, int RS, int R>
__device__ __forceinline__ void torus_stencil(const TorusArgs& A,
                                              const Slice<LW, false, RS>& s,
                                              const float (&em)[R + 1],
                                              float w9, float (&x)[R]) {
  constexpr int NR = Slice<LW, false, RS>::NR;
  const float ml = s.ml * w9, mr = s.mr * w9;
  float pn = NR == 2 ? __shfl_xor(x[R - 1], 32) : x[R - 1];
  const float fn = NR == 2 ? __shfl_xor(x[0], 32) : x[0];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const float a0 = x[r], a1 = r + 1 < R ? x[r + 1 < R ? r + 1 : 0] : fn;
    const float sum = fmaf(a1, em[r + 1], fmaf(pn, em[r], a0));
    float y = sum * w9;
    add_lr<LW>(y, sum, ml, mr);
    pn = a0;
    x[r] = y;
  }
}

constexpr int vjp_waves(int lw) { return lw == 32 ? 8 : (lw == 16 ? 4 : 1); }
constexpr int vjp_pairs(int lw) { return lw == 8 ? 4 : 1; }

// Arrays of R rows that a wave parks: y of the layers before the last, and u
// where the layer has an ntk input.
__host__ __device__ constexpr int vjp_parked(int L, bool ntk, bool img) {
  int n = 0;
  for (int l = 0; l + 1 < L; ++l) n += 1 + (ntk && (l > 0 || !img) ? 1 : 0);
  return n;
}

// A workgroup takes one pair (LW = 8: four) and a share of its e; a wave walks
// d upwards for one e after the other.  The normaliser cotangents of image i
// stay in the lanes' (h, w); those of image j move by a row with every d
// (h' = h - d) and by a lane with every e, so they are accumulated into the
// next row's register and both stay in registers for the whole pair, summed
// over the waves in LDS, in a fixed order, at the end.
// Bound: the vector ALU (about 140 instructions per element of a two-layer
// segment from images, two waves a SIMD).  512 pairs of 32x32 images, 2
// layers: 2.8 ms here and 0.35 ms in k_torus_pixels (3.35 ms while the layer
// before the last was mapped again on the way back instead of keeping s and
// pk, cuts were worked out per stencil and s and 1 / s took a root and a
// reciprocal); with the pixels' sums in the same registers 5.7 ms (336 bytes a
// lane spilled).  The per-layer kernels of the general path stream states of
// 4 MiB a pair and tensor through k_relu_bwd_rows, the stencils and two GEMMs:
// the gradients of 20 x 20 and 20 x 64 pairs through Myrtle-5 took 43.2 ms
// with them, 16.0 ms with these (forward included).
// part[pair][split]: side i, then side j: [L][H W]; wbp[pair][split][L][2].
// gin: the cotangent of the input, from a state in its layout, from images
// (of the input covariance) [pair][e - e0][d - d0][h][w].
template <int LW, int RS, int L, bool NTK, bool IMG>
__global__ __launch_bounds__(LW == 32 ? 512 : 256)
__attribute__((amdgpu_waves_per_eu(2))) void k_torus_vjp(
    TorusArgs A, VjpArgs V, const float* __restrict__ x1,
    const float* __restrict__ x2, const float2* __restrict__ tab,
    const float* __restrict__ in_n, const float* __restrict__ in_t,
    const float* __restrict__ g_n, const float* __restrict__ g_t,
    const float* __restrict__ seed, float* __restrict__ gin_n,
    float* __restrict__ gin_t, float* __restrict__ part,
    double* __restrict__ wbp) {
  using S = Slice<LW, false, RS>;
  constexpr int R = RS, SPW = S::SPW;
  constexpr int WPP = vjp_waves(LW), PPB = vjp_pairs(LW);
  constexpr int NPK = vjp_parked(L, NTK, IMG);
  constexpr int H = S::NR * RS, S2 = H * H;   // square, P = Q = H = W
  constexpr int PR = H, TR = 2 * H;
  constexpr int sz_x = IMG ? (PR + TR) * LW * 4 : 0;
  constexpr int sz_t = L * (PR + TR) * LW * 2;
  constexpr int sz_p = NPK * R * 64 * WPP;
  extern __shared__ __align__(16) float lds[];
  __shared__ double redw[LW == 32 ? 8 : 4][L][2];
  constexpr int Ks = L * S2;
  constexpr int body = sz_x + sz_t + sz_p;
  constexpr int per = body > Ks ? body : Ks;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int slot = PPB == 1 ? 0 : wave;
  const int k = PPB == 1 ? wave : 0;
  const int tid = PPB == 1 ? (int)threadIdx.x : lane;
  constexpr int NT = WPP * 64;
  float* base = lds + slot * per;
  float4* xi = reinterpret_cast<float4*>(base);
  float4* xj = xi + PR * LW;
  float2* ti = reinterpret_cast<float2*>(base + sz_x);
  float2* tj = ti + L * PR * LW;
  float* park = base + sz_x + sz_t + k * NPK * R * 64 + lane;
  const long long blk = blockIdx.x;
  const long long pb = blk / V.nsplit;
  const int split = (int)(blk - pb * V.nsplit);
  const long long want = pb * PPB + slot;
  const bool live = want < A.np;
  const long long pl = live ? want : A.np - 1;
  const PairIdx pr = torus_pair(A, A.p0 + pl);

  if constexpr (IMG) {
    const float* xa = torus_image(A, x1, x2, pr.i);
    const float* xb = torus_image(A, x1, x2, pr.j);
    for (int q = tid; q < (PR + TR) * LW; q += NT) {
      const bool jj = q >= PR * LW;
      const int o = jj ? q - PR * LW : q;
      const int h = o / LW;
      (jj ? xj : xi)[o] = torus_pixel(A, jj ? xb : xa, h, o - h * LW);
    }
  }
  // The layers' constants for the pair's scaled values (nta_torus.h), their
  // scales and those taken off again.
  float we[L], be[L], ze[L], zr[L];
#pragma unroll
  for (int l = 0; l < L; ++l) {
    const float2* si = tab + ((long long)l * A.nimg + pr.i) * A.TS;
    const float2* sj = tab + ((long long)l * A.nimg + pr.j) * A.TS;
    const TorusWB wb = torus_wb<true>(A, l, si[TR * LW], sj[TR * LW]);
    we[l] = wb.w;
    be[l] = wb.b;
    ze[l] = wave_uniform(si[TR * LW].y * sj[TR * LW].y);
    zr[l] = wave_uniform(torus_unscale<true>(si + TR * LW, sj + TR * LW));
    for (int q = tid; q < PR * LW; q += NT) ti[l * PR * LW + q] = si[q];
    for (int q = tid; q < TR * LW; q += NT) tj[l * TR * LW + q] = sj[q];
  }
  __syncthreads();

  S s;
  s.lane_init();
  const int w = s.w;
  const int row0 = S::NR == 2 ? s.part * RS : 0;
  float ga[L][R], gb[L][R];
  double sw[L], sb[L];
#pragma unroll
  for (int l = 0; l < L; ++l) {
    sw[l] = sb[l] = 0.0;
#pragma unroll
    for (int r = 0; r < R; ++r) ga[l][r] = gb[l][r] = 0.0f;
  }

  // the pooled state's periods are its sides
  constexpr int Ph = H / 2, go_h = Ph * Ph, go_d = Ph * go_h;
  constexpr long long per_in = (long long)S2 * S2;
  constexpr long long per_out = (long long)go_h * go_h;
  constexpr int RB = R < 4 ? R : 4;       // rows whose loads are in flight
  auto in_band = [&](int E) {
    const int v = E <= Ph / 2 ? E : E - Ph;
    return V.bo < 0 || (v <= V.bo && -v <= V.bo);
  };
  const float2* pi0 = ti + row0 * LW + w;
  const float* gpn = g_n ? g_n + (V.uniform ? pl : pl * per_out) : nullptr;
  const float* gpt = NTK && g_t ? g_t + (V.uniform ? pl : pl * per_out)
                                : nullptr;
  const bool pooled = gpn && !V.uniform;
  const float osc = V.osc * zr[L - 1];
  float un = 0.0f, ut = 0.0f;
  if (gpn && V.uniform) {
    un = gpn[0] * osc;
    if constexpr (NTK) ut = gpt[0] * osc;
  }

  // The value at row r - 1 of an accumulator of image j (the row before this
  // lane's first one is the other half's, or its own, last).
  auto before = [&](float v) { return S::NR == 2 ? __shfl_xor(v, 32) : v; };

#pragma nounroll
  for (int st = 0; st < V.nE; ++st) {
    const int job = ((split * WPP + k) * V.nE + st) * SPW + s.grp;
    int e = V.e0 + job;
    e = e < 0 ? e + H : (e >= H ? e - H : e);
    s.set_cols(A, job < V.ne ? e : A.Q);
    if (LW == 32 && st > 0) {
      const int src = 4 * ((lane & 32) | ((lane - 1) & 31));
#pragma unroll
      for (int r = 0; r < R; ++r) {
#pragma unroll
        for (int l = 0; l < L; ++l) gb[l][r] = lane_value(gb[l][r], src);
      }
    }
    if (!__any(s.vw)) continue;
    // pooled columns of even and odd e
    const int E0 = e >> 1;
    int Ew = (e & 1) && !(w & 1) ? E0 + 1 : E0;
    if (Ew >= Ph) Ew = 0;
    const bool okE = s.vw && in_band(Ew);
    const int colo = Ew * Ph + (w >> 1);
#pragma nounroll
    for (int dd = 0; dd < V.nd; ++dd) {
      int d = V.d0 + dd;
      d = d < 0 ? d + H : (d >= H ? d - H : d);
      s.set_rows(A, d);
      const float keep = pr.i == pr.j && d == 0 && s.e == 0 ? 0.0f : 1.0f;
      const int jrow = (H - d + row0) * LW + s.wq;
      const float2* pj0 = tj + jrow;
      float em[R + 1];
#pragma unroll
      for (int r = 0; r <= R; ++r) em[r] = s.edge(s.cut0, s.cut1, r);
      float n[R], t[R];
      float ks[R], kp[R];       // s, pk of the last layer but one
      float last;
      if constexpr (IMG) {
        torus_gram_lds<LW>(A, RS, xi + row0 * LW + w, xj + jrow, n, last);
      } else {
        torus_load(A, s, true, in_n + pl * per_in, n, last);
        if constexpr (NTK)
          torus_load(A, s, true, in_t + pl * per_in, t, last);
      }
      // forward
      int pk = 0;
#pragma unroll
      for (int l = 0; l < L; ++l) {
        const bool hu = NTK && (l > 0 || !IMG);
        torus_stencil<LW, RS>(A, s, em, we[l], n);
        if (hu) torus_stencil<LW, RS>(A, s, em, we[l], t);
        if (l + 1 < L) {
          const float bias = be[l], kk = A.k[l];
#pragma unroll
          for (int r = 0; r < R; ++r) {
            park[(pk * R + r) * 64] = n[r];
            if (hu) park[((pk + 1) * R + r) * 64] = t[r];
            const float c = n[r] + bias;
            const VjpAngle g = vjp_angle(c, pi0[l * PR * LW + r * LW],
                                         pj0[l * TR * LW + r * LW], kk, keep);
            if constexpr (NTK) t[r] = (hu ? t[r] + c : c) * g.pk;
            n[r] = fmaf(g.pk, c, g.s);
            if (l + 2 == L) {
              ks[r] = g.s;
              kp[r] = g.pk;
            }
          }
          pk += hu ? 2 : 1;
        }
      }
      // cotangents of the segment's output: pooled diagonal De for the even
      // rows, Do for the odd ones.  What is not needed is read from somewhere
      // in the same rows of the buffer and dropped.
      const int De = (d + 1) >> 1 >= Ph ? 0 : (d + 1) >> 1, Do = d >> 1;
      const bool dead = V.skip00 && d == 0 && s.e == 0;
      const bool ok_e = okE && in_band(De) && !dead;
      const bool ok_o = okE && in_band(Do) && !dead;
      const int ob = (row0 >> 1) * go_h;
      const int oe = ob + (ok_e ? De * go_d + colo : 0);
      const int oo = ob + (ok_o ? Do * go_d + colo : 0);
      const bool head = s.vw && !dead;
      auto cots = [&](const float* p, float u, int r, float (&v)[RB]) {
        if (pooled) {
#pragma unroll
          for (int q = 0; q < RB; ++q)
            v[q] = p[((q & 1) ? oo : oe) + ((r + q) >> 1) * go_h];
#pragma unroll
          for (int q = 0; q < RB; ++q)
            v[q] = ((q & 1) ? ok_o : ok_e) ? v[q] * osc : 0.0f;
        } else {
#pragma unroll
          for (int q = 0; q < RB; ++q) v[q] = head ? u : 0.0f;
        }
      };
      // back
#pragma unroll
      for (int l = L - 1; l >= 0; --l) {
        const bool hu = NTK && (l > 0 || !IMG);
        if (l + 1 < L) {
          pk -= hu ? 2 : 1;
          torus_stencil<LW, RS>(A, s, em, we[l + 1], n);
          if constexpr (NTK) torus_stencil<LW, RS>(A, s, em, we[l + 1], t);
        }
        const float bias = be[l], kk = A.k[l];
        const float wrap = before(gb[l][R - 1]);
        float cn[RB], ct[RB];
#pragma unroll
        for (int r = R - 1; r >= 0; --r) {
          float y, u = 0.0f, gn, gt = 0.0f;
          if (l + 1 == L && (r & (RB - 1)) == RB - 1) {
            cots(gpn, un, r - (RB - 1), cn);
            if constexpr (NTK) cots(gpt, ut, r - (RB - 1), ct);
          }
          if (l + 1 < L) {
            y = park[(pk * R + r) * 64];
            if (hu) u = park[((pk + 1) * R + r) * 64];
            gn = n[r];
            if constexpr (NTK) gt = t[r];
          } else {
            y = n[r];
            if (hu) u = t[r];
            gn = cn[r & (RB - 1)];
            if constexpr (NTK) gt = ct[r & (RB - 1)];
          }
          const float c = y + bias;
          VjpAngle g;
          if (l + 2 == L) {
            g.s = ks[r];
            g.pk = kp[r];
            g.rs = g.s > 0.0f ? __builtin_amdgcn_rcpf(g.s) : 0.0f;
          } else {
            g = vjp_angle(c, pi0[l * PR * LW + r * LW],
                          pj0[l * TR * LW + r * LW], kk, keep);
          }
          float f = gn * g.s, gct = gn * g.pk;
          if constexpr (NTK) {
            const float tr = gt * (hu ? u + c : c) * g.rs;
            f = fmaf(-tr, c, f);
            gt *= g.pk;
            gct += tr + gt;
            t[r] = gt;
          } else if (V.seeded) {
            if (s.vw)
              gct += zr[l] *
                     seed[((long long)pr.i * (L + (IMG ? A.C : 0)) + l) * S2 +
                          (row0 + r) * H + w];
          }
          n[r] = gct;
          ga[l][r] += f;
          gb[l][r] = (r > 0 ? gb[l][r > 0 ? r - 1 : 0] : wrap) + f;
          sw[l] += (double)(hu ? fmaf(gt, u, gct * y) : gct * y);
          sb[l] += (double)gct;
          // here, not after the loop (which would keep the addends of all
          // rows in registers)
          asm volatile(""
                       : "+v"(ga[l][r]), "+v"(gb[l][r]), "+v"(sw[l]),
                         "+v"(sb[l]));
        }
      }
      torus_stencil<LW, RS>(A, s, em, we[0], n);
      if constexpr (!IMG && NTK) torus_stencil<LW, RS>(A, s, em, we[0], t);
      if (live && s.vw) {
        const long long o =
            IMG ? ((pl * V.ne + job) * V.nd + dd) * S2 + row0 * H + w
                : pl * per_in + (long long)d * H * S2 + row0 * S2 + s.e * H + w;
        constexpr int pitch = IMG ? H : S2;
#pragma unroll
        for (int r = 0; r < R; ++r) {
          gin_n[o + r * pitch] = n[r];
          if constexpr (!IMG && NTK) gin_t[o + r * pitch] = t[r];
        }
      }
    }
  }

  // Sums over the waves (and lane groups), one after the other.
  int dl = V.d0 + V.nd - 1;
  dl = dl < 0 ? dl + H : (dl >= H ? dl - H : dl);
  float* out = part + (pl * V.nsplit + split) * (2LL * Ks);
  for (int side = 0; side < 2; ++side) {
    __syncthreads();
    for (int q = tid; q < Ks; q += NT) base[q] = 0.0f;
    __syncthreads();
    for (int turn = 0; turn < WPP * SPW; ++turn) {
      if (k == turn / SPW && s.grp == turn % SPW && s.vw) {
#pragma unroll
        for (int r = 0; r < R; ++r) {
          int h = row0 + r;
          if (side) {
            h -= dl;
            if (h < 0) h += H;
          }
          const int o = h * H + (side ? s.wq : w);
#pragma unroll
          for (int l = 0; l < L; ++l)
            base[l * S2 + o] += side ? gb[l][r] : ga[l][r];
        }
      }
      __syncthreads();
    }
    const int img = side ? pr.j : pr.i;
    if (live)
      for (int q = tid; q < Ks; q += NT) {
        const int l = q / S2, o = q - l * S2;
        const float2* tl = tab + ((long long)l * A.nimg + img) * A.TS;
        const float qv = tl[o / H * LW + (o & (H - 1))].x;
        const float z = tl[TR * LW].y;           // qv = z^2 q
        out[side * Ks + q] = qv > 0.0f ? base[q] * 0.5f / qv * (z * z) : 0.0f;
      }
  }
#pragma unroll
  for (int l = 0; l < L; ++l) {
    double a = sw[l], b = sb[l] * (double)ze[l];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      a += __shfl_xor(a, o);
      b += __shfl_xor(b, o);
    }
    if (lane == 0) {
      redw[wave][l][0] = a;
      redw[wave][l][1] = b;
    }
  }
  __syncthreads();
  if (live && tid < 2 * L) {
    double v = 0.0;
    for (int q = 0; q < WPP; ++q) v += redw[slot + q][tid >> 1][tid & 1];
    wbp[(pl * V.nsplit + split) * 2 * L + tid] = v;
  }
}

// Pixel cotangents from those G of the input covariance (k_torus_vjp's gin;
// first layer's 1 / C included): side i sum G x_j[h - d, w - e], side j
// sum G x_i[h, w], kept as the normalisers' are in k_torus_vjp.
// Bound: reading G (4 MiB a 32x32 pair, 6.2 TB/s partly from the cache that
// k_torus_vjp left it in).
// part[pair][split]: side i, then side j: [H W][C].
template <int LW, int RS>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2)))
void k_torus_pixels(TorusArgs A, VjpArgs V, const float* __restrict__ x1,
                    const float* __restrict__ x2,
                    const float* __restrict__ G, float* __restrict__ part) {
  using S = Slice<LW, false, RS>;
  constexpr int R = RS, SPW = S::SPW;
  constexpr int PPB = vjp_pairs(LW), WPP = 4 / PPB;
  constexpr int H = S::NR * RS, S2 = H * H;
  constexpr int TR = 2 * H;
  constexpr int body = TR * LW * 4;           // >= 3 S2
  extern __shared__ __align__(16) float lds[];
  const int C = A.C, Ks = C * S2;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int slot = PPB == 1 ? 0 : wave;
  const int k = PPB == 1 ? wave : 0;
  const int tid = PPB == 1 ? (int)threadIdx.x : lane;
  constexpr int NT = WPP * 64;
  float* base = lds + slot * body;
  float4* xj = reinterpret_cast<float4*>(base);
  const long long blk = blockIdx.x;
  const long long pb = blk / V.xsplit;
  const int split = (int)(blk - pb * V.xsplit);
  const long long want = pb * PPB + slot;
  const bool live = want < A.np;
  const long long pl = live ? want : A.np - 1;
  const PairIdx pr = torus_pair(A, A.p0 + pl);
  const float* xa = torus_image(A, x1, x2, pr.i);
  const float* xb = torus_image(A, x1, x2, pr.j);
  for (int q = tid; q < TR * LW; q += NT)
    xj[q] = torus_pixel(A, xb, q / LW, q % LW);
  __syncthreads();
  S s;
  s.lane_init();
  const int w = s.w;
  const int row0 = S::NR == 2 ? s.part * RS : 0;
  float xi[3][R], gi[3][R], gj[3][R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const float4 v = torus_pixel(A, xa, row0 + r, w);
    xi[0][r] = v.x;
    xi[1][r] = v.y;
    xi[2][r] = v.z;
#pragma unroll
    for (int c = 0; c < 3; ++c) gi[c][r] = gj[c][r] = 0.0f;
  }
#pragma nounroll
  for (int st = 0; st < V.xE; ++st) {
    const int job = ((split * WPP + k) * V.xE + st) * SPW + s.grp;
    int e = V.e0 + job;
    e = e < 0 ? e + H : (e >= H ? e - H : e);
    s.set_cols(A, job < V.ne ? e : A.Q);
    if (LW == 32 && st > 0) {
      const int src = 4 * ((lane & 32) | ((lane - 1) & 31));
#pragma unroll
      for (int r = 0; r < R; ++r)
#pragma unroll
        for (int c = 0; c < 3; ++c) gj[c][r] = lane_value(gj[c][r], src);
    }
    if (!__any(s.vw)) continue;
    const float* g0 = G + (pl * V.ne + (s.vw ? job : 0)) * V.nd * S2 +
                      row0 * H + w;
    float nx[R];
#pragma unroll
    for (int r = 0; r < R; ++r) nx[r] = g0[r * H];
#pragma nounroll
    for (int dd = 0; dd < V.nd; ++dd) {
      int d = V.d0 + dd;
      d = d < 0 ? d + H : (d >= H ? d - H : d);
      float n[R];
#pragma unroll
      for (int r = 0; r < R; ++r) n[r] = s.vw ? nx[r] : 0.0f;
      g0 += dd + 1 < V.nd ? S2 : 0;
#pragma unroll
      for (int r = 0; r < R; ++r) nx[r] = g0[r * H];
      const float4* rj = xj + (H - d + row0) * LW + s.wq;
      float wr[3];
#pragma unroll
      for (int c = 0; c < 3; ++c)
        wr[c] = S::NR == 2 ? __shfl_xor(gj[c][R - 1], 32) : gj[c][R - 1];
#pragma unroll
      for (int r = R - 1; r >= 0; --r) {
        const float4 b = rj[r * LW];
        const int m = r > 0 ? r - 1 : 0;
        gi[0][r] = fmaf(n[r], b.x, gi[0][r]);
        gi[1][r] = fmaf(n[r], b.y, gi[1][r]);
        gi[2][r] = fmaf(n[r], b.z, gi[2][r]);
#pragma unroll
        for (int c = 0; c < 3; ++c)
          gj[c][r] = fmaf(n[r], xi[c][r], r > 0 ? gj[c][m] : wr[c]);
      }
    }
  }
  int dl = V.d0 + V.nd - 1;
  dl = dl < 0 ? dl + H : (dl >= H ? dl - H : dl);
  float* out = part + (pl * V.xsplit + split) * (2LL * Ks);
  for (int side = 0; side < 2; ++side) {
    __syncthreads();
    for (int q = tid; q < Ks; q += NT) base[q] = 0.0f;
    __syncthreads();
    for (int turn = 0; turn < WPP * SPW; ++turn) {
      if (k == turn / SPW && s.grp == turn % SPW && s.vw) {
#pragma unroll
        for (int r = 0; r < R; ++r) {
          int h = row0 + r;
          if (side) {
            h -= dl;
            if (h < 0) h += H;
          }
          float* o = base + (h * H + (side ? s.wq : w)) * C;
          o[0] += side ? gj[0][r] : gi[0][r];
          if (C > 1) o[1] += side ? gj[1][r] : gi[1][r];
          if (C > 2) o[2] += side ? gj[2][r] : gi[2][r];
        }
      }
      __syncthreads();
    }
    if (live)
      for (int q = tid; q < Ks; q += NT) out[side * Ks + q] = base[q];
  }
}

template <int LW, int RS>
int vjp_pixels(const TorusArgs& A, const VjpArgs& V, const float* x1,
               const float* x2, const float* G, float* part, hipStream_t st) {
  constexpr int H = (LW == 32 ? 2 : 1) * RS;
  constexpr size_t bytes = sizeof(float) * vjp_pairs(LW) * 2 * H * LW * 4;
  const long long blocks =
      (A.np + vjp_pairs(LW) - 1) / vjp_pairs(LW) * V.xsplit;
  hipLaunchKernelGGL((k_torus_pixels<LW, RS>), dim3((unsigned)blocks),
                     dim3(256), bytes, st, A, V, x1, x2, G, part);
  return check_launch("nta_torus_vjp");
}

template <int LW, int RS, int L, bool NTK, bool IMG>
int vjp_run(const TorusArgs& A, const VjpArgs& V, const float* x1,
            const float* x2, const float2* tab, const float* in_n,
            const float* in_t, const float* g_n, const float* g_t,
            const float* seed, float* gin_n, float* gin_t, float* part,
            double* wbp, hipStream_t st) {
  constexpr int H = (LW == 32 ? 2 : 1) * RS;
  constexpr int body = (IMG ? 3 * H * LW * 4 : 0) + L * 3 * H * LW * 2 +
                       vjp_parked(L, NTK, IMG) * RS * 64 * vjp_waves(LW);
  constexpr int Ks = L * H * H;
  constexpr size_t bytes =
      sizeof(float) * vjp_pairs(LW) * (size_t)(body > Ks ? body : Ks);
  if (bytes > 64 * 1024) {
    hipError_t e = hipFuncSetAttribute(
        reinterpret_cast<const void*>(k_torus_vjp<LW, RS, L, NTK, IMG>),
        hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
    if (e != hipSuccess)
      return set_error((int)e, "nta_torus_vjp: %s", hipGetErrorString(e));
  }
  const long long blocks =
      (A.np + vjp_pairs(LW) - 1) / vjp_pairs(LW) * V.nsplit;
  hipLaunchKernelGGL((k_torus_vjp<LW, RS, L, NTK, IMG>),
                     dim3((unsigned)blocks),
                     dim3(LW == 32 ? 512 : 256), bytes, st, A, V, x1, x2, tab,
                     in_n, in_t, g_n, g_t, seed, gin_n, gin_t, part, wbp);
  return check_launch("nta_torus_vjp");
}

// LDS of a workgroup (the kernel's static sums aside) within 160 KB?
inline bool vjp_fits(int side, bool img, int L) {
  const int lw = side == 32 ? 32 : (side == 16 ? 16 : 8);
  const int rs = side == 32 ? 16 : side;
  const long long body = (img ? 3 * side * lw * 4 : 0) + L * 3 * side * lw * 2 +
                         vjp_parked(L, true, img) * rs * 64 * vjp_waves(lw);
  return body * 4 * vjp_pairs(lw) <= 159 * 1024;
}

int vjp_images(int side, int L, bool ntk, const TorusArgs& A,
               const VjpArgs& V, const float* x1, const float* x2,
               const float2* tab, const float* g_n, const float* g_t,
               const float* seed, float* G, float* part, double* wbp,
               float* xpart, hipStream_t st);
int vjp_state(int side, int L, bool ntk, const TorusArgs& A, const VjpArgs& V,
              const float2* tab, const float* in_n, const float* in_t,
              const float* g_n, const float* g_t, const float* seed,
              float* gin_n, float* gin_t, float* part, double* wbp,
              hipStream_t st);

}  // namespace nta
