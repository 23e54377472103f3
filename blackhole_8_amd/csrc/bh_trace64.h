// bh_trace64.h — the whole FP64 reference march of one pixel
// (include/blackhole/blackhole_solution_test.cc:167-298, with the escape
// extension) and its replay for a known outcome, in the reference's operation
// order.  The device code of march64_kernel and of the FP64 pass's fallbacks.
#pragma once

#include "bh_math.h"

namespace bh {

// 1.0 / sqrt(x), both correctly rounded (the IEEE square root, then the IEEE
// reciprocal of it), for 2^-600 <= x < 2^600, where neither operation needs
// scaling: Goldschmidt's iteration from the hardware estimate, with Markstein's
// fused residual corrections for the last bit of the root and of its
// reciprocal, which starts from the same estimate: 16 instructions in place of
// about 30.  (A root whose significand is all ones has a reciprocal so near a
// midpoint that the last correction may leave it one ulp off: one value in
// 2^52.)
__device__ __forceinline__ bool inv_sqrt_in_range(double x) {
  const uint32_t hi = (uint32_t)(__builtin_bit_cast(uint64_t, x) >> 32);
  return hi - 0x1a700000u < 0x65800000u - 0x1a700000u;
}
__device__ __forceinline__ double inv_sqrt_ranged(double x) {
  double y = __builtin_amdgcn_rsq(x);
  double s = x * y, h = 0.5 * y;
  const double r = __builtin_fma(-h, s, 0.5);
  s = __builtin_fma(s, r, s);
  h = __builtin_fma(h, r, h);
  s = __builtin_fma(__builtin_fma(-s, s, x), h, s);
  s = __builtin_fma(__builtin_fma(-s, s, x), h, s);
  y = h + h;
  y = __builtin_fma(y, __builtin_fma(-s, y, 1.0), y);
  return __builtin_fma(y, __builtin_fma(-s, y, 1.0), y);
}

// Steps of u taken together: their G and w form independent chains.
constexpr int kChunk64 = 4;

// w = 1 / sqrt(G(u)) (InvSqrtG, blackhole_solution.h:31-33) of the chunk's u.
__device__ __forceinline__ void inv_sqrt_g64(const double* u, double M2, double ib2, double* w) {
  bool ok = true;
#pragma unroll
  for (int k = 0; k < kChunk64; ++k) {
    w[k] = (u[k] * u[k] * (M2 * u[k] - 1.0)) + ib2;
    ok = ok && inv_sqrt_in_range(w[k]);
  }
  if (ok) {
#pragma unroll
    for (int k = 0; k < kChunk64; ++k) w[k] = inv_sqrt_ranged(w[k]);
  } else {  // zero, negative, huge, NaN
#pragma unroll 1
    for (int k = 0; k < kChunk64; ++k) {
      const double v = 1.0 / sqrt(w[0]);  // (one copy: the values rotate)
      w[0] = w[1];
      w[1] = w[2];
      w[2] = w[3];
      w[3] = v;
    }
  }
}

// The point of the march at (u, phi) in frame f.
__device__ __forceinline__ d3 place64(const DevScene& s, const Frame64& f, double u, double phi) {
  const double r = 1. / u;
  double sn, cs;
  sincos(phi, &sn, &cs);  // the values of sin and cos, from one reduction
  const d3 lv = mk3(0, r * cs, r * sn);
  return matrow(f.R, lv) + ld3(s.B);
}

// The spheres (a bit each) that a chord of the march in frame f can meet.
// Every point of the march is B + yv r cos(phi) + xv r sin(phi) (matrow with
// the first component 0) or the camera or B, all in the plane through B
// spanned by yv and xv (R's second and third columns) up to rounding of
// ~1e-15 (r + |B|), with r <= reach when du > 0 (u only grows from u0, or
// the escape march stops short of r_esc).  A sphere whose centre lies farther
// from that plane than R + tol misses every chord in exact arithmetic by
// D^2 - R^2 >= 1e-12 L^2, L bounding |q - c| over the march's points q, far
// above the rounding of seg_sphere64's discriminant (~1e-15 |Q|^2 L^2 against
// its exact |Q|^2 (R^2 - D^2)), so its test would return false on every
// chord: skipping it changes no outcome.  With du <= 0 (or not finite) the
// points are not bounded and every sphere is kept.
__device__ inline uint32_t plane_spheres64(const DevScene& s, const Frame64& f) {
  if (s.n_spheres == 0) return 0u;
  if (!(f.du > 0.0) || !(f.r0 < 1e300)) return ~0u;
  const d3 yv = mk3(f.R[1], f.R[4], f.R[7]), xv = mk3(f.R[2], f.R[5], f.R[8]);
  const d3 n = normalize(cross(yv, xv));
  if (!(dot(n, n) > 0.5)) return ~0u;
  const d3 B = ld3(s.B);
  const double reach = s.escape ? fmax(f.r0, s.r_esc) : f.r0;
  const double bs = sqrt(dot(B, B));
  uint32_t m = 0u;
  for (int i = 0; i < s.n_spheres; ++i) {
    const d3 c = ld3(s.sc[i]) - B;
    const double R = s.sr[i];
    const double tol = 1e-6 * (sqrt(dot(c, c)) + reach + R) + 1e-9 * bs;
    if (!(fabs(dot(n, c)) > R + tol)) m |= 1u << i;
  }
  return m;
}

// Which chords of a ray can meet an object at all.  In its orbit plane the
// march's points are r (cos phi, sin phi), r = 1/u, and with du > 0 the angle
// phi only grows, so a chord from (u_a, phi_a) to (u_b, phi_b), d = phi_b -
// phi_a < pi, lies in the wedge [phi_a, phi_b], no nearer to the hole than
// min(r_a, r_b) cos(d/2) >= (1 - d^2/8) / max(u_a, u_b) and no farther than
// 1 / min(u_a, u_b).  So the reference's tests can only succeed
//   horizon  when that distance reaches R_h,
//   disc     when n.(P - B) = r A cos(phi - psi) (a disc centred on the hole)
//            changes sign in the wedge, within a guard far above the rounding
//            of the reference's own points, and the chord's radii meet the
//            disc's,
//   spheres  when the wedge meets a sphere's angles.
// Every other chord is left out with its points; the tests of the chords that
// remain are the reference's own.  Each condition is written so that a NaN
// keeps the chord.  `every`: the geometry above does not hold (camera at or
// inside the photon sphere, a disc off the hole, points so far from the
// origin that their rounding could matter): every chord is tested.
struct Cull64 {
  bool every;      // test every chord
  bool first;      // the first chord does not start at phi0
  double a_disc;   // the disc's next crossing angle, less the guard
  double a_sph;    // the next sphere's first angle
  double psi, guard;
  uint32_t spheres;
};

// First crossing of the disc plane after a - guard, less the guard.
__device__ __forceinline__ double next_cross64(const Cull64& c, double a) {
  const double k = floor((a - c.guard - c.psi) * kInvPiD) + 1.0;
  return c.psi + k * kPiD - c.guard;
}

// Earliest start of a sphere's wedge (theta_c -+ asin(rho / D), widened by
// 1e-4 of itself and 1e-4 rad against the FP32 angles) among those that end
// at or after phi.
__device__ inline double next_sphere64(const DevScene& s, const Frame64& f, const Cull64& c,
                                       double phi) {
  const d3 yv = mk3(f.R[1], f.R[4], f.R[7]), xv = mk3(f.R[2], f.R[5], f.R[8]);
  const d3 B = ld3(s.B);
  double next = 1e308;
  for (int i = 0; i < s.n_spheres; ++i) {
    if (!((c.spheres >> i) & 1u)) continue;
    const d3 v = ld3(s.sc[i]) - B;
    const double X = dot(v, yv), Y = dot(v, xv);
    // the sphere's own radius bounds the circle it cuts from the plane
    const float q = (float)(s.sr[i] / sqrt(X * X + Y * Y));
    double lo = -1e308;  // around the hole: every angle
    if (q < 0.999f) {
      const double w = (double)(asinf(q) * 1.0001f + 1e-4f);
      lo = (double)atan2_fast((float)Y, (float)X) - w;
      lo += 2.0 * kPiD * ceil((phi - (lo + 2.0 * w)) * (0.5 * kInvPiD));
      if (!(lo == lo)) lo = -1e308;
    }
    next = fmin(next, lo);
  }
  return next;
}

__device__ inline void cull64(const DevScene& s, const Frame64& f, Cull64& c) {
  c.spheres = plane_spheres64(s, f);
  c.first = !(f.Y0 > 0.0) || !(fabs(f.X0) <= 1e-7 * f.r0);
  const d3 B = ld3(s.B);
  const double far = sqrt(dot(B, B)) * f.u_end;  // |B| over the smallest radius
  c.every = !(f.du > 0.0) || !(f.du < 1e300) || !(fabs(f.phi0) < 4.0) || !(far < 1e6);
  c.a_disc = c.a_sph = 1e308;
  c.psi = c.guard = 0.0;
  if (s.has_disc) {
    const d3 n = ld3(s.dn);
    const d3 yv = mk3(f.R[1], f.R[4], f.R[7]), xv = mk3(f.R[2], f.R[5], f.R[8]);
    const float ny = (float)dot(n, yv), nx = (float)dot(n, xv);
    const float nn = (float)(fabs(n.x) + fabs(n.y) + fabs(n.z));
    const float amp2 = ny * ny + nx * nx;
    c.psi = (double)atan2_fast(nx, ny) + kPiD / 2.0;
    // FP32 angle (2e-7) and the rounding of n.P (1e-14 |n| (1 + |B| / r))
    c.guard = 4e-6 + (4e-7 + 1e-13 * (1.0 + far)) * (double)(nn * __builtin_amdgcn_rsqf(amp2));
    c.every = c.every || !(s.dv0[0] == s.B[0] && s.dv0[1] == s.B[1] && s.dv0[2] == s.B[2]) ||
              !(amp2 > 1e-30f) || !(nn < 1e15f) || !(c.guard < 0.5);
    c.a_disc = next_cross64(c, f.phi0);
  }
  if (c.spheres != 0u) c.a_sph = next_sphere64(s, f, c, f.phi0);
}

// Whether the chord that ends at (u, phi), d = its angle, can meet an object.
__device__ __forceinline__ bool chord_meets64(const DevScene& s, const Cull64& c, double u_a,
                                              double u, double phi, double d) {
  const double umax = fmax(u_a, u);
  const double near = __builtin_fma(-0.125 * d, d, 1.0);  // <= cos(d/2)
  bool meets = c.every || !(near > s.Rcull * umax);
  if (!(phi < c.a_disc)) {
    const double umin = fmin(u_a, u);
    meets = meets || !(umin * s.r_in > 1.0 + 1e-6 || umax * s.r_out < near * (1.0 - 1e-6));
  }
  if (c.spheres != 0u) meets = meets || !(phi < c.a_sph) || !(d < 1.0);
  return meets;
}

// The whole march of one pixel (blackhole_solution_test.cc:167-298) with the
// escape extension.  Returns through px.  With CULL only the chords that can
// meet an object are placed and tested (Cull64); the sums of u, w and phi,
// and so every output, are the same to the bit either way.
//
// Bound by FP64 vector issue, and by latency where the frame is small.  A lane
// steps on its own, four steps' G and w at a time, up to its next chord that
// can meet something (or the end of a phase of the step rule); once every lane
// of the wave waits at such a chord or has ended, all of them place and test
// theirs together.  So the tests (about 300 instructions) run as often as the
// ray with the most such chords needs, not once for every step at which some
// lane has one.  The reference's 960x540 scene takes 72 us; with every chord
// of every step placed and tested it took 153.
template <bool CULL = true>
__device__ inline void trace64(const DevScene& s, int x, int y, Pixel64& px) {
  Frame64 f;
  frame64(s, x, y, f);
  const double nan = __builtin_nan("");
  px.q = mk3(nan, nan, nan);
  px.rgb = 0;
  px.cls = BH_HIT_NONE;
  if (f.degenerate) {
    px.cls = BH_HIT_HORIZON;
    px.phi = nan;
    px.steps = 0;
    return;
  }
  const double M2 = 2.0 * s.M, ib2 = 1.0 / (f.b * f.b);
  const int nstep = s.nstep;
  double u = f.u0, w_prev = 0, phi = f.phi0;
  double u_a = u, phi_a = phi;       // the start of the last chord
  d3 P_prev = ld3(s.C);
  int placed = 1;                    // P_prev is the start of chord `placed`
  Cull64 c;
  if constexpr (CULL) {
    cull64(s, f, c);
  } else {
    c.every = true;
    c.spheres = plane_spheres64(s, f);
  }
  Hit64 h;
  bool live = true, hit = false;
  bool centre = false;  // chord n is a captured ray's, to the centre (:264-272)
  bool ends = false;    // the march ended without a hit before step n
  int n = 1;
#pragma unroll 1
  do {
    bool meets = !live;  // wait for the others
#pragma unroll 1
    do {
      if (!meets) {
        // the steps n .. n + m - 1 of the current phase; inc is their u's
        int last = nstep;
        double inc = f.du * 0.9;
        if (n < nstep) {
          last = nstep - 1;
          inc = f.du;
        } else if (n > nstep) {
          last = n < 2 * nstep ? 2 * nstep - 1 : s.escape ? s.step_cap : 0;
          inc = -f.du;
        }
        centre = f.captured && n > nstep;
        ends = !centre && n > last;
        int m = centre || ends ? 0 : last - n + 1;
        if (c.every) m = min(m, 1);
        meets = m == 0;
        double uk[kChunk64], w[kChunk64];
        double v = u;
#pragma unroll
        for (int k = 0; k < kChunk64; ++k) {
          if (k < m) v = v + inc;
          uk[k] = v;
        }
        inv_sqrt_g64(uk, M2, ib2, w);
#pragma unroll
        for (int k = 0; k < kChunk64; ++k) {
          if (k < m && !meets) {
            if (n >= 2 * nstep && uk[k] * s.r_esc <= 1.0) {
              ends = meets = true;
            } else {
              const double d = (w_prev + w[k]) * f.du_h;
              u_a = u;
              phi_a = phi;
              u = uk[k];
              phi += d;
              w_prev = w[k];
              meets = !CULL || (c.first && n == 1) || chord_meets64(s, c, u_a, u, phi, d);
              if (!meets) ++n;
            }
          }
        }
        if (ends && !(s.escape && s.has_bg)) live = false;
      }
    } while (__any(!meets));
    if (live) {
      // the chord's ends: P_prev unless it is the last chord's end, and P (B
      // itself for a chord to the centre; the last chord's of an escaped ray)
      d3 P = ld3(s.B);
      if (centre) {
        u_a = u;
        phi_a = phi;
      }
      const bool have = placed == n && !ends;
#pragma unroll 1
      for (int k = have ? 1 : 0; k < (centre ? 1 : 2); ++k) {
        const d3 Q = place64(s, f, k == 0 ? u_a : u, k == 0 ? phi_a : phi);
        if (k == 0)
          P_prev = Q;
        else
          P = Q;
      }
      if (ends) {
        px.rgb = equirect64(s.bg, normalize(P - P_prev));
        live = false;
      } else {
        hit = find_collision64(s, P_prev, P, &h, c.spheres);
        live = !hit && !centre;
        if (live) {
          P_prev = P;
          if constexpr (CULL) {
            if (!(phi < c.a_disc)) c.a_disc = next_cross64(c, phi);
            if (!(phi < c.a_sph)) c.a_sph = next_sphere64(s, f, c, phi);
          }
          ++n;
          placed = n;
        }
      }
    }
  } while (__any(live));
  px.phi = phi;
  px.steps = centre ? nstep : ends ? n - 1 : n;
  if (hit) {
    px.rgb = hit_color64(s, h);
    px.cls = h.cls;
    px.q = h.q;
  }
}

// The reference march of pixel (x, y) replayed for a known outcome: the march
// ends at step n with a disc hit (cls BH_HIT_DISC) or with no hit (escape
// background along the last chord).  The swept angle of steps 1..n follows
// trace64's to the bit (the same updates of u, w and phi in the same order);
// only the last chord's two end points are placed, and the colour is taken as
// trace64 takes it, without the per-step object tests.  Returns false when the
// last chord does not cross the disc after all (the outcome was not the
// reference's); px is then unset.
__device__ inline bool replay64(const DevScene& s, int x, int y, int n, int cls, Pixel64& px) {
  if (n < 1 || (cls != BH_HIT_DISC && cls != BH_HIT_NONE)) return false;
  Frame64 f;
  frame64(s, x, y, f);
  if (f.degenerate) return false;
  const double M2 = 2.0 * s.M, ib2 = 1.0 / (f.b * f.b);
  const int nstep = s.nstep;
  double u = f.u0, w_prev = 0, phi = f.phi0;
  double u_a = u, phi_a = phi;  // state at the start of the last chord
#pragma unroll 1
  for (int k0 = 1; k0 <= n; k0 += kChunk64) {
    double uk[kChunk64], w[kChunk64];
    double v = u;
#pragma unroll
    for (int k = 0; k < kChunk64; ++k) {
      if (k0 + k <= n)
        v = v + (k0 + k < nstep ? f.du : k0 + k == nstep ? f.du * 0.9 : -f.du);
      uk[k] = v;
    }
    inv_sqrt_g64(uk, M2, ib2, w);
#pragma unroll
    for (int k = 0; k < kChunk64; ++k) {
      if (k0 + k <= n) {
        u_a = u;
        phi_a = phi;
        u = uk[k];
        phi += (w_prev + w[k]) * f.du_h;
        w_prev = w[k];
      }
    }
  }
  d3 Pa = ld3(s.C), Pb = Pa;
#pragma unroll 1
  for (int k = n == 1 ? 1 : 0; k < 2; ++k) {
    const d3 Q = place64(s, f, k == 0 ? u_a : u, k == 0 ? phi_a : phi);
    if (k == 0)
      Pa = Q;
    else
      Pb = Q;
  }
  const double nan = __builtin_nan("");
  px.phi = phi;
  px.steps = n;
  if (cls == BH_HIT_DISC) {
    Hit64 h;
    if (!s.has_disc || !annulus64(s, Pa, Pb, &h.q)) return false;
    px.rgb = s.disc_tex.data ? disc_color64(s, h.q) : 0u;
    px.cls = BH_HIT_DISC;
    px.q = h.q;
    return true;
  }
  px.rgb = 0;
  px.cls = BH_HIT_NONE;
  px.q = mk3(nan, nan, nan);
  if (s.escape && s.has_bg) px.rgb = equirect64(s.bg, normalize(Pb - Pa));
  return true;
}

}  // namespace bh
