// bh_flat.hip — the flat-space march of the ray_tracer_test entry point
// (include/blackhole/ray_tracer.h:52-96): from the camera through the pixel
// point, straight chords of a fixed vector (BasicLinearRayRecurrence,
// ray_tracer.h:17-35), each chord tested against every object for the nearest
// hit (object_manager.h:69-85).  FP64 in the reference's operation order, one
// lane per pixel.
//
// Only the chords that can cross an object are tested: a height over an
// object's plane changes by a fixed amount a chord, so the chord of its sign
// change is known up to rounding, and a rectangle whose plane is crossed
// outside it is left out.  A ray takes two or three rounds over the objects in
// place of one a chord, and three additions for each chord between; what is
// constant of an object is formed on the host, one record an object, so that a
// round's constants are a few wide scalar loads.  Bound by those loads'
// latency in small frames and by FP64 issue in large ones.  800x450, 10 chords,
// 3 rectangles and a plane: 20.2 us with every chord tested, 11.4 here;
// 3840x2160, 20 chords: 590 and 135.  (Keeping the last chord's heights in
// registers and testing each chord: 17.9 and 397.)
#include "bh_internal.h"
#include "bh_fp64.h"

#include <cmath>

namespace bh {
namespace {

// Signed height of a point over a rectangle's plane (n.(P - p1)) and over a
// plane (its axis z).
__device__ __forceinline__ double height(const DevRect& r, d3 p) {
  return dot(ld3(r.n), p - ld3(r.p));
}
__device__ __forceinline__ double height(const DevPlane& s, d3 p) {
  return s.z[0] * (p.x - s.p[0]) + s.z[1] * (p.y - s.p[1]) + s.z[2] * (p.z - s.p[2]);
}

// Rectangle::Collide (vector_object.h:107-127) for a chord whose ends' heights
// q1, q2 differ in sign: crossing by linear interpolation, inside the
// parallelogram p1 + [0,1] s1 + [0,1] s3.
__device__ __forceinline__ bool rect_collide(const DevRect& r, d3 aa, d3 bb, double q1, double q2,
                                             d3* inter) {
  const d3 p0 = ld3(r.p);
  const d3 Q1 = aa - p0;
  const d3 Q2 = bb - p0;
  const d3 Q = (Q1 * fabs(q2) + Q2 * fabs(q1)) * (1.0 / (fabs(q1) + fabs(q2)));
  const double e1 = dot(ld3(r.e1), Q), e3 = dot(ld3(r.e3), Q);
  *inter = Q + p0;
  return e1 > 0 && r.d1 > e1 && e3 > 0 && r.d3 > e3;
}

// InfinitePlane::Collide (vector_object.h:210-225) for such a chord; a chord
// lying in the plane (t1 = t2 = 0) gives the reference's 0/0 crossing.
__device__ __forceinline__ d3 plane_collide(d3 p1, d3 p2, double t1, double t2) {
  const double d1 = fabs(t1), d2 = fabs(t2);
  return (p1 * d2 + p2 * d1) * (1.0 / (d1 + d2));
}

// The chords on which a height can change sign.  From point `st` on the
// points are equally spaced up to rounding, so a height of h there grows by D
// a chord and vanishes j chords further, j = -h / D.  Rounding moves a height
// by at most err (a few units in the last place a chord of the largest terms;
// tiny heights, whose products could underflow, are within it), so chord st +
// i can cross only for j - w <= i <= j + w + 1, w = err / |D|.  Every
// comparison keeps the chord when something is not a number.
struct Window {
  double j, w;
  __device__ __forceinline__ bool past() const { return j + w < 0.0; }
  // the first such chord after chord st (beyond last: last + 1)
  __device__ __forceinline__ int first(int st, int last) const {
    const double i = ceil(j - w);
    if (!(i > 1.0)) return st + 1;
    return i > (double)(last - st) ? last + 1 : st + (int)i;
  }
};

__device__ __forceinline__ double sum_abs(d3 a) { return fabs(a.x) + fabs(a.y) + fabs(a.z); }

// size: the sum of the absolute coordinates of the march's largest point.
__device__ __forceinline__ Window window(d3 n, d3 o, d3 vec, double h, double size, int steps) {
  const double D = n.x * vec.x + n.y * vec.y + n.z * vec.z;
  const double err = 1e-15 * (double)(steps + 16) * sum_abs(n) * (size + sum_abs(o)) + 1e-140;
  double r = __builtin_amdgcn_rcp(D);
  r = r * __builtin_fma(-D, r, 2.0);
  const double j = -h * r;
  return Window{j, err * fabs(r) + 1e-9 * fabs(j) + 1e-9};
}

// ChessPattern2D::mod (pattern.h:44-47): |a| minus whole multiples of
// 2 size, with C++ integer division of truncated values; size is a whole
// number >= 1 (checked on the host).  Beyond the int range, where the
// reference's (int) cast is undefined, the same truncated quotient is taken
// in double arithmetic.
__device__ inline double chess_mod(double a, double ps) {
  const double b = fabs(a);
  if (!(b < 2147483648.0)) return b - floor(floor(b) / (ps * 2)) * (ps * 2);
  return b - (double)((int)b / (int)(ps * 2)) * (ps * 2);
}

// InfinitePlane::color (vector_object.h:227-232) with ChessPattern2D
// (pattern.h:22-42): plane coordinates (a, b) of (x, y), then the checker.
__device__ inline uint32_t plane_color(const DevPlane& s, d3 q) {
  if (!(s.size > 0)) return 0u;
  const double* vx = s.x;
  const double* vy = s.y;
  const double b = (vx[0] * q.y - vx[1] * q.x) / (vx[0] * vy[1] - vx[1] * vy[0]);
  const double a = (q.x - b * vy[0]) / vx[0];
  const double ps = s.size;
  const double x2 = chess_mod(a, ps), y2 = chess_mod(b, ps);
  const bool in = (x2 <= ps && y2 <= ps) || (ps <= x2 && ps <= y2);
  const bool white = (a * b > 0) ? in : !in;
  return white ? 0xffffffu : 0u;
}

// Rectangle::color (vector_object.h:159-179), nearest texel, clamped.
__device__ inline uint32_t rect_color(const DevRect& s, const DevTex& t, d3 p) {
  const d3 v = p - ld3(s.p);
  const double r = sqrt(dot(v, v));
  double theta = acos(dot(ld3(s.e1), v) / (s.l1 * r));
  theta = isnan(theta) ? 0 : theta;
  double sn, cs;
  sincos(theta, &sn, &cs);  // the values of sin and cos, from one reduction
  const double a = (r * cs / s.l1) * t.cols;
  const double b = (r * sn / s.l3) * t.rows;
  return texel(t, tex_index(a, t.cols), tex_index(b, t.rows));
}

__global__ __launch_bounds__(256) void flat_kernel(DevFlat s, DevOut out) {
  const int x = blockIdx.x * 16 + (threadIdx.x & 15);
  const int y = blockIdx.y * 16 + (threadIdx.x >> 4);
  if (x >= s.W || y >= s.H) return;
  const size_t idx = (size_t)y * s.W + x;
  // Camera::PixelVector (camera.h:55-63), treated as a point (the chord from
  // the camera to it is the first one)
  const double sx = s.W / 2.0 - x, sy = s.H / 2.0 - y;
  d3 old = ld3(s.C);
  d3 present = (ld3(s.fv) - ld3(s.vy) * sx) - ld3(s.vz) * sy;
  d3 vec = present - old;
  const double d2 = dot(vec, vec);
  if (d2 < 100) vec = vec * (100.0 / d2);
  const double size = sum_abs(present) + (double)s.steps * sum_abs(vec);
  int st = 1, kind = -1, which = -1;
  d3 q = mk3(__builtin_nan(""), __builtin_nan(""), __builtin_nan(""));
  bool live = true;
  do {
    // chord st against every object (object_manager.h:69-85: the nearest hit,
    // rectangles first), and the next chord that can cross one
    int next = s.steps + 1;
    bool found = false;
    double best = 0;
    const auto nearest = [&](int k, int i, d3 c) {
      const d3 d = old - c;
      const double kk = dot(d, d);
      if (!found || kk < best) {
        best = kk;
        found = true;
        kind = k;
        which = i;
        q = c;
      }
    };
    if (live) {
#pragma unroll 1
      for (int i = 0; i < s.n_rects; ++i) {
        const DevRect& r = s.rect[i];
        const double q1 = height(r, old), q2 = height(r, present);
        d3 c;
        if (!(q1 * q2 >= 0) && rect_collide(r, old, present, q1, q2, &c)) nearest(0, i, c);
        const Window w = window(ld3(r.n), ld3(r.p), vec, q2, size, s.steps);
        if (!w.past()) {
          // left out where the crossing lies outside the rectangle by more than
          // the window's length and rounding
          const d3 X = (present - ld3(r.p)) + vec * w.j;
          const double m = 1e-9 * (size + fabs(w.j) * sum_abs(vec) + sum_abs(ld3(r.p))) +
                           w.w * sum_abs(vec);
          const double x1 = dot(ld3(r.e1), X), x3 = dot(ld3(r.e3), X);
          const double m1 = m * sum_abs(ld3(r.e1)), m3 = m * sum_abs(ld3(r.e3));
          if (!(x1 < -m1 || x1 > r.d1 + m1 || x3 < -m3 || x3 > r.d3 + m3))
            next = min(next, w.first(st, s.steps));
        }
      }
#pragma unroll 1
      for (int i = 0; i < s.n_planes; ++i) {
        const DevPlane& p = s.plane[i];
        const double t1 = height(p, old), t2 = height(p, present);
        if (!(t1 * t2 > 0)) nearest(1, i, plane_collide(old, present, t1, t2));
        const Window w = window(ld3(p.z), ld3(p.p), vec, t2, size, s.steps);
        if (!w.past()) next = min(next, w.first(st, s.steps));
      }
      if (found) {
        live = false;
      } else if (next > s.steps) {
        st = s.steps;
        live = false;
      } else {
        for (; st < next; ++st) {
          old = present;
          present = present + vec;
        }
      }
    }
  } while (__any(live));
  const int cls = kind >= 0 ? BH_HIT_OBJECT : BH_HIT_NONE;
  uint32_t rgb = 0;
#pragma unroll 1
  for (int i = 0; i < s.n_rects; ++i)
    if (kind == 0 && which == i) rgb = rect_color(s.rect[i], s.rtex[i], q);
#pragma unroll 1
  for (int i = 0; i < s.n_planes; ++i)
    if (kind == 1 && which == i) rgb = plane_color(s.plane[i], q);
  if (out.rgb) {
    out.rgb[3 * idx + 0] = (uint8_t)(rgb & 0xff);
    out.rgb[3 * idx + 1] = (uint8_t)((rgb >> 8) & 0xff);
    out.rgb[3 * idx + 2] = (uint8_t)((rgb >> 16) & 0xff);
  }
  if (out.hit) out.hit[idx] = (uint8_t)cls;
  if (out.phi) out.phi[idx] = __builtin_nan("");
  if (out.hitpt) {
    out.hitpt[3 * idx + 0] = q.x;
    out.hitpt[3 * idx + 1] = q.y;
    out.hitpt[3 * idx + 2] = q.z;
  }
  if (out.steps) out.steps[idx] = st;
}

}  // namespace

// In the kernel's own operation order (IEEE operations, contraction off).
void flat_rect(DevRect* r, const double (*v)[3]) {
  for (int k = 0; k < 3; ++k) {
    r->p[k] = v[1][k];
    r->e1[k] = v[2][k] - v[1][k];
    r->e3[k] = v[4][k] - v[1][k];
  }
  const double *a = r->e1, *b = r->e3;
  const double n[3] = {a[1] * b[2] - a[2] * b[1], a[2] * b[0] - a[0] * b[2],
                       a[0] * b[1] - a[1] * b[0]};
  auto dot3 = [](const double* x, const double* y) {
    return x[0] * y[0] + x[1] * y[1] + x[2] * y[2];
  };
  const double nv = std::sqrt(dot3(n, n));
  const double k = nv != 0.0 ? 1. / nv : 0.;
  for (int j = 0; j < 3; ++j) r->n[j] = n[j] * k;
  r->d1 = dot3(a, a);
  r->d3 = dot3(b, b);
  r->l1 = std::sqrt(r->d1);
  r->l3 = std::sqrt(r->d3);
}

hipError_t launch_flat(const DevFlat& s, const DevOut& out, hipStream_t stream) {
  dim3 grid((s.W + 15) / 16, (s.H + 15) / 16);
  hipLaunchKernelGGL(flat_kernel, grid, dim3(256), 0, stream, s, out);
  return hipGetLastError();
}

}  // namespace bh
