// The FP64 march's choice of the chords it tests (trace64<true>) against the
// march that tests every chord (trace64<false>), lane by lane on the host, over
// random scenes of every form the FP64 precision accepts: turned-away cameras,
// cameras at and inside the photon sphere, tilted, off-centre and degenerate
// discs, spheres near and around the hole, escape, holes far from the origin.
// Prints the scene class, the rays and the rays whose outcome differs.
#include <cfloat>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>

#include "bh_trace64.h"

using namespace bh;

static std::mt19937_64 rng;
static double uni(double a, double b) {
  return a + (b - a) * (double)(rng() >> 11) * 0x1p-53;
}
static d3 dir() {
  for (;;) {
    const d3 v = mk3(uni(-1, 1), uni(-1, 1), uni(-1, 1));
    if (dot(v, v) < 1.0 && dot(v, v) > 1e-4) return normalize(v);
  }
}
static void put(double* p, d3 v) {
  p[0] = v.x;
  p[1] = v.y;
  p[2] = v.z;
}

static uint32_t texture[64 * 64];

static DevScene make(const char* cls) {
  const auto is = [&](const char* c) { return !strcmp(cls, c); };
  DevScene s;
  memset(&s, 0, sizeof s);
  const DevTex tex{texture, 64, 64};
  const double rs = uni(0.5, 2.0);
  s.M = rs / 2.0;
  const d3 B = dir() * (is("far") ? uni(1e3, 1e7) : uni(0.0, 1.0) < 0.5 ? 0.0 : uni(0.0, 30.0));
  const double dist = rs * (is("inside") ? uni(1.05, 1.6) : uni(1.6, 40.0));
  const d3 out = dir();
  const d3 C = B + out * dist;
  // the pixel plane is that of a camera at the origin: the axes' frame looks
  // toward or past the hole from C
  const d3 x = normalize(normalize(B - C) * (is("away") ? -1.0 : 1.0) + dir() * uni(0.0, 0.7));
  const d3 z = normalize(cross(x, dir()));
  const d3 y = cross(z, x);
  s.W = 64;
  s.H = 48;
  put(s.C, C);
  put(s.B, B);
  put(s.F, C - B);
  put(s.vy, y);
  put(s.vz, z);
  put(s.fv, x * (s.W / (2 * tan(uni(0.3, 1.2)))));
  s.bc = 3.0 * sqrt(3.0) * s.M;
  s.Rh = 2 * s.M;
  s.Rcull = s.Rh * (1.0 + 1e-6);
  s.l0 = std::cbrt(DBL_EPSILON);
  s.u0 = 1.0 / sqrt(dot(C - B, C - B));
  s.nstep = uni(0, 1) < 0.5 ? 20 : 2 + (int)uni(0, 40);
  s.root = BH_ROOT_BISECT20;
  if (!is("hole")) {
    s.has_disc = 1;
    const d3 n = uni(0, 1) < 0.3 ? mk3(0, 0, 1) : uni(0, 1) < 0.2 ? normalize(cross(out, dir())) : dir();
    const d3 a = normalize(cross(n, dir())), b = cross(n, a);
    const double R = rs * uni(4.0, 15.0);
    const d3 c0 = is("offdisc") ? B + dir() * uni(0.1, 3.0) : B;
    put(s.dv0, c0);
    put(s.dv1, c0 + (a + b) * R);
    put(s.dv2, c0 + (b - a) * R);
    put(s.dv4, c0 + (a - b) * R);
    put(s.dn, is("normal") ? n * (uni(0, 1) < 0.3 ? 0.0 : uni(0, 1) < 0.5 ? 1e-9 : NAN) : n);
    s.r_out = is("radii") ? (uni(0, 1) < 0.5 ? NAN : uni(-1.0, 1.0)) : R;
    s.r_in = is("radii") ? uni(-1.0, 2.0) * R : rs * uni(0.0, 4.0);
    s.disc_tex = tex;
  }
  if (is("spheres") || is("escape")) {
    s.n_spheres = 1 + (int)uni(0, 12);
    for (int i = 0; i < s.n_spheres; ++i) {
      s.sr[i] = uni(0.1, 3.0);
      // some around the hole, some far, some at the camera's distance
      put(s.sc[i], B + dir() * (uni(0, 1) < 0.2 ? uni(0.0, s.sr[i] * 1.2) : uni(2.0, 1.3 * dist)));
      s.stex[i] = tex;
    }
  }
  if (is("escape")) {
    s.escape = 1;
    s.step_cap = uni(0, 1) < 0.3 ? (int)uni(1, 90) : 400;
    s.r_esc = dist * uni(0.5, 6.0);
    s.has_bg = 1;
    s.bg = tex;
  }
  return s;
}

static bool same(double a, double b) { return memcmp(&a, &b, 8) == 0 || (a != a && b != b); }

int main(int argc, char** argv) {
  const int scenes = argc > 1 ? atoi(argv[1]) : 60;
  for (uint32_t i = 0; i < 64 * 64; ++i) texture[i] = i * 2654435761u;
  const char* classes[] = {"hole", "disc", "away", "inside", "offdisc", "normal",
                           "radii", "far", "spheres", "escape"};
  long bad = 0;
  for (const char* cls : classes) {
    long rays = 0, diff = 0, hits = 0;
    for (int k = 0; k < scenes; ++k) {
      rng.seed(1000003ull * (unsigned)k + 17);
      const DevScene s = make(cls);
      for (int i = 0; i < 400; ++i) {
        const int x = (int)(rng() % (uint64_t)s.W), y = (int)(rng() % (uint64_t)s.H);
        Pixel64 a, b;
        memset(&a, 0, sizeof a);
        memset(&b, 0, sizeof b);
        trace64<true>(s, x, y, a);
        trace64<false>(s, x, y, b);
        ++rays;
        hits += b.cls != 0;
        const bool eq = a.cls == b.cls && a.rgb == b.rgb && a.steps == b.steps &&
                        same(a.phi, b.phi) && same(a.q.x, b.q.x) && same(a.q.y, b.q.y) &&
                        same(a.q.z, b.q.z);
        if (!eq && ++diff <= 3)
          printf("  %s scene %d (%d, %d): cls %d %d steps %d %d phi %.17g %.17g\n", cls, k, x, y,
                 a.cls, b.cls, a.steps, b.steps, a.phi, b.phi);
        // a replay of a disc hit or a miss must give the march's outcome
        Pixel64 r;
        memset(&r, 0, sizeof r);
        if (b.cls == BH_HIT_DISC && replay64(s, x, y, b.steps, b.cls, r) &&
            !(r.rgb == b.rgb && r.steps == b.steps && same(r.phi, b.phi) && same(r.q.x, b.q.x)))
          ++diff;
      }
    }
    printf("%s rays %ld hits %ld differ %ld\n", cls, rays, hits, diff);
    bad += diff;
  }
  return bad ? 1 : 0;
}
