// The replay of a ray whose outcome is known (replay64) against the march that
// found it (trace64<false>), lane by lane on the host, over the random scenes of
// trace64_host.cpp: every disc hit, and every ray that ends without a hit and
// was not captured, escaped ones with a background among them, must replay, with
// the march's colour, angle, steps and point.  A hit named one step early, and
// a class that is not replayed, must be refused.  Prints the class, the replays
// of both kinds and those that differ.
#define main chords_main
#include "trace64_host.cpp"
#undef main

static bool same3(d3 a, d3 b) { return same(a.x, b.x) && same(a.y, b.y) && same(a.z, b.z); }

int main(int argc, char** argv) {
  const int scenes = argc > 1 ? atoi(argv[1]) : 60;
  for (uint32_t i = 0; i < 64 * 64; ++i) texture[i] = i * 2654435761u;
  const char* classes[] = {"hole", "disc", "away", "inside", "offdisc", "normal",
                           "radii", "far", "spheres", "escape"};
  long bad = 0;
  for (const char* cls : classes) {
    long disc = 0, miss = 0, diff = 0;
    for (int k = 0; k < scenes; ++k) {
      rng.seed(777767777ull * (unsigned)k + 31);
      DevScene s = make(cls);
      if (k % 6 == 0) s.nstep = 2 + k % 4;
      for (int i = 0; i < 400; ++i) {
        const int x = (int)(rng() % (uint64_t)s.W), y = (int)(rng() % (uint64_t)s.H);
        Pixel64 b, r;
        memset(&b, 0, sizeof b);
        memset(&r, 0, sizeof r);
        trace64<false>(s, x, y, b);
        Frame64 f;
        frame64(s, x, y, f);
        const bool is_disc = b.cls == BH_HIT_DISC && b.steps > 0;
        const bool is_miss = b.cls == BH_HIT_NONE && !f.captured && !f.degenerate;
        if (!is_disc && !is_miss) continue;
        const bool ok = replay64(s, x, y, b.steps, b.cls, r);
        // (a captured ray's last chord, to the centre, is not a step's)
        if (!ok && is_disc && f.captured && b.steps == s.nstep) continue;
        disc += is_disc;
        miss += is_miss;
        const bool eq = ok && r.cls == b.cls && r.rgb == b.rgb && r.steps == b.steps &&
                        same(r.phi, b.phi) && same3(r.q, b.q);
        if (!eq && ++diff <= 3)
          printf("  %s scene %d (%d, %d): replayed %d cls %d %d steps %d %d rgb %x %x\n", cls, k, x,
                 y, ok, r.cls, b.cls, r.steps, b.steps, r.rgb, b.rgb);
        if (replay64(s, x, y, b.steps, BH_HIT_HORIZON, r) ||
            (is_disc && replay64(s, x, y, b.steps - 1, BH_HIT_DISC, r)))
          ++diff;
      }
    }
    printf("%s disc %ld miss %ld differ %ld\n", cls, disc, miss, diff);
    bad += diff;
  }
  return bad ? 1 : 0;
}
