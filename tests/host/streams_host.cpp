// The order that a context's calls have on the GPU, shown on the host: the
// library's bh_api.cpp on a model of the HIP runtime.  The model runs nothing;
// it keeps, for each stream, how much of every other stream's work its work
// follows (a vector clock), moved by launches, event records and waits and by
// the host's own waits.  Work that the host has not waited for counts as still
// running.  Two launches that touch the same memory, one of them writing, must
// be ordered; a launch's memory is what its arguments name.
// Prints one line a scenario and returns the number of those that failed.
#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

#include "bh_api.h"
#include "bh_internal.h"

namespace {

using Clock = std::map<int, int>;  // stream id -> its launches that are followed

void merge(Clock& a, const Clock& b) {
  for (const auto& [k, v] : b)
    if (a[k] < v) a[k] = v;
}
bool covers(const Clock& a, const Clock& b) {
  for (const auto& [k, v] : b) {
    const auto it = a.find(k);
    if (v > 0 && (it == a.end() || it->second < v)) return false;
  }
  return true;
}

struct Stream {
  int id = 0;
  Clock clock;
  bool capturing = false, dead = false;
};
struct Event {
  Clock clock;
  bool captured = false;
};
struct Launch {
  std::string what;
  int stream = 0, seq = 0;
  Clock clock;
  std::vector<const void*> reads, writes;
};

std::map<hipStream_t, Stream> streams;
Clock host;  // what the host has waited for
std::vector<Launch> launches;
int next_id = 1;
int refused = 0;  // calls that a capture does not allow

// What a capture refuses: the state of a capturing stream, and waits of the
// host and frees while any stream captures.
bool refuse(hipStream_t st, bool any) {
  bool no = streams[st].capturing;
  for (const auto& [h, s] : streams) no = no || (any && s.capturing);
  refused += no;
  return no;
}

Stream& at(hipStream_t s) { return streams[s]; }

hipStream_t new_stream() {
  const hipStream_t h = (hipStream_t) new int;
  streams[h].id = next_id++;
  return h;
}

void launch(const char* what, hipStream_t st, std::vector<const void*> reads,
            std::vector<const void*> writes) {
  Stream& s = at(st);
  merge(s.clock, host);
  Launch l{what, s.id, ++s.clock[s.id], s.clock, std::move(reads), std::move(writes)};
  if (!s.capturing) launches.push_back(std::move(l));
}

// Pairs of launches that touch the same memory, one writing it, unordered.
int conflicts() {
  int n = 0;
  for (size_t i = 0; i < launches.size(); ++i)
    for (size_t j = 0; j < i; ++j) {
      const Launch &a = launches[j], &b = launches[i];
      const auto hit = [](const std::vector<const void*>& x, const std::vector<const void*>& y) {
        for (const void* p : x)
          for (const void* q : y)
            if (p && p == q) return true;
        return false;
      };
      if (!hit(a.writes, b.writes) && !hit(a.writes, b.reads) && !hit(a.reads, b.writes)) continue;
      const auto it = b.clock.find(a.stream);
      if (it == b.clock.end() || it->second < a.seq) {
        printf("  unordered: %s on %d, %s on %d\n", a.what.c_str(), a.stream, b.what.c_str(),
               b.stream);
        ++n;
      }
    }
  return n;
}

// Whether the last launch named b follows the last one named a.
bool follows(const char* b, const char* a) {
  const Launch *la = nullptr, *lb = nullptr;
  for (const Launch& l : launches) {
    if (l.what == a) la = &l;
    if (l.what == b) lb = &l;
  }
  if (!la || !lb) return false;
  const auto it = lb->clock.find(la->stream);
  return it != lb->clock.end() && it->second >= la->seq;
}

}  // namespace

// ---- the HIP runtime ---------------------------------------------------------
extern "C" {
hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
  memset(p, 0, sizeof *p);
  p->multiProcessorCount = 256;
  return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { *v = 100000; return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "error"; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipMalloc(void** p, size_t n) { *p = malloc(n); return hipSuccess; }
hipError_t hipFree(void* p) { free(p); return hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { *p = malloc(n); return hipSuccess; }
hipError_t hipHostFree(void* p) { free(p); return hipSuccess; }
hipError_t hipMemcpy(void*, const void*, size_t, hipMemcpyKind) { return hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t, hipMemcpyKind, hipStream_t st) {
  launch("copy", st, {s}, {d});
  return hipSuccess;
}
hipError_t hipMemsetAsync(void*, int, size_t, hipStream_t) { return hipSuccess; }

hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { *s = new_stream(); return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) {
  if (refuse(s, true)) return hipErrorStreamCaptureUnsupported;
  at(s).dead = true;
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) {
  if (at(s).dead) return hipErrorContextIsDestroyed;
  if (refuse(s, true)) return hipErrorStreamCaptureUnsupported;
  merge(host, at(s).clock);
  return hipSuccess;
}
hipError_t hipDeviceSynchronize() {
  if (refuse(nullptr, true)) return hipErrorStreamCaptureUnsupported;
  for (auto& [h, s] : streams) merge(host, s.clock);
  return hipSuccess;
}
hipError_t hipStreamQuery(hipStream_t s) {
  if (at(s).dead) return hipErrorContextIsDestroyed;
  if (refuse(s, false)) return hipErrorStreamCaptureUnsupported;
  return covers(host, at(s).clock) ? hipSuccess : hipErrorNotReady;
}
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus* c) {
  if (at(s).dead) return hipErrorContextIsDestroyed;
  *c = at(s).capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
  return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
  if (at(s).dead) return hipErrorContextIsDestroyed;
  // (a wait for captured work draws the stream into the capture)
  at(s).capturing = at(s).capturing || ((Event*)e)->captured;
  merge(at(s).clock, ((Event*)e)->clock);
  return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t* e) { *e = (hipEvent_t) new Event; return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) { delete (Event*)e; return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  if (at(s).dead) return hipErrorContextIsDestroyed;
  ((Event*)e)->clock = at(s).clock;
  ((Event*)e)->captured = at(s).capturing;
  return hipSuccess;
}
hipError_t hipEventQuery(hipEvent_t e) {
  return covers(host, ((Event*)e)->clock) ? hipSuccess : hipErrorNotReady;
}
hipError_t hipEventSynchronize(hipEvent_t e) { merge(host, ((Event*)e)->clock); return hipSuccess; }
// (every launch takes 1 ms)
hipError_t hipEventElapsedTime(float* ms, hipEvent_t a, hipEvent_t b) {
  *ms = 0.f;
  for (const auto& [k, v] : ((Event*)b)->clock) *ms += (float)v;
  for (const auto& [k, v] : ((Event*)a)->clock) *ms -= (float)v;
  return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t s, hipStreamCaptureMode) { at(s).capturing = true; return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t s, hipGraph_t* g) {
  at(s).capturing = false;
  *g = (hipGraph_t)1;
  return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t, hipGraphNode_t*, char*, size_t) {
  *e = (hipGraphExec_t)1;
  return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t st) {
  launch("graph", st, {}, {});
  return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
}

// ---- the kernels ---------------------------------------------------------------
namespace bh {
hipError_t launch_scene(const DevScene&, DevScene* dst, uint32_t* count, hipStream_t st) {
  launch("scene", st, {}, {dst, count});
  return hipSuccess;
}
hipError_t launch_march_fp32(const DevScene* s, const DevOut& o, int, int, const DevQueue& q,
                             hipStream_t st, bool, bool, int) {
  launch("march", st, {s}, {o.rgb, q.count, q.items});
  return hipSuccess;
}
hipError_t launch_march_fp64(const DevScene* s, const DevOut& o, int, int, hipStream_t st) {
  launch("march64", st, {s}, {o.rgb});
  return hipSuccess;
}
hipError_t launch_band(const DevScene* s, const DevOut& o, const DevQueue& q, hipStream_t st, bool,
                       bool) {
  launch("band", st, {s, q.count, q.items}, {o.rgb});
  return hipSuccess;
}
hipError_t launch_march_frames(const DevScene* s, const DevOut& o, int, int, int, int,
                               const DevQueue& q, hipStream_t st, bool, bool, int) {
  launch("march frames", st, {s}, {o.rgb, q.count, q.items});
  return hipSuccess;
}
hipError_t launch_band_frames(const DevScene* s, const DevOut& o, int, int, int, int,
                              const DevQueue& q, hipStream_t st, bool, bool) {
  launch("band frames", st, {s, q.count, q.items}, {o.rgb});
  return hipSuccess;
}
hipError_t launch_zero_u32(uint32_t* p, int, hipStream_t st) {
  launch("zero", st, {}, {p});
  return hipSuccess;
}
hipError_t launch_turning(const DevScene* s, double* l, int, int, hipStream_t st) {
  launch("turning", st, {s}, {l});
  return hipSuccess;
}
hipError_t launch_steps_taken(const DevScene* s, int32_t* n, int, int, int, hipStream_t st) {
  launch("steps taken", st, {s}, {n});
  return hipSuccess;
}
hipError_t launch_chord_sincos(const float* x, float* o, int, hipStream_t st) {
  launch("sincos", st, {x}, {o});
  return hipSuccess;
}
hipError_t launch_flat(const DevFlat&, const DevOut& o, hipStream_t st) {
  launch("flat", st, {}, {o.rgb});
  return hipSuccess;
}
hipError_t launch_batch_clear(const BatchDev& b, hipStream_t st) {
  launch("batch clear", st, {b.scenes}, {b.head});
  return hipSuccess;
}
hipError_t launch_batch(const BatchDev& b, int, int, int, hipStream_t st) {
  launch("batch", st, {b.scenes}, {b.head, b.band.count});
  return hipSuccess;
}
hipError_t launch_batch_band(const BatchDev& b, int, hipStream_t st) {
  launch("batch band", st, {b.scenes, b.band.count}, {});
  return hipSuccess;
}
hipError_t launch_batch_grid_finish(const BatchDev& b, hipStream_t st) {
  launch("batch finish", st, {b.head}, {b.scene_end});
  return hipSuccess;
}
hipError_t launch_diff_forward(const DiffScene& d, bool, float* rgb, uint8_t*, hipStream_t st) {
  launch("diff", st, {d.tex.data}, {rgb});
  return hipSuccess;
}
hipError_t launch_diff_adjoint(const DiffScene& d, bool, const float* g, float* rgb, uint8_t*,
                               double* work, double* grad, uint32_t*, hipStream_t st) {
  launch("adjoint", st, {d.tex.data, g}, {rgb, work, grad});
  return hipSuccess;
}
int diff_partial_blocks(int W, int H) { return ((W + 15) / 16) * ((H + 15) / 16); }
void flat_rect(DevRect*, const double (*)[3]) {}
hipError_t noalloc_scratch(void** p) { *p = malloc(64); return hipSuccess; }
NoallocLayout noalloc_layout(void* p) {
  return NoallocLayout{(DevScene*)p, (uint32_t*)p, (uint64_t*)p};
}
template <typename T> hipError_t fma_probe(int, hipStream_t st, T* sink, double* tf) {
  launch("probe", st, {}, {sink});
  *tf = 1.0;
  return hipSuccess;
}
template hipError_t fma_probe<float>(int, hipStream_t, float*, double*);
template hipError_t fma_probe<double>(int, hipStream_t, double*, double*);
}  // namespace bh

// ---- scenarios -----------------------------------------------------------------
namespace {

struct Setup {
  bh_ctx* ctx = nullptr;
  bh_scene sc;
  bh_options opt;
  bh_diff_params dp;
  uint8_t rgb1[4], rgb2[4];
  float image[4], image2[4], grad_rgb[4];
  double grad[4], work[64];

  Setup() {
    streams.clear();
    host.clear();
    launches.clear();
    next_id = 1;
    refused = 0;
    at(nullptr).id = 0;
    if (bh_ctx_create(0, &ctx)) abort();
    memset(&sc, 0, sizeof sc);
    memset(&opt, 0, sizeof opt);
    memset(&dp, 0, sizeof dp);
    sc.camera.width = 64;
    sc.camera.height = 48;
    sc.camera.fov = 1.0;
    sc.camera.position[0] = -20.0;
    sc.camera.axis_x[0] = sc.camera.axis_y[1] = sc.camera.axis_z[2] = 1.0;
    sc.hole.mass = 0.5;
    sc.background = -1;
    opt.precision = BH_PREC_FP32;
    dp.r_s = 1.0;
    dp.incl = 1.2;
    dp.dist = 18.0;
    dp.r_inner = 3.0;
    dp.r_outer = 12.0;
    dp.fov = 1.0;
    dp.edge_width = 0.2;
    dp.width = dp.height = 16;
    dp.texture = -1;
  }
  ~Setup() { bh_ctx_destroy(ctx); }
  bool frame(uint8_t* rgb) {
    const bh_outputs o{rgb, nullptr, nullptr, nullptr, nullptr};
    const bool ok = bh_render_device(ctx, &sc, &opt, &o) == BH_OK;
    if (!ok) printf("  frame: %s\n", bh_last_error(ctx));
    return ok;
  }
  bool batch(uint8_t* rgb) {
    const bh_outputs o{rgb, nullptr, nullptr, nullptr, nullptr};
    return bh_render_batch_device(ctx, 1, &sc, &opt, &o, nullptr, nullptr, nullptr) == BH_OK;
  }
  bool set(hipStream_t s) { return bh_ctx_set_stream(ctx, s) == BH_OK; }
  bool image_on(hipStream_t s) {
    const bool ok = bh_diff_render_stream(ctx, s, &dp, BH_PREC_FP32, image, nullptr) == BH_OK;
    if (!ok) printf("  image: %s\n", bh_last_error(ctx));
    return ok;
  }
  bool adjoint_on(hipStream_t s) {
    return bh_diff_adjoint_stream(ctx, s, &dp, BH_PREC_FP32, grad_rgb, image2, nullptr, grad,
                                  nullptr, work, sizeof work) == BH_OK;
  }
};

// Frames before and after an image on another stream, the context's stream
// moved in between: the frames share the context's scene record and queue.
bool frames_around_an_image() {
  Setup s;
  const hipStream_t a = new_stream(), b = new_stream(), c = new_stream();
  return s.set(a) && s.frame(s.rgb1) && s.set(b) && s.image_on(c) && s.frame(s.rgb2) &&
         conflicts() == 0;
}

bool frames_on_two_streams() {
  Setup s;
  const hipStream_t a = new_stream(), b = new_stream();
  return s.set(a) && s.frame(s.rgb1) && s.set(b) && s.frame(s.rgb2) && s.set(nullptr) &&
         s.frame(s.rgb1) && s.set(a) && s.frame(s.rgb2) && conflicts() == 0;
}

bool batches_on_two_streams() {
  Setup s;
  const hipStream_t a = new_stream(), b = new_stream();
  return s.set(a) && s.batch(s.rgb1) && s.set(b) && s.batch(s.rgb2) && conflicts() == 0;
}

// The context's later work follows the image, and the image the context's
// earlier work; so do images on two streams.
bool calls_keep_their_order() {
  Setup s;
  const hipStream_t b = new_stream(), c = new_stream();
  bool ok = s.frame(s.rgb1) && s.image_on(c) && follows("diff", "band");
  ok = ok && s.frame(s.rgb2) && follows("scene", "diff") && conflicts() == 0;
  ok = ok && s.image_on(c) && s.adjoint_on(b) && follows("adjoint", "diff");
  ok = ok && s.set(c) && s.frame(s.rgb1) && follows("scene", "adjoint");
  return ok && conflicts() == 0;
}

// The first image and gradient of a context under capture, the context's
// stream set to the capturing one and a frame on it; then a frame after it.
bool first_calls_in_a_capture() {
  Setup s;
  const hipStream_t c = new_stream();
  bool ok = s.frame(s.rgb1);
  at(c).capturing = true;
  ok = ok && s.image_on(c) && s.adjoint_on(c) && s.set(c) && s.frame(s.rgb2) && refused == 0;
  at(c).capturing = false;
  return ok && s.frame(s.rgb1) && conflicts() == 0 && refused == 0;
}

// An image on a stream that does not capture while the context's stream does.
bool image_beside_a_capture() {
  Setup s;
  const hipStream_t a = new_stream(), b = new_stream();
  bool ok = s.set(a) && s.frame(s.rgb1);
  at(a).capturing = true;
  ok = ok && s.image_on(b) && refused == 0 && !at(b).capturing;
  at(a).capturing = false;
  return ok && s.frame(s.rgb2) && follows("scene", "diff") && conflicts() == 0;
}

// A wait for the context's work (a texture about to be replaced) covers all of
// it and no other stream's, also once a caller has destroyed its stream.
bool waits_for_its_own_work() {
  Setup s;
  const hipStream_t a = new_stream(), b = new_stream(), c = new_stream(), x = new_stream();
  uint8_t texel[3] = {1, 2, 3};
  const bh_image img{texel, 1, 1, 3};
  const auto done = [](hipStream_t st) { return covers(host, at(st).clock); };
  launch("other", x, {}, {});
  bool ok = s.set(a) && s.frame(s.rgb1) && s.set(b) && s.image_on(c);
  ok = ok && bh_texture_set(s.ctx, 1, &img) == BH_OK && done(a) && done(c) && !done(x);
  ok = ok && s.frame(s.rgb1) && s.set(a) && bh_synchronize(s.ctx) == BH_OK && done(b) && !done(x);
  ok = ok && s.image_on(c) && s.adjoint_on(b) && bh_texture_clear(s.ctx, 1) == BH_OK && done(b) &&
       done(c) && !done(x);
  ok = ok && s.image_on(c) && hipStreamSynchronize(c) == hipSuccess &&
       hipStreamDestroy(c) == hipSuccess;
  return ok && bh_texture_set(s.ctx, 1, &img) == BH_OK && s.image_on(b) && s.frame(s.rgb2) &&
         bh_synchronize(s.ctx) == BH_OK && done(a) && done(b);
}

// The reported times of a path's replay hold all its launches.
bool path_times_hold_every_launch() {
  Setup s;
  const bh_camera cams[2] = {s.sc.camera, s.sc.camera};
  bh_path* p = nullptr;
  if (bh_path_create(s.ctx, &s.sc, &s.opt, cams, 2, &p) != BH_OK) return false;
  float ms = 0.f;
  double march = 0.0, band = 0.0, march2 = 0.0, band2 = 0.0;
  const size_t n0 = launches.size();
  bool ok = bh_path_launch(p, &ms) == BH_OK && bh_path_last_ms(p, &march, &band) == BH_OK;
  const size_t n1 = launches.size();
  ok = ok && bh_path_time(p, 1, &march2, &band2) == BH_OK;
  const size_t n2 = launches.size();
  bh_path_destroy(p);
  return ok && n1 > n0 && ms == (float)(n1 - n0) && march + band == (double)(n1 - n0) &&
         march2 + band2 == (double)(n2 - n1);
}

}  // namespace

int main() {
  const struct {
    const char* name;
    bool (*run)();
  } all[] = {
      {"frames_around_an_image", frames_around_an_image},
      {"frames_on_two_streams", frames_on_two_streams},
      {"batches_on_two_streams", batches_on_two_streams},
      {"calls_keep_their_order", calls_keep_their_order},
      {"first_calls_in_a_capture", first_calls_in_a_capture},
      {"image_beside_a_capture", image_beside_a_capture},
      {"waits_for_its_own_work", waits_for_its_own_work},
      {"path_times_hold_every_launch", path_times_hold_every_launch},
  };
  int bad = 0;
  for (const auto& t : all) {
    const bool ok = t.run();
    printf("%s %s\n", t.name, ok ? "ok" : "FAILED");
    bad += !ok;
  }
  return bad;
}
