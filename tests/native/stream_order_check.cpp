// Order between the library's launches on several streams and threads, checked
// on a recording HIP runtime (hip_recorder.h).  One check per run, named by the
// argument; prints "ok" and exits 0 when it holds.
#include <cstdio>
#include <cstring>

#include "convfpga/convfpga_ext.h"
#include "hip_recorder.h"

// (convfpga.h and the HIP headers both name a float2)
extern "C" int fpga_initialize(const char*, const char*, bool);

static int failures = 0;
#define CHECK(c)                                            \
  do {                                                      \
    if (!(c)) {                                             \
      printf("line %d: %s\n", __LINE__, #c);                \
      ++failures;                                           \
    }                                                       \
  } while (0)

static size_t cube(unsigned n) { return (size_t)n * n * n * 8; }
static void forget() {
  rec::launches.clear();
  rec::faults.clear();
  rec::device_waits = rec::captured_launches = 0;
}
struct Bufs {
  char *in, *out;
  explicit Bufs(unsigned n, unsigned count = 1) : in(rec::alloc(cube(n) * count)), out(rec::alloc(cube(n) * count)) {}
};
static int fft(unsigned n, const Bufs& b, hipStream_t s, int inverse = 0) {
  return cf_fft3d_device(n, b.in, b.out, 1, inverse, s);
}

// Transforms on hipStreamPerThread, which is another stream in every thread: they
// meet in no memory, and neither do one on it and one on a stream of another thread.
static void fft_per_thread() {
  for (unsigned n : {256u, 512u})
    for (int inverse : {0, 1}) {
      Bufs a(n), b(n), c(n);
      fft(n, a, hipStreamPerThread, inverse);
      forget();
      std::thread([&] { CHECK(fft(n, a, hipStreamPerThread, inverse) == CF_OK); }).join();
      std::thread([&] { CHECK(fft(n, b, hipStreamPerThread, inverse) == CF_OK); }).join();
      CHECK(fft(n, c, rec::new_stream(), inverse) == CF_OK);
      CHECK(rec::races() == 0);
      CHECK(rec::faults.empty());
    }
}

// Transforms on different streams have nothing to do with each other: no memory in
// common, no order between them, no wait, whatever was queued or is being captured
// on the others.
static void fft_streams() {
  hipStream_t s[20];
  for (auto& x : s) x = rec::new_stream();
  const size_t held = rec::held;
  for (unsigned n : {256u, 512u, 256u}) {
    forget();
    for (auto x : s) {
      Bufs b(n);
      for (int k = 0; k < 2; ++k) CHECK(fft(n, b, x, k) == CF_OK);
    }
    std::set<int> axis;  // the streams that have no workspace
    for (auto& l : rec::launches)
      if (l.name.rfind("cf_coly_inv_", 0) == 0 && l.name.find("slab") == std::string::npos) axis.insert(l.stream);
    CHECK(axis.size() == (n == 256 ? 4 : 20));  // (16 at 256^3 leave nothing for 512^3)
    CHECK(rec::races() == 0);
    CHECK(rec::faults.empty() && rec::device_waits == 0);
    for (auto& a : rec::launches)
      for (auto& b : rec::launches) CHECK(a.stream == b.stream || !rec::ordered(a, b));
  }
  CHECK(rec::held - held < (size_t(2) << 30) + (1 << 20));  // (and twiddles)
}
static void fft_beside_capture() {
  for (unsigned n : {256u, 512u}) {
    hipStream_t a = rec::new_stream(), b = rec::new_stream();
    Bufs x(n), y(n);
    fft(n, y, b);
    fft(n, x, a);  // the last user of what transforms may share
    forget();
    rec::begin_capture(a);
    CHECK(fft(n, x, a) == CF_OK);
    CHECK(rec::captured_launches > 0 && rec::launches.empty());
    const unsigned captured = rec::captured_launches;
    CHECK(fft(n, y, b) == CF_OK);
    rec::end_capture(a);
    CHECK(rec::faults.empty());
    CHECK(rec::captured_launches == captured && !rec::launches.empty());
  }
}

// A stream's first transform, which makes its workspace, is as free to be called as
// a later one: beside a capture, with no memory left, and with nothing waited for.
static void fft_first_call() {
  for (unsigned n : {256u, 512u}) {
    Bufs x(n), y(n);
    cf_spectrum_t kept = nullptr;
    CHECK(cf_set_plan(n, CF_PLAN_AXIS5) == CF_OK);
    CHECK(cf_spectrum_create(n, 1, x.in, 1, nullptr, &kept) == CF_OK);
    cf_spectrum_destroy(kept);
    hipStream_t a = rec::new_stream();
    forget();
    rec::begin_capture(a);
    CHECK(fft(n, y, rec::new_stream()) == CF_OK);
    rec::end_capture(a);
    CHECK(rec::faults.empty() && rec::device_waits == 0 && rec::launches.size() > 0);
    CHECK(cf_set_plan(7, CF_PLAN_AUTO) < 0);
    const std::string text = cf_last_error();
    rec::alloc_limit = 0;
    CHECK(fft(n, y, rec::new_stream()) == CF_OK);
    rec::alloc_limit = ~size_t(0);
    CHECK(rec::device_waits == 0 && text == cf_last_error() && hipGetLastError() == hipSuccess);
  }
}

// Convolutions through the common workspace (a four-step plan) are ordered, whoever
// calls: threads on their hipStreamPerThread, other streams before and after them.
static void conv_per_thread() {
  CHECK(cf_set_plan(256, CF_PLAN_SPLIT3_G24) == CF_OK);
  Bufs f(256), x(256), y(256), z(256);
  cf_spectrum_t h = nullptr;
  CHECK(cf_spectrum_create(256, 1, f.in, 1, nullptr, &h) == CF_OK);
  hipStream_t s = rec::new_stream();
  forget();
  auto conv = [&](const Bufs& b, hipStream_t st) {
    CHECK(cf_conv3d_device(h, b.in, b.out, 1, CF_SCALE_INV_N3, CF_PREC_FP32, st) == CF_OK);
  };
  conv(z, s);
  for (int k = 0; k < 2; ++k) {
    std::thread([&] { conv(x, hipStreamPerThread), conv(x, hipStreamPerThread); }).join();
    std::thread([&] { conv(y, hipStreamPerThread); }).join();
    if (k == 0) conv(z, s);
  }
  conv(z, nullptr);
  CHECK(rec::launches.size() == 3 * 9);
  CHECK(rec::races() == 0);
  CHECK(rec::faults.empty() && rec::device_waits == 0);
  cf_spectrum_destroy(h);
}

// A destroyed spectrum's memory is written again only after the convolutions queued
// with it: at once on the one stream that used it, which orders them; on no other.
// What several streams, or others, may be reading is freed, which waits for them.
// Making a spectrum waits for no stream but its own.
static void spectrum_reuse() {
  CHECK(cf_set_plan(128, CF_PLAN_AXIS5) == CF_OK);
  Bufs f(128), x(128), y(128);
  hipStream_t a = rec::new_stream(), b = rec::new_stream(), capture = rec::new_stream();
  auto make = [&](hipStream_t s) {
    cf_spectrum_t h = nullptr;
    CHECK(cf_spectrum_create(128, 1, f.in, 1, s, &h) == CF_OK);
    return h;
  };
  auto conv = [&](cf_spectrum_t h, const Bufs& u, hipStream_t s) {
    CHECK(cf_conv3d_device(h, u.in, u.out, 1, CF_SCALE_INV_N3, CF_PREC_FP32, s) == CF_OK);
  };
  enum { ONE, TWO_STREAMS, PER_THREAD, ADDRESS, CAPTURED, VIEW };
  make(a);  // (the edge is set up)
  for (int use : {ONE, TWO_STREAMS, PER_THREAD, ADDRESS, CAPTURED, VIEW})
    for (hipStream_t next : {a, b, (hipStream_t)hipStreamPerThread}) {
      cf_spectrum_t h = make(a), v = h;
      forget();
      const size_t blocks = rec::allocs.size();
      if (use == VIEW) CHECK(cf_spectrum_view(h, 0, &v) == CF_OK);
      conv(v, x, a);
      if (use == TWO_STREAMS) conv(h, y, b);
      if (use == PER_THREAD) conv(h, y, hipStreamPerThread);
      if (use == ADDRESS) CHECK(cf_spectrum_data(h) != nullptr);
      if (use == CAPTURED) {
        rec::begin_capture(capture, hipStreamCaptureModeRelaxed);
        conv(h, y, capture);
        rec::end_capture(capture);
      }
      if (v != h) cf_spectrum_destroy(v);
      const bool sole = use == ONE || use == VIEW;
      cf_spectrum_destroy(h);
      CHECK(rec::device_waits == (sole ? 0 : 1));
      rec::begin_capture(capture, hipStreamCaptureModeRelaxed);  // which a wait for the device would end
      rec::mode = hipStreamCaptureModeRelaxed;
      h = make(next);
      rec::mode = hipStreamCaptureModeGlobal;
      rec::end_capture(capture);
      CHECK(rec::device_waits == (sole ? 0 : 1));
      if (use == ONE && next == a) CHECK(rec::allocs.size() == blocks);
      conv(h, y, next);
      CHECK(rec::races() == 0 && rec::faults.empty());
      CHECK(cf_spectrum_data(h) != nullptr);  // (freed, not kept)
      cf_spectrum_destroy(h);
    }
}

// A batch whose output overlaps its signal at another place: a plan that takes the
// signal into the workspace reads every cube before it is overwritten.
static void conv_overlap() {
  const struct {
    unsigned n, plan, count;
    int precision;
  } cases[] = {{128, CF_PLAN_SPLIT3_G24, 20, CF_PREC_FP32},
               {256, CF_PLAN_SPLIT3_G24, 4, CF_PREC_FP32},
               {256, CF_PLAN_SPLIT3_G24M2, 4, CF_PREC_SPLIT_FP16}};
  for (auto& c : cases)
    for (unsigned own : {0u, 1u})
      for (bool timed : {false, true})
        for (double shift : {1.0, -1.0, 2.5, -2.5, (double)c.count}) {
          const size_t V = cube(c.n);
          char* const buf = rec::alloc(V * 3 * c.count);
          char* const sig = buf + V * c.count;
          char* const out = sig + (long long)(shift * V);
          cf_spectrum_t h = nullptr, one = nullptr;
          CHECK(cf_set_plan(c.n, c.plan) == CF_OK);
          CHECK(cf_spectrum_create(c.n, own ? c.count : 1, rec::alloc(V * c.count), 1, nullptr, &h) == CF_OK);
          CHECK(cf_spectrum_create(c.n, 1, rec::alloc(V), 1, nullptr, &one) == CF_OK);
          Bufs single(c.n);
          forget();
          CHECK(cf_conv3d_device(one, single.in, single.out, 1, CF_SCALE_INV_N3, c.precision, nullptr) == CF_OK);
          std::map<std::string, int> tiles;
          for (auto& l : rec::launches) tiles[l.name] = l.ntotal;
          forget();
          cf_pass_times_t t;
          CHECK((timed ? cf_conv3d_device_timed(h, sig, out, c.count, CF_SCALE_INV_N3, c.precision, nullptr, &t)
                       : cf_conv3d_device(h, sig, out, c.count, CF_SCALE_INV_N3, c.precision, nullptr)) == CF_OK);
          unsigned read = 0, written = 0;
          for (size_t j = 0; j < rec::launches.size(); ++j) {
            const rec::Launch& l = rec::launches[j];
            const unsigned nb = l.ntotal / tiles[l.name];
            if (rec::base(l.out) == buf) written += nb;
            if (rec::base(l.in) != buf) continue;
            read += nb;
            for (size_t i = 0; i <= j; ++i) {
              const rec::Launch& w = rec::launches[i];
              if (rec::base(w.out) == buf)
                CHECK(w.out >= l.in + nb * V || l.in >= w.out + w.ntotal / tiles[w.name] * V);
            }
          }
          CHECK(read == c.count && written == c.count);
          cf_spectrum_destroy(h);
          cf_spectrum_destroy(one);
        }
}

// What is kept for later calls can be given back, and is made again when needed.
static void trim() {
  CHECK(cf_set_plan(256, CF_PLAN_AXIS5) == CF_OK);
  Bufs b(256);
  cf_spectrum_t h = nullptr;
  CHECK(cf_spectrum_create(256, 1, b.in, 1, nullptr, &h) == CF_OK);
  const size_t held = rec::held - cube(256);
  hipStream_t s = rec::new_stream();
  for (int k = 0; k < 2; ++k) {
    CHECK(fft(256, b, s) == CF_OK);
    if (h) cf_spectrum_destroy(h);
    h = nullptr;
    CHECK(rec::held > held);
    rec::begin_capture(s, hipStreamCaptureModeRelaxed);
    rec::mode = hipStreamCaptureModeRelaxed;
    CHECK(cf_trim() < 0 && rec::held > held);  // (refused, nothing freed)
    rec::mode = hipStreamCaptureModeGlobal;
    rec::end_capture(s);
    rec::faults.clear();
    rec::device_waits = 0;
    CHECK(cf_trim() == CF_OK);
    CHECK(rec::held == held && rec::device_waits > 0 && rec::faults.empty());
  }
  CHECK(cf_spectrum_create(256, 1, b.in, 1, nullptr, &h) == CF_OK);
  CHECK(rec::races() == 0);
}

int main(int argc, char** argv) {
  const struct {
    const char* name;
    void (*run)();
  } checks[] = {{"fft_per_thread", fft_per_thread},
                {"fft_streams", fft_streams},
                {"fft_beside_capture", fft_beside_capture},
                {"fft_first_call", fft_first_call},
                {"conv_per_thread", conv_per_thread},
                {"spectrum_reuse", spectrum_reuse},
                {"conv_overlap", conv_overlap},
                {"trim", trim}};
  CHECK(fpga_initialize("gfx950", "recorded", false) == 0);
  bool found = false;
  for (auto& c : checks)
    if (argc == 2 && !strcmp(argv[1], c.name)) {
      c.run();
      found = true;
    }
  CHECK(found);
  for (auto& f : rec::faults) printf("%s\n", f.c_str());
  if (failures) return 1;
  printf("ok %s\n", argv[1]);
  return 0;
}
