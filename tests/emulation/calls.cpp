// calls [-o name=value]... kind:n:m:data[:populations][:rows kept][:repeats][:poisoned] ...
// Calls of the library on the emulated device, each against the C checker.  The workspace starts out filled with a pattern
// and is used by one call after the other, as a program does.  poisoned: a wait of the call runs out, its results say so.
#include <unistd.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>
#include <vector>
#include <random>
#include <cmath>
#include <chrono>
#include "evox_hip.h"
#include <sanitizer/asan_interface.h>
extern "C" int oracle_nd_rank(const float* f, int64_t n, int m, int32_t* rank);
extern "C" int oracle_first_front(const float* f, int64_t n, int m, uint8_t* mask);
extern "C" int oracle_crowding(const float* costs, int64_t n, int m, const uint8_t* mask, float* dist);
extern "C" int oracle_select(const float* f, int64_t n, int m, int64_t topk, int32_t* rank, float* dist, int64_t* order);
extern "C" __attribute__((no_sanitize("address"))) const char* __asan_default_options() { return "detect_stack_use_after_return=0:detect_leaks=0:abort_on_error=0:allocator_may_return_null=1:quarantine_size_mb=64:use_sigaltstack=0:print_legend=0"; }
static std::mt19937_64 rng;
static double U() { return (rng() >> 11) * (1.0 / 9007199254740992.0); }
static double N() { double u = U(), v = U(); return std::sqrt(-2 * std::log(1 - u)) * std::cos(6.283185307179586 * v); }
static void fill(const std::string& data, float* f, int64_t n, int m) {
  for (int64_t i = 0; i < n; ++i) {
    float* r = f + i * m;
    if (data == "uniform") for (int k = 0; k < m; ++k) r[k] = (float)U();
    else if (data == "grid") for (int k = 0; k < m; ++k) r[k] = (float)(rng() % 8);
    else if (data == "equal") for (int k = 0; k < m; ++k) r[k] = 1.0f;
    else if (data == "chain") for (int k = 0; k < m; ++k) r[k] = (float)((i * 7919) % n);
    else if (data == "nan") for (int k = 0; k < m; ++k) r[k] = (rng() % 50) ? (float)U() : (rng() % 2 ? NAN : (rng() % 2 ? INFINITY : -INFINITY));
    else if (data == "inf") for (int k = 0; k < m; ++k) r[k] = (rng() % 5) ? (float)(rng() % 4) : INFINITY;
    else if (data == "layers") { float l = (float)(i * 20 / n) + 1; r[0] = std::round((float)U() * l * 64) / 64; r[1] = l - r[0]; for (int k = 2; k < m; ++k) r[k] = 0; }
    else {
      double s = 0, q = 0; std::vector<double> d(m); for (auto& v : d) { v = std::fabs(N()); s += v; q += v * v; }
      const double mean = m <= 3 ? 0.1 : 0.05, rad = data == "simplex" ? 1 / s : (1 - mean * std::log1p(-U())) / std::sqrt(q);
      for (int k = 0; k < m; ++k) r[k] = (float)(d[k] * rad);
    }
  }
}
template <class T> struct Buf { T* p; size_t n; Buf(size_t c) : n(c) { p = (T*)aligned_alloc(256, 256); free(p); if (posix_memalign((void**)&p, 16, c * sizeof(T) ? c * sizeof(T) : 1)) abort(); memset(p, 0xC7, c * sizeof(T)); } ~Buf() { free(p); } };
static uint8_t* ws = nullptr; static size_t ws_bytes = 0;
static uint8_t* workspace(size_t need) {
  if (need > ws_bytes) { if (ws) { __asan_unpoison_memory_region(ws, ws_bytes); free(ws); } void* p; if (posix_memalign(&p, 256, need)) abort(); ws = (uint8_t*)p; ws_bytes = need; for (size_t i = 0; i < need; i += 8) { uint64_t v = 0xC7C7C7C7C7C7C7C7ull; memcpy(ws + i, &v, std::min<size_t>(8, need - i)); } }
  else { __asan_unpoison_memory_region(ws, ws_bytes); }
  return ws;
}
static double now() { return std::chrono::duration<double>(std::chrono::steady_clock::now().time_since_epoch()).count(); }
#define DIE(...) do { fprintf(stderr, __VA_ARGS__); fprintf(stderr, "\n"); fflush(stdout); _exit(1); } while (0)
int main(int argc, char** argv) {
  for (int a = 1; a < argc; ++a) {
    std::string s = argv[a];
    if (s == "-o") { std::string o = argv[++a]; auto q = o.find('='); if (evox_hip_set_option(o.substr(0, q).c_str(), atoll(o.c_str() + q + 1))) DIE("option %s", o.c_str()); continue; }
    std::vector<std::string> p; size_t at = 0; for (;;) { auto q = s.find(':', at); p.push_back(s.substr(at, q == std::string::npos ? q : q - at)); if (q == std::string::npos) break; at = q + 1; }
    const std::string kind = p[0]; const int64_t n = atoll(p[1].c_str()); const int m = atoi(p[2].c_str()); const std::string data = p[3];
    const int64_t b = p.size() > 4 && !p[4].empty() ? atoll(p[4].c_str()) : 1; int64_t k = p.size() > 5 && !p[5].empty() ? atoll(p[5].c_str()) : (n / 2 > 0 ? n / 2 : 1);
    const int repeats = p.size() > 6 && !p[6].empty() ? atoi(p[6].c_str()) : 1;
    const bool poisoned = p.size() > 7 && p[7] == "poisoned";
    const int d = 7;
    rng.seed(1234 + n * 31 + m);
    Buf<float> f((size_t)b * n * m), x((size_t)b * n * d);
    for (size_t i = 0; i < x.n; ++i) x.p[i] = (float)i;
    for (int64_t c = 0; c < b; ++c) fill(data, f.p + c * n * m, n, m);
    std::vector<std::vector<int32_t>> orank(b); std::vector<std::vector<float>> odist(b); std::vector<std::vector<int64_t>> oorder(b);
    double t0 = now();
    const bool sel = kind == "select" || kind == "batch" || kind == "twopart" || kind == "select64";
    if (sel) for (int64_t c = 0; c < b; ++c) { orank[c].resize(n); odist[c].resize(n); oorder[c].resize(n); if (oracle_select(f.p + c * n * m, n, m, k, orank[c].data(), odist[c].data(), oorder[c].data()) < 0) DIE("oracle"); }
    double t1 = now();
    for (int rep = 0; rep < repeats; ++rep) {
      fprintf(stderr, "%s rep %d\n", s.c_str(), rep);
      int e = 0;
      if (sel) {
        Buf<float> ox((size_t)b * k * d), of((size_t)b * k * m), od((size_t)b * k); Buf<int32_t> orr((size_t)b * k);
        Buf<double> f64(kind == "select64" ? (size_t)n * m : 0), of64(kind == "select64" ? (size_t)k * m : 0), od64(kind == "select64" ? (size_t)k : 0);
        if (kind == "select") {
          uint8_t* w = workspace(evox_hip_workspace_bytes(n, m));
          e = evox_hip_nd_environmental_selection(x.p, d * 4, d * 4, f.p, n, m, m, 1, k, ox.p, of.p, orr.p, od.p, nullptr, w, ws_bytes, nullptr);
        } else if (kind == "twopart") {
          uint8_t* w = workspace(evox_hip_workspace_bytes(n, m)); const int64_t h = n / 3;
          e = evox_hip_nd_environmental_selection_two_part(x.p, d * 4, x.p + h * d, d * 4, d * 4, f.p, h, m, 1, f.p + h * m, n - h, m, 1, m, k, ox.p, of.p, orr.p, od.p, nullptr, w, ws_bytes, nullptr);
        } else if (kind == "select64") {
          for (size_t i = 0; i < f64.n; ++i) f64.p[i] = f.p[i];
          uint8_t* w = workspace(evox_hip_workspace_bytes(n, m));
          e = evox_hip_nd_environmental_selection_wide_whole(x.p, d * 4, d * 4, f64.p, m * 8, m * 8, f64.p, 0, n, m, m, 1, k, ox.p, of64.p, orr.p, od64.p, 0, w, ws_bytes, nullptr);
          for (size_t i = 0; i < of.n; ++i) of.p[i] = (float)of64.p[i];
          for (size_t i = 0; i < od.n; ++i) od.p[i] = (float)od64.p[i];
        } else if (n <= evox_hip_batched_max_rows(m)) {
          e = evox_hip_batched_nd_environmental_selection(x.p, d * 4, d * 4, n * d * 4, f.p, b, n, m, n * m, m, 1, k, ox.p, of.p, orr.p, od.p, nullptr);
        } else {
          const int64_t per = evox_hip_many_populations_per_launch(b, n, m, k);
          size_t need = evox_hip_many_workspace_bytes(b, n, m, k);
          uint8_t* w = workspace(need);
          for (int64_t b0 = 0; b0 < b && !e; b0 += per) { const int64_t nb = std::min(per, b - b0);
            __asan_unpoison_memory_region(ws, ws_bytes);
            e = evox_hip_many_nd_environmental_selection(x.p + b0 * n * d, d * 4, d * 4, n * d * 4, f.p + b0 * n * m, nb, n, m, n * m, m, 1, k, ox.p + b0 * k * d, of.p + b0 * k * m, orr.p + b0 * k, od.p + b0 * k, w, ws_bytes, nullptr); }
        }
        if (e) DIE("error %d", e);
        if (poisoned) { for (size_t i = 0; i < orr.n; ++i) if (orr.p[i] != -1 || od.p[i] == od.p[i]) DIE("a result in place %ld", (long)i); int32_t status[8]; if (evox_hip_read_status(ws, nullptr, status) != -3) DIE("the status tells nothing"); continue; }
        for (int64_t c = 0; c < b; ++c) for (int64_t i = 0; i < k; ++i) {
          const int64_t o = oorder[c][i];
          const float* px = ox.p + (c * k + i) * d;
          if (orr.p[c * k + i] != orank[c][o]) DIE("rank differs pop %ld place %ld: %d want %d", (long)c, (long)i, orr.p[c * k + i], orank[c][o]);
          if (memcmp(of.p + (c * k + i) * m, f.p + (c * n + o) * m, m * 4) && kind != "select64") DIE("fitness differs pop %ld place %ld", (long)c, (long)i);
          if (kind != "select64" && px[0] != x.p[(c * n + o) * d]) DIE("row differs pop %ld place %ld", (long)c, (long)i);
          const float a = od.p[c * k + i], w = odist[c][o];
          if (!(a == w || (a != a && w != w) || std::fabs(a - w) <= 1e-4f * std::fabs(w))) DIE("dist differs pop %ld place %ld %g want %g", (long)c, (long)i, a, w);
        }
      } else if (kind == "rank" || kind == "until") {
        Buf<int32_t> r(n); std::vector<int32_t> want(n);
        uint8_t* w = workspace(evox_hip_workspace_bytes(n, m));
        if (oracle_nd_rank(f.p, n, m, want.data()) < 0) DIE("oracle");
        e = kind == "rank" ? evox_hip_non_dominate_rank(f.p, n, m, m, 1, r.p, w, ws_bytes, nullptr) : evox_hip_non_dominate_rank_until(f.p, n, m, m, 1, k, r.p, w, ws_bytes, nullptr);
        if (e) DIE("error %d", e);
        for (int64_t i = 0; i < n; ++i) if (r.p[i] != want[i] && !(kind == "until" && r.p[i] == 0x7FFFFFFF)) DIE("rank differs %ld: %d want %d", (long)i, r.p[i], want[i]);
      } else if (kind == "mask") {
        Buf<uint8_t> r(n); std::vector<uint8_t> want(n);
        uint8_t* w = workspace(evox_hip_first_front_workspace_bytes(n, m));
        oracle_first_front(f.p, n, m, want.data());
        e = evox_hip_first_front_mask(f.p, n, m, m, 1, r.p, w, ws_bytes, nullptr);
        if (e) DIE("error %d", e);
        for (int64_t i = 0; i < n; ++i) if ((r.p[i] != 0) != (want[i] != 0)) DIE("mask differs %ld", (long)i);
      } else if (kind == "crowd") {
        Buf<float> r(n); std::vector<float> want(n); Buf<uint8_t> mk(n); for (int64_t i = 0; i < n; ++i) mk.p[i] = rng() % 4 != 0;
        uint8_t* w = workspace(evox_hip_workspace_bytes(n, m));
        oracle_crowding(f.p, n, m, mk.p, want.data());
        e = evox_hip_crowding_distance(f.p, n, m, m, 1, mk.p, 1, r.p, w, ws_bytes, nullptr);
        if (e) DIE("error %d", e);
        for (int64_t i = 0; i < n; ++i) { const float a = r.p[i], v = want[i]; if (!(a == v || (a != a && v != v) || std::fabs(a - v) <= 1e-4f * std::fabs(v))) DIE("dist differs %ld %g want %g", (long)i, a, v); }
      } else DIE("kind");
    }
    printf("ok %s  (checker %.1f s, here %.1f s)\n", s.c_str(), t1 - t0, now() - t1); fflush(stdout);
  }
  fflush(stdout); _exit(0);
}
