// Runs the workgroups of a launch on the CPU (see hip/hip_runtime.h).
//
// A workgroup is a thread, so that workgroups that wait for each other make progress together; its lanes are fibers, each
// run until it waits: for its wave (a shuffle, a ballot, a DPP move), for its workgroup (a barrier) or for another
// workgroup (a sleep, or an atomic load that may be polling).  A wave operation is carried out once no lane of the wave
// can run, for the lanes that wait at the same call; of several calls the one that stands first in the code goes first,
// which lets the lanes still inside a loop finish it before those behind it go on.
//
// EMU_CUS: compute units of the device (256).  EMU_TRACE: print every launch.  EMU_GIVE_UP: waits inside launches of the
// kernel of this name run out at their first look at the clock.  EMU_ERROR_BEHIND=name:launch:block:look: in that
// launch (1, 2, ...) of those with this in their names, another workgroup sets the error word right behind that look (1, 2, ...) that
// the first wave of that workgroup takes at it; a wave of the workgroup that sees it at the same point ends the run.
#include <hip/hip_runtime.h>

#include <sched.h>
#include <sys/mman.h>
#include <time.h>

#include <chrono>
#include <condition_variable>
#include <mutex>
#include <thread>
#include <vector>

int emu_cus = getenv("EMU_CUS") ? atoi(getenv("EMU_CUS")) : 256;

// Callee-saved registers on the stack, then the other stack.
extern "C" void emu_switch(void** save, void* to);
asm(R"(
.text
.globl emu_switch
.type emu_switch,@function
emu_switch:
  pushq %rbp
  pushq %rbx
  pushq %r12
  pushq %r13
  pushq %r14
  pushq %r15
  movq %rsp,(%rdi)
  movq %rsi,%rsp
  popq %r15
  popq %r14
  popq %r13
  popq %r12
  popq %rbx
  popq %rbp
  ret
)");

namespace emu {

thread_local Lane* cur;
thread_local dim3 bid;
dim3 bdim, gdim;
thread_local void* dyn;

enum State { kReady, kWave, kBlock, kSpin, kDone };
struct Fiber {
  Lane l;
  void* sp;
  State st;
  const void* site;
  uint64_t v, mask;
  const uint64_t* all;
  int any, every;
};
struct Worker {
  std::vector<std::pair<const void*, void*>> shared;
  std::vector<Fiber> f;
  std::vector<uint64_t> vals;
  const std::function<void()>* body;
  void* main_sp;
  Fiber* now = nullptr;
  char* stacks = nullptr;
  size_t n_stacks = 0;
  unsigned loads = 0, barriers = 0;  // (barriers: that the workgroup has passed)
  bool spinning;
};
static thread_local Worker* W;
static const bool g_trace = getenv("EMU_TRACE") != nullptr;
static bool g_give_up;
static int g_look;          // the look at the error word behind which it is set; 0: none
static unsigned g_look_block;
static unsigned g_look_barriers;
static int g_looks_of[1024];  // looks that the lanes of that workgroup have taken
constexpr size_t kStack = 64 * 1024;

static void to_main() {
  Fiber* f = W->now;
  emu_switch(&f->sp, W->main_sp);
}
extern "C" void emu_fiber_main() {
  (*W->body)();
  W->now->st = kDone;
  to_main();
  abort();
}
uint64_t wave_op(const void* site, uint64_t v, const uint64_t** all) {
  Fiber* f = W->now;
  f->site = site;
  f->v = v;
  f->st = kWave;
  to_main();
  *all = f->all;
  return f->mask;
}
void block_op(const void* site, int v, int* any, int* every) {
  Fiber* f = W->now;
  f->site = site;
  f->v = (uint64_t)(v != 0);
  f->st = kBlock;
  to_main();
  *any = f->any;
  *every = f->every;
}
void yield_spin() {
  if (!W) return;
  W->now->st = kSpin;
  W->spinning = true;
  to_main();
}
void load_yield() {
  if (W && (++W->loads & 7) == 0) yield_spin();
}
// Static LDS: an allocation of its own per workgroup, so that the sanitizer sees its end.
void* shared_at(const void* key, size_t bytes) {
  for (auto& e : W->shared)
    if (e.first == key) return e.second;
  const size_t n = (bytes + 15) / 16 * 16;
  void* p = aligned_alloc(16, n);
  memset(p, 0xC7, n);
  W->shared.push_back({key, p});
  return p;
}

static void run_block(Worker& w, int threads) {
  if (w.n_stacks < (size_t)threads) {
    if (w.stacks) munmap(w.stacks, w.n_stacks * kStack);
    w.stacks = (char*)mmap(nullptr, threads * kStack, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
    w.n_stacks = threads;
  }
  w.barriers = 0;
  const int waves = (threads + 63) / 64;
  w.f.resize(threads);
  w.vals.resize((size_t)waves * 64);
  for (int t = 0; t < threads; ++t) {
    Fiber& f = w.f[t];
    f.l.tid = dim3(t % bdim.x, t / bdim.x % bdim.y, t / bdim.x / bdim.y);
    f.l.lane = t & 63;
    f.st = kReady;
    void** sp = (void**)(w.stacks + (size_t)(t + 1) * kStack - 64);
    *--sp = nullptr;
    *--sp = (void*)emu_fiber_main;
    for (int i = 0; i < 6; ++i) *--sp = nullptr;
    f.sp = sp;
  }
  for (int done = 0, idle = 0; done < threads;) {
    bool progress = false;
    w.spinning = false;
    for (int a = 0; a < threads; a += 64) {
      const int b = std::min(threads, a + 64);
      for (;;) {
        bool spin = false;
        for (int t = a; t < b; ++t) {
          Fiber& f = w.f[t];
          if (f.st != kReady && f.st != kSpin) continue;
          const bool was_spin = f.st == kSpin;
          w.now = &f;
          cur = &f.l;
          f.st = kReady;
          emu_switch(&w.main_sp, f.sp);
          if (f.st == kSpin) spin = true;
          if (!(was_spin && f.st == kSpin)) progress = true;
          if (f.st == kDone) ++done;
        }
        if (spin) break;  // (come back to it in the next round)
        const void* site = nullptr;
        for (int t = a; t < b; ++t)
          if (w.f[t].st == kWave && (!site || w.f[t].site < site)) site = w.f[t].site;
        if (!site) break;
        uint64_t mask = 0;
        for (int t = a; t < b; ++t)
          if (w.f[t].st == kWave && w.f[t].site == site) {
            mask |= 1ull << (t - a);
            w.vals[t] = w.f[t].v;
          }
        for (int t = a; t < b; ++t)
          if (mask >> (t - a) & 1) {
            w.f[t].mask = mask;
            w.f[t].all = &w.vals[a];
            w.f[t].st = kReady;
          }
        progress = true;
      }
    }
    bool all_wait = true;
    int waiting = 0, any = 0, every = 1;
    const void* site = nullptr;
    for (auto& f : w.f) {
      if (f.st == kDone) continue;
      if (f.st != kBlock) {
        all_wait = false;
        break;
      }
      if (waiting++ && site != f.site) {
        fprintf(stderr, "emulator: the lanes of a workgroup stand at different barriers\n");
        abort();
      }
      site = f.site;
      any |= (int)f.v;
      every &= (int)f.v;
    }
    if (all_wait && waiting) {
      ++w.barriers;
      for (auto& f : w.f)
        if (f.st == kBlock) {
          f.any = any;
          f.every = every;
          f.st = kReady;
        }
      progress = true;
    }
    if (progress) {
      idle = 0;
    } else if (w.spinning) {
      sched_yield();
      if (++idle > 64) {
        timespec ts{0, 20000};
        nanosleep(&ts, nullptr);
      }
    } else {
      fprintf(stderr, "emulator: no lane of a workgroup can go on\n");
      abort();
    }
  }
}

// The threads take the workgroups of a launch in order.
static std::mutex mu;
static std::condition_variable cv, cv_done;
static std::vector<std::thread> pool;
static uint64_t epoch;
static std::atomic<int64_t> next_block;
static int64_t n_blocks;
static int busy, wanted;
static const std::function<void()>* g_body;
static size_t g_lds;

static void worker(int id) {
  Worker w;
  W = &w;
  uint64_t seen = 0;
  for (;;) {
    {
      std::unique_lock<std::mutex> l(mu);
      cv.wait(l, [&] { return epoch != seen; });
      seen = epoch;
      if (id >= wanted) continue;
    }
    for (;;) {
      const int64_t b = next_block.fetch_add(1);
      if (b >= n_blocks) break;
      bid = dim3((unsigned)(b % gdim.x), (unsigned)(b / gdim.x % gdim.y), (unsigned)(b / gdim.x / gdim.y));
      const size_t bytes = (g_lds + 15) / 16 * 16;
      dyn = bytes ? aligned_alloc(16, bytes) : nullptr;
      if (bytes) memset(dyn, 0xC7, bytes);
      w.body = g_body;
      run_block(w, bdim.x * bdim.y * bdim.z);
      free(dyn);
      for (auto& e : w.shared) free(e.second);
      w.shared.clear();
    }
    std::lock_guard<std::mutex> l(mu);
    if (--busy == 0) cv_done.notify_all();
  }
}
void run(const char* name, dim3 g, dim3 b, size_t lds, const std::function<void()>& body) {
  if (g_trace) fprintf(stderr, "launch %.90s grid %u %u %u block %u lds %zu\n", name, g.x, g.y, g.z, b.x, lds);
  if (b.x * b.y * b.z > 1024 || !g.x || !g.y || !g.z || lds > 160 * 1024 || g.y > 65535 || g.z > 65535) {
    fprintf(stderr, "emulator: a launch of %s that the device would refuse\n", name);
    abort();
  }
  const char* give_up = getenv("EMU_GIVE_UP");
  g_give_up = give_up != nullptr && strcmp(give_up, name) == 0;
  char behind[100] = "";
  int launch = 0, look = 0;
  g_look = 0;
  if (const char* e = getenv("EMU_ERROR_BEHIND"); e && sscanf(e, "%99[^:]:%d:%u:%d", behind, &launch, &g_look_block, &look) == 4 && strstr(name, behind)) {
    static int launches;
    if (++launches == launch) g_look = look;
    memset(g_looks_of, 0, sizeof(g_looks_of));
    g_look_barriers = ~0u;
  }
  std::unique_lock<std::mutex> l(mu);
  gdim = g;
  bdim = b;
  g_body = &body;
  g_lds = lds;
  n_blocks = (int64_t)g.x * g.y * g.z;
  next_block = 0;
  // (a grid whose workgroups wait for each other is resident at once: at most a few hundred)
  wanted = (int)(n_blocks <= 1200 ? n_blocks : 8);
  while ((int)pool.size() < wanted) {
    const int id = (int)pool.size();
    pool.emplace_back(worker, id);
    pool.back().detach();
  }
  busy = wanted;
  ++epoch;
  cv.notify_all();
  cv_done.wait(l, [&] { return busy == 0; });
}

}  // namespace emu

// A slow clock (workgroups take turns on the CPU), or one on which every wait runs out.
long long wall_clock64() {
  static std::atomic<long long> leap{0};
  if (emu::g_give_up) return (leap += 1ll << 40) | 1;
  return (std::chrono::duration_cast<std::chrono::nanoseconds>(std::chrono::steady_clock::now().time_since_epoch()).count() / 100000) | 1;
}

int emu_error_word(const int* p, int failed) {
  if (emu::g_look == 0 || blockIdx.x != emu::g_look_block) return emu_aload(p);
  const int v = __atomic_load_n(p, __ATOMIC_SEQ_CST);  // (no lane lets the others go on here: the first wave looks first)
  const int look = ++emu::g_looks_of[threadIdx.x];
  if (threadIdx.x == 0 && look == emu::g_look) {
    fprintf(stderr, "another workgroup gives up\n");
    emu_astore(const_cast<int*>(p), failed);
    emu::g_look_barriers = emu::W->barriers;
  } else if (threadIdx.x < 64) {
    return look == emu::g_look ? 0 : v;  // (the lanes of a wave look together)
  } else if (v != 0 && look <= emu::g_look && emu::W->barriers == emu::g_look_barriers) {
    fprintf(stderr, "emulator: the waves of a workgroup see different error words\n");
    abort();
  }
  return v;
}

using emu::block_op;
using emu::wave_op;
constexpr uint64_t kNobody = 0xDEADBEEFDEADBEEFull;  // what a lane reads from a lane that takes no part

uint64_t emu_ballot(bool p) {
  const uint64_t* a;
  const uint64_t m = wave_op(EMU_SITE, p, &a);
  uint64_t r = 0;
  for (int i = 0; i < 64; ++i)
    if ((m >> i & 1) && a[i]) r |= 1ull << i;
  return r;
}
uint64_t emu_read(uint64_t v, int lane) {
  const uint64_t* a;
  const uint64_t m = wave_op(EMU_SITE, v, &a);
  return (m >> (lane & 63) & 1) ? a[lane & 63] : kNobody;
}
uint64_t emu_first(uint64_t v) {
  const uint64_t* a;
  const uint64_t m = wave_op(EMU_SITE, v, &a);
  return a[__builtin_ctzll(m)];
}
uint64_t emu_shfl(uint64_t v, int x, int mode) {
  const uint64_t* a;
  const uint64_t m = wave_op(EMU_SITE, v, &a);
  const int me = emu::cur->lane, s = mode == 0 ? x & 63 : mode == 1 ? me - x : me ^ x;
  if (s < 0 || s > 63) return v;
  return (m >> s & 1) ? a[s] : kNobody;
}
int emu_dpp(int old, int v, int ctrl, int row_mask, int bank_mask, bool bound) {
  const uint64_t* a;
  const uint64_t m = wave_op(EMU_SITE, (uint32_t)v, &a);
  const int me = emu::cur->lane, row = me >> 4, in = me & 15, by = ctrl & 15;
  int s = -1;
  if (ctrl < 0x100)
    s = (me & ~3) | ((ctrl >> (2 * (me & 3))) & 3);  // quad_perm
  else if (ctrl >= 0x101 && ctrl <= 0x10F)
    s = in + by < 16 ? me + by : -1;  // row_shl
  else if (ctrl >= 0x111 && ctrl <= 0x11F)
    s = in >= by ? me - by : -1;  // row_shr
  else if (ctrl >= 0x121 && ctrl <= 0x12F)
    s = (me & ~15) | ((in - by) & 15);  // row_ror
  else if (ctrl == 0x130)
    s = me < 63 ? me + 1 : -1;  // wave_shl
  else if (ctrl == 0x138)
    s = me - 1;  // wave_shr
  else if (ctrl == 0x140)
    s = (me & ~15) | (15 - in);  // row_mirror
  else if (ctrl == 0x141)
    s = (me & ~7) | (7 - (me & 7));  // row_half_mirror
  else if (ctrl == 0x142)
    s = row == 0 ? -1 : row * 16 - 1;  // row_bcast 15
  else if (ctrl == 0x143)
    s = row < 2 ? -1 : 31;  // row_bcast 31
  else
    abort();
  if (!(row_mask >> row & 1) || !(bank_mask >> (in >> 2) & 1)) return old;
  if (s < 0 || !(m >> s & 1)) return bound ? 0 : old;
  return (int)(uint32_t)a[s];
}
void emu_sync() {
  int any, every;
  block_op(EMU_SITE, 0, &any, &every);
}
int emu_sync_or(int x) {
  int any, every;
  block_op(EMU_SITE, x, &any, &every);
  return any;
}
int emu_sync_and(int x) {
  int any, every;
  block_op(EMU_SITE, x, &any, &every);
  return every;
}
