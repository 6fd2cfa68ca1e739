// Lockstep block execution for the CPU emulation header (hip/hip_runtime.h): every
// thread of a block is a fiber of the calling host thread.  A wavefront's fibers run
// one after another up to its next lane exchange and go on together; wavefronts meet at
// block barriers.  Every second block walks its wavefronts last to first, so that a
// value read in the same phase as it is written shows whichever side runs first.
#include "hip/hip_runtime.h"
#include <sys/mman.h>
#include <cstdio>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <vector>
#if defined(__SANITIZE_ADDRESS__)
#include <sanitizer/common_interface_defs.h>
#endif
thread_local uint3e blockIdx, threadIdx, blockDim, gridDim;
thread_local int emu_lane = 0;

// Saves this stack's registers and its pointer in *from, and goes on where `to` was
// saved (the x86-64 calling convention's kept registers; no system call).
extern "C" void emu_switch(void** from, void* to);
asm(R"(
.text
.type emu_switch, @function
emu_switch:
  pushq %rbp
  pushq %rbx
  pushq %r12
  pushq %r13
  pushq %r14
  pushq %r15
  movq %rsp, (%rdi)
  movq %rsi, %rsp
  popq %r15
  popq %r14
  popq %r13
  popq %r12
  popq %rbx
  popq %rbp
  ret
.size emu_switch, .-emu_switch
)");

namespace {
enum class At { kReady, kExchange, kBarrier, kDone };
constexpr size_t kStack = 512 * 1024;

struct Fiber {
  char* stack = nullptr;
  void* sp = nullptr;
  At at = At::kDone;
  uint3e thread{};
  int lane = 0, wave = 0;
  void* fake = nullptr;
};

struct Block {
  std::vector<Fiber*> fibers;  // made on first use and kept
  void* home = nullptr;  // the scheduler's stack pointer while a fiber runs
  const void* home_bottom = nullptr;
  size_t home_size = 0;
  Fiber* cur = nullptr;
  const std::function<void()>* job = nullptr;
  struct Wave {
    float value[2][64];
    uint64_t ballot[2];
    int phase;  // exchanges of the wavefront so far
  } waves[16];
  long blocks = 0;
};
thread_local Block the_block;

void finish_switch(void* fake) {
#if defined(__SANITIZE_ADDRESS__)
  const void* bottom;
  size_t size;
  __sanitizer_finish_switch_fiber(fake, &bottom, &size);
  if (the_block.cur) {  // arrived in a fiber: the stack left is the scheduler's
    the_block.home_bottom = bottom;
    the_block.home_size = size;
  }
#endif
}

void enter(Fiber* f) {
  Block& b = the_block;
  b.cur = f;
  threadIdx = f->thread;
  emu_lane = f->lane;
  void* fake = nullptr;
#if defined(__SANITIZE_ADDRESS__)
  __sanitizer_start_switch_fiber(&fake, f->stack, kStack);
#endif
  emu_switch(&b.home, f->sp);
  b.cur = nullptr;
  finish_switch(fake);
}

void leave(At at) {
  Block& b = the_block;
  Fiber* f = b.cur;
  f->at = at;
#if defined(__SANITIZE_ADDRESS__)
  __sanitizer_start_switch_fiber(&f->fake, b.home_bottom, b.home_size);
#endif
  emu_switch(&f->sp, b.home);
  finish_switch(f->fake);
}

void fiber_main() {
  finish_switch(nullptr);
  for (;;) {
    (*the_block.job)();
    leave(At::kDone);
  }
}

Fiber* make_fiber() {
  Fiber* f = new Fiber;
  f->stack = (char*)mmap(nullptr, kStack, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
  if (f->stack == MAP_FAILED) { std::fprintf(stderr, "emulation: no stack\n"); std::abort(); }
  void** top = (void**)(f->stack + kStack) - 8;  // six registers, the entry, its (absent) return address
  top[6] = (void*)fiber_main;
  f->sp = top;
  return f;
}

// Runs wavefront w (fibers [lo, hi)) until its live lanes wait at the block barrier
// or are done; true while some are live.
bool run_wave(Block& b, int w, int lo, int hi) {
  for (;;) {
    int exchange = 0, barrier = 0;
    for (int t = lo; t < hi; ++t) {
      Fiber* f = b.fibers[t];
      if (f->at == At::kReady) enter(f);
      exchange += f->at == At::kExchange;
      barrier += f->at == At::kBarrier;
    }
    if (exchange > 0 && barrier > 0) {
      std::fprintf(stderr, "emulation: lanes of one wavefront at an exchange and at a barrier\n");
      std::abort();
    }
    if (exchange == 0) return barrier > 0;
    for (int t = lo; t < hi; ++t)
      if (b.fibers[t]->at == At::kExchange) b.fibers[t]->at = At::kReady;
    b.waves[w].phase += 1;
    b.waves[w].ballot[b.waves[w].phase & 1] = 0;
  }
}

void run_block(const std::function<void()>& job, dim3 b3) {
  Block& b = the_block;
  const int threads = (int)(b3.x * b3.y * b3.z), waves = (threads + 63) / 64;
  if (threads > 1024) { std::fprintf(stderr, "emulation: block of %d threads\n", threads); std::abort(); }
  while ((int)b.fibers.size() < threads) b.fibers.push_back(make_fiber());
  b.job = &job;
  for (int t = 0; t < threads; ++t) {
    Fiber* f = b.fibers[t];
    f->at = At::kReady;
    f->thread = {t % b3.x, (t / b3.x) % b3.y, t / (b3.x * b3.y)};
    f->lane = t % 64;
    f->wave = t / 64;
  }
  for (int w = 0; w < waves; ++w) b.waves[w].phase = 0, b.waves[w].ballot[0] = b.waves[w].ballot[1] = 0;
  const bool backward = (b.blocks++ & 1) != 0;
  for (bool live = true; live;) {
    live = false;
    for (int q = 0; q < waves; ++q) {
      const int w = backward ? waves - 1 - q : q;
      live = run_wave(b, w, w * 64, std::min(threads, w * 64 + 64)) || live;
    }
    for (int t = 0; t < threads; ++t)
      if (b.fibers[t]->at == At::kBarrier) b.fibers[t]->at = At::kReady;
  }
}
}  // namespace

float emu_exchange(float v, int src) {
  Block::Wave& w = the_block.waves[the_block.cur->wave];
  const int slot = w.phase & 1;
  w.value[slot][emu_lane] = v;
  leave(At::kExchange);
  return w.value[slot][src];
}

uint64_t emu_ballot(bool v) {
  Block::Wave& w = the_block.waves[the_block.cur->wave];
  const int slot = w.phase & 1;
  if (v) w.ballot[slot] |= (uint64_t)1 << emu_lane;
  leave(At::kExchange);
  return w.ballot[slot];
}

void emu_barrier() { leave(At::kBarrier); }

void emu_run_grid(dim3 g, dim3 b, const std::function<void()>& job) {
  gridDim = {g.x, g.y, g.z};
  blockDim = {b.x, b.y, b.z};
  for (unsigned z = 0; z < g.z; ++z)
    for (unsigned y = 0; y < g.y; ++y)
      for (unsigned x = 0; x < g.x; ++x) {
        blockIdx = {x, y, z};
        run_block(job, b);
      }
}

namespace {
std::mutex launch_mutex;
std::map<std::string, long>& launch_counts() { static std::map<std::string, long> m; return m; }
}  // namespace

void emu_note_launch(const char* name) {
  std::lock_guard<std::mutex> lock(launch_mutex);
  ++launch_counts()[name];
}

// launches so far of the kernels whose launch expression contains `part`
extern "C" long emu_kernel_launches(const char* part) {
  std::lock_guard<std::mutex> lock(launch_mutex);
  long n = 0;
  for (const auto& kv : launch_counts())
    if (std::strstr(kv.first.c_str(), part)) n += kv.second;
  return n;
}
