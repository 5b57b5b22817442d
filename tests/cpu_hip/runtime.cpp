// Fibers for the threads of a workgroup, and guarded memory (x86-64).
#include <csignal>
#include <map>
#include <string>

#include <sys/mman.h>
#include <unistd.h>

#include "hip/hip_runtime.h"
#include "user_source.h"

namespace cpu_hip {
Index tid, bid;
dim3 grid, block;

namespace {
enum State { RUN, AT_BARRIER, IN_EXCHANGE, DONE };
struct Fiber {
  void* sp;
  char* stack;
  State state;
  unsigned ops;  // wave exchanges entered
};
constexpr size_t STACK = 256 << 10;
std::vector<Fiber> fibers;
void* main_sp;
int cur, nthr;
const char* kernel = "";
const std::function<void()>* body;
uint64_t passed[2][1024];
}  // namespace

extern "C" void cpu_hip_switch(void** save, void* load);
asm(R"(
.globl cpu_hip_switch
cpu_hip_switch:
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

static void yield() {
  cpu_hip_switch(&fibers[cur].sp, main_sp);
  tid = {unsigned(cur), 0, 0};
}

extern "C" void cpu_hip_entry() {
  (*body)();
  fibers[cur].state = DONE;
  cpu_hip_switch(&fibers[cur].sp, main_sp);
  abort();
}

void barrier() {
  fibers[cur].state = AT_BARRIER;
  yield();
}

// Two slots suffice: a lane enters operation op + 1 only when every lane of
// the wave has entered op, and leaves it only when all have entered op + 1.
uint64_t exchange(uint64_t v, int (*src)(int, int), int arg, bool* valid) {
  const int me = cur, w0 = me & ~63;
  const unsigned op = fibers[me].ops++;
  passed[op & 1][me] = v;
  for (;;) {
    bool all = true;
    for (int l = w0; l < w0 + 64 && l < nthr && all; ++l) all = fibers[l].state == DONE || fibers[l].ops > op;
    if (all) break;
    fibers[me].state = IN_EXCHANGE;
    yield();
    fibers[me].state = RUN;
  }
  const int s = src(me & 63, arg);
  *valid = s >= 0 && w0 + s < nthr && fibers[w0 + s].ops > op;
  return *valid ? passed[op & 1][w0 + s] : 0;
}

static void on_fault(int, siginfo_t* si, void*) {
  char b[400];
  const int n = snprintf(b, sizeof b, "out of range at %p: %s, block %u, thread %u\n", si->si_addr, kernel, bid.x, tid.x);
  (void)!write(2, b, n);
  _exit(99);
}

static void catch_faults() {
  static bool done = false;
  if (done) return;
  done = true;
  static char alt[1 << 16];
  stack_t ss{};
  ss.ss_sp = alt;
  ss.ss_size = sizeof alt;
  sigaltstack(&ss, nullptr);
  struct sigaction sa {};
  sa.sa_sigaction = on_fault;
  sa.sa_flags = SA_SIGINFO | SA_ONSTACK;
  sigaction(SIGSEGV, &sa, nullptr);
  sigaction(SIGBUS, &sa, nullptr);
}

static void run_block() {
  for (int t = 0; t < nthr; ++t) {
    Fiber& f = fibers[t];
    void** sp = (void**)(((uintptr_t(f.stack) + STACK) & ~uintptr_t(63)) - 64);
    *sp = (void*)cpu_hip_entry;  // where the first switch returns to
    for (int k = 1; k <= 6; ++k) sp[-k] = nullptr;
    f.sp = sp - 6;
    f.state = RUN;
    f.ops = 0;
  }
  for (int left = nthr; left > 0;) {
    bool ran = false;
    int waiting = 0;
    for (int t = 0; t < nthr; ++t) {
      const State s = fibers[t].state;
      if (s == RUN || s == IN_EXCHANGE) {
        cur = t;
        tid = {unsigned(t), 0, 0};
        ran = true;
        cpu_hip_switch(&main_sp, fibers[t].sp);
        left -= fibers[t].state == DONE;
      }
      waiting += fibers[t].state == AT_BARRIER;
    }
    if (left && waiting == left) {
      for (int t = 0; t < nthr; ++t)
        if (fibers[t].state == AT_BARRIER) fibers[t].state = RUN;
    } else if (!ran) {
      fprintf(stderr, "no thread can go on: %s\n", kernel);
      abort();
    }
  }
}

void launch(const char* name, dim3 g, dim3 b, const std::function<void()>& f) {
  catch_faults();
  kernel = name;
  grid = g;
  block = b;
  body = &f;
  nthr = int(b.x);
  if (g.x == 0 || g.y == 0 || g.z == 0 || nthr == 0 || nthr > 1024 || b.y != 1 || b.z != 1) {
    fprintf(stderr, "bad launch: %s\n", name);
    abort();
  }
  while (fibers.size() < size_t(nthr))
    fibers.push_back({nullptr, (char*)mmap(nullptr, STACK, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0), DONE, 0});
  for (bid.z = 0; bid.z < g.z; ++bid.z)
    for (bid.y = 0; bid.y < g.y; ++bid.y)
      for (bid.x = 0; bid.x < g.x; ++bid.x) run_block();
}
}  // namespace cpu_hip

// 256 pages that fault before and behind; the memory ends at the one behind
// (CPU_HIP_FRONT: begins at the one before) and holds NaN.
static std::map<void*, std::pair<char*, size_t>>& allocations() {
  static std::map<void*, std::pair<char*, size_t>> m;
  return m;
}
extern "C" hipError_t cpu_hip_malloc(void** p, size_t n) {
  const size_t page = 4096, room = (std::max<size_t>(n, 1) + page - 1) / page * page, len = room + 512 * page;
  char* base = (char*)mmap(nullptr, len, PROT_NONE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
  if (base == MAP_FAILED) return hipErrorOutOfMemory;
  char* s = base + 256 * page;
  mprotect(s, room, PROT_READ | PROT_WRITE);
  memset(s, 0xff, room);
  static const bool front = getenv("CPU_HIP_FRONT") != nullptr;
  *p = front ? s : s + room - (n + 15) / 16 * 16;
  allocations()[*p] = {base, len};
  return 0;
}
extern "C" hipError_t cpu_hip_free(void* p) {
  if (!p) return 0;
  const auto it = allocations().find(p);
  if (it == allocations().end()) return hipErrorInvalidValue;
  munmap(it->second.first, it->second.second);
  allocations().erase(it);
  return 0;
}

namespace amr {
int compile_user_source(const char*, int, hipModule_t*, hipFunction_t*, std::string* log) {
  *log = "not on the CPU";
  return 1;
}
const char* user_source_prelude() { return ""; }
}  // namespace amr
