// host_exec.cpp -- runs the library's kernels on the CPU and checks what they
// touch (built with the address sanitizer against hip/hip_runtime.h):
//   * every device buffer is an exact-size heap block, and the LDS of a launch
//     is the first `lds` bytes of an array whose rest is poisoned: an access
//     out of range ends the program with its stack;
//   * buffers start as NaN patterns, LDS too at the start of each block, and
//     so do automatic variables (compiler flag): a value that is used before
//     it is written shows in the result;
//   * blocks and the threads of a block run in three orders (ascending,
//     descending, shuffled); a thread runs until its next barrier, so a
//     missing barrier makes the results differ between the orders;
//   * all threads of a block must wait at the same barrier.
// Input (stdin), a case a line: fields, then the files that hold the input and
// receive the output of each order:
//   plan  name kind n howmany dtype dir r2r is id os od adjoint inplace bytes in out
//         (no bytes: the plan is described only)
//   mixed name count dtype dir inplace lengths bytes in out
//   fault which path   (a small kernel with a fault that must be found)
// Sizes and the values are the caller's (test_host_exec.py).
#include <hip/hip_runtime.h>

#include <sanitizer/asan_interface.h>
#include <sys/mman.h>

#include <algorithm>
#include <cstdio>
#include <fstream>
#include <iostream>
#include <random>
#include <set>
#include <sstream>
#include <string>
#include <vector>

#include "plfft.h"
#include "plfft_gpu.h"

SimIdx threadIdx, blockIdx, blockDim, gridDim;
int sim_cus = 256;
constexpr size_t kLds = 160 * 1024;
namespace plf {
alignas(4096) unsigned char plf_dyn_lds[kLds];
}
using plf::plf_dyn_lds;

// ---------------------------------------------------------------------------
// threads of a block: one stack each, switched by hand
// ---------------------------------------------------------------------------
extern "C" void sim_switch(void **from, void *to);
asm(R"(
.text
.globl sim_switch
sim_switch:
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
)");

namespace {

constexpr size_t kStack = 512 * 1024;
enum { RUN, AT_BLOCK, AT_WAVE, DONE };
struct Thread {
  char *stack = nullptr;
  void *sp = nullptr, *where = nullptr;
  int state = DONE, value = 0;
};
std::vector<Thread> threads;
void *scheduler_sp;
int current;
const std::function<void()> *body_now;
const char *kernel_now;
int order_now;  // 0 ascending, 1 descending, 2 shuffled
std::mt19937 shuffle_rng;

[[noreturn]] void die(const std::string &what) {
  std::fprintf(stderr, "host_exec: %s: block %u thread %u of %s\n", what.c_str(), blockIdx.x,
               threadIdx.x, kernel_now ? kernel_now : "?");
  std::abort();
}

void yield(int state, void *where) {
  Thread &t = threads[current];
  t.state = state;
  t.where = where;
  sim_switch(&t.sp, scheduler_sp);
}

void entry() {
  (*body_now)();
  yield(DONE, nullptr);
}

void start(Thread &t) {
  if (!t.stack) {
    t.stack = static_cast<char *>(mmap(nullptr, kStack, PROT_READ | PROT_WRITE,
                                       MAP_PRIVATE | MAP_ANONYMOUS, -1, 0));
    if (t.stack == MAP_FAILED) die("no memory for a stack");
  }
  __asan_unpoison_memory_region(t.stack, kStack);
  void **sp = reinterpret_cast<void **>(t.stack + kStack - 64);
  *--sp = nullptr;  // alignment: entry() starts as if called
  *--sp = reinterpret_cast<void *>(&entry);
  for (int i = 0; i < 6; ++i) *--sp = nullptr;
  t.sp = sp;
  t.state = RUN;
}

std::vector<int> in_order(int count) {
  std::vector<int> v(count);
  for (int i = 0; i < count; ++i) v[i] = order_now == 1 ? count - 1 - i : i;
  if (order_now == 2) std::shuffle(v.begin(), v.end(), shuffle_rng);
  return v;
}

void run_block(int count) {
  if ((int)threads.size() < count) threads.resize(count);
  for (int i = 0; i < count; ++i) start(threads[i]);
  for (;;) {
    bool ran = false;
    for (int i : in_order(count)) {
      if (threads[i].state != RUN) continue;
      ran = true;
      current = i;
      threadIdx.x = i;
      sim_switch(&scheduler_sp, threads[i].sp);
    }
    for (int w = 0; w < count; w += 64) {  // waves that have met
      const int end = std::min(w + 64, count);
      bool met = true;
      for (int i = w; i < end; ++i) met = met && threads[i].state == AT_WAVE;
      for (int i = w; met && i < end; ++i) {
        if (threads[i].where != threads[w].where) die("lanes of a wave at two places");
        threads[i].state = RUN;
        ran = true;
      }
    }
    if (ran) continue;
    int waiting = 0, done = 0;
    void *where = nullptr;
    for (int i = 0; i < count; ++i) {
      const Thread &t = threads[i];
      threadIdx.x = i;
      if (t.state == DONE) ++done;
      else if (t.state != AT_BLOCK) die("a wave never meets");
      else if (where && t.where != where) die("threads wait at two barriers");
      else where = t.where, ++waiting;
    }
    if (!waiting) return;
    if (done) die("a barrier that some threads have left behind");
    for (int i = 0; i < count; ++i) threads[i].state = RUN;
  }
}

std::set<std::string> kernels_run;

}  // namespace

__attribute__((noinline)) void sim_block_barrier() {
  yield(AT_BLOCK, __builtin_return_address(0));
}
__attribute__((noinline)) void sim_wave_barrier() {
  yield(AT_WAVE, __builtin_return_address(0));
}
__attribute__((noinline)) int sim_lane(int v, int src) {
  void *where = __builtin_return_address(0);
  threads[current].value = v;
  yield(AT_WAVE, where);
  const int got = threads[(current & ~63) + src].value;
  yield(AT_WAVE, where);
  return got;
}
void sim_unsupported(const char *what) { die(std::string("not simulated: ") + what); }

void sim_launch(const char *name, dim3 grid, dim3 block, size_t lds,
                const std::function<void()> &body) {
  kernel_now = name;
  kernels_run.insert(name);
  if (block.x < 1 || block.x > 1024 || lds > kLds || grid.x < 1) die("launch out of range");
  body_now = &body;
  blockDim.x = block.x;
  gridDim.x = grid.x;
  for (int b : in_order((int)grid.x)) {
    blockIdx.x = b;
    __asan_unpoison_memory_region(plf_dyn_lds, kLds);
    memset(plf_dyn_lds, 0xff, kLds);
    __asan_poison_memory_region(plf_dyn_lds + lds, kLds - lds);
    run_block((int)block.x);
  }
}

hipError_t sim_malloc(void **p, size_t bytes) {
  if (posix_memalign(p, 256, bytes ? bytes : 1)) return hipErrorInvalidValue;
  memset(*p, 0xff, bytes);
  return hipSuccess;
}
hipError_t hipFree(void *p) {
  free(p);
  return hipSuccess;
}

// ---------------------------------------------------------------------------
// cases
// ---------------------------------------------------------------------------
namespace {

std::vector<char> read_file(const std::string &path) {
  std::ifstream f(path, std::ios::binary);
  if (!f) die("cannot read " + path);
  return std::vector<char>(std::istreambuf_iterator<char>(f), {});
}
void write_file(const std::string &path, const char *p, size_t n) {
  std::ofstream f(path, std::ios::binary);
  f.write(p, (std::streamsize)n);
}

// The output in three orders: all must agree. `out_bytes` of output start as
// 0xA5; in place, the output starts as the input (then padded).
template <class Run>
void in_three_orders(const std::string &name, const std::string &in_path,
                     const std::string &out_path, size_t out_bytes, bool inplace, Run &&run) {
  const std::vector<char> in = read_file(in_path);
  std::vector<char> first;
  for (order_now = 0; order_now < 3; ++order_now) {
    const size_t ib = inplace ? std::max(in.size(), out_bytes) : in.size();
    char *di, *dout;
    sim_malloc(reinterpret_cast<void **>(&di), ib);
    if (ib > in.size()) memset(di + in.size(), 0xa5, ib - in.size());
    memcpy(di, in.data(), in.size());
    if (inplace) {
      dout = di;
    } else {
      sim_malloc(reinterpret_cast<void **>(&dout), out_bytes);
      memset(dout, 0xa5, out_bytes);
    }
    run(di, dout);
    const std::vector<char> got(dout, dout + out_bytes);
    if (!inplace && memcmp(di, in.data(), in.size())) die(name + ": the input was written");
    if (order_now == 0) {
      first = got;
      write_file(out_path, got.data(), got.size());
    } else if (got != first) {
      die(name + ": the result depends on the order of the threads");
    }
    if (!inplace) hipFree(dout);
    hipFree(di);
  }
  order_now = 0;
}

plfft_data_type_t type_of(const std::string &s) {
  if (s == "f32") return PLFFT_DATA_TYPE_FP32;
  if (s == "f64") return PLFFT_DATA_TYPE_FP64;
  if (s == "f16") return PLFFT_DATA_TYPE_FP16;
  if (s == "bf16") return (plfft_data_type_t)5;
  if (s == "q15") return PLFFT_DATA_TYPE_Q15;
  return PLFFT_DATA_TYPE_Q7;
}

void run_plan(std::istringstream &l) {
  std::string name, kind, dtype, in, out;
  int64_t n, hm, is, id, os, od, bytes;
  int dir, r2r, adjoint, inplace;
  l >> name >> kind >> n >> hm >> dtype >> dir >> r2r >> is >> id >> os >> od >> adjoint >>
      inplace >> bytes >> in >> out;
  plfft_config_t *c = nullptr;
  const plfft_status_t made = kind == "c2c"   ? plfft_config_create(&c, n, (plfft_direction_t)dir)
                              : kind == "r2c" ? plfft_config_create_r2c(&c, n)
                              : kind == "c2r" ? plfft_config_create_c2r(&c, n)
                                              : plfft_config_create_r2r(&c, n, (plfft_r2r_kind_t)r2r);
  if (made != PLFFT_OK) die(name + ": no configuration");
  plfft_config_set_data_type(c, type_of(dtype));
  plfft_config_set_io_alias(c, inplace ? PLFFT_IO_MAY_ALIAS : PLFFT_IO_NO_ALIAS);
  plfft_config_set_batch(c, hm, is, id, os, od);
  plfft_config_set_rigor(c, PLFFT_ESTIMATE);
  plfft_plan_t *p = nullptr;
  const plfft_status_t st = plfft_plan_create_from_config(&p, c);
  if (st != PLFFT_OK) die(name + ": no plan: " + plfft_last_error());
  char buf[4096];
  plfft_plan_describe(p, buf, sizeof(buf));
  std::printf("%s %s\n", name.c_str(), buf);
  std::fflush(stdout);
  if (bytes) in_three_orders(name, in, out, (size_t)bytes, inplace, [&](void *di, void *dout) {
    const plfft_status_t e = adjoint
                                 ? plfft_plan_execute_adjoint_async(p, di, dout, nullptr, nullptr)
                                 : plfft_plan_execute_async(p, di, dout, nullptr, nullptr);
    if (e != PLFFT_OK) die(name + ": " + plfft_last_error());
  });
  plfft_plan_destroy(p);
  plfft_config_destroy(c);
}

void run_mixed(std::istringstream &l) {
  std::string name, dtype, in, out;
  int64_t count, bytes;
  int dir, inplace;
  l >> name >> count >> dtype >> dir >> inplace;
  std::vector<int64_t> n((size_t)count);
  for (auto &v : n) l >> v;
  l >> bytes >> in >> out;
  plfft_mixed_plan_t *p = nullptr;
  if (plfft_mixed_plan_create(&p, count, n.data(), nullptr, nullptr, (plfft_direction_t)dir,
                              type_of(dtype), PLFFT_ESTIMATE) != PLFFT_OK)
    die(name + ": no plan: " + plfft_last_error());
  char buf[4096];
  plfft_mixed_plan_describe(p, buf, sizeof(buf));
  std::printf("%s %s\n", name.c_str(), buf);
  std::fflush(stdout);
  in_three_orders(name, in, out, (size_t)bytes, inplace, [&](void *di, void *dout) {
    if (plfft_mixed_plan_execute_async(p, di, dout, nullptr, nullptr) != PLFFT_OK)
      die(name + ": " + plfft_last_error());
  });
  plfft_mixed_plan_destroy(p);
}

// Kernels with one fault each; `out` holds 64 ints. 0: none.
void run_fault(int which, const std::string &path) {
  write_file(path + ".in", reinterpret_cast<const char *>(&which), sizeof(which));
  in_three_orders("fault", path + ".in", path, 64 * sizeof(int), false, [&](void *, void *dout) {
    int *out = static_cast<int *>(dout);
    sim_launch("fault", dim3(1), dim3(64), 64 * sizeof(int), [=] {
      volatile int *l = reinterpret_cast<volatile int *>(plf_dyn_lds);
      const int t = (int)threadIdx.x;
      l[t] = t;
      if (which == 1) l[t + 1] = t;                  // past the launch's LDS
      if (which != 2) __syncthreads();               // 2: no barrier
      if (which == 3 && t < 32) __syncthreads();     // a barrier for some
      out[which == 4 ? t + 1 : t] = l[63 - t];       // 4: past the buffer
    });
  });
}

}  // namespace

int main() {
  std::string line;
  while (std::getline(std::cin, line)) {
    std::istringstream l(line);
    std::string what;
    if (!(l >> what)) continue;
    if (what == "cus") l >> sim_cus;
    else if (what == "plan") run_plan(l);
    else if (what == "mixed") run_mixed(l);
    else {
      int which;
      std::string path;
      l >> which >> path;
      run_fault(which, path);
    }
  }
  for (const std::string &k : kernels_run) std::printf("kernel %s\n", k.c_str());
  return 0;
}
