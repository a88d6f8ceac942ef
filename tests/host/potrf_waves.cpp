// Runs the diagonal-block Cholesky kernel on the CPU, one fiber per thread of
// the workgroup, with the waves of every barrier interval one after the other
// in an order of the caller's choice: what a wave reads and another one writes
// between the same two barriers then shows in the result.
//   potrf_waves <32|64> <live> <order of the 8 waves, e.g. 01234567> < A (128 x 128) > L, X, info
// The kernel itself is KERNEL_SRC, cut out of the HIP source by the test.
#include <ucontext.h>
#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <vector>

#define __device__
#define __forceinline__ inline
using std::max;
using std::min;
typedef float f4v __attribute__((ext_vector_type(4)));
typedef double d4v __attribute__((ext_vector_type(4)));

constexpr int DB = 128, WAVES = 8, LANES = 64, THREADS = WAVES * LANES;
constexpr size_t STACK = 128 << 10;

enum State { READY, AT_WAVE, AT_BARRIER, DONE };
static ucontext_t sched, ctx[THREADS];
static State state[THREADS];
static int cur;
// what the lanes of a wave bring to a cross-lane operation, and the site of it
static double opa[THREADS], opb[THREADS];
static int64_t opi[THREADS], site[THREADS];

struct Dim { int x; };
#define threadIdx (Dim{cur})

static void yield(State s) {
  const int me = cur;
  state[me] = s;
  swapcontext(&ctx[me], &sched);
}
// All lanes of a wave meet here; a wave whose lanes stand at different
// operations is an error of the harness or of the kernel.
static void meet(int64_t where) {
  site[cur] = where;
  yield(AT_WAVE);
}
static int wave0() { return cur / LANES * LANES; }

static int emu_readlane(int v, int l) {
  opi[cur] = v;
  meet(1);
  const int r = (int)opi[wave0() + l];
  meet(2);                               // nobody overwrites before all have read
  return r;
}
static int emu_readfirstlane(int v) { return emu_readlane(v, 0); }
#define __builtin_amdgcn_readlane emu_readlane
#define __builtin_amdgcn_readfirstlane emu_readfirstlane
#define __builtin_amdgcn_rcpf(x) (1.0f / (x))
#define __builtin_amdgcn_sqrtf(x) std::sqrt(x)
#define __builtin_amdgcn_rsqf(x) (1.0f / std::sqrt(x))
#define __builtin_amdgcn_rsq(x) ((double)(float)(1.0 / std::sqrt(x)))      // a seed good to 2^-24
#define __builtin_amdgcn_sched_barrier(x) ((void)0)
static int __float_as_int(float f) { int i; memcpy(&i, &f, 4); return i; }
static float __int_as_float(int i) { float f; memcpy(&f, &i, 4); return f; }
static int __double2loint(double d) { int64_t i; memcpy(&i, &d, 8); return (int)i; }
static int __double2hiint(double d) { int64_t i; memcpy(&i, &d, 8); return (int)(i >> 32); }
static double __hiloint2double(int hi, int lo) {
  const int64_t i = (int64_t)((uint64_t)(uint32_t)hi << 32 | (uint32_t)lo);
  double d;
  memcpy(&d, &i, 8);
  return d;
}
static unsigned __umul24(int a, int b) { return (unsigned)a * (unsigned)b; }
static int atomicAdd(int* p, int v) { const int o = *p; *p += v; return o; }
static int atomicCAS(int32_t* p, int c, int v) { const int o = *p; if (o == c) *p = v; return o; }
static void __syncthreads() { yield(AT_BARRIER); }

// 16 x 16 x 4 matrix product of a wave: A[l % 16][l / 16], B[l / 16][l % 16];
// lane l holds column l % 16 of C, its rows 4 (l / 16) + r (float) or l / 16 + 4 r (double)
template <typename T, typename V>
static V emu_mfma(T a, T b, V c) {
  opa[cur] = a;
  opb[cur] = b;
  meet(3);
  const int w = wave0(), l = cur - w;
  for (int r = 0; r < 4; ++r) {
    const int row = sizeof(T) == 4 ? 4 * (l / 16) + r : l / 16 + 4 * r;
    T s = c[r];
    for (int k = 0; k < 4; ++k) s += (T)opa[w + 16 * k + row] * (T)opb[w + 16 * k + l % 16];
    c[r] = s;
  }
  meet(4);
  return c;
}
template <typename T> struct Mfma;
template <> struct Mfma<float> {
  using acc_t = f4v;
  static acc_t mma(float a, float b, acc_t c) { return emu_mfma(a, b, c); }
};
template <> struct Mfma<double> {
  using acc_t = d4v;
  static acc_t mma(double a, double b, acc_t c) { return emu_mfma(a, b, c); }
};

#include KERNEL_SRC

template <typename T> struct Job { static T *S, *A, *X; };
template <typename T> T* Job<T>::S;
template <typename T> T* Job<T>::A;
template <typename T> T* Job<T>::X;
static int live;
static int32_t info;

template <typename T>
static void thread_main() {
  potrf_blocked<T, THREADS>(BlkStore<T>{Job<T>::S}, Job<T>::A, DB, Job<T>::X, DB, &info, 0, live);
  yield(DONE);
}

template <typename T>
static int run(const char* order) {
  alignas(16) static T S[BlkStore<T>::SIZE], A[DB * DB], X[DB * DB];
  static_assert(GK_POTRF_NT == THREADS, "the harness runs the kernel's own number of threads");
  std::fill(S, S + BlkStore<T>::SIZE, T(NAN));             // LDS holds nothing of use at the start
  if (fread(A, sizeof(T), DB * DB, stdin) != DB * DB) return 2;
  Job<T>::S = S; Job<T>::A = A; Job<T>::X = X;
  std::vector<char> stacks(STACK * THREADS);
  for (int t = 0; t < THREADS; ++t) {
    getcontext(&ctx[t]);
    ctx[t].uc_stack.ss_sp = &stacks[STACK * t];
    ctx[t].uc_stack.ss_size = STACK;
    ctx[t].uc_link = &sched;
    makecontext(&ctx[t], thread_main<T>, 0);
  }
  while (state[0] != DONE) {                               // one barrier interval
    for (int o = 0; o < WAVES; ++o) {
      const int w = (order[o] - '0') * LANES;
      for (;;) {                                           // the wave, from one meeting to the next
        for (int l = 0; l < LANES; ++l) {
          cur = w + l;
          swapcontext(&sched, &ctx[cur]);
        }
        for (int l = 1; l < LANES; ++l)
          if (state[w + l] != state[w] || (state[w] == AT_WAVE && site[w + l] != site[w])) return 3;
        if (state[w] != AT_WAVE) break;
      }
    }
    for (int t = 1; t < THREADS; ++t)
      if (state[t] != state[0]) return 4;                  // a barrier that not every wave reaches
  }
  fwrite(A, sizeof(T), DB * DB, stdout);
  fwrite(X, sizeof(T), DB * DB, stdout);
  fwrite(&info, sizeof(info), 1, stdout);
  return 0;
}

int main(int argc, char** argv) {
  if (argc != 4 || strlen(argv[3]) != WAVES) return 1;
  live = atoi(argv[2]);
  return atoi(argv[1]) == 64 ? run<double>(argv[3]) : run<float>(argv[3]);
}
