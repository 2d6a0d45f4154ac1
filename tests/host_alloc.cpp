// Failed allocations and fills in the library's host code, without a GPU: this file includes the
// source under test (SOURCE) and defines the HIP calls it makes over host memory, so that a
// chosen one can fail.  Prints "ok", or what went wrong.
#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>

static int fail_malloc = 0, fail_memset = 0;  // the n-th call from now fails (0: none)
static bool counts_down(int &n) { return n > 0 && --n == 0; }

extern "C" {
hipError_t hipMalloc(void **p, size_t n) {
  *p = nullptr;
  if (counts_down(fail_malloc)) return hipErrorOutOfMemory;
  *p = malloc(n);
  memset(*p, 0xA5, n);
  return hipSuccess;
}
hipError_t hipFree(void *p) {
  free(p);
  return hipSuccess;
}
hipError_t hipMemsetAsync(void *p, int v, size_t n, hipStream_t) {
  if (counts_down(fail_memset)) return hipErrorUnknown;
  if (!p) return hipErrorInvalidValue;
  memset(p, v, n);
  return hipSuccess;
}
}

#include SOURCE

static bool zero(const void *p, size_t n) {
  const char *c = static_cast<const char *>(p);
  for (size_t i = 0; i < n; i++)
    if (c[i]) return false;
  return n == 0 || p;
}
#define EXPECT(c, ...)                                \
  do {                                                \
    if (!(c)) return printf(__VA_ARGS__), puts(""), 1; \
  } while (0)

#ifdef CFM
static int fail_rope = 0;
namespace itts {
hipError_t cfm_rope_table(int T, float *tab, hipStream_t) {
  if (counts_down(fail_rope)) return hipErrorUnknown;
  for (int i = 0; i < T * 64; i++) tab[i] = (float)T;
  return hipSuccess;
}
itts_status set_error_text(itts_status st, const char *) { return st; }
size_t cfm_frag_pieces(long rows, int nk) { return (size_t)((rows + 127) / 128 * 4) * nk * 128; }
size_t cfm_q_pieces(int, int T, int H) { return (size_t)H * T; }
size_t cfm_kv_pieces(int, int T, int H) { return (size_t)H * T; }
}  // namespace itts

// What a forward of the shape finds: the padded planes all zero (nothing has written them) and
// the rope table of T.
static int check(itts_cfm &m, int B, int T, const char *when, int k) {
  EXPECT(ensure_rows(&m, B, T) == ITTS_OK, "%s %d: the next call fails", when, k);
  EXPECT(zero(m.hpP.p, sizeof(uint4) * B * hp_pieces(m.c, T)), "%s %d: padding rows not zero", when, k);
  EXPECT(m.rope.p && m.rope.p[0] == (float)T && m.rope.p[64 * T - 1] == (float)T, "%s %d: rope table", when, k);
  return 0;
}

int main() {
  const int B = 2;
  for (int T : {20, 100}) {  // the few-row path's buffers, the planes'
    for (int k = 1, failed = 1; failed; k++) {
      itts_cfm m;
      m.c = itts_cfm_config{64, 3, 1, 96, 8, 16, 2, 5};
      m.skips.resize(1);
      m.skipP.resize(1);
      if (check(m, B, T, "first", 0)) return 1;
      fail_malloc = k;  // a longer call that runs out of memory at its k-th growth
      failed = ensure_rows(&m, B, 300) != ITTS_OK;
      fail_malloc = 0;
      if (check(m, B, T, "after a failed allocation", k)) return 1;
    }
    itts_cfm m;
    m.c = itts_cfm_config{64, 3, 1, 96, 8, 16, 2, 5};
    m.skips.resize(1);
    m.skipP.resize(1);
    for (int *f : {&fail_memset, &fail_rope}) {
      *f = 1;
      EXPECT(ensure_rows(&m, B, T) != ITTS_OK, "a failed fill goes unnoticed");
      *f = 0;
      if (check(m, B, T, "after a failed fill", T)) return 1;
      if (check(m, B, 2 * T, "longer", T)) return 1;
      *f = 1;
      EXPECT(ensure_rows(&m, B, T) != ITTS_OK, "a failed fill goes unnoticed");
      *f = 0;
      if (check(m, B, 2 * T, "back after a failed fill", T)) return 1;
    }
  }
  puts("ok");
  return 0;
}
#endif

#ifdef RUNTIME
namespace itts {
size_t rows_planes_pieces(int M, int K) { return (size_t)M * K / 4; }
}  // namespace itts

int main() {
  itts_gpt g;
  for (int *f : {&fail_malloc, &fail_memset}) {
    DevBuf b;
    EXPECT(ensure_planes(&g, b, 32, 64) == hipSuccess && zero(b.p, b.bytes), "first planes");
    *f = 1;
    EXPECT(ensure_planes(&g, b, 96, 64) != hipSuccess, "a failure goes unnoticed");
    *f = 0;
    for (int M : {32, 96}) {
      EXPECT(ensure_planes(&g, b, M, 64) == hipSuccess, "the next call fails");
      EXPECT(b.bytes >= sizeof(uint4) * rows_planes_pieces(M, 64) && zero(b.p, b.bytes), "planes not zero at %d rows", M);
    }
  }
  puts("ok");
  return 0;
}
#endif
