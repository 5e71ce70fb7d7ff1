// Counts the heap allocations of kspace_field_noalloc calls without sites,
// which validate and count wave vectors and stop before the device.
#include <cstdio>
#include <cstdlib>
#include <initializer_list>
#include <new>

extern "C" int kspace_field_noalloc(double, int, const void *, const double *, const void *, double,
                                    double, double *, void *, void *);

static long count;
void *operator new(std::size_t n) {
  count++;
  if (void *p = std::malloc(n)) return p;
  std::abort();
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, std::size_t) noexcept { std::free(p); }

int main() {
  const double latv[9] = {0.3, 0, 0, 0, 0.3, 0, 0, 0, 0.3};
  for (double kc : {1.0, 7.0, 12.0}) {
    count = 0;
    const int rc = kspace_field_noalloc(kc, 0, nullptr, nullptr, latv, 9000.0, 0.32, nullptr, nullptr, nullptr);
    std::printf("kc %g rc %d allocations %ld\n", kc, rc, count);
    if (rc != 0 || count != 0) return 1;
  }
  return 0;
}
