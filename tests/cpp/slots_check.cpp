// Record slots of the binning (pme_slots.hpp) at atom counts up to the largest an
// int holds: the first and last slot of the last chunk, through the list type in
// which the spread reorders a batch, against 128-bit arithmetic.  Prints "ok" and
// exits 0, or names the first wrong slot and exits 1.
#include <cstdio>
#include <initializer_list>

#include "pme_slots.hpp"

int main() {
  const int counts[] = {1, 511, 512, 262144, 262145, 33554431, 268435455, 268435456, 268435457, 536870912, 2147483647};
  for (int n : counts) {
    // plan_chunks: 512 atoms per chunk, doubled until 512 chunks do
    int chunk = 512;
    while ((long long)chunk * 512 < n) chunk *= 2;
    const int nchunk = (int)(((long long)n + chunk - 1) / chunk);
    const int stride = 8 * chunk;
    for (int at : {0, stride - 1}) {
      const __int128 want = (__int128)(nchunk - 1) * stride + at;
      pme::RecordList list[1];
      list[0] = pme::record_slot(nchunk - 1, stride, at);
      const pme::RecordSlot got = list[0];
      if ((__int128)got != want || got == pme::kNoSlot) {
        std::printf("%d atoms, slot %d of chunk %d: %zu\n", n, at, nchunk - 1, (size_t)got);
        return 1;
      }
    }
  }
  std::puts("ok");
  return 0;
}
