// Enumerates on the host every row offset that the elementwise scans' kernels load
// (mg_rows.h) and reports those outside the tensors.  Built and run by
// test_host_checks.py with hipcc's host pass alone: nothing here touches a GPU.
#include "mg_rows.h"

#include <cstdio>

static long bad = 0, seen = 0;

// `o` as the offset of a row of D elements in a tensor of `rows` rows `ld` apart.
static void check(const char* what, int64_t o, int64_t rows, int64_t ld, int64_t B, int64_t T,
                  int64_t t) {
  ++seen;
  if (o >= 0 && o % ld == 0 && o / ld < rows) return;
  if (bad++ < 5)
    printf("%s: offset %lld of B=%lld T=%lld ld=%lld at step %lld\n", what, (long long)o,
           (long long)B, (long long)T, (long long)ld, (long long)t);
}

int main() {
  const int64_t lengths[] = {1, 2, 3, 4, 5, 7, 8, 9, 31, 32, 33, 63, 64, 65, 127, 129};
  const int waves[] = {4, 8}, subs[] = {4, 8, 16};
  for (int64_t T : lengths)
    for (int64_t B = 1; B <= 3; ++B)
      for (int64_t ld : {1, 6, 64, 259})
        for (int W : waves)
          for (int S : subs)
            for (int64_t c = 0; c * W * S < T; ++c)
              for (int w = 0; w < W; ++w)
                for (int64_t b = 0; b < B; ++b) {
                  const int64_t t0 = (c * W + w) * S, b0 = b * T;
                  EwRows rows(b0, t0, T, ld);
                  for (int s = 0; s < S; ++s) {
                    const int64_t t = t0 + s, o = rows.next();
                    check("row", o, B * T, ld, B, T, t);
                    check("row before", rows.before(o), B * T, ld, B, T, t);
                    if (t < T && o != (b0 + t) * ld) check("row of the step", -1, 0, ld, B, T, t);
                    if (t > 0 && t < T && rows.before(o) != (b0 + t - 1) * ld)
                      check("row before the step", -1, 0, ld, B, T, t);
                    // parallel_scan_log's values have a row more per batch row.
                    check("log value", o + (b + 1) * ld, B * (T + 1), ld, B, T, t);
                  }
                  check("row before the wave", ew_row(b0, t0 > 0 ? t0 - 1 : 0, T) * ld, B * T, ld,
                        B, T, t0);
                }
  printf("%ld offsets, %ld outside\n", seen, bad);
  return bad != 0;
}
