// Host check of rai_amd/csrc/stream_addr.h: every weight load of k_gemv_stream
// for `rows` x `groups` groups of `gs`, with the range check taken as it is
// documented (each dword's VGPR offset against the buffer's bytes).  Prints the
// loads checked, the dwords read outside their array and the dwords of real
// groups that are not where the layout has them.
// Built and run by tests/test_cpu_pins.py (test infrastructure only).
#include <cstdio>
#include <initializer_list>

#include "stream_addr.h"

int main() {
  long long loads = 0, outside = 0, wrong = 0;
  auto load = [&](rai::BufOff o, long long bytes, long long want, int valid) {
    ++loads;
    for (int d = 0; d < 4; ++d) {
      const bool dropped = o.v + 4 * d >= bytes;  // answered with zero
      const long long at = (long long)o.v + o.s + 4 * d;
      if (!dropped && (at < 0 || at + 4 > bytes)) ++outside;
      if (d < valid && (dropped || at != want + 4 * d)) ++wrong;
    }
  };
  for (int gs : {32, 64, 128})
    for (int groups = 1; groups <= 70; ++groups)
      for (int rows : {1, 2, 15, 16, 17, 33}) {
        const int cols = groups * gs, nq = (groups + 3) / 4, nst = (nq + 3) / 4;
        const long long nib = (long long)rows * (cols / 2), par = 4LL * rows * groups;
        for (int r = 0; r < (rows + 15) / 16 * 16 + 48; ++r) {  // tiles of a block past the matrix as well
          const int row = r < rows - 1 ? r : rows - 1;
          for (int S = 0; S < nst + 3; ++S)  // the ring asks past the last stage
            for (int step = 0; step < 4; ++step) {
              const int q = 4 * S + step, left = groups - 4 * q;
              load(rai::stream_param_off(row, groups, S, step), par, 4LL * (row * groups + 4 * q),
                   left < 0 ? 0 : left > 4 ? 4 : left);
              for (int g = 0; g < 4; ++g)
                for (int piece = 0; piece < gs / 32; ++piece)
                  load(rai::stream_code_off(row, cols, gs, q, g, piece), nib,
                       (long long)row * (cols / 2) + (4LL * q + g) * (gs / 2) + 16 * piece, g < left ? 4 : 0);
            }
        }
      }
  std::printf("%lld %lld %lld\n", loads, outside, wrong);
  return 0;
}
