// Byte offsets of k_gemv_stream's weight loads (gemv_stream.hip), apart from
// the kernel so that the host can check them for every shape.  A raw buffer
// load drops each dword whose VGPR offset lies past the buffer; the SGPR offset
// is added behind that check, so it may only carry what stays inside.
#ifndef RAI_STREAM_ADDR_H
#define RAI_STREAM_ADDR_H

#ifdef __HIPCC__
#define RAI_HD __host__ __device__ __forceinline__
#else
#define RAI_HD inline
#endif

namespace rai {

struct BufOff {
  int v, s;  // VGPR and SGPR offset
};

// 16 bytes of codes: unit `piece` of group 4 * q + group of a row, the step
// and the group clamped to the row's last ones.
RAI_HD BufOff stream_code_off(int row, int cols, int gs, int q, int group, int piece) {
  const int groups = cols / gs, nq = (groups + 3) / 4;
  const int qc = q < nq - 1 ? q : nq - 1;
  const int left = groups - 1 - 4 * qc;  // last group of the step
  const int g = group < left ? group : left;
  return {row * (cols / 2) + g * (gs / 2) + piece * 16, qc * (2 * gs)};
}

// 16 bytes of parameters, step 4 * S + step of a row: what lies past the row's
// groups is the next row's, or past the array, where the range check drops it.
RAI_HD BufOff stream_param_off(int row, int groups, int S, int step) {
  const int nst = ((groups + 3) / 4 + 3) / 4;
  return {row * groups * 4 + 16 * step + 64 * (S < nst - 1 ? S : nst - 1), 0};
}

}  // namespace rai

#endif
