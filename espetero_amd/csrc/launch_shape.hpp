// How a pass's shape becomes workgroups: the facts of the attention kernels that the host planner counts with too. No device
// code and no HIP header: the kernels, the C ABI and espetero_amd/engine/planner.hpp read the same lines.
#pragma once

#include <cstddef>
#include <cstdint>

namespace esp {

constexpr int kComputeUnits = 256;  // of one MI355X

// Which kernel serves rows_per_tile x G packed rows: 1 or 2, the streaming kernel with that many column tiles; -1, the tiled
// kernel. (Two column tiles: in one wavefront's registers at head dim 128, as two wavefront pairs of one workgroup at head dim 512.)
constexpr int kernel_family(int head_dim, int rows_per_tile, int G) {
  const int nc = (rows_per_tile * G + 15) / 16;
  return nc == 1 || (nc == 2 && (head_dim == 128 || head_dim == 512)) ? nc : -1;
}

// Resident workgroups per compute unit of each variant: the single-column-tile head_dim-128 kernel fits two; the wider ones
// need more than 256 VGPRs and run one.
constexpr int stream_occ(int HD, int NC) { return (HD == 128 && NC == 1) ? 2 : 1; }  // wavefronts per SIMD
// Head dim 512: workgroups of one wavefront pair per column tile, one wavefront per SIMD: two pairs fill a compute unit.
constexpr int stream_workgroups_per_cu(int HD, int NC) { return HD >= 512 ? 2 / NC : stream_occ(HD, NC); }
constexpr int tiled_occ(int HD) { return HD == 128 ? 2 : 1; }
constexpr int tiled_workgroups_per_cu(int HD) { return tiled_occ(HD); }

// Does the tiled kernel give a tile of `rows` live rows one workgroup per KV head, all G query heads' rows in it, instead of one
// per query head? Where they fit its 128 places, and the grid is more than a workgroup per compute unit; why the line lies there:
// at the kernel. (Head dim 512 has a kernel of its own, which does not.)
constexpr bool tiled_fits(int rows, int G) { return rows * G <= 128; }
template <typename N>
constexpr bool tiled_packs_grid(N grid) {
  return grid > N(kComputeUnits);
}
constexpr bool tiled_packs(int HD, int rows, int G, long long grid) { return HD != 512 && tiled_fits(rows, G) && tiled_packs_grid(grid); }

// Where a pass's partial records and, for the tiled kernels, its transposed batch V lie in the workspace.
struct Carve {
  size_t parts_o, parts_ml, vt_stage, total;
};
constexpr Carve carve_workspace(int H, int Hkv, int head_dim, int rows_per_tile, int n_rows, int64_t n_parts) {
  const size_t cols = size_t(rows_per_tile) * size_t(H / Hkv);
  const size_t recs = size_t(n_parts > 0 ? n_parts : 0) * Hkv * cols;
  auto up = [](size_t x) { return (x + 255) & ~size_t(255); };
  Carve c{};
  c.parts_o = 0;
  c.parts_ml = up(recs * head_dim * sizeof(float));
  c.vt_stage = c.parts_ml + up(recs * 2 * sizeof(float));
  const size_t groups = size_t(n_rows > 0 ? (n_rows + 15) / 16 : 0);
  c.total = c.vt_stage + (kernel_family(head_dim, rows_per_tile, H / Hkv) < 0 ? up(groups * 16 * Hkv * head_dim * sizeof(uint16_t)) : 0);
  if (c.total == 0) c.total = 256;
  return c;
}

}  // namespace esp
