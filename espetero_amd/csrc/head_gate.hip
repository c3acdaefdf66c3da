// head_gate: the head-wise output gate that follows the attention of a layer,
// O[row, h, :] *= sigmoid(x[row] . Wg[h]) (sp_head_gate, kernels/85_spark.metal:96-128;
// dispatched at src/model/impl/gemma.h:481-492). The reference runs one threadgroup
// of scalar dots per (head, row); its own note says a GEMM dispatch cost more than
// the dots at 16 rows (src/model/impl/gemma_load.h:292-294).
//
// Mapping to gfx950: HBM bound (X once, O there and back; Wg stays in L2). One
// workgroup takes 16 rows. The dots of 16 rows x 16 heads x 32 model dims are one
// v_mfma_f32_16x16x32 whose operands are 16-byte loads straight from X and Wg; the
// four wavefronts take a quarter of the model dims each and their sums meet in LDS. Then
// the workgroup streams its 16 rows of O through registers, 16 bytes per lane and
// 16 loads in flight per lane (the first 16 issued before the dots, so that their
// latency lies under the dots'). The dots alone, for the attention kernels' own
// epilogue to use, have a kernel of their own below.
#include "lds_direct.hpp"

namespace esp {

constexpr int kGateRows = 16;

template <int DT>
__device__ __forceinline__ float2 unpack2(uint32_t u) {
  if constexpr (DT == ESP_F16) {
    const f16x2 v = __builtin_bit_cast(f16x2, u);
    return make_float2(float(v[0]), float(v[1]));
  } else {
    return make_float2(__builtin_bit_cast(float, u << 16), __builtin_bit_cast(float, u & 0xffff0000u));
  }
}

template <int DT, int NB>  // NB: blocks of 16 heads
__global__ __launch_bounds__(256) void head_gate_kernel(const GateArgs a) {
  constexpr int R = kGateRows, U = NB == 1 ? 8 : (NB == 2 ? 4 : 2), B = 16;
  __shared__ float sums[4][R][16 * NB + 1];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int c16 = lane & 15, q4 = lane >> 4;
  const int row0 = blockIdx.x * R;
  const int rows = min(R, a.n_rows - row0);

  // The workgroup's part of O is rows x vpr 16-byte vectors; a thread takes every 256th of them in
  // row-major order, B at a time: with rows that follow one another in memory a batch is one
  // contiguous 64 KB. (r, v) walk that order without a division.
  const int vpr = a.H * a.hd / 8;
  int r_ld = 0, v_ld = tid;
  auto normalise = [&](int& r, int& v) {
    while (v >= vpr) {
      v -= vpr;
      ++r;
    }
  };
  normalise(r_ld, v_ld);
  u32x4 o[B];
  auto load_batch = [&]() {
#pragma unroll
    for (int j = 0; j < B; ++j) {
      o[j] = (a.O && r_ld < rows) ? *reinterpret_cast<const u32x4*>(a.O + size_t(row0 + r_ld) * a.q_ld + 8 * v_ld) : u32x4{0, 0, 0, 0};
      v_ld += 256;
      normalise(r_ld, v_ld);
    }
  };
  load_batch();  // in flight while the dots are formed

  // ---- dots: rows past the end repeat the last row, heads past H repeat the last head; neither is read back
  const uint16_t* xp = a.X + size_t(row0 + min(c16, rows - 1)) * a.x_ld + 8 * q4;
  const uint16_t* wp[NB];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) wp[nb] = a.Wg + size_t(min(16 * nb + c16, a.H - 1)) * a.D + 8 * q4;
  f32x4 acc[NB];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) acc[nb] = f32x4{0, 0, 0, 0};
  // A wavefront's chunks follow one another; each workgroup starts its walk somewhere else, so that
  // the workgroups of an XCD do not all ask its L2 for the same lines of Wg at the same moment.
  const int n_chunks = (a.D + 31) / 32, per_wave = (n_chunks + 3) / 4;
  const int rot = int((blockIdx.x * 7u) % unsigned(per_wave));
  for (int i = 0; i < per_wave; i += U) {
    u32x4 xa[U], wb[NB][U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      int ci = i + u + rot;
      if (ci >= per_wave) ci -= per_wave;
      const int k = 32 * (wave * per_wave + ci);
      const bool ok = i + u < per_wave && k + 8 * q4 < a.D;  // D is a multiple of 8: a lane's 8 dims exist or do not
      xa[u] = ok ? *reinterpret_cast<const u32x4*>(xp + k) : u32x4{0, 0, 0, 0};
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) wb[nb][u] = ok ? *reinterpret_cast<const u32x4*>(wp[nb] + k) : u32x4{0, 0, 0, 0};
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) acc[nb] = mfma16x32<DT>(xa[u], wb[nb][u], acc[nb]);
  }
#pragma unroll
  for (int nb = 0; nb < NB; ++nb)
#pragma unroll
    for (int i = 0; i < 4; ++i) sums[wave][4 * q4 + i][16 * nb + c16] = acc[nb][i];
  __syncthreads();
  for (int i = tid; i < R * 16 * NB; i += 256) {
    const int r = i / (16 * NB), h = i % (16 * NB);
    const float dot = (sums[0][r][h] + sums[1][r][h]) + (sums[2][r][h] + sums[3][r][h]);
    if (a.dots && r < rows && h < a.H) a.dots[size_t(row0 + r) * a.H + h] = dot;
    sums[0][r][h] = 1.0f / (1.0f + __expf(-dot));
  }
  if (!a.O) return;
  __syncthreads();

  // ---- O = storage(float(O) * gate), 8 elements per lane and load
  int r_st = 0, v_st = tid;
  normalise(r_st, v_st);
  while (r_st < rows) {
#pragma unroll
    for (int j = 0; j < B; ++j) {
      if (r_st < rows) {
        const int h = a.hd_shift >= 0 ? (8 * v_st) >> a.hd_shift : (8 * v_st) / a.hd;
        const float g = sums[0][r_st][h];
        u32x4 out;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float2 f = unpack2<DT>(o[j][e]);
          out[e] = pack2<DT>(f.x * g, f.y * g);
        }
        *reinterpret_cast<u32x4*>(a.O + size_t(row0 + r_st) * a.q_ld + 8 * v_st) = out;
      }
      v_st += 256;
      normalise(r_st, v_st);
    }
    if (r_ld < rows) load_batch();
  }
}

// The dots alone, for the attention kernels' epilogue. Bound: one CU's path to its caches (64 bytes a clock; 16 rows x 4096 dims
// and 32 heads are 384 KB, 2.6 us at that rate), so the loads must be the kind that reach it: neighbouring lanes of the operand
// layout (row = lane % 16) are different rows, and such a load takes a clock per lane, a quarter of the rate. Here eight
// neighbouring lanes take one row's 128 bytes, straight to LDS, and the operands are read from there. A wavefront takes every
// eighth piece of 64 dims and keeps DP of them in flight in LDS of its own, so no barrier stands between loads and products;
// a row's eight 16-byte parts are turned by its number, which spreads an operand read over the banks. The eight sums of a dot
// meet in LDS, in pairs. Against the kernel above (replayed graph, fp16): 4096 dims and 32 heads, 1 row 10.7 -> 5.3 us, 500 rows 14.1
// -> 6.4, 2600 rows 14.5 -> 7.4, 8192 rows 29.9 -> 19.9; 2560 dims and 16 heads, 2600 rows 8.4 -> 5.3; 1024 dims and 8 heads, 16
// rows 4.6 -> 2.7. Eight or sixteen wavefronts with the register loads above gave 13.2 and 13.0 at 2600 rows.
template <int DT, int NB>  // NB: blocks of 16 heads
struct GateDots {
  static constexpr int W = 8, T = 1 + NB, DP = NB == 1 ? 4 : (NB == 2 ? 3 : 2);
  static constexpr int kTile = kGateRows * 128, kPiece = T * kTile, kLds = W * DP * kPiece;
  static_assert(kLds <= 160 * 1024 && W * kGateRows * (16 * NB + 1) * 4 <= kLds);
};

template <int DT, int NB>
__global__ __launch_bounds__(512) void gate_dots_kernel(const GateArgs a) {
  using G = GateDots<DT, NB>;
  constexpr int R = kGateRows, W = G::W, T = G::T, DP = G::DP;
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c16 = lane & 15, q4 = lane >> 4;
  const int row0 = blockIdx.x * R;
  const int rows = min(R, a.n_rows - row0);

  // A load takes eight rows of a piece: lane l the part (l % 8) ^ (row % 8) of row l / 8. Rows past the end repeat the last
  // row, heads past H the last head, parts past D the row's first; none of them is read back.
  const int lr = lane >> 3, part = (lane & 7) ^ lr;
  const char* base[T];
  uint32_t off[T][2];
#pragma unroll
  for (int t = 0; t < T; ++t) {
    base[t] = reinterpret_cast<const char*>(t ? a.Wg : a.X + size_t(row0) * a.x_ld);
#pragma unroll
    for (int h = 0; h < 2; ++h)
      off[t][h] = t ? uint32_t(min(16 * (t - 1) + 8 * h + lr, a.H - 1)) * uint32_t(a.D) * 2 : uint32_t(min(8 * h + lr, rows - 1)) * uint32_t(a.x_ld) * 2;
  }
  const int n_pieces = (a.D + 63) / 64, own = (n_pieces - wave + W - 1) / W;  // 0 where there are fewer pieces than wavefronts
  const int rot = own > 0 ? int((blockIdx.x * 7u) % unsigned(own)) : 0;  // the workgroups of an XCD ask its L2 for different lines of Wg
  auto dim_of = [&](int i) {
    const int p = i + rot < own ? i + rot : i + rot - own;
    return 64 * (wave + W * p);
  };
  const uint32_t lds0 = uint32_t(uintptr_t(lds)) + uint32_t(wave * DP * G::kPiece);
  auto request = [&](int i, int st) {
    const int k = dim_of(i) + 8 * part;
    const uint32_t kb = k < a.D ? 2u * uint32_t(k) : 0u;
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
      for (int h = 0; h < 2; ++h) load_to_lds16(base[t], off[t][h] + kb, lds0 + uint32_t(st * G::kPiece + t * G::kTile + h * 1024));
  };
  f32x4 acc[NB];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) acc[nb] = f32x4{0, 0, 0, 0};
#pragma unroll
  for (int d = 0; d < DP - 1; ++d)
    if (d < own) request(d, d);
  int st = 0;
  for (int i = 0; i < own; ++i) {
    const int ahead = i + DP - 1;  // into the stage that iteration i - 1 has read
    if (ahead < own) request(ahead, st == 0 ? DP - 1 : st - 1);
    // piece i has landed when no more than the loads of the pieces behind it are out
    const int behind = min(own - 1 - i, DP - 1);
    if (behind == 0) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    else if (behind == 1) asm volatile("s_waitcnt vmcnt(%0)" : : "n"(2 * T) : "memory");
    else if (behind == 2) asm volatile("s_waitcnt vmcnt(%0)" : : "n"(4 * T) : "memory");
    else asm volatile("s_waitcnt vmcnt(%0)" : : "n"(6 * T) : "memory");
    const char* piece = lds + (wave * DP + st) * G::kPiece + c16 * 128;
    const int k = dim_of(i) + 8 * q4;
    u32x4 x[2], w[NB][2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int at = ((4 * h + q4) ^ (c16 & 7)) * 16;
      x[h] = *reinterpret_cast<const u32x4*>(piece + at);
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) w[nb][h] = *reinterpret_cast<const u32x4*>(piece + (1 + nb) * G::kTile + at);
      if (k + 32 * h >= a.D) {  // both sides: a value of another dim may be an infinity
        x[h] = u32x4{0, 0, 0, 0};
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) w[nb][h] = u32x4{0, 0, 0, 0};
      }
    }
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) acc[nb] = mfma16x32<DT>(x[h], w[nb][h], acc[nb]);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the stage is read before its next request
    st = st + 1 == DP ? 0 : st + 1;
  }
  __syncthreads();
  constexpr int S = 16 * NB + 1;
  float* sums = reinterpret_cast<float*>(lds);
#pragma unroll
  for (int nb = 0; nb < NB; ++nb)
#pragma unroll
    for (int i = 0; i < 4; ++i) sums[(wave * R + 4 * q4 + i) * S + 16 * nb + c16] = acc[nb][i];
  __syncthreads();
  for (int i = tid; i < R * 16 * NB; i += 64 * W) {
    const int r = i / (16 * NB), h = i % (16 * NB);
    float s[W];
#pragma unroll
    for (int w = 0; w < W; ++w) s[w] = sums[(w * R + r) * S + h];
    if (r < rows && h < a.H) a.dots[size_t(row0 + r) * a.H + h] = ((s[0] + s[1]) + (s[2] + s[3])) + ((s[4] + s[5]) + (s[6] + s[7]));
  }
}

template <int DT, int NB>
hipError_t launch_gate(const GateArgs& a, dim3 grid, hipStream_t st) {
  // The dots kernel's addresses: 16-byte parts, and 32-bit offsets from a workgroup's first row. O is scaled by the kernel above,
  // whose dots lie under O's loads.
  const bool parts = (reinterpret_cast<uintptr_t>(a.X) | reinterpret_cast<uintptr_t>(a.Wg)) % 16 == 0;
  if (!a.O && parts && a.x_ld < (1 << 26) && a.D < (1 << 24)) {
    const hipError_t e = allow_dynamic_lds<gate_dots_kernel<DT, NB>>(GateDots<DT, NB>::kLds);
    if (e != hipSuccess) return e;
    launch_timed(gate_dots_kernel<DT, NB>, grid, dim3(512), size_t(GateDots<DT, NB>::kLds), st, a);
  } else {
    launch_timed(head_gate_kernel<DT, NB>, grid, dim3(256), 0, st, a);
  }
  return hipGetLastError();
}

// The dots kernels' dynamic LDS limits on the current device, ahead of their first launch.
template <int DT, int... NBs>
hipError_t gate_attributes_t() {
  hipError_t e = hipSuccess;
  ((e = e == hipSuccess ? allow_dynamic_lds<gate_dots_kernel<DT, NBs>>(GateDots<DT, NBs>::kLds) : e), ...);
  return e;
}
hipError_t gate_init_attributes() {
  const hipError_t e = gate_attributes_t<ESP_F16, 1, 2, 3, 4>();
  return e != hipSuccess ? e : gate_attributes_t<ESP_BF16, 1, 2, 3, 4>();
}

hipError_t launch_head_gate(int dt, const GateArgs& a, hipStream_t st) {
  const dim3 grid((a.n_rows + kGateRows - 1) / kGateRows);
  const int nb = (a.H + 15) / 16;
#define ESP_GATE_CASE(DT, NB) \
  if (dt == DT && nb == NB) return launch_gate<DT, NB>(a, grid, st);
  ESP_GATE_CASE(ESP_F16, 1) ESP_GATE_CASE(ESP_F16, 2) ESP_GATE_CASE(ESP_F16, 3) ESP_GATE_CASE(ESP_F16, 4)
  ESP_GATE_CASE(ESP_BF16, 1) ESP_GATE_CASE(ESP_BF16, 2) ESP_GATE_CASE(ESP_BF16, 3) ESP_GATE_CASE(ESP_BF16, 4)
#undef ESP_GATE_CASE
  return hipErrorInvalidValue;
}

}  // namespace esp
