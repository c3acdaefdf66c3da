// attn_prep: what runs between the fused in-projection and the attention of a
// layer. Per (row, head) of the fp32 projection: RMSNorm over the head with a
// learned weight (queries and keys), rotary embedding of the leading
// `rope_dims` dims in the half-split pairing (d, d + rope_dims / 2), cast to the
// storage type; values are cast (or normalised without weight); the rows' K / V
// also go straight into their pool entries, so no kv_save dispatch follows.
//
// One kernel for the reference's three: attn_prep (kernels/40_attention.metal:9-102:
// head_dim 256, 64 rotating dims, the gate beside each query head, the folded
// append), g4_attn_prep<HD> (kernels/80_gemma.metal:52-108: all dims rotate,
// values normalised) and q3m_attn_prep<HD> (kernels/82_qwen3_omni.metal:30-88:
// per-frequency position component, query scale).
//
// Mapping to gfx950: HBM bound (fp32 in, 16-bit out). One workgroup = 8 consecutive rows x 2048 columns (16 heads of 128
// dims, 8 of 256); a lane owns two chunks of 4 dims that are each other's partners in the rotation (two 16-byte loads, two
// 8-byte stores), so the rotation stays inside the lane and only the norm's sum is a lane exchange, through the vector
// unit. A thread works on the same (head, dims) of all 8 rows at once: 16 independent loads in flight, issued ahead of the
// rows' cos / sin tables (rope_dims / 2 entries each, worked out once per workgroup into LDS: the reference computes them
// once per (row, head)), and no branch between the rows. With half as many columns per workgroup, the loads behind the
// tables and the exchanges through LDS the same passes took, before -> now: 8192 rows of 16 + 8 + 8 heads of 256 dims
// (402 MB) 106 -> 70 us (5.7 TB/s), 2048 rows of 40 + 8 + 8 heads of 128 with the append 26.9 -> 18.7 us, 1500 rows of
// 16 + 2 + 2 heads of 512 37.6 -> 24.2 us, 524 rows of 32 + 4 + 4 heads of 128 13.6 -> 8.6 us.
// The folded append writes K rows as they are. V lies transposed in the pool (16-token sub-blocks, tokens contiguous per
// dim): when the 8 rows go to 8 consecutive, 8-aligned positions of one block - every full group of a prefill chunk - a
// lane holds 8 tokens of its dims and stores 16 bytes per dim; any other arrangement (decode rows of different sequences,
// a row saved into two slots) takes element stores.
#include "common.hpp"
#include "prep_math.hpp"

namespace esp {

constexpr int kPrepRows = 8;

template <int DT, int HD>
__global__ __launch_bounds__(256) void attn_prep_kernel(const PrepArgs a, int n_rows, bool deal) {
  constexpr int R = kPrepRows;
  constexpr int LPH = HD / kPrepDims;  // lanes per head
  constexpr int HPW = 64 / LPH;        // heads of a wavefront
  __shared__ __attribute__((aligned(16))) float2 cs[R][HD / 2];  // (cos, sin) per row and frequency
  const esp_prep_params& p = a.p;
  const int row0 = blockIdx.x * R;
  const int rows = min(R, n_rows - row0);
  const int tid = threadIdx.x;
  const int half = p.rope_dims / 2;
  const int n_slots = p.H + 2 * p.Hkv;
  // This lane's head: queries, then keys, then values
  const int slot = (deal ? (tid / 64) * int(gridDim.y) + int(blockIdx.y) : 4 * int(blockIdx.y) + tid / 64) * HPW + tid % 64 / LPH;
  const bool live = slot < n_slots;
  const int kind = slot < p.H ? 0 : (slot < p.H + p.Hkv ? 1 : 2);  // q, k, v
  const int h = kind == 0 ? slot : (kind == 1 ? slot - p.H : slot - p.H - p.Hkv);
  const int li = tid % LPH;
  const PrepDims pd = prep_dims<HD>(p, li);
  // What the angles need is asked for ahead of the projection: loads come back in order.
  int f = 0, sel = 0, r_first = R, r_step = R;
  float freq = 0.0f;
  int4 pos_r = make_int4(0, 0, 0, 0);
  if (half > 0) {
    f = tid & (half - 1);
    r_first = tid / half;
    r_step = max(1, 256 / half);
    freq = a.inv_freq[f];
    if (a.rope_sel) sel = a.rope_sel[f];
    pos_r = a.pos[row0 + min(r_first, rows - 1)];
  }
  // The rows' projection is on its way while the angles below are worked out; a row past the last one repeats it and is
  // not stored.
  f32x4 xv[R][2];
  float w[kPrepDims];
#pragma unroll
  for (int i = 0; i < kPrepDims; ++i) w[i] = 1.0f;
  if (live) {
    if (kind != 2) {
      const float* wn = kind == 0 ? a.qn_w : a.kn_w;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        w[i] = wn[pd.a + i];
        w[4 + i] = wn[pd.b + i];
      }
    }
    const float* xc = a.X + size_t(kind == 0 ? p.q_off + h * p.q_hs : (kind == 1 ? p.k_off : p.v_off) + h * HD);
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const float* xr = xc + size_t(row0 + min(r, rows - 1)) * p.x_ld;
      // read once: no reason to keep it in a cache
      xv[r][0] = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(xr + pd.a));
      xv[r][1] = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(xr + pd.b));
    }
  }
  // Do the 8 rows go to positions ps0 .. ps0 + 7 (ps0 a multiple of 8) of one block, nowhere else? (The same entries for the
  // whole workgroup, read through the scalar cache, as some of the positions below: no kernel writes either while this one
  // runs. chain_advance_kernel does between the steps of a chain, in a dispatch of its own.)
  using const_int = const int __attribute__((address_space(4)));
  const_int* ents = (const_int*)(a.row_table + row0);
  bool run = a.row_table && rows == R;
  if (run) {
    const int b0 = ents[0], ps0 = ents[1];
    run = b0 >= 0 && (ps0 & (R - 1)) == 0;
#pragma unroll
    for (int r = 0; r < R; ++r) run = run & (ents[4 * r] == b0) & (ents[4 * r + 1] == ps0 + r) & (ents[4 * r + 2] < 0);
  }
  // half is a power of two of at most 256: a thread's angles are all of one frequency, a row further on each turn. Turns
  // after the first exist for half >= 64 only, where a wavefront's row is one: its position comes through the scalar
  // cache, whose counter the projection's loads in flight do not hold up.
  for (int r = r_first; r < rows; r += r_step) {
    if (r != r_first) {
      const_int* pr = (const_int*)(a.pos + row0 + __builtin_amdgcn_readfirstlane(r));
      pos_r = make_int4(pr[0], pr[1], pr[2], 0);
    }
    cs[r][f] = prep_cos_sin(pos_r, sel, freq);
  }
  __syncthreads();
  if (!live) return;
  u32x2 out[R][2];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    float x[kPrepDims];
#pragma unroll
    for (int i = 0; i < kPrepDims; ++i) x[i] = xv[r][i / 4][i % 4];
    prep_lane<HD>(x, kind, w, cs[min(r, rows - 1)], p, li, pd.rot);
    out[r][0] = u32x2{pack2<DT>(x[0], x[1]), pack2<DT>(x[2], x[3])};
    out[r][1] = u32x2{pack2<DT>(x[4], x[5]), pack2<DT>(x[6], x[7])};
  }
  // Kb / Vb may be left out when the rows go to the pool anyway (a pass whose attention reads them from there)
  uint16_t* dst = kind == 0 ? a.Q : (kind == 1 ? a.Kb : a.Vb);
  if (dst) {
    const size_t ld = size_t(kind == 0 ? p.q_ld : p.kv_ld);
    dst += size_t(row0) * ld + size_t(h) * HD;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      if (r >= rows) break;
      *reinterpret_cast<u32x2*>(dst + size_t(r) * ld + pd.a) = out[r][0];
      *reinterpret_cast<u32x2*>(dst + size_t(r) * ld + pd.b) = out[r][1];
    }
  }
  if (kind == 0 || !a.row_table) return;
  // The folded append: the same bits into the rows' pool entries (a row saved into two slots has two).
  if (kind == 2 && run) {
    // 8 tokens of one dim are 16 contiguous bytes of the transposed V plane, and this lane has all of them.
    uint16_t* vt = a.pool + p.kv_base + (size_t(ents[0]) * p.Hkv + h) * size_t(2 * p.bt * HD) + vt_elem(p.bt, HD, ents[1], 0);
#pragma unroll
    for (int i = 0; i < kPrepDims; ++i) {
      u32x4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint32_t t0 = out[2 * e][i / 4][(i % 4) / 2], t1 = out[2 * e + 1][i / 4][(i % 4) / 2];
        v[e] = i & 1 ? (t0 >> 16) | (t1 & 0xffff0000u) : (t0 & 0xffffu) | (t1 << 16);
      }
      *reinterpret_cast<u32x4*>(vt + size_t((i < 4 ? pd.a : pd.b) + i % 4) * kVtDim) = v;
    }
    return;
  }
#pragma unroll
  for (int r = 0; r < R; ++r) {
    if (r >= rows) break;
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const int b = ents[4 * r + 2 * e], ps = ents[4 * r + 2 * e + 1];
      if (b < 0) continue;
      uint16_t* hb = a.pool + p.kv_base + (size_t(b) * p.Hkv + h) * size_t(2 * p.bt * HD);
      prep_append<HD>(hb, kind, p.bt, ps, pd.a, out[r][0]);
      prep_append<HD>(hb, kind, p.bt, ps, pd.b, out[r][1]);
    }
  }
}

hipError_t launch_attn_prep(const PrepArgs& a, int n_rows, hipStream_t st) {
  const int dt = a.p.dtype, HD = a.p.head_dim;
  const int hpp = 4 * (64 / (HD / kPrepDims)), n_slots = a.p.H + 2 * a.p.Hkv;  // heads of a workgroup's four wavefronts
  // Few rows, and value heads that are more than one wavefront: the heads are dealt to the rows' workgroups a wavefront at a time.
  // A value row that goes to a block of its own takes an element store per dim, which consecutive heads put into one workgroup:
  // 16 decode rows of 16 + 8 + 8 heads of 256 dims 14.1 us, dealt 7.6; 4 rows of 40 + 8 + 8 of 128 5.8 and 5.1. With many rows a
  // workgroup's consecutive 8 KB of each row read faster: 2048 rows in whole groups 22.8 us, dealt 30.1; the two meet between
  // 500 and 1000 rows (524: 11.6 and 10.6; 40 + 8 + 8 heads of 128 7.9 and 8.2). Value heads of one wavefront gain nothing
  // (16 rows of 32 + 4 + 4 of 128 6.4 us, dealt 6.8).
  const bool deal = n_rows <= 512 && a.p.Hkv > 64 / (HD / kPrepDims);
  const dim3 grid((n_rows + kPrepRows - 1) / kPrepRows, (n_slots + hpp - 1) / hpp), block(256);
  if (dt == ESP_F16 && HD == 128) launch_timed(attn_prep_kernel<ESP_F16, 128>, grid, block, 0, st, a, n_rows, deal);
  else if (dt == ESP_F16 && HD == 256) launch_timed(attn_prep_kernel<ESP_F16, 256>, grid, block, 0, st, a, n_rows, deal);
  else if (dt == ESP_BF16 && HD == 128) launch_timed(attn_prep_kernel<ESP_BF16, 128>, grid, block, 0, st, a, n_rows, deal);
  else if (dt == ESP_BF16 && HD == 256) launch_timed(attn_prep_kernel<ESP_BF16, 256>, grid, block, 0, st, a, n_rows, deal);
  else if (dt == ESP_F16 && HD == 512) launch_timed(attn_prep_kernel<ESP_F16, 512>, grid, block, 0, st, a, n_rows, deal);
  else if (dt == ESP_BF16 && HD == 512) launch_timed(attn_prep_kernel<ESP_BF16, 512>, grid, block, 0, st, a, n_rows, deal);
  else return hipErrorInvalidValue;
  return hipGetLastError();
}

}  // namespace esp
