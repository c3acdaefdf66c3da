// Tiled MFMA attention at head dim 512: prefill and chunked prefill of the
// full-attention layers whose heads are 512 wide (the reference's
// g4_attention512_s{1,2,4,8}, kernels/80_gemma.metal:157-342, :355-358).
//
// Semantics as in the tiled kernel of the narrower heads: cached keys [k0, k1)
// through the block table or ring, then the tree's batch keys (`last` tiles) under
// the tree mask (80_:284) and the window (80_:285), online softmax in fp32, P
// rounded to the storage type before P.V, output O / l (0 when no key is visible)
// with the optional sigmoid gate, or a partial record for the merge.
//
// Mapping to gfx950. A 512-dim head does not fit one wavefront (32 rows x 512 dims
// of fp32 accumulators alone are 256 registers), so a workgroup is one tile of up to
// 64 query rows x one query head, and its 4 wavefronts are 2 row groups of 32 rows x 2.
// Keys advance in steps of 32 (two 16-key sub-blocks). The two wavefronts of a row group
// share a step's scores by keys and its output by dims: wavefront (rg, w) computes
//   S^T[16 keys][32 rows] of sub-block w over all 512 dims   v_mfma_f32_16x16x32, A = K from LDS, B = Q^T in registers
//   P^T = exp2(S^T - m)                                      of its 16 keys, left in LDS in 16 bits
//   O^T[256 dims][32 rows] += V^T . P^T                      its 256 dims, all 32 keys; A = V^T and B = P^T from LDS
// (The reference's simdgroups split the dims of the scores and sum partials through threadgroup memory, 80_:272-282. So did
// this kernel: 4 KB of fp32 partials there and back per wavefront and step and the whole softmax in both wavefronts of a pair,
// 370 issued instructions around 1024 clocks of matrix work. By keys, 1 KB of P goes through LDS and each score has one owner.)
// Steps overlap: iteration i multiplies Q K^T of step i and P V of step i - 1, so that one barrier per step publishes the
// staged data and the P at once and the softmax of step i stands beside P V instructions that do not depend on it. K runs
// one step ahead of V in the staging (global_load_lds_dwordx4, no staging registers).
// The row's reference m moves only where a lane's share of a step's sum says so, and in the whole workgroup at once: the two
// wavefronts of a row group multiply each other's P.
// What bounds it: one wavefront per SIMD (accumulators 128 registers, Q 128, the rest 130), which issues in order, and the 64 KB a
// step brings through the compute unit's vector memory path at 64 B per clock. A step of whole cached sub-blocks is 242
// instructions, 48 of them matrix ones, and takes 880 ns of a lone workgroup (910 with the 293 it had, 2150 clocks by the counter then:
// 1010 in the 32 instructions of Q K^T (512 clocks) with 12 of a wavefront's 16 loads between them, 690 in 12 of P V (384) with
// the softmax, 170 in the wait and the barrier, 280 in the last 4 of P V with the other 4 loads); with all 16 loads in a row behind
// the barrier that stretch alone was 990, with four of them beside P V they landed too late (a wait of 440). Two prompt
// chunks of 700 .. 1024 rows over 3000 .. 7000 keys, 16 / 2 heads: kernel 412 us before, 325 so (the step's scores by dims halves 3340
// clocks; a lone branch that moved the reference inside the step's matrix instructions cost 70 register moves in every step).
//
// LDS layout: K of stage 0, K of stage 1, V^T of stage 0, V^T of stage 1 (an operand read is a per-lane base
// register plus an immediate, which takes 16 bits), P. K of a stage: 32 rows of 1024 bytes, unpadded; the 16-byte chunk c of
// row r of a sub-block lies at chunk position c ^ r: the 16 lanes that read a chunk of 16 rows hit 16 different positions.
// V^T per sub-block: [dim][2 halves of 8 keys], the two 16-byte halves of dim d swapped when bit 3 of d is set
// (lanes d and d + 8 of an operand read would otherwise share banks). P: [row][32 keys], rows 80 bytes apart.
#include <utility>

#include "common.hpp"
#include "lds_direct.hpp"

namespace esp {

namespace {
constexpr int kHD = 512, kHW = 256;                  // dims of a head; dims one wavefront accumulates
constexpr int kKStage = 32 * kHD * 2;                // K of one stage: 32 rows
constexpr int kVSub = kHD * 32;                      // V^T of one sub-block
constexpr int kVStage = 2 * kVSub;                   // V^T of one stage: two sub-blocks
constexpr int kVBase = 2 * kKStage;                  // layout: K stage 0, K stage 1, V^T stage 0, V^T stage 1
constexpr int kPRow = 80, kPBuf = 2 * 32 * kPRow;    // P of one step: 2 row groups x 32 rows
constexpr int kPBase = kVBase + 2 * kVStage;
constexpr int kMax = kPBase + 2 * kPBuf;             // a row's maximum in either wavefront: [row group][wavefront][32] floats
constexpr int kFlags = kMax + 2 * 2 * 32 * 4;        // [buffer][wavefront] ints
constexpr int kLds = kFlags + 2 * 4 * 4;
}  // namespace

template <int DT>
__global__ __launch_bounds__(256, 1) void attn_tiled512_kernel(const KArgs a, int n_tiles) {
  constexpr int NT = kHW / 32, KK = kHD / 32;
  extern __shared__ __attribute__((aligned(16))) char lds[];
  int(*flags)[4] = reinterpret_cast<int(*)[4]>(lds + kFlags);

  // Workgroup -> (KV head, head in group, tile): consecutive ids differ in KV head first, the heads
  // sharing a KV head land on the same XCD's L2; tiles run last to first (longest key ranges first).
  const int kvh = blockIdx.x % a.Hkv;
  const int rest = blockIdx.x / a.Hkv;
  const int hg = rest % a.G;
  const int tile_i = n_tiles - 1 - rest / a.G;
  const int h = kvh * a.G + hg;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int rg = wave >> 1, half = wave & 1, dw = half * kHW;
  const int l32 = lane & 31, hb = lane >> 5;   // P V: this lane's row of the group, half of a sub-block's keys
  const int c16 = lane & 15, q4 = lane >> 4;   // scores: rows c16 and 16 + c16 of the group, keys 4 q4 .. + 3 of sub-block `half`
  esp_tile tile = a.tiles[tile_i];
  const esp_tree tree = a.trees[tile.tree];
  if (tile.k1 == INT32_MAX) tile.k1 = tree.P;  // open-ended range: up to the tree's cached length as it is now
  const int table = tile.pad > 0 ? tile.pad - 1 : tree.table;
  const int end = tree.base + tree.M;
  const int rows_live = min(a.R, end - tile.r0);
  const int rr0 = tile.r0 - tree.base;

  // ---- Q rows of the tile: a whole row to a load, then through the V^T stages, row r's chunk c at position c ^ (r % 16) as in K.
  // Loads of the fragments themselves, whose neighbouring lanes are different rows, take the memory path a clock per lane, and every
  // wavefront needs all dims of its 32 rows: 8192 clocks in front of a tile of 64. One pass of 64 fresh rows (16 / 2 heads) took
  // 16.7 us so and takes 14.7 through LDS, 32 rows 10.9 and 10.3, 64 rows behind 1000 keys 50.4 and 48.0.
  u32x4 qrow[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int r = 4 * i + wave;
    if (r < rows_live) qrow[i] = *reinterpret_cast<const u32x4*>(a.Q + size_t(tile.r0 + r) * a.q_ld + size_t(h) * kHD + 8 * lane);
  }

  // ---- this lane's two rows of the scores
  int rr[2], qpos[2];
  int4 d[2];
  u32x4 qf[2][KK];
  int kl = -1;  // the last batch key they see
#pragma unroll
  for (int rt = 0; rt < 2; ++rt) {
    const int m = 32 * rg + 16 * rt + c16;
    const bool ok = m < rows_live;
    const int row = ok ? tile.r0 + m : tile.r0;
    rr[rt] = rr0 + m;
    d[rt] = a.desc ? a.desc[row] : make_int4(0, 0, 0, 0);
    qpos[rt] = a.window > 0 ? a.pos[row].x : 0;
    if (ok) kl = max(kl, max(rr[rt], max(d[rt].z - 1, a.bidi ? d[rt].w - 1 : -1)));
  }

  // ---- the last batch key any row of the tile sees
  int k_last = -1;
  {
#pragma unroll
    for (int o = 8; o >= 1; o >>= 1) kl = max(kl, __shfl_xor(kl, o));  // the lanes of a quarter hold all rows
    if (lane == 0) flags[0][wave] = kl;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int r = 4 * i + wave;
      if (r < rows_live) *reinterpret_cast<u32x4*>(lds + kVBase + r * 1024 + ((lane ^ (r & 15)) << 4)) = qrow[i];
    }
    __syncthreads();
#pragma unroll
    for (int rt = 0; rt < 2; ++rt) {
      const int m = 32 * rg + 16 * rt + c16;
      const char* qr = lds + kVBase + m * 1024;
#pragma unroll
      for (int kk = 0; kk < KK; ++kk) qf[rt][kk] = m < rows_live ? *reinterpret_cast<const u32x4*>(qr + (((4 * kk + q4) ^ c16) << 4)) : u32x4{0, 0, 0, 0};
    }
    k_last = max(flags[0][0], flags[0][2]);
    k_last = __builtin_amdgcn_readfirstlane(min(min(k_last, tree.M - 1), tile.last >= 2 ? tile.last - 2 : INT32_MAX));  // last >= 2: the part's batch range ends at row last - 2
  }

  // ---- the key range as 16-key sub-blocks: cached [k0, k1), then batch rows [b0, k_last]
  const int c0 = tile.k0 >> 4;
  const int n_c = tile.k1 > tile.k0 ? ((tile.k1 + 15) >> 4) - c0 : 0;
  const int a0 = (tree.base + tile.b0) >> 4;  // batch sub-blocks are groups of 16 absolute rows
  const int n_b = (tile.last && k_last >= tile.b0) ? ((tree.base + k_last) >> 4) - a0 + 1 : 0;
  const int n_sb = n_c + n_b;
  const int n_steps = (n_sb + 1) >> 1;
  const int n_groups = (a.n_rows + 15) >> 4;
  // Batch rows in the pool (no Kb / Vb): row j of a tree lies at position P + j of the tree's block list, P - base a
  // multiple of 16: a batch sub-block of 16 absolute rows is one 16-token sub-block of the pool, staged like a cached one.
  const bool in_pool = a.Kb == nullptr;
  const int pool_shift = tree.P - tree.base;

  // ---- staging, 16 bytes per lane straight into LDS. K: this wavefront brings rows 4 wave .. + 3 of each
  // sub-block; the lane that fills chunk position `lane` of row r brings chunk lane ^ r.
  // V^T: this wavefront brings pieces 256 wave .. + 255 of each sub-block's
  // 1024 (piece c: keys 8 (c % 2) .. + 7 of dim c / 2); position p holds piece p ^ ((p >> 4) & 1).
  constexpr uint32_t lds_base = 0;  // the dynamic array is the only LDS object
  // Pool addresses of the sub-blocks, 64 at a time: lane l holds the byte address of the K rows of sub-block adr0 + l
  // (block list entry, the head's place in the block, the sub-block's place in the head, worked out by 64 lanes at
  // once), so that in front of a sub-block's staging loads stand two lane reads instead of a dependent memory access
  // and the scalar arithmetic behind it. V^T of a sub-block lies bt rows' worth of bytes behind its K rows.
  uint32_t kadr_lo = 0, kadr_hi = 0;
  int adr0 = -64;
  auto pool_k = [&](int sidx) __attribute__((always_inline)) {
    if (sidx - adr0 >= 64) {  // (sub-blocks are asked for in order)
      adr0 = sidx;
      const int sl = sidx + lane;
      const int js = sl < n_c ? (c0 + sl) << 4 : (in_pool && sl < n_sb) ? ((a0 + sl - n_c) << 4) + pool_shift : -1;
      uint64_t adr = 0;
      if (js >= 0) {
        const int b = block_of(a, table, js);
        adr = reinterpret_cast<uint64_t>(a.pool + head_base(a, kHD, b, kvh)) + uint64_t(js % a.bt) * 1024;
      }
      kadr_lo = uint32_t(adr);
      kadr_hi = uint32_t(adr >> 32);
      asm volatile("" : "+v"(kadr_lo), "+v"(kadr_hi));  // arrived here: a wait at the lane reads below would drain the staging loads
    }
    const int idx = sidx - adr0;
    const uint32_t lo = uint32_t(__builtin_amdgcn_readlane(int(kadr_lo), idx)), hi = uint32_t(__builtin_amdgcn_readlane(int(kadr_hi), idx));
    return reinterpret_cast<const char*>(uint64_t(lo) | (uint64_t(hi) << 32));
  };
  const uint32_t kx = uint32_t(4 * wave);
  const uint32_t voff = uint32_t((lane ^ ((lane >> 4) & 1)) << 4);
  // Staging of a step whose sub-blocks the pool holds: where this wavefront's share of the K of sub-block t lies (and, bt rows' worth
  // of bytes behind it, of its V^T: kept for an iteration later), and its four loads of either, on one LDS base. fill_k and fill_v: the same, whatever
  // the sub-block (v_src null: past the range).
  const char* k_src = nullptr;
  const char* v_src[2] = {nullptr, nullptr};
  auto locate_k = [&](int t, int step) __attribute__((always_inline)) {
    k_src = pool_k(2 * step + t) + wave * 4096;
    v_src[t] = k_src + size_t(a.bt) * 1024;  // the 16-token sub-block: 16 KB contiguous
  };
  auto load_k = [&](int t, int stage) __attribute__((always_inline)) {
    const uint32_t kl = uint32_t(lane);
    load_to_lds16_x4(k_src, (kl ^ kx) << 4, (kl ^ (kx + 1)) << 4, (kl ^ (kx + 2)) << 4, (kl ^ (kx + 3)) << 4,
                     lds_base + stage * kKStage + (16 * t + 4 * wave) * 1024);
  };
  auto load_v = [&](int t, int stage) __attribute__((always_inline)) {
    load_to_lds16_x4(v_src[t], voff, voff, voff, voff, lds_base + kVBase + stage * kVStage + t * kVSub + wave * 4096);
  };
  auto fill_k = [&](int t, int step, int stage) __attribute__((always_inline)) {
    const int sidx = 2 * step + t;
    if (sidx < n_c || (in_pool && sidx < n_sb)) {
      locate_k(t, step);
      load_k(t, stage);
    } else if (sidx < n_sb) {
      const int g = a0 + (sidx - n_c);
      const int lim = a.n_rows - 1 - 16 * g;  // batch rows past the pass's last row do not exist: repeat the last (masked)
      const char* kb = reinterpret_cast<const char*>(a.Kb + size_t(16 * g) * a.kv_ld + size_t(kvh) * kHD);
      v_src[t] = reinterpret_cast<const char*>(a.vt_stage + (size_t(kvh) * n_groups + g) * size_t(kHD) * 16) + wave * 4096;
#pragma unroll
      for (int q = 0; q < 4; ++q)
        load_to_lds16(kb + size_t(min(4 * wave + q, lim)) * size_t(a.kv_ld) * 2, (uint32_t(lane) ^ (kx + q)) << 4,
                      lds_base + stage * kKStage + (16 * t + 4 * wave + q) * 1024);
    } else {
      v_src[t] = nullptr;  // past the range: K stays whatever it was (S is masked)
    }
  };
  auto fill_v = [&](int t, int stage) __attribute__((always_inline)) {
    if (v_src[t]) {
      load_v(t, stage);
    } else {  // V^T must be finite
#pragma unroll
      for (int q = 0; q < 4; ++q)
        *reinterpret_cast<u32x4*>(lds + kVBase + stage * kVStage + t * kVSub + wave * 4096 + q * 1024 + lane * 16) = u32x4{0, 0, 0, 0};
    }
  };
  // After this wavefront's loads of V^T of `step` have landed: cached keys outside [k0, k1) may be memory
  // never written, and rows beside the tree's are another's; their V must not reach the products (0 x infinity).
  auto fix = [&](int step, int stage) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const int sidx = 2 * step + t;
      // keys [v0, v1) of the sub-block's own numbering count: the tile's cached range, or the tree's rows. (In the pool what
      // lies below its first row is the end of its cached keys; in Kb / Vb the staged V^T past the pass's last row is zero.)
      int j0, v0, v1;
      if (sidx < n_c) {
        j0 = (c0 + sidx) << 4;
        v0 = tile.k0;
        v1 = tile.k1;
      } else if (sidx < n_sb) {
        j0 = ((a0 + sidx - n_c) << 4) - tree.base;
        v0 = in_pool ? INT32_MIN : 0;
        v1 = !in_pool && tree.base + tree.M == a.n_rows ? 1 << 30 : tree.M;
      } else {
        continue;
      }
      if (j0 >= v0 && j0 + 16 <= v1) continue;
      const int jv = j0 + 8 * ((lane & 1) ^ ((lane >> 4) & 1));  // the half of the piece at this lane's position
      u32x4 msk;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const bool lo = jv + 2 * e >= v0 && jv + 2 * e < v1;
        const bool hi = jv + 2 * e + 1 >= v0 && jv + 2 * e + 1 < v1;
        msk[e] = (lo ? 0xffffu : 0u) | (hi ? 0xffff0000u : 0u);
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        u32x4* p = reinterpret_cast<u32x4*>(lds + kVBase + stage * kVStage + t * kVSub + wave * 4096 + q * 1024 + lane * 16);
        *p = *p & msk;
      }
    }
  };

  // ---- operand reads: LDS byte addresses (base register + immediate)
  using lds_u32x4 = const __attribute__((address_space(3))) u32x4;
  auto lds_ptr = [](uint32_t addr) __attribute__((always_inline)) { return reinterpret_cast<lds_u32x4*>(addr); };
  // K slice kk is chunk 4 kk + q4 of key row c16 of sub-block `half`.
  uint32_t kaddr[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) kaddr[j] = lds_base + uint32_t((16 * half + c16) * 1024 + (((4 * j + q4) ^ c16) << 4));
  // V^T operand nt of sub-block t: keys 8 hb .. + 7 of dim dw + 32 nt + l32.
  const uint32_t vaddr = lds_base + uint32_t(kVBase + (dw + l32) * 32 + ((hb ^ ((l32 >> 3) & 1)) << 4));
  // P operand of sub-block t: keys 8 hb .. + 7 of row l32. This lane's own P: keys 4 q4 .. + 3 of sub-block `half`, rows c16 and 16 + c16.
  const uint32_t paddr = lds_base + uint32_t(kPBase + (32 * rg + l32) * kPRow + 16 * hb);
  char* const p_own = lds + kPBase + (32 * rg + c16) * kPRow + 32 * half + 8 * q4;

  f32x16 acc[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[nt][i] = 0.0f;
  // Per score row of this lane: the running reference in log2 units of the scaled score and this lane's share of the row's sum. A
  // row begins at kUnset, the lowest value of the type: the first visible score gives an infinite P and with it a sum that asks for
  // a reference (a score of kUnset itself has it already), and keys the row does not see give 0 as always. ps: the lane's share of
  // the sum of the step whose P is in LDS, not yet in l_run.
  constexpr float kUnset = -__FLT_MAX__;
  float m_run[2], l_run[2], ps[2];
#pragma unroll
  for (int rt = 0; rt < 2; ++rt) {
    m_run[rt] = kUnset;
    l_run[rt] = ps[rt] = 0.0f;
  }
  f32x4 s[2];        // scores of the step: s[rt][e] is key 4 q4 + e of sub-block `half`, row 16 rt + c16
  u32x4 ring[2][4];  // operands on their way from LDS
  int out_of_range = 0;  // did any lane of the workgroup find its share of the last step's sum beyond 2^8?

  // P of the step's scores into buffer `buf`, and this lane's shares of its sums. The row sum is that of the rounded P the products
  // use: under a lazily moved reference the dominant P is not exactly 1, and O = sum(P~ v) / sum(P~) keeps its rounding out of
  // a row that one key dominates. No maximum is taken: all P >= 0, so a share of the sum <= 2^8 bounds every one of them.
  auto exp_pack = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int rt = 0; rt < 2; ++rt) {
      float p[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) p[e] = fast_exp2(__builtin_fmaf(s[rt][e], a.scale_log2, -m_run[rt]));
      const u32x2 w = {pack2<DT>(p[0], p[1]), pack2<DT>(p[2], p[3])};
      ps[rt] = sum2<DT>(w.y, sum2<DT>(w.x, 0.0f));
      *reinterpret_cast<u32x2*>(p_own + buf * kPBuf + 16 * rt * kPRow) = w;
    }
  };
  // Some lane of the workgroup found a reference too low for the step whose P is in buffer `buf` (or not set): every row takes
  // the maximum of that step over both wavefronts of its group, moves its reference, rescales what is accumulated, and the step's P is
  // written again. Every wavefront of the workgroup comes through here together.
  auto settle = [&](int buf) __attribute__((always_inline)) {
    asm volatile("s_nop 0");  // a real branch: this block must not be speculated into the loop body
    float* mx_sh = reinterpret_cast<float*>(lds + kMax) + rg * 64;
    float mx[2];
#pragma unroll
    for (int rt = 0; rt < 2; ++rt) {
      mx[rt] = fmaxf(fmaxf(s[rt][0], s[rt][1]), fmaxf(s[rt][2], s[rt][3]));
      mx[rt] = fmaxf(mx[rt], __shfl_xor(mx[rt], 16));
      mx[rt] = fmaxf(mx[rt], __shfl_xor(mx[rt], 32));
      if (q4 == 0) mx_sh[half * 32 + 16 * rt + c16] = mx[rt];
    }
    __syncthreads();
    float corr[2];
#pragma unroll
    for (int rt = 0; rt < 2; ++rt) {
      const float other = mx_sh[(half ^ 1) * 32 + 16 * rt + c16];
      const float m_new = fmaxf(m_run[rt], fmaxf(mx[rt], other) * a.scale_log2);  // scale > 0: the max commutes with it
      corr[rt] = fast_exp2(m_run[rt] - m_new);
      m_run[rt] = m_new;
      l_run[rt] *= corr[rt];
    }
    const float c = (lane & 16) ? corr[1] : corr[0];  // of row l32
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) acc[nt] *= c;
    exp_pack(buf);
    __syncthreads();
  };
  // Visibility of the step's keys of this wavefront's sub-block.
  auto mask = [&](int step) __attribute__((always_inline)) {
    const int sidx = 2 * step + half;
    const bool cached = sidx < n_c, batch = !cached && sidx < n_sb;
    const int j0 = cached ? (c0 + sidx) << 4 : ((a0 + sidx - n_c) << 4) - tree.base;
    if (cached && a.window == 0 && j0 >= tile.k0 && j0 + 16 <= tile.k1) return;  // every key visible to every row
#pragma unroll
    for (int rt = 0; rt < 2; ++rt) {
      // Visible keys of the sub-block for this row: j in [lo, hi], or b0 <= j < anc.
      int lo, hi, anc = 0;
      if (cached) {
        lo = tile.k0;
        hi = tile.k1 - 1;
        if (a.window > 0) lo = max(lo, qpos[rt] - a.window + 1);
      } else if (batch) {
        lo = max(d[rt].x, tile.b0);  // below b0 (the window's lower edge over the tile's rows) nothing is visible
        hi = min(k_last, (a.bidi && d[rt].w > 0) ? max(rr[rt], d[rt].w - 1) : rr[rt]);
        anc = min(d[rt].z, k_last + 1);
      } else {
        lo = 1;
        hi = 0;
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int j = j0 + 4 * q4 + e;
        bool vis = (j >= lo && j <= hi) || (j >= tile.b0 && j < anc);
        if (batch && a.window > 0 && vis) vis = qpos[rt] - a.pos[tree.base + j].x < a.window;
        s[rt][e] = vis ? s[rt][e] : -INFINITY;
      }
    }
  };
  auto mul_v = [&](const u32x4 (&buf)[4], int nt0, u32x4 p) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[nt0 + j] = mfma32x16<DT>(buf[j], p, acc[nt0 + j]);
  };

  // Iteration i. At its top the barrier has been passed that publishes K of step i, V^T and P of step i - 1; the first sub-block of V^T
  // of step i is on its way, and so are the first K operands. It requests the rest of V^T of step i and K of step i + 1, multiplies
  // Q K^T of step i, then P V of step i - 1 but for four instructions, with the softmax of step i between them, and leaves P of step i.
  // Those four instructions stand behind the barrier that publishes it and cover the first reads and requests of the next.
  // plain: every key of steps i and i + 1 is a cached key inside [k0, k1) of a layer without a window, i >= 1, and no reference has to
  // move. The loads stand between the matrix instructions there, a sub-block's four at a time.
  auto iter = [&](int i, auto plain) __attribute__((always_inline)) {
    constexpr bool PLAIN = decltype(plain)::value;
    const int S = i & 1;
    auto read_k = [&](u32x4 (&buf)[4], uint32_t off) __attribute__((always_inline)) {
#pragma unroll
      for (int j = 0; j < 4; ++j) buf[j] = *lds_ptr(kaddr[j] + off);
    };
    const uint32_t va = vaddr + uint32_t((S ^ 1) * kVStage), pa = paddr + uint32_t((S ^ 1) * kPBuf);
    auto read_v = [&](u32x4 (&buf)[4], int t, int nt0) __attribute__((always_inline)) {
#pragma unroll
      for (int j = 0; j < 4; ++j) buf[j] = *lds_ptr(va + uint32_t(t * kVSub + (nt0 + j) * 1024));
    };
    if constexpr (!PLAIN) {
      if (i > 0 && out_of_range) settle(S ^ 1);
      fill_v(1, S);
      if (i + 1 < n_steps) {
        fill_k(0, i + 1, S ^ 1);
        fill_k(1, i + 1, S ^ 1);
      }
    }
#pragma unroll
    for (int rt = 0; rt < 2; ++rt) {
      l_run[rt] += ps[rt];
      s[rt] = f32x4{0, 0, 0, 0};
    }
    u32x4 pf[2], carry[4];
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      if (g < 3) {
        read_k(ring[(g + 1) & 1], uint32_t(256 * (g + 1)));
      } else {
        read_v(ring[0], 0, 0);
#pragma unroll
        for (int t = 0; t < 2; ++t) pf[t] = *lds_ptr(pa + uint32_t(32 * t));
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
#pragma unroll
        for (int rt = 0; rt < 2; ++rt) s[rt] = mfma16x32<DT>(ring[g & 1][j], qf[rt][4 * g + j], s[rt]);
        if (PLAIN && (j & 1)) {
          const int slot = 2 * g + (j >> 1);
          __builtin_amdgcn_sched_barrier(0);
          if (slot == 0) load_v(1, S);
          if (slot == 2) locate_k(0, i + 1), load_k(0, S ^ 1);
          if (slot == 4) locate_k(1, i + 1), load_k(1, S ^ 1);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    read_v(ring[1], 0, 4);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (!PLAIN) {
      mfma_settle(s[0]);
      mfma_settle(s[1]);
      mask(i);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (PLAIN || i > 0) {
      mul_v(ring[0], 0, pf[0]);
      read_v(ring[0], 1, 0);
      mul_v(ring[1], 4, pf[0]);
      read_v(carry, 1, 4);
      if constexpr (PLAIN) exp_pack(S);
      mul_v(ring[0], 0, pf[1]);
    }
    if constexpr (PLAIN) {
#pragma unroll
      for (int j = 0; j < 12; ++j) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, 5, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      }
    } else {
      exp_pack(S);
    }
    const int mine = __any(ps[0] > 256.0f || ps[1] > 256.0f);
    *reinterpret_cast<__attribute__((address_space(3))) int*>(uint32_t(kFlags + S * 16 + wave * 4)) = mine;  // (every lane the same: cheaper than one alone)
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");  // own loads landed, own reads of this iteration's stages done
    if constexpr (!PLAIN) fix(i, S);
    __syncthreads();
    const int fl = *reinterpret_cast<const __attribute__((address_space(3))) int*>(uint32_t(kFlags + S * 16 + (lane & 3) * 4));
#pragma unroll
    for (int j = 0; j < 4; ++j) kaddr[j] ^= uint32_t(kKStage);  // the other stage
    read_k(ring[0], 0);
    __builtin_amdgcn_sched_barrier(0);
    auto left = [&](int j) __attribute__((always_inline)) {
      if (PLAIN || i > 0) acc[4 + j] = mfma32x16<DT>(carry[j], pf[1], acc[4 + j]);
      __builtin_amdgcn_sched_barrier(0);
    };
    left(0);
    left(1);
    if constexpr (PLAIN) {
      load_v(0, S ^ 1);
    } else {
      if (i + 1 < n_steps) fill_v(0, S ^ 1);
    }
    __builtin_amdgcn_sched_barrier(0);
    left(2);
    left(3);
    out_of_range = __any(fl != 0);
  };
  constexpr std::false_type general{};
  constexpr std::true_type plain{};
  float l = 0.0f;  // the row's sum
  if (n_steps > 0) {
#pragma unroll
    for (int t = 0; t < 2; ++t) fill_k(t, 0, 0);
    wait_loads();
    __syncthreads();
    fill_v(0, 0);
#pragma unroll
    for (int j = 0; j < 4; ++j) ring[0][j] = *lds_ptr(kaddr[j]);
    // Plain iterations lie below p1: steps up to i + 1 are sub-blocks wholly inside the cached range.
    const int p1 = a.window == 0 && n_c > 0 ? ((n_c - ((tile.k1 & 15) ? 1 : 0)) >> 1) - 1 : 0;
    for (int i = 0; i < n_steps;) {
      iter(i++, general);
#pragma nounroll
      for (; i < p1 && !out_of_range; ++i) iter(i, plain);
    }
    // ---- what is left: P V of the last step
    const int S = (n_steps - 1) & 1;
    if (out_of_range) settle(S);
    // The row's sum: over the lanes that share the row, then over both wavefronts of the group (settle has left the place).
#pragma unroll
    for (int rt = 0; rt < 2; ++rt) {
      l_run[rt] += ps[rt];
      l_run[rt] += __shfl_xor(l_run[rt], 16);
      l_run[rt] += __shfl_xor(l_run[rt], 32);
    }
    float* l_sh = reinterpret_cast<float*>(lds + kMax) + rg * 64;
    const float l_mine = (lane & 16) ? l_run[1] : l_run[0];
    if (hb == 0) l_sh[half * 32 + l32] = l_mine;
    __syncthreads();
    l = half ? l_sh[l32] + l_mine : l_mine + l_sh[32 + l32];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const u32x4 p = *lds_ptr(paddr + uint32_t(S * kPBuf + 32 * t));
#pragma unroll
      for (int nt0 = 0; nt0 < NT; nt0 += 4) {
#pragma unroll
        for (int j = 0; j < 4; ++j) ring[0][j] = *lds_ptr(vaddr + uint32_t(S * kVStage + t * kVSub + (nt0 + j) * 1024));
        mul_v(ring[0], nt0, p);
      }
    }
  }

  // ---- output: lane (row l32, half hb) holds dims dw + 32 nt + 8 i + 4 hb + j at acc[nt][4 i + j].
  const float m_mine = (lane & 16) ? m_run[1] : m_run[0];
  const int m_row = 32 * rg + l32;
  const int row = tile.r0 + m_row;
  if (m_row >= rows_live) return;
  if (tile.part >= 0) {
    const size_t rec = (size_t(tile.part) * a.Hkv + kvh) * a.cols + size_t(m_row) * a.G + hg;
    float* po = a.parts_o + rec * kHD + dw;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int i4 = 0; i4 < 4; ++i4)
        *reinterpret_cast<f32x4*>(po + 32 * nt + 8 * i4 + 4 * hb) =
            f32x4{acc[nt][4 * i4], acc[nt][4 * i4 + 1], acc[nt][4 * i4 + 2], acc[nt][4 * i4 + 3]};
    if (hb == 0 && dw == 0) {
      a.parts_ml[rec * 2] = m_mine == kUnset && !(l > 0.0f) ? -INFINITY : m_mine;  // no key seen: the merge passes the part over
      a.parts_ml[rec * 2 + 1] = l;
    }
    return;
  }
  uint16_t* op = a.O + size_t(row) * a.q_ld + size_t(h) * kHD + dw + 4 * hb;
  finish_output<DT>(a, acc, l > 0.0f ? 1.0f / l : 0.0f, row, h, dw, hb, [&](int i, u32x2 v) { *reinterpret_cast<u32x2*>(op + 8 * i) = v; });
}

// The dynamic LDS limit of both variants on the current device, ahead of the first launch.
hipError_t tiled512_init_attributes() {
  const hipError_t e = allow_dynamic_lds<attn_tiled512_kernel<ESP_F16>>(kLds);
  return e != hipSuccess ? e : allow_dynamic_lds<attn_tiled512_kernel<ESP_BF16>>(kLds);
}

hipError_t launch_tiled512(int dt, const KArgs& a, int n_tiles, hipStream_t st) {
  constexpr auto kf = attn_tiled512_kernel<ESP_F16>;
  constexpr auto kb = attn_tiled512_kernel<ESP_BF16>;
  const hipError_t e = dt == ESP_F16 ? allow_dynamic_lds<kf>(kLds) : allow_dynamic_lds<kb>(kLds);
  if (e != hipSuccess) return e;
  launch_timed(dt == ESP_F16 ? kf : kb, dim3(unsigned(n_tiles) * a.H), dim3(256), size_t(kLds), st, a, n_tiles);
  return hipGetLastError();
}

}  // namespace esp
