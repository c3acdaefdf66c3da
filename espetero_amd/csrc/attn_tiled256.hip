// Tiled MFMA attention at head dim 256: prefill, chunked prefill, large verify batches.
//
// Semantics, key order and operand layouts as in the tiled kernel of 128 dims: cached keys [k0, k1) through the block table or
// ring, then the tree's batch keys (`last` tiles) under the tree mask (kernels/80_gemma.metal:284) and the window (80_:285), online
// softmax in fp32, P rounded to the storage type before P.V, output O / l (0 when no key is visible) with the optional
// sigmoid gate, or a partial record for the merge.
//
// Mapping to gfx950. A workgroup is one tile of up to 128 query rows x one query head (of a short tile: x all query heads of a KV
// head), its 4 wavefronts are 2 row groups of 64 rows x 2. Keys advance in steps of 64 (four 16-key sub-blocks; wavefront w stages
// sub-block w with global_load_lds_dwordx4). The two wavefronts of a row group share a step's scores by keys and its output by dims:
// wavefront (rg, half) computes
//   S^T[32 keys][64 rows] of sub-blocks 2 half, 2 half + 1 over all 256 dims   A = K from LDS, B = Q^T in registers
//   P^T = exp2(S^T - m)                                                        left in LDS in 16 bits
//   O^T[128 dims][64 rows] += V^T . P^T                                        its 128 dims, all 64 keys; A = V^T and B = P^T from LDS
// so that every operand read from LDS feeds two matrix instructions. P V runs one step behind Q K^T: one barrier per step publishes
// the staged data and the P at once, and the softmax of step i stands beside P V instructions that do not depend on it. K runs one step
// ahead of V in the staging. The row's reference m moves only where a lane's share of a step's sum says so, and in the whole workgroup at
// once: the two wavefronts of a row group multiply each other's P.
//
// What bounds it: the issue of a lone wavefront per SIMD (accumulators 128 registers, Q 128, the rest 143). Such a wavefront issues an
// instruction every 8 clocks (measured: 2, 4, 6, 8 multiply-adds behind every v_mfma_f32_32x32x16 make it 33, 38, 51, 66 clocks; two
// wavefronts on the SIMD 32, 33, 37, 45), so three instructions hide behind a matrix instruction's 32 clocks and every further one is
// matrix time lost; a v_dot2 waits for the matrix pipe to drain, 14 clocks wherever one stands alone. A step of mask-free keys in the pool
// is 64 matrix instructions (2048 clocks) and 331 others as compiled, 39 of them waits and s_nops: 139 beyond three each, 1100 clocks, and
// 3300 were measured, of which 1300 in Q K^T with 12 of the 16 loads, 1450 in three quarters of P V with the softmax, 180 in wait and
// barrier, 370 in the rest of P V with the other loads. So an instruction taken out of the step counts more than one moved: loads in pairs on
// one LDS base, one form of the loop for masked and mask-free steps (a second copy cost spills and what a workgroup waits for instructions it
// has not run before), masks worked out as bits. The form before, wavefronts of 32 rows with all keys and all dims, had 310 others but read
// 256 KB of operands per step through an LDS path of 128 bytes a clock, where this one reads 160: 4400 clocks.
// Behind a window, rows whose first key lies past their tile's first step have no reference until then: their first P is infinite, and the
// workgroup settles (four barriers, 128 multiplications, the step's softmax again) in one or two of a tile's 18 steps.
// 8 x 1024 rows over 15360 keys, 16 / 8 heads: 2180 us before, 1930 so; with a window of 1024 232 and 217; 100 rows over 6871 keys 44.5 and
// 40.4, with the window 47.2 and 41.1; prompts of 300 rows 24.8 and 22.9, of 32 10.7 and 9.6, one of 48 10.4 and 10.1, one of 128 14.2 and
// 12.8; of 2 .. 7 rows side by side from Kb / Vb 12.1 and 12.5 (their groups of 16 hold each other's rows, whose V is zeroed in LDS).
//
// LDS layout (all 160 KB). K of a stage: 64 rows of 512 bytes, unpadded; the 16-byte chunk c of row r lies at chunk position
// c ^ (pi(r) & 15), where pi swaps bits 2 and 3 of a row index. The lane with S^T row l reads key row pi(l): its chunk position is
// c ^ (l & 15), distinct over any 16 consecutive lanes -> no bank conflicts, and the 8 P values a lane packs for one P V instruction are
// 8 consecutive keys, which is how V^T lies in memory. V^T per sub-block, per group of 32 dims: [half of the 16 keys][32 dims][8 keys].
// P: the very 16 bytes per lane that are the operand.
#include <utility>

#include "common.hpp"
#include "lds_direct.hpp"
#include "rows_out.hpp"

namespace esp {

namespace {
constexpr int kHD = 256, kHW = 128;                  // dims of a head; dims one wavefront accumulates
constexpr int kRowB = kHD * 2;                       // bytes of a K row
constexpr int kKSub = 16 * kRowB;                    // K of one sub-block
constexpr int kKStage = 4 * kKSub;                   // K of one stage: 64 rows
constexpr int kVSub = kHD * 32;                      // V^T of one sub-block
constexpr int kVStage = 4 * kVSub;
constexpr int kVBase = 2 * kKStage;                  // layout: K stage 0, K stage 1, V^T stage 0, V^T stage 1, P of two steps
constexpr int kPBase = kVBase + 2 * kVStage;
constexpr int kPWave = 4 * 1024;                     // a wavefront's P of one step: [row tile][sub-block][lane] 16 bytes
constexpr int kPBuf = 4 * kPWave;
constexpr int kLds = kPBase + 2 * kPBuf;             // all of a compute unit's 160 KB
constexpr int kFlagAt = 3 * 1024 + 12;               // in a wavefront's P: lane 0's last word of the last piece carries its flag
}  // namespace

template <int DT>
__global__ __launch_bounds__(256, 1) void attn_tiled256_kernel(const KArgs a, int n_tiles) {
  constexpr int NT = kHW / 32, KS = kHD / 16;
  extern __shared__ __attribute__((aligned(16))) char lds[];  // the only LDS object: it begins at LDS address 0
  int(*red)[4] = reinterpret_cast<int(*)[4]>(lds + kVBase + kVStage);  // in the prologue, V^T stage 1 being free

  // Workgroup -> (KV head, head in group, tile): consecutive ids differ in KV head first, so the heads
  // sharing a KV head land on the same XCD's L2; tiles run last to first (longest key ranges first).
  const int kvh = blockIdx.x % a.Hkv;
  const int rest = blockIdx.x / a.Hkv;
  const int hg = rest % a.G;
  const int tile_i = n_tiles - 1 - rest / a.G;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int rg = wave >> 1, half = wave & 1, dw = half * kHW;
  const int l32 = lane & 31, hb = lane >> 5;
  esp_tile tile = a.tiles[tile_i];

  // ---- Q rows of the tile: whole rows, two to a load, through K stage 1 (rows 0 .. 63) and the place of P (row r's 16-byte chunk c at
  // position c ^ (r % 16)).
  // Loads of the fragments themselves, whose neighbouring lanes are different rows, take the memory path a clock per lane, and
  // both wavefronts of a row group need all dims of its 64 rows. The loads need the tile's record only: a row past the
  // pass's last one reads that row instead, one past the tree's is zeroed once the tree's record says so.
  // Tiles of up to 32 rows take four of the 16, of up to 64 eight, and a row group without rows reads no fragments: what a short prompt waits for.
  u32x4 qrow[16];
  auto q_loads = [](int rows, auto&& f) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 4; ++i) f(i);
    if (rows > 32) {
#pragma unroll
      for (int i = 4; i < 8; ++i) f(i);
    }
    if (rows > 64) {
#pragma unroll
      for (int i = 8; i < 16; ++i) f(i);
    }
  };
  {
    const char* q0 = reinterpret_cast<const char*>(a.Q + size_t(tile.r0) * a.q_ld + size_t(kvh * a.G + hg) * kHD);
    const uint32_t ld = uint32_t(a.q_ld) * 2, last = uint32_t(min(a.n_rows - 1 - tile.r0, 127)) * ld + uint32_t(l32) * 16;
    uint32_t at = uint32_t(2 * wave + hb) * ld + uint32_t(l32) * 16;
    q_loads(a.n_rows - tile.r0, [&](int i) __attribute__((always_inline)) {
      qrow[i] = *reinterpret_cast<const u32x4*>(q0 + min(at, last));
      at += 8 * ld;
    });
  }
  // ---- this lane's two rows of the scores: places 64 rg + 32 rt + l32
  int m[2], row_of[2], qpos[2];
  int4 d[2];
  auto load_facts = [&](int rt) __attribute__((always_inline)) {
    row_of[rt] = min(tile.r0 + m[rt], a.n_rows - 1);
    d[rt] = a.desc ? a.desc[row_of[rt]] : make_int4(0, 0, 0, 0);
    qpos[rt] = a.window > 0 ? a.pos[row_of[rt]].x : 0;
  };
#pragma unroll
  for (int rt = 0; rt < 2; ++rt) {
    m[rt] = 64 * rg + 32 * rt + l32;
    load_facts(rt);
  }

  const esp_tree tree = a.trees[tile.tree];
  if (tile.k1 == INT32_MAX) tile.k1 = tree.P;  // open-ended range: up to the tree's cached length as it is now
  const int table = tile.pad > 0 ? tile.pad - 1 : tree.table;
  const int end = tree.base + tree.M;
  const int rows_live = min(a.R, end - tile.r0);
  const int rr0 = tile.r0 - tree.base;
  // A short tile whose rows of all G query heads fit the tile's 128 places is one workgroup per KV head: place x of it is
  // row x / G, query head x % G, and the workgroups of the other heads end here (as in the kernel of 128 dims).
  const bool packed = tiled_fits(rows_live, a.G) && tiled_packs_grid(gridDim.x) && a.G > 1;
  const int places = packed ? rows_live * a.G : rows_live;
  if (packed) {
    if (hg != 0) return;
#pragma unroll
    for (int rt = 0; rt < 2; ++rt) {
      m[rt] = (64 * rg + 32 * rt + l32) / a.G;
      load_facts(rt);
    }
    int pr = (2 * wave + hb) / a.G, ph = 2 * wave + hb - pr * a.G;
    const int step_r = 8 / a.G, step_h = 8 - step_r * a.G;
    q_loads(places, [&](int i) __attribute__((always_inline)) {
      const int row = min(tile.r0 + pr, a.n_rows - 1);
      qrow[i] = *reinterpret_cast<const u32x4*>(a.Q + size_t(row) * a.q_ld + size_t(kvh * a.G + ph) * kHD + 8 * l32);
      pr += step_r;
      ph += step_h;
      if (ph >= a.G) ph -= a.G, ++pr;
    });
  }
  const int rr[2] = {rr0 + m[0], rr0 + m[1]};

  // ---- the key range as 16-key sub-blocks: cached [k0, k1), then batch rows [b0, k_last]
  const int c0 = tile.k0 >> 4;
  const int n_c = tile.k1 > tile.k0 ? ((tile.k1 + 15) >> 4) - c0 : 0;
  const int a0 = (tree.base + tile.b0) >> 4;  // batch sub-blocks are groups of 16 absolute rows
  // Batch rows in the pool (no Kb / Vb): row j of a tree lies at position P + j of the tree's block list, P - base a multiple of 16:
  // a batch sub-block of 16 absolute rows is one 16-token sub-block of the pool, staged like a cached one.
  const bool in_pool = a.Kb == nullptr;
  const int pool_shift = tree.P - tree.base;
  // Sub-blocks the tree's block list can name for this tile: at least those of the range that the pool holds.
  const int n_sb_list = n_c + ((in_pool && tile.last && tree.M > tile.b0) ? ((end - 1) >> 4) - a0 + 1 : 0);

  // Pool addresses of this wavefront's sub-blocks, 64 steps at a time: lane l holds the byte address of the K rows of sub-block
  // 4 (adr_step0 + l) + wave, or of the last one there is. V^T lies bt rows' worth of bytes behind. Steps are asked for in order.
  uint32_t kadr_lo = 0, kadr_hi = 0;
  int adr_step0 = -64;
  auto pool_k = [&](int step) __attribute__((always_inline)) {
    if (step - adr_step0 >= 64) {
      adr_step0 = step;
      const int sl = min(4 * (step + lane) + wave, n_sb_list - 1);
      uint64_t adr = 0;
      if (sl >= 0) {
        const int js = sl < n_c ? (c0 + sl) << 4 : ((a0 + sl - n_c) << 4) + pool_shift;
        const int b = block_of(a, table, js);
        const int t0 = a.bt == 16 ? 0 : js % a.bt;
        adr = reinterpret_cast<uint64_t>(a.pool + head_base(a, kHD, b, kvh)) + uint64_t(t0) * kRowB;
      }
      kadr_lo = uint32_t(adr);
      kadr_hi = uint32_t(adr >> 32);
      asm volatile("" : "+v"(kadr_lo), "+v"(kadr_hi));  // arrived here: a wait at the lane reads below would drain the staging loads
    }
    const int idx = step - adr_step0;
    const uint32_t lo = uint32_t(__builtin_amdgcn_readlane(int(kadr_lo), idx)), hi = uint32_t(__builtin_amdgcn_readlane(int(kadr_hi), idx));
    return reinterpret_cast<const char*>(uint64_t(lo) | (uint64_t(hi) << 32));
  };

  // ---- staging of this wavefront's sub-block. K instruction q brings rows 2 q, 2 q + 1: lane l row 2 q + l / 32, and there the
  // chunk that belongs at position l % 32, which is that ^ pi(row) (pi swaps bits 2 and 3 of a row). V^T instruction q brings dims 32 q ..:
  // keys 8 (l / 32) .. + 7 of dim 32 q + l % 32. Two instructions go with one LDS base (the immediate offset moves the global
  // address too: k_row makes up for it where rows are not 512 bytes apart).
  const uint32_t kcol0 = uint32_t((l32 ^ hb) << 4);
  const uint32_t voff = uint32_t(l32 * 32 + hb * 16);
  auto kswz = [](int q) constexpr { return uint32_t(swap23(2 * q) << 4); };
  const char *k_src = nullptr, *v_src = nullptr;
  uint32_t k_ld = kRowB, k_row = uint32_t(hb) * kRowB;
  int n_sb = 0;
  const int n_groups = (a.n_rows + 15) >> 4;
  // The pass's last group where not all of its 16 rows exist: its K rows are brought one instruction at a time once the others of
  // the step have landed (rows past the end are masked).
  const char* cut_src = nullptr;
  int cut_lim = 0;
  // Steps whose sub-block of this wavefront the pool holds.
  const int pool_steps = in_pool ? INT32_MAX : (n_c - wave + 3) >> 2;
  // Where the sub-block of `step` lies. Past the range: the last one of the range (its scores are masked, its V^T zeroed in `fix`).
  auto locate = [&](int step) __attribute__((always_inline)) {
    const int s = min(4 * step + wave, n_sb - 1);
    if (step < pool_steps || s < n_c) {
      k_src = pool_k(step);
      v_src = k_src + size_t(a.bt) * kRowB;
    } else {
      const int g = a0 + (s - n_c);
      k_src = reinterpret_cast<const char*>(a.Kb + size_t(16 * g) * a.kv_ld + size_t(kvh) * kHD);
      v_src = reinterpret_cast<const char*>(a.vt_stage + (size_t(kvh) * n_groups + g) * size_t(kHD) * 16);
      k_ld = uint32_t(a.kv_ld) * 2;
      if (16 * g + 15 >= a.n_rows) {
        if (4 * step + wave < n_sb) {
          cut_src = k_src;
          cut_lim = a.n_rows - 1 - 16 * g;
        }
        k_src = v_src;  // something that is there
        k_ld = kRowB;
      }
      k_row = hb ? k_ld : 0u;
    }
  };
  // K instructions q = 2 Q2, 2 Q2 + 1 and V^T instructions 2 Q2, 2 Q2 + 1.
  auto load_k = [&]<int Q2>(int stage) __attribute__((always_inline)) {
    constexpr int q = 2 * Q2, r = q & 3;
    uint32_t kc = kcol0;
    asm volatile("" : "+v"(kc));  // worked out where it is used, not kept in a register per instruction
    const uint32_t d = 2 * k_ld - 1024;
    load_to_lds16_x2<r / 2>(q < 4 ? k_src : k_src + size_t(8) * k_ld, (kc ^ kswz(q)) + (k_row + r * d), (kc ^ kswz(q + 1)) + (k_row + (r + 1) * d),
                            uint32_t(stage * kKStage + wave * kKSub + (q & 4) * 1024));
  };
  auto load_v = [&]<int Q2>(int stage) __attribute__((always_inline)) {
    constexpr int q = 2 * Q2;
    load_to_lds16_x2<(q & 3) / 2>(v_src + (q & 4) * 1024, voff, voff, uint32_t(kVBase + stage * kVStage + wave * kVSub + (q & 4) * 1024));
  };
  // What is left of the K of the step located last, once its loads have landed.
  auto load_cut = [&](int stage) __attribute__((always_inline)) {
#pragma nounroll
    for (int q = 0; 2 * q <= cut_lim; ++q)
      load_to_lds16(cut_src, uint32_t(min(2 * q + hb, cut_lim)) * (uint32_t(a.kv_ld) * 2) + (kcol0 ^ uint32_t(swap23(2 * q) << 4)),
                    uint32_t(stage * kKStage + wave * kKSub + q * 1024));
    cut_src = nullptr;
  };
  auto load_k_all = [&](int stage) __attribute__((always_inline)) {
    load_k.template operator()<0>(stage);
    load_k.template operator()<1>(stage);
    load_k.template operator()<2>(stage);
    load_k.template operator()<3>(stage);
  };

  // Step 0 leaves now, behind the Q rows, and has landed at the first barrier with them (the store of the last Q row waits on the same
  // counter). The rows' facts may show that the range ends sooner than the tree: what is brought beyond it is there all the same, and masked.
  n_sb = n_c + ((tile.last && tree.M > tile.b0) ? ((end - 1) >> 4) - a0 + 1 : 0);
  if (n_sb > 0) {
    locate(0);
    if (cut_src) load_cut(0);
    else load_k_all(0);
    load_v.template operator()<0>(0);
    load_v.template operator()<1>(0);
    load_v.template operator()<2>(0);
    load_v.template operator()<3>(0);
  }

  bool row_ok[2];
#pragma unroll
  for (int rt = 0; rt < 2; ++rt) {
    row_ok[rt] = m[rt] < rows_live;
    if (!row_ok[rt]) {
      d[rt] = make_int4(0, 0, 0, 0);
      qpos[rt] = 0;
    }
  }

  // ---- tile-wide facts about the rows (for the batch range and the no-mask fast path), and the rows into LDS
  int k_last = -1, seg_max = 0, qpos_max = 0;
  bool anc_any = false;  // does any row of the tile see ancestors (keys below its segment)?
  {
    const bool plain = !a.desc && a.window == 0;  // rows below their own row's number, and that is all
    if (!plain) {
      int kl = -1, sm = 0, am = 0, qm = INT32_MIN;
#pragma unroll
      for (int rt = 0; rt < 2; ++rt)
        if (row_ok[rt]) {
          kl = max(kl, max(rr[rt], max(d[rt].z - 1, a.bidi ? d[rt].w - 1 : -1)));
          sm = max(sm, d[rt].x);
          am = max(am, d[rt].z);
          qm = max(qm, qpos[rt]);
        }
#pragma unroll
      for (int o = 16; o >= 1; o >>= 1) {
        kl = max(kl, __shfl_xor(kl, o));
        sm = max(sm, __shfl_xor(sm, o));
        am = max(am, __shfl_xor(am, o));
        qm = max(qm, __shfl_xor(qm, o));
      }
      if (lane == 0) {
        red[wave][0] = kl;
        red[wave][1] = sm;
        red[wave][2] = am;
        red[wave][3] = qm;
      }
    }
    auto q_place = [&](int i) __attribute__((always_inline)) {
      const int r = 8 * i + 2 * wave + hb;
      return reinterpret_cast<u32x4*>(lds + (i < 8 ? kKStage : kPBase - 64 * kRowB) + r * kRowB + ((l32 ^ (r & 15)) << 4));
    };
    q_loads(places, [&](int i) __attribute__((always_inline)) { *q_place(i) = qrow[i]; });
#pragma nounroll
    for (int i = places >> 3; i < (places > 64 ? 16 : 8); ++i)
      if (8 * i + 2 * wave + hb >= places) *q_place(i) = u32x4{0, 0, 0, 0};
    __syncthreads();
    int anc_max = 0;
    if (plain) {
      k_last = rr0 + rows_live - 1;
    } else {
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        k_last = max(k_last, red[w][0]);
        seg_max = max(seg_max, red[w][1]);
        anc_max = max(anc_max, red[w][2]);
        qpos_max = max(qpos_max, red[w][3]);
      }
    }
    // The same in every lane; saying so keeps everything derived from them in scalar registers.
    // a part whose batch range is cut ends at row last - 2 of the tree (last = 1: open, up to what its rows see)
    k_last = __builtin_amdgcn_readfirstlane(min(min(k_last, tree.M - 1), tile.last >= 2 ? tile.last - 2 : INT32_MAX));
    seg_max = __builtin_amdgcn_readfirstlane(seg_max);
    anc_max = __builtin_amdgcn_readfirstlane(anc_max);
    qpos_max = __builtin_amdgcn_readfirstlane(qpos_max);
    if (anc_max > 0 || a.bidi) seg_max = INT32_MAX;  // rows that see beyond the causal rule: always mask
    anc_any = anc_max > 0;
  }
  // Q fragments as stored: the scale (times log2 e) is applied to the fp32 score in the fused multiply-add that subtracts the
  // row's reference.
  u32x4 qf[2][KS];
  const int q_at = rg == 0 ? kKStage : kPBase - 64 * kRowB;
  if (64 * rg < places) {
#pragma unroll
    for (int rt = 0; rt < 2; ++rt) {
      const int r = 64 * rg + 32 * rt + l32;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) qf[rt][ks] = *reinterpret_cast<const u32x4*>(lds + q_at + r * kRowB + (((2 * ks + hb) ^ (r & 15)) << 4));
    }
  }
#pragma unroll
  for (int rt = 0; rt < 2; ++rt)
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) asm volatile("" : "+a"(qf[rt][ks]));

  const int n_b = (tile.last && k_last >= tile.b0) ? ((tree.base + k_last) >> 4) - a0 + 1 : 0;
  n_sb = n_c + n_b;
  const int n_steps = (n_sb + 3) >> 2;
  // A tile none of whose rows reaches b0: step 0 may have left with batch rows all the same; the sub-blocks that follow are the pool's.
  if (n_b == 0) {
    k_ld = kRowB;
    k_row = uint32_t(hb) * kRowB;
  }

  // Windowed layers: do this tile's batch keys need a window test at all? Not when the oldest position among
  // them is inside the window of the row with the largest position. Where they do and their positions rise by
  // one per row (position of row j = j + const: a plain chunk of prompt), the window is one more lower
  // bound in row numbers, j >= qpos - w_off, and a step whose rows lie at or above bw_lo is inside every row's
  // window; only other position patterns (trees) take the per-key position test.
  bool batch_window = false;
  int w_off = 1 << 30, bw_lo = INT32_MIN;
  if (a.window > 0 && n_b > 0) {
    int kp = INT32_MAX, dmin = INT32_MAX, dmax = INT32_MIN;
    for (int j = tile.b0 + int(threadIdx.x); j <= k_last; j += 256) {
      const int p = a.pos[tree.base + j].x;
      kp = min(kp, p);
      dmin = min(dmin, p - j);
      dmax = max(dmax, p - j);
    }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
      kp = min(kp, __shfl_xor(kp, o));
      dmin = min(dmin, __shfl_xor(dmin, o));
      dmax = max(dmax, __shfl_xor(dmax, o));
    }
    __syncthreads();  // every wavefront has read the facts above
    if (lane == 0) {
      red[wave][0] = kp;
      red[wave][1] = dmin;
      red[wave][2] = dmax;
    }
    __syncthreads();
    kp = __builtin_amdgcn_readfirstlane(min(min(red[0][0], red[1][0]), min(red[2][0], red[3][0])));
    dmin = __builtin_amdgcn_readfirstlane(min(min(red[0][1], red[1][1]), min(red[2][1], red[3][1])));
    dmax = __builtin_amdgcn_readfirstlane(max(max(red[0][2], red[1][2]), max(red[2][2], red[3][2])));
    if (qpos_max - kp >= a.window) {
      if (dmin == dmax) {
        w_off = a.window - 1 + dmin;
        bw_lo = qpos_max - w_off;
      } else {
        batch_window = true;
      }
    }
  }

  // After this wavefront's loads of V^T of `step` have landed: cached keys outside [k0, k1) may be memory never written, other trees' rows
  // and keys past the range are not its own; their V must not reach the products (0 x infinity).
  auto fix = [&](int step, int stage) __attribute__((always_inline)) {
    const int s = 4 * step + wave;
    // keys [v0, v1) of the sub-block's own numbering count: the tile's cached range, or the tree's rows. (In Kb / Vb the
    // rows beside them are other trees'; in the pool what lies below its first row is the end of its cached keys.)
    int j0 = 0, v0 = 0, v1 = 0;
    if (s < n_c) {
      j0 = (c0 + s) << 4;
      v0 = tile.k0;
      v1 = tile.k1;
    } else if (s < n_sb) {
      j0 = ((a0 + s - n_c) << 4) - tree.base;
      v0 = in_pool ? -16 : 0;  // (a sub-block begins less than 16 rows in front of the tree)
      v1 = !in_pool && end == a.n_rows ? 1 << 30 : tree.M;  // (past the pass's last row the staged V^T is zero)
    }
    if (j0 >= v0 && j0 + 16 <= v1) return;
    const int jv = j0 + 8 * hb;
    const int e0 = min(max(v0 - jv, 0), 8), e1 = min(max(v1 - jv, e0), 8);
    const uint32_t in = (1u << e1) - (1u << e0);  // this lane's 8 keys, a bit each
    u32x4 msk;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      msk[e] = (uint32_t(__builtin_amdgcn_sbfe(int(in), 2 * e, 1)) & 0xffffu) | uint32_t(__builtin_amdgcn_sbfe(int(in), 2 * e + 1, 1)) << 16;
#pragma unroll 4
    for (int q = 0; q < 8; ++q) {
      u32x4* p = reinterpret_cast<u32x4*>(lds + kVBase + stage * kVStage + wave * kVSub + q * 1024 + lane * 16);
      *p = *p & msk;
    }
  };

  // ---- operand reads: LDS byte addresses (base register + immediate)
  using lds_u32x4 = const __attribute__((address_space(3))) u32x4;
  using lds_i32 = const __attribute__((address_space(3))) int;
  auto lds_ptr = [](uint32_t addr) __attribute__((always_inline)) { return reinterpret_cast<lds_u32x4*>(addr); };
  // K slice ks: chunk 2 ks + hb of key row pi(l32) of the wavefront's 32 keys; slices ks and ks + 8 are 256 bytes apart. The stage is
  // bit 15 of the address and changes by it.
  uint32_t kaddr[8];
  {
    const int prow = (l32 & 0x13) | ((l32 & 4) << 1) | ((l32 & 8) >> 1);  // pi(l32)
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) kaddr[ks] = uint32_t(half * 2 * kKSub + prow * kRowB + (((2 * ks + hb) ^ (l32 & 15)) << 4));
  }
  // V^T operand (sub-block t, nt): the lane's 16 bytes of dims dw + 32 nt ..
  const uint32_t vaddr = uint32_t(kVBase + half * (kVSub / 2) + lane * 16);
  // P operand (row tile rt, sub-block t): this lane's 16 bytes, as wavefront (rg, t / 2) left them.
  const uint32_t paddr = uint32_t(kPBase + 2 * rg * kPWave + lane * 16);
  char* const p_own = lds + kPBase + wave * kPWave + lane * 16;

  f32x16 acc[2][NT];
  // (by matrix instructions: 8, where moves would be 128)
  auto clear = [&]() __attribute__((always_inline)) {
    u32x4 z = {0, 0, 0, 0};
    asm volatile("" : "+v"(z));
    const f32x16 none = {};
#pragma unroll
    for (int n = 0; n < 2 * NT; ++n) acc[n & 1][n >> 1] = mfma32x16<DT>(z, z, none);
  };
  // Per row of this lane: the running reference in log2 units of the scaled score and this lane's share of the row's sum. A row
  // begins at kUnset, the lowest value of the type. ps: the lane's share of the sum of the step whose P is in LDS, not yet in l_run.
  constexpr float kUnset = -__FLT_MAX__;
  float m_run[2], l_run[2], ps[2];
#pragma unroll
  for (int rt = 0; rt < 2; ++rt) {
    m_run[rt] = kUnset;
    l_run[rt] = ps[rt] = 0.0f;
  }
  f32x16 s[2];       // scores of the step: s[rt][4 i + j] is key 16 (i / 2) + 8 hb + 4 (i % 2) + j of the wavefront's 32, row 32 rt + l32
  u32x4 ring[2][4];  // operands on their way from LDS
  u32x4 pf[2][2];    // P operands of two sub-blocks: [sub-block % 2][rt]
  bool out_of_range = false;  // did any lane of the workgroup find its share of the last step's sum beyond 2^8?

  // P of the step's scores in 16 slices, one pair of scores each: slice q takes the exponentials of pair q and packs, sums and leaves pair
  // q - 1. The row sum is that of the rounded P the products use. No maximum is taken: all P >= 0, so a share of the sum <= 2^8 bounds
  // every one of them. The last piece waits for the comparison of the sums: a set sign in lane 0's last word (P has none) is the
  // wavefront's flag.
  float pv[4];
  u32x4 pw[2];
  auto slice_pack = [&]<int Q>(int buf) __attribute__((always_inline)) {
    constexpr int rt = Q >> 3, e = Q & 7;
    uint32_t w = pack2<DT>(pv[2 * (Q & 1)], pv[2 * (Q & 1) + 1]);
    asm volatile("" : "+v"(w));  // packed here, not sunk to the block of its first use
    pw[e >> 2][e & 3] = w;
    if constexpr ((e & 3) == 3 && Q != 15) *reinterpret_cast<u32x4*>(p_own + buf * kPBuf + (2 * rt + (e >> 2)) * 1024) = pw[e >> 2];
    // A row tile's sums in a row: v_dot2 waits for the matrix instruction in front of it and holds up the one behind, 14 clocks
    // wherever it stands alone, and 4 for each that follows.
    if constexpr (e == 7) {
      __builtin_amdgcn_sched_barrier(0);
      const float x = sum2<DT>(pw[1][0], sum2<DT>(pw[0][0], 0.0f)), y = sum2<DT>(pw[1][1], sum2<DT>(pw[0][1], 0.0f));
      const float z = sum2<DT>(pw[1][2], sum2<DT>(pw[0][2], 0.0f)), u = sum2<DT>(pw[1][3], sum2<DT>(pw[0][3], 0.0f));
      ps[rt] = (x + y) + (z + u);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  auto slice = [&]<int Q>(int buf) __attribute__((always_inline)) {
    constexpr int rt = Q >> 3, e = Q & 7;
    pv[2 * (Q & 1)] = fast_exp2(__builtin_fmaf(s[rt][2 * e], a.scale_log2, -m_run[rt]));
    pv[2 * (Q & 1) + 1] = fast_exp2(__builtin_fmaf(s[rt][2 * e + 1], a.scale_log2, -m_run[rt]));
    if constexpr (Q > 0) slice_pack.template operator()<Q - 1>(buf);
  };
  auto leave_last = [&](int buf, bool flag) __attribute__((always_inline)) {
    pw[1][3] = (pw[1][3] & 0x7fffffffu) | (flag ? 0x80000000u : 0u);
    *reinterpret_cast<u32x4*>(p_own + buf * kPBuf + 3 * 1024) = pw[1];
  };
  auto sums_beyond = [&]() __attribute__((always_inline)) { return __any(ps[0] > 256.0f || ps[1] > 256.0f) != 0; };
  // The rows' maxima over this wavefront's keys, left for the group's other one.
  auto leave_max = [&](char* mx_sh, float (&mx)[2]) __attribute__((always_inline)) {
#pragma unroll
    for (int rt = 0; rt < 2; ++rt) {
      mx[rt] = s[rt][0];
#pragma unroll
      for (int i = 1; i < 16; ++i) mx[rt] = fmaxf(mx[rt], s[rt][i]);
      mx[rt] = fmaxf(mx[rt], __shfl_xor(mx[rt], 32));
      if (hb == 0) *reinterpret_cast<float*>(mx_sh + wave * kPWave + (32 * rt + l32) * 4) = mx[rt];
    }
  };
  auto new_reference = [&](const char* mx_sh, const float (&mx)[2], int rt) __attribute__((always_inline)) {
    const float other = *reinterpret_cast<const float*>(mx_sh + (wave ^ 1) * kPWave + (32 * rt + l32) * 4);
    return fmaxf(m_run[rt], fmaxf(mx[rt], other) * a.scale_log2);  // scale > 0: the max commutes with it
  };
  auto all_slices = [&](int buf) __attribute__((always_inline)) {
    [&]<int... Q>(std::integer_sequence<int, Q...>) __attribute__((always_inline)) {
      (slice.template operator()<Q>(buf), ...);
    }(std::make_integer_sequence<int, 16>{});
    slice_pack.template operator()<15>(buf);
    leave_last(buf, false);
  };
  // Some lane of the workgroup found a reference too low for the step whose P is in buffer `buf` (or not set): every row takes the
  // maximum of that step over both wavefronts of its group, moves its reference, rescales what is accumulated, and the step's P is
  // written again. Every wavefront of the workgroup comes through here together (one whose group has ended only to its barriers).
  auto settle = [&](int buf) __attribute__((always_inline)) {
    asm volatile("s_nop 0");  // a real branch: this block must not be speculated into the loop body
    char* mx_sh = lds + kPBase + buf * kPBuf;
    __syncthreads();  // every wavefront has read the flags
    float mx[2];
    leave_max(mx_sh, mx);
    __syncthreads();
#pragma unroll
    for (int rt = 0; rt < 2; ++rt) {
      const float m_new = new_reference(mx_sh, mx, rt);
      const float corr = fast_exp2(m_run[rt] - m_new);
      m_run[rt] = m_new;
      l_run[rt] *= corr;
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) acc[rt][nt] *= corr;
    }
    __syncthreads();
    all_slices(buf);
    __syncthreads();
  };
  auto settle_beside = [&]() __attribute__((always_inline)) {
#pragma nounroll
    for (int k = 0; k < 4; ++k) __syncthreads();
  };

  const int wave_first[2] = {__builtin_amdgcn_readfirstlane(rr[0]), __builtin_amdgcn_readfirstlane(rr[1])};  // of either row tile
  // Steps this row group computes: batch steps past its last row hold nothing it can see, and their V, infinities among them, must not
  // reach its products. A group without a row (or with nothing to see) has only its share of the staging to do. `both`: the first
  // row tile sees something of the group's last step too.
  int my_steps = wave_first[0] < rr0 + rows_live ? n_steps : 0;
  bool both = true;
  if (seg_max != INT32_MAX) {
    auto step_end = [&](int rt) __attribute__((always_inline)) {  // one past the last step with a key at or below the row tile's last row
      const int last = min(__builtin_amdgcn_readlane(rr[rt], 31), rr0 + rows_live - 1);
      return last < tile.b0 ? (n_c + 3) >> 2 : (n_c + ((tree.base + last) >> 4) - a0 + 4) >> 2;
    };
    my_steps = min(my_steps, step_end(1));
    both = step_end(0) >= my_steps;
  }
  // Keys this lane's rows see: cached ones [lo_c, k1), batch ones [lo_b, end_b), or b0 <= j < anc. b0 is the first batch key any
  // row of the tile sees (the window's lower edge; 0 without one): the first sub-block starts at a multiple of 16 rows at or below it,
  // and what lies below b0 is invisible.
  int lo_c[2], lo_b[2], end_b[2];
#pragma unroll
  for (int rt = 0; rt < 2; ++rt) {
    lo_c[rt] = a.window > 0 ? max(tile.k0, qpos[rt] - a.window + 1) : tile.k0;
    lo_b[rt] = max(max(d[rt].x, tile.b0), qpos[rt] - w_off);
    end_b[rt] = n_b > 0 ? 1 + min(k_last, (a.bidi && d[rt].w > 0) ? max(rr[rt], d[rt].w - 1) : rr[rt]) : tile.b0;  // (a part without batch keys)
  }
  // Visibility of the step's keys of this wavefront.
  auto mask = [&](int step) __attribute__((always_inline)) {
    const int s0 = 4 * step + 2 * half;
    bool full[2] = {false, false};  // all 32 keys visible to every row of the row tile?
    if (s0 + 2 <= n_c) {
      const int j0 = (c0 + s0) << 4;
      full[0] = full[1] = j0 >= tile.k0 && j0 + 32 <= tile.k1 && (a.window == 0 || qpos_max - j0 < a.window);
    } else if (s0 >= n_c && s0 + 2 <= n_sb) {
      const int j0 = ((a0 + s0 - n_c) << 4) - tree.base;
      const bool most = !batch_window && j0 >= seg_max && j0 >= tile.b0 && j0 >= bw_lo;
#pragma unroll
      for (int rt = 0; rt < 2; ++rt) full[rt] = most && j0 + 31 <= min(wave_first[rt], k_last);
    }
    // first key of either sub-block (past the range: rows beyond the last one, which no row sees)
    int j0[2];
    bool cached[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      cached[t] = s0 + t < n_c;
      j0[t] = cached[t] ? (c0 + s0 + t) << 4 : ((a0 + s0 + t - n_c) << 4) - tree.base;
    }
#pragma unroll
    for (int rt = 0; rt < 2; ++rt) {
      if (full[rt]) continue;
      uint32_t vis = 0;  // this lane's 16 keys, a bit each
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const int jb = j0[t] + 8 * hb;
        const int e0 = min(max((cached[t] ? lo_c[rt] : lo_b[rt]) - jb, 0), 8);
        const int e1 = min(max((cached[t] ? tile.k1 : end_b[rt]) - jb, e0), 8);
        vis |= ((1u << e1) - (1u << e0)) << (8 * t);
      }
      if (anc_any || batch_window) {  // ancestors, per-key positions: the rare shapes
        const int anc = n_b > 0 ? min(d[rt].z, k_last + 1) : tile.b0;
#pragma nounroll
        for (int i = 0; i < 16; ++i) {
          if (i < 8 ? cached[0] : cached[1]) continue;
          const int j = (i < 8 ? j0[0] : j0[1]) + 8 * hb + (i & 7);
          bool v = (vis >> i & 1) || (j >= tile.b0 && j < anc);
          if (batch_window && v) v = qpos[rt] - a.pos[tree.base + j].x < a.window;
          vis = (vis & ~(1u << i)) | uint32_t(v) << i;
        }
      }
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const uint32_t v = uint32_t(__builtin_amdgcn_sbfe(int(vis), i, 1));  // all bits where visible
        const float x = s[rt][i];
        s[rt][i] = __builtin_bit_cast(float, (__builtin_bit_cast(uint32_t, x) & v) | (0xff800000u & ~v));
      }
    }
  };

  // ---- the pieces of an iteration
  auto k_operand = [&]<int KSL>(int more = 0) __attribute__((always_inline)) { return *lds_ptr(kaddr[(KSL + more) & 7] + uint32_t(KSL >> 3) * 256u); };
  // V^T and P operands of sub-block t of the step whose V^T lies at va and whose P at pa.
  auto v_operand = [&](uint32_t va, int t, int nt) __attribute__((always_inline)) { return *lds_ptr(va + uint32_t(t * kVSub + nt * 1024)); };
  auto p_operand = [&](uint32_t pa, int t, int rt) __attribute__((always_inline)) { return *lds_ptr(pa + uint32_t((t >> 1) * kPWave + (2 * rt + (t & 1)) * 1024)); };
  auto mul_v1 = [&](const u32x4 (&buf)[4], const u32x4 (&pb)[2], int n) __attribute__((always_inline)) {  // one of the 8 instructions of a sub-block
    acc[n & 1][n >> 1] = mfma32x16<DT>(buf[n >> 1], pb[n & 1], acc[n & 1][n >> 1]);
  };
  auto flags_of = [&](int buf) __attribute__((always_inline)) {
    return *reinterpret_cast<lds_i32*>(uint32_t(kPBase + buf * kPBuf + (lane & 3) * kPWave + kFlagAt));
  };

  // Iteration i. At its top the barrier has been passed that publishes K of step i, V^T and P of step i - 1; half of V^T of step i is
  // on its way, and so are the first K operands. It requests the rest of V^T of step i and K of step i + 1 between the instructions
  // of Q K^T of step i, multiplies P V of step i - 1 but for its last sub-block with the softmax of step i between, and leaves P of step i.
  // The last sub-block's instructions stand behind the barrier that publishes it and cover the first reads and requests of the next.
  // FIRST: i = 0 has no P V yet; it sets the rows' references. (What is requested past the last step goes to
  // stages that nobody reads any more.)
  auto iter = [&]<bool FIRST>(int i, bool clean) __attribute__((always_inline)) {
    const int S = i & 1;
    const uint32_t va = vaddr + uint32_t((S ^ 1) * kVStage), pa = paddr + uint32_t((S ^ 1) * kPBuf);
#pragma unroll
    for (int rt = 0; rt < 2; ++rt) {
      l_run[rt] += ps[rt];
#pragma unroll
      for (int e = 0; e < 16; ++e) s[rt][e] = 0.0f;
    }
    // (the next operands' reads come first in a group of eight matrix instructions, the loads behind them)
    auto qk = [&]<int N>() __attribute__((always_inline)) {
      constexpr int G = N >> 3, J = (N & 7) >> 1, rt = N & 1, gap = N & 7;
      s[rt] = mfma32x16<DT>(ring[G & 1][J], qf[rt][4 * G + J], s[rt]);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (G < 3) {
        if constexpr (gap < 4) ring[(G + 1) & 1][gap] = k_operand.template operator()<4 * G + 4 + gap>();
      } else if constexpr (!FIRST) {
        if constexpr (gap < 4) ring[0][gap] = v_operand(va, 0, gap);
        else if constexpr (gap < 6) pf[0][gap - 4] = p_operand(pa, 0, gap - 4);
      }
      if constexpr (N == 4 && !FIRST) load_v.template operator()<2>(S);
      if constexpr (N == 6 && !FIRST) load_v.template operator()<3>(S);
      if constexpr (N == 8) locate(i + 1);
      if constexpr (N == 12) load_k.template operator()<0>(S ^ 1);
      if constexpr (N == 14) load_k.template operator()<1>(S ^ 1);
      if constexpr (N == 20) load_k.template operator()<2>(S ^ 1);
      if constexpr (N == 22) load_k.template operator()<3>(S ^ 1);
      __builtin_amdgcn_sched_barrier(0);
    };
    [&]<int... N>(std::integer_sequence<int, N...>) __attribute__((always_inline)) {
      (qk.template operator()<N>(), ...);
    }(std::make_integer_sequence<int, 32>{});
    // Matrix instruction n of the first three sub-blocks of P V. The slices of the softmax stand behind the fourth and those that follow.
    constexpr int AHEAD = 3;
    auto pv_step = [&]<int N>() __attribute__((always_inline)) {
      constexpr int t = N >> 3, gap = N & 7;
      mul_v1(ring[t & 1], pf[t & 1], gap);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (gap < 4) ring[(t + 1) & 1][gap] = v_operand(va, t + 1, gap);
      else if constexpr (gap < 6) pf[(t + 1) & 1][gap - 4] = p_operand(pa, t + 1, gap - 4);
      constexpr int Q = N - AHEAD;
      if constexpr (Q >= 0 && Q < 16) slice.template operator()<Q>(S);
      if constexpr (Q == 16) slice_pack.template operator()<15>(S);
      __builtin_amdgcn_sched_barrier(0);
    };
    if constexpr (!FIRST) {
      [&]<int... N>(std::integer_sequence<int, N...>) __attribute__((always_inline)) {
        (pv_step.template operator()<N>(), ...);
      }(std::make_integer_sequence<int, AHEAD>{});
    }
    if (FIRST || !clean) {
      mfma_settle(s[0]);
      mfma_settle(s[1]);
      mask(i);
    }
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (!FIRST) {
      bool flag = false;
      [&]<int... N>(std::integer_sequence<int, N...>) __attribute__((always_inline)) {
        ([&]<int NN>() __attribute__((always_inline)) {
          if constexpr (NN == 22) {
            flag = sums_beyond();  // (two instructions ahead of its use: the comparison has come back)
            __builtin_amdgcn_sched_barrier(0);
          }
          pv_step.template operator()<NN>();
        }.template operator()<AHEAD + N>(), ...);
      }(std::make_integer_sequence<int, 24 - AHEAD>{});
      leave_last(S, flag);
    } else {  // the first step: its maxima are the rows' references
      char* mx_sh = lds + kPBase + kPBuf;
      float mx[2];
      leave_max(mx_sh, mx);
      __syncthreads();
#pragma unroll
      for (int rt = 0; rt < 2; ++rt) m_run[rt] = new_reference(mx_sh, mx, rt);
      clear();  // (beside the softmax)
      all_slices(0);
    }
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");  // own loads landed, own reads of this iteration's stages done
    if (cut_src) {
      load_cut(S ^ 1);
      wait_loads();
    }
    if (FIRST || !clean) fix(i, S);
    __syncthreads();
    const int fl = FIRST ? 0 : flags_of(S);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      kaddr[j] ^= uint32_t(kKStage);
      ring[0][j] = k_operand.template operator()<0>(j);
    }
    __builtin_amdgcn_sched_barrier(0);
    auto last = [&](int n) __attribute__((always_inline)) {
      mul_v1(ring[1], pf[1], 2 * n);
      mul_v1(ring[1], pf[1], 2 * n + 1);
      __builtin_amdgcn_sched_barrier(0);
    };
    if constexpr (!FIRST) last(0);
    load_v.template operator()<0>(S ^ 1);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (!FIRST) last(1);
    load_v.template operator()<1>(S ^ 1);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (!FIRST) last(2);
#pragma unroll
    for (int j = 4; j < 8; ++j) kaddr[j] ^= uint32_t(kKStage);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (!FIRST) last(3);
    out_of_range = !FIRST && __any(fl < 0) != 0;
  };

  // Mask-free steps: every key is one that every row of the tile sees and nothing needs fixing up. Two runs
  // of them: cached steps [int_lo, c_hi) - inside [k0, k1) and inside every row's window - and batch steps
  // [b_lo, b_hi), whose rows all lie below the tile's first row (and at or above b0, inside every segment,
  // with no ancestors and no per-key window test pending). Where the cached range ends on a step boundary
  // the two runs are one.
  int int_lo, c_hi, b_lo = 0, b_hi = 0;
  {
    const int first = c0 << 4;  // key of sub-block 0
    int lo_key = tile.k0;
    if (a.window > 0) lo_key = max(lo_key, qpos_max - a.window + 1);
    int_lo = lo_key <= first ? 0 : (lo_key - first + 63) >> 6;
    c_hi = ((tile.k1 >> 4) - c0) >> 2;  // steps wholly inside the cached range
    if (n_b > 0 && !batch_window && !anc_any && seg_max != INT32_MAX) {
      const int lo_b = max(max(max(tile.b0, seg_max), bw_lo), 0);
      const int g_lo = (tree.base + lo_b + 15) >> 4;           // first group of 16 rows wholly at or above lo_b
      const int g_hi = min(((tree.base + rr0) >> 4), ((tree.base + k_last + 1) >> 4)) - 1;  // last group wholly below the tile's first row (and inside the part's batch range)
      const int s_lo = n_c + g_lo - a0, s_hi = n_c + g_hi - a0;  // as sub-blocks of the range
      b_lo = (s_lo + 3) >> 2;
      b_hi = max(b_lo, (s_hi + 1) >> 2);
      if (b_lo == c_hi && (n_c & 3) == 0 && (tile.k1 & 15) == 0 && c_hi > int_lo) {  // one run
        c_hi = b_hi;
        b_lo = b_hi = 0;
      }
    }
  }

  // Where a row group's sums cross: each wavefront's in its own P, in the buffer that the last step's does not take.
  auto l_sh = [&](int w) __attribute__((always_inline)) { return reinterpret_cast<float*>(lds + kPBase + (my_steps & 1) * kPBuf + w * kPWave); };
  if (n_steps > 0) {
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");  // K of step 0 landed, Q fragments read
    __syncthreads();
    if (my_steps > 0) {
#pragma unroll
      for (int j = 0; j < 4; ++j) ring[0][j] = k_operand.template operator()<0>(j);
      iter.template operator()<true>(0, false);
#pragma nounroll
      for (int i = 1; i < my_steps; ++i) {
        if (__builtin_expect(out_of_range, 0)) settle((i - 1) & 1);  // (out of the loop's way: 1406 ns a step otherwise, 1388 so)
        iter.template operator()<false>(i, (i >= int_lo && i < c_hi) || (i >= b_lo && i < b_hi));
      }
      if (out_of_range) settle((my_steps - 1) & 1);
      out_of_range = false;
    } else {
      clear();
      if (lane < 2) *reinterpret_cast<int*>(lds + kPBase + lane * kPBuf + wave * kPWave + kFlagAt) = 0;  // its P never asks for a reference
    }
    // ---- what is left: P V of the group's last step, and its share of the staging of those that the other group goes on with. (Its own
    // flags stay clear from here on: a settled step's are, and the other buffer's it clears itself.)
    bool left = my_steps > 0;
    for (int i = my_steps;; ++i) {
      const int S = i & 1;
      if (out_of_range) settle_beside();
      if (i < n_steps) {
        if (i > 0) {
          load_v.template operator()<2>(S);
          load_v.template operator()<3>(S);
        }
        locate(i + 1);
        load_k_all(S ^ 1);
      }
      if (left) {
        left = false;
        const uint32_t va = vaddr + uint32_t((S ^ 1) * kVStage), pa = paddr + uint32_t((S ^ 1) * kPBuf);
#pragma unroll
        for (int rt = 0; rt < 2; ++rt) {
          l_run[rt] += ps[rt];
          l_run[rt] += __shfl_xor(l_run[rt], 32);
          if (hb == 0) l_sh(wave)[32 * rt + l32] = l_run[rt];
        }
        if (lane == 0) l_sh(wave)[kFlagAt / 4] = 0.0f;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
#pragma unroll
          for (int nt = 0; nt < 4; ++nt) ring[0][nt] = v_operand(va, t, nt);
#pragma unroll
          for (int rt = 0; rt < 2; ++rt) pf[0][rt] = p_operand(pa, t, rt);
          if (both) {
#pragma unroll
            for (int n = 0; n < 8; n += 2) mul_v1(ring[0], pf[0], n);
          }
#pragma unroll
          for (int n = 1; n < 8; n += 2) mul_v1(ring[0], pf[0], n);
        }
      }
      if (i >= n_steps) break;
      if (i == 0) __syncthreads();  // (the maxima of the first step)
      asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
      if (cut_src) {
        load_cut(S ^ 1);
        wait_loads();
      }
      fix(i, S);
      __syncthreads();
      out_of_range = __any(flags_of(S) < 0) != 0;
      load_v.template operator()<0>(S ^ 1);
      load_v.template operator()<1>(S ^ 1);
    }
  } else {
    clear();
  }
  wait_loads();  // nothing is on its way to LDS any more (step 0 left before it was known whether there is one)

  __syncthreads();  // every wavefront is through with the stages and with P
  float l[2] = {0.0f, 0.0f};
  if (my_steps > 0) {
#pragma unroll
    for (int rt = 0; rt < 2; ++rt) {
      const float other = l_sh(wave ^ 1)[32 * rt + l32];
      l[rt] = half ? other + l_run[rt] : l_run[rt] + other;
    }
  }

  // ---- output: lane (row l32, half hb) holds dims dw + 32 nt + 8 i + 4 hb + j at acc[rt][nt][4 i + j]. A wavefront's rows go through
  // its quarter of the stages, which all four have read, so that neighbouring lanes store one row's bytes.
  // The lane's number anew: addresses made from it before the loop would be carried through it.
  int ln;
  asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(ln));
  const int r32 = ln & 31, hq = ln >> 5;
  char* ob = lds + wave * kKStage;
  const bool direct = tile.part >= 0 && (packed || rows_live <= 96);
#pragma unroll
  for (int rt = 0; rt < 2; ++rt) {
    if (64 * rg + 32 * rt >= places) break;
    const int place = 64 * rg + 32 * rt + r32;
    const int mm = packed ? place / a.G : place, hh = packed ? place - mm * a.G : hg;
    const bool ok = place < places;
    if (tile.part >= 0) {
      const size_t rec = (size_t(tile.part) * a.Hkv + kvh) * a.cols + size_t(mm) * a.G + hh;
      float* po = a.parts_o + rec * kHD + dw;
      if (ok) {
#pragma unroll
        for (int i = 0; i < NT * 4; ++i) {
          const f32x4 v = {acc[rt][i / 4][4 * (i % 4)], acc[rt][i / 4][4 * (i % 4) + 1], acc[rt][i / 4][4 * (i % 4) + 2], acc[rt][i / 4][4 * (i % 4) + 3]};
          if (direct) *reinterpret_cast<f32x4*>(po + 8 * i + 4 * hq) = v;
          else *reinterpret_cast<f32x4*>(RowsOut<4 * kHW>::at(ob + rt * 16384, r32, 2 * i + hq)) = v;
        }
        if (hq == 0 && half == 0) {
          a.parts_ml[rec * 2] = m_run[rt] == kUnset && !(l[rt] > 0.0f) ? -INFINITY : m_run[rt];  // no key seen: the merge passes the part over
          a.parts_ml[rec * 2 + 1] = l[rt];
        }
      }
      if (!direct) RowsOut<4 * kHW>::store(ob + rt * 16384, ok ? reinterpret_cast<uint64_t>(po) : 0, ln);
    } else {
      const int row = tile.r0 + mm, h = kvh * a.G + hh;
      if (ok)
        finish_output<DT>(a, acc[rt], l[rt] > 0.0f ? 1.0f / l[rt] : 0.0f, row, h, dw, hq, [&](int i, u32x2 v) __attribute__((always_inline)) {
          *reinterpret_cast<u32x2*>(RowsOut<2 * kHW>::at(ob + rt * 16384, r32, i) + 8 * hq) = v;
        });
      if (packed) {
        RowsOut<2 * kHW>::store(ob + rt * 16384, ok ? reinterpret_cast<uint64_t>(a.O + size_t(row) * a.q_ld + size_t(h) * kHD + dw) : 0, ln);
      } else {
        RowsOut<2 * kHW>::store_even(ob + rt * 16384, a.O + size_t(tile.r0 + 64 * rg + 32 * rt) * a.q_ld + size_t(kvh * a.G + hg) * kHD + dw,
                                     uint32_t(a.q_ld) * 2, places - (64 * rg + 32 * rt), ln);
      }
    }
  }
}

// The dynamic LDS limit of both variants on the current device, ahead of the first launch.
hipError_t tiled256_init_attributes() {
  const hipError_t e = allow_dynamic_lds<attn_tiled256_kernel<ESP_F16>>(kLds);
  return e != hipSuccess ? e : allow_dynamic_lds<attn_tiled256_kernel<ESP_BF16>>(kLds);
}

hipError_t launch_tiled256(int dt, const KArgs& a, int n_tiles, hipStream_t st) {
  constexpr auto kf = attn_tiled256_kernel<ESP_F16>;
  constexpr auto kb = attn_tiled256_kernel<ESP_BF16>;
  const hipError_t e = dt == ESP_F16 ? allow_dynamic_lds<kf>(kLds) : allow_dynamic_lds<kb>(kLds);
  if (e != hipSuccess) return e;
  launch_timed(dt == ESP_F16 ? kf : kb, dim3(unsigned(n_tiles) * a.H), dim3(256), size_t(kLds), st, a, n_tiles);
  return hipGetLastError();
}

}  // namespace esp
