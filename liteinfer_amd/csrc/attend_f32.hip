// Paged attention over fp32 pools on the fp32 matrix cores (head_dim 64 or
// 128, any grouping): decode partitions and packed query blocks, the same
// attention as the general-shape kernel (attend_generic.hip; the reference's
// Triton body, liteinfer/models/paged_kernels.py:216-371) with every product
// and sum in fp32. fp32 pools keep their 1e-5 parity bar, so nothing here is
// rounded to 16 bits.
//
// v_mfma_f32_16x16x4_f32: A is 16 x 4, B 4 x 16, one value per lane: lane
// (n, g) = (lane % 16, lane / 16) holds row (column) n, contraction index g.
// The result gives lane (n, g) column n, rows 4g .. 4g + 3.
//
//   S^T = K Q^T     A = K, B = Q^T, 16 keys x 16 (query, head) rows. The order
//                   of the contraction is free, so step (j, e) takes dim
//                   16 j + 4 g + e: a lane's operands of four steps are one
//                   16-byte load of its key's row. Lane (n, g) gets the
//                   scores of keys 4g .. 4g + 3 for row n.
//   O^T += V^T P^T  step r multiplies keys 4g + r: the lane's own weight r is
//                   its B operand, no lane exchange. A = V^T: block (h, e)
//                   is dims 64 h + 4 m + e, m = 0 .. 15, so a lane's operands
//                   of four blocks are one 16-byte load of key 4g + r's row.
//                   Lane (n, g) ends with dims 64 h + 16 g .. + 15 of row n.
//
// A tile's K goes straight into a wave's own LDS stage and its V into
// registers, the next tile's loads in flight while a tile is folded (16 keys
// of 16 rows take D / 64 * 1024 cycles of one SIMD's matrix core for D / 64 *
// 8 KiB of loads). The matrix cores are the bound of packed passes (157
// TFLOP/s in fp32), HBM of decode. Tiles shared by the waves of a work-group
// would save L2 reads, which are not the bound, and cost its barriers.
//
// A work-group is four waves on one (sequence, KV head, block of 16 rows,
// key range): the waves split the block's 16-key tiles (interleaved, so that
// a causal block's work is even) and merge their softmax states in LDS, as
// the reference's cross-partition reduce does (paged_kernels.py:574-629).
//
// Measured (MI355X), three chunks of 281 .. 336 queries over 300 .. 1,100
// cached keys beside five one-query rows, 32 / 8 heads, head_dim 64 (7.1
// GFLOP, 51 us at the rate of a large fp32 GEMM): 94 us, against 35.5 ms on
// the general-shape kernel. What is left is a unit's start and end (its
// descriptor, query and slots, the masked tile, the merge: as long as eight
// of its ~20 tiles a wave), the last units' imbalance, and the key loop's
// mid-step wait for the next tile's K.
#include "li_attention.h"
#include "li_mfma.h"

#include <type_traits>

namespace li {
namespace {

constexpr int kF32Waves = 4;
// (query, head) rows of a block: a 50-query chunk over 1,200 keys takes 22
// us, against 37 / 68 us in blocks of 32 / 64 rows whose row groups share the
// waves, and passes that fill the GPU the same within 3% (64 rows 10% more).
constexpr int kF32Rows = 16;

// The loads of one 16-key tile. Lane (n, g) brings keys 4g + i, i < 4 (their
// slots in `slot`), 16 lanes side by side on a row, so that an instruction
// reads whole 256-byte runs.
//
// K goes into LDS: its operands are one lane per key, and loaded that way
// every lane of an instruction would read another row. A stage is D / 64
// planes of 16 rows x 64 dims; instruction (h, i) fills rows 4i + g of plane
// h, 16-byte chunk c of key k at c ^ k, so that the 16 keys of one operand
// read lie in 16 different bank groups.
constexpr int kPlaneBytes = 16 * 256;

template <int D>
__device__ __forceinline__ void issue_k_f32(uint32_t stage, const char* kpool, const int (&slot)[4],
                                            uint32_t row_bytes, int n, int g) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const char* row = row_ptr(kpool + 16 * (n ^ (4 * g + i)), (uint32_t)slot[i], row_bytes);
#pragma unroll
    for (int h = 0; h < D / 64; ++h) dma16(row + 256 * h, stage + h * kPlaneBytes + 1024 * i);
  }
}

// V into registers, as the lane's operands of four output blocks are 16
// bytes of one row (dims 64 h + 4 n ..).
template <int D>
__device__ __forceinline__ void load_v_f32(u32x4_t (&v)[4][D / 64], const char* vpool, const int (&slot)[4],
                                           uint32_t row_bytes, int n) {
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const char* vrow = vpool + (uint64_t)(uint32_t)slot[r] * row_bytes + 16 * n;
#pragma unroll
    for (int h = 0; h < D / 64; ++h) v[r][h] = *reinterpret_cast<const u32x4_t*>(vrow + 256 * h);
  }
}

// V rows stay integers up to the matrix cores: the sources build with
// -fno-honor-nans, under which a test of a float's bits may lose its NaNs.
__device__ __forceinline__ bool not_finite(uint32_t bits) { return (bits & 0x7f800000u) == 0x7f800000u; }

template <int D>
__global__ __launch_bounds__(64 * kF32Waves) __attribute__((amdgpu_waves_per_eu(2))) void attend_f32(
    AttnArgs a) {
  constexpr int kJ = D / 16, kH = D / 64;
  // The waves' K stages (two each), then their states for the merge.
  constexpr int kStage = kH * kPlaneBytes;
  __shared__ __attribute__((aligned(1024))) union {
    char k[kF32Waves][2][kStage];
    float acc[kF32Waves][16][D + 4];  // rows 16 bytes past a multiple of the banks
  } lds;
  __shared__ float s_m[kF32Waves][16], s_l[kF32Waves][16];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int n = lane & 15, g = lane >> 4;

  // Units (KV head fastest, so that at 8 heads one XCD's L2 serves a head):
  // a decode step's are (sequence, partition, block), one a work-group. A
  // packed pass's are the blocks its sequences really have, found from the
  // query counts, the last block of a sequence (most keys) first; a grid of
  // about twice what the GPU holds walks them. (A grid sized by the longest
  // chunk is mostly empty beside short ones, and an empty work-group costs
  // its launch: 27 us for 2,990 of them beside three 300-query chunks.)
  const int kvh = (int)(blockIdx.x % (unsigned)a.num_kv_heads);
  // The first 64 sequences' query rows and blocks, kept for every unit.
  auto info_of = [&](int sq, int& first, int& count) -> int {  // returns the sequence's blocks
    first = count = 0;
    if (sq >= a.batch) return 0;
    first = a.qsl[sq];
    count = a.qsl[sq + 1] - first;
    return count > 0 ? (int)(((int64_t)count * a.groups + kF32Rows - 1) / kF32Rows) : 0;
  };
  int first0 = 0, count0 = 0;
  const int blocks0 = a.qsl ? info_of(lane, first0, count0) : 0;
  for (unsigned at = blockIdx.x / (unsigned)a.num_kv_heads;; at += gridDim.x / (unsigned)a.num_kv_heads) {
  int seq, part = 0, block, first_tok, nq = 1;
  if (!a.qsl) {
    if (at >= (unsigned)(a.batch * a.num_parts * a.num_qblocks)) break;
    seq = first_tok = (int)(at % (unsigned)a.batch);
    part = (int)(at / (unsigned)a.batch % (unsigned)a.num_parts);
    block = (int)(at / (unsigned)a.batch / (unsigned)a.num_parts);
  } else {
    int before = 0, s0 = 0;
    uint64_t hit = 0;
    int first = first0, count = count0, nb = blocks0, incl = 0;
    for (;;) {
      incl = nb;
#pragma unroll
      for (int off = 1; off < 64; off <<= 1) {
        const int up = __shfl_up(incl, off, 64);
        if (lane >= off) incl += up;
      }
      hit = __ballot(before + incl > (int)at);
      if (hit) break;
      before += __shfl(incl, 63, 64);
      if ((s0 += 64) >= a.batch) break;
      nb = info_of(s0 + lane, first, count);
    }
    if (!hit) break;
    const int src = __ffsll((long long)hit) - 1;
    seq = s0 + src;
    first_tok = __builtin_amdgcn_readfirstlane(__shfl(first, src, 64));
    nq = __builtin_amdgcn_readfirstlane(__shfl(count, src, 64));
    block = __builtin_amdgcn_readfirstlane(before + __shfl(incl, src, 64) - 1 - (int)at);
  }
  const int ctx = a.ctx[seq];
  // Rows of the sequence are (query, head) pairs, head fastest; this block's
  // are [row0, row1).
  const int G = a.groups;
  const int64_t rows = (int64_t)nq * G;
  const int64_t row0 = (int64_t)block * kF32Rows;
  const int nrows = (int)min((int64_t)kF32Rows, rows - row0);

  int kb = 0, ke = ctx, nparts = 1;
  if (a.part_o) {
    const int plen = a.part_len > 0 ? a.part_len : max(1, (ctx + a.num_parts - 1) / a.num_parts);
    kb = part * plen;
    if (kb >= max(ctx, 1)) continue;  // (an empty context: partition 0 writes 0 / 0)
    ke = min(kb + plen, ctx);
    nparts = (ctx + plen - 1) / plen;
  }
  const int pos0 = ctx - nq;  // position of the sequence's first query
  // Keys any row of the block sees end at the last row's own position.
  ke = min(ke, pos0 + (int)((row0 + nrows - 1) / G) + 1);

  const int64_t row = row0 + n;
  const bool real = n < nrows;
  const int ql = (int)((real ? row : row0) / G), head = kvh * G + (int)((real ? row : row0) % G);
  const int lim = pos0 + ql;               // last key the row sees
  const int lim_lo = pos0 + (int)(row0 / G);  // the first row sees the fewest keys

  // The row's query, the softmax scale times log2(e) folded in: scores are in
  // log2 units.
  const float sc = a.scale * kLog2eMfma;
  floatx4_t q[kJ];
  {
    const float* qrow = static_cast<const float*>(a.q) + (int64_t)(first_tok + ql) * a.q_s0 + (int64_t)head * a.q_s1;
#pragma unroll
    for (int j = 0; j < kJ; ++j) {
      q[j] = *reinterpret_cast<const floatx4_t*>(qrow + 16 * j + 4 * g);
#pragma unroll
      for (int e = 0; e < 4; ++e) q[j][e] = real ? q[j][e] * sc : 0.f;
    }
  }
  const char* kpool = reinterpret_cast<const char*>(static_cast<const float*>(a.kp) + (int64_t)kvh * a.p_s1);
  const char* vpool = reinterpret_cast<const char*>(static_cast<const float*>(a.vp) + (int64_t)kvh * a.p_s1);
  const uint32_t row_bytes = (uint32_t)(a.p_s0 * (int64_t)sizeof(float));
  const int64_t* srow = a.st + (int64_t)seq * a.st_s;

  float m = -INFINITY, l = 0.f;  // running maximum (log2 units); this lane's part of the denominator
  floatx4_t acc[kH][4];          // block (h, e), result rows 4g + r: dim 64 h + 16 g + 4 r + e
#pragma unroll
  for (int h = 0; h < kH; ++h)
#pragma unroll
    for (int e = 0; e < 4; ++e) acc[h][e] = floatx4_t{0.f, 0.f, 0.f, 0.f};

  // This lane's K operands in a stage: key n's chunk 4 (j % 4) + g of plane j / 4.
  uint32_t koff[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) koff[j] = (uint32_t)(256 * (4 * (n & 3) + (n >> 2)) + 16 * ((4 * j + g) ^ n));
  const uint32_t stage0 = lds_addr(lds.k[w][0]), stage1 = stage0 + kStage;

  // One tile: with kMasked, some of its keys lie past some row's last one.
  auto fold = [&](auto masked_tag, uint32_t kst, const u32x4_t (&v)[4][kH], int slot, int t0)
      __attribute__((always_inline)) {
    constexpr bool kMasked = decltype(masked_tag)::value;
    floatx4_t k[kJ];
#pragma unroll
    for (int j = 0; j < kJ; ++j) k[j] = lds_read_frag<floatx4_t>(kst + koff[j % 4] + (j / 4) * kPlaneBytes);
    floatx4_t s0 = {0.f, 0.f, 0.f, 0.f}, s1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < kJ; j += 2)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        s0 = __builtin_amdgcn_mfma_f32_16x16x4f32(k[j][e], q[j][e], s0, 0, 0, 0);
        s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(k[j + 1][e], q[j + 1][e], s1, 0, 0, 0);
      }
    float x[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) x[r] = s0[r] + s1[r];
    if constexpr (kMasked) {
#pragma unroll
      for (int r = 0; r < 4; ++r) x[r] = (t0 + 4 * g + r <= lim && t0 + 4 * g + r < ke) ? x[r] : -INFINITY;
    }
    const float mx = li_group_max(fmaxf(fmaxf(x[0], x[1]), fmaxf(x[2], x[3])));
    const float mnew = fmaxf(m, mx);
    // A row that has seen no key yet keeps m = -inf and zero weights.
    const float base = mnew == -INFINITY ? 0.f : mnew;
    if (__any(mnew != m)) {
      const float alpha = __builtin_amdgcn_exp2f(m - base);
      l *= alpha;
#pragma unroll
      for (int h = 0; h < kH; ++h)
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[h][e][r] *= alpha;
      m = mnew;
    }
    float p[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) p[r] = __builtin_amdgcn_exp2f(x[r] - base);
    l += (p[0] + p[1]) + (p[2] + p[3]);
    if constexpr (kMasked) {
      // V rows some row of the group does not see: a zero weight times an
      // infinity or a NaN would reach that row's sum, so a tile that holds
      // one is folded row by row with those keys left out.
      bool odd = false;
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int h = 0; h < kH; ++h)
#pragma unroll
          for (int e = 0; e < 4; ++e) odd |= not_finite(v[r][h][e]);
      if (__any(odd)) {
#pragma unroll 1
        for (int g2 = 0; g2 < 4; ++g2) {
#pragma unroll
          for (int r2 = 0; r2 < 4; ++r2) {
            const int key = t0 + 4 * g2 + r2;
            const float pk = __shfl(p[r2], n + 16 * g2, 64);
            const uint32_t sees = key <= lim && key < ke ? 0xffffffffu : 0u;
            const float* vrow = reinterpret_cast<const float*>(
                vpool + (uint64_t)(uint32_t)__shfl(slot, 4 * g2 + r2, 64) * row_bytes);
#pragma unroll
            for (int h = 0; h < kH; ++h)
#pragma unroll
              for (int r = 0; r < 4; ++r) {
                const u32x4_t vv = *reinterpret_cast<const u32x4_t*>(vrow + 64 * h + 16 * g + 4 * r);
#pragma unroll
                for (int e = 0; e < 4; ++e)
                  acc[h][e][r] = fmaf(pk, __uint_as_float(vv[e] & sees), acc[h][e][r]);
              }
          }
        }
        return;
      }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int h = 0; h < kH; ++h)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          acc[h][e] = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(v[r][h][e]), p[r], acc[h][e], 0, 0, 0);
  };

  // This wave's tiles: kb + 16 (w + 4 i). The first `clear` tiles of the
  // range are seen whole by every row; they run with slots two tiles ahead
  // of the fold and rows one. Look-ahead past the range reads the last key's
  // slot, a real row. (As compiled it reaches less far: `slot_of` narrows its
  // load at once, and the wait for that, which the compiler places in
  // mid-step, is also one for the next tile's K.)
  const int ntiles = ke > kb ? (ke - kb + 15) / 16 : 0;
  const int clear = max(0, min(lim_lo + 1, ke) - kb) / 16;
  auto slot_of = [&](int tile) -> int { return (int)srow[min(kb + 16 * tile + n, ke - 1)]; };
  // The V rows a lane loads of a tile: keys 4g + r.
  auto spread = [&](int slot, int (&vs)[4]) {
#pragma unroll
    for (int r = 0; r < 4; ++r) vs[r] = __shfl(slot, 4 * g + r, 64);
  };
  int tile = w;
  if (tile < clear) {
    u32x4_t va[4][kH], vn[4][kH];
    int sa = slot_of(tile), sb = slot_of(tile + kF32Waves), vs[4];
    spread(sa, vs);
    issue_k_f32<D>(stage0, kpool, vs, row_bytes, n, g);
    load_v_f32<D>(va, vpool, vs, row_bytes, n);
    __builtin_amdgcn_sched_barrier(0);
    auto step = [&](uint32_t kst, const u32x4_t (&v)[4][kH], uint32_t knext, u32x4_t (&vnext)[4][kH], int& s0, int s1)
        __attribute__((always_inline)) {
      const int s2 = slot_of(tile + 2 * kF32Waves);
      spread(s1, vs);
      issue_k_f32<D>(knext, kpool, vs, row_bytes, n, g);
      load_v_f32<D>(vnext, vpool, vs, row_bytes, n);
      // Newer than the tile's K: its V (4 kH loads), this step's slot, K and
      // V (1 + 8 kH). With 8 kH + 1 in flight its K has landed, and needs no
      // more of this step's loads for that than K's (assembly, never dropped)
      // and one other: a step whose look-ahead nobody reads may not use this
      // count, since the compiler drops such loads.
      li_wait_vm<8 * kH + 1>();
      // (Left to itself the scheduler sinks the loads between the MFMAs.)
      __builtin_amdgcn_sched_barrier(0);
      fold(std::false_type{}, kst, v, s0, kb + 16 * tile);
      // The stage's reads are done before the next step's loads fill it.
      __builtin_amdgcn_sched_barrier(0);
      s0 = s2;
      tile += kF32Waves;
    };
    // (Two tiles an iteration and no way out between them: with one, the
    // compiler waits for every load at the loop's head.)
    while (tile + kF32Waves < clear) {
      step(stage0, va, stage1, vn, sa, sb);
      step(stage1, vn, stage0, va, sb, sa);
    }
    // The odd tile has nothing to look ahead to.
    li_wait_vm<0>();
    __builtin_amdgcn_sched_barrier(0);
    if (tile < clear) {
      fold(std::false_type{}, stage0, va, sa, kb + 16 * tile);
      __builtin_amdgcn_sched_barrier(0);
      tile += kF32Waves;
    }
  }
  for (; tile < ntiles; tile += kF32Waves) {
    u32x4_t v[4][kH];
    const int slot = slot_of(tile);
    int vs[4];
    spread(slot, vs);
    issue_k_f32<D>(stage0, kpool, vs, row_bytes, n, g);
    load_v_f32<D>(v, vpool, vs, row_bytes, n);
    li_wait_vm<0>();
    fold(std::true_type{}, stage0, v, slot, kb + 16 * tile);
    __builtin_amdgcn_sched_barrier(0);
  }

  // The waves' states, merged through LDS.
  const float lt = li_group_sum(l);
  __syncthreads();  // every wave is done with its stages
#pragma unroll
  for (int h = 0; h < kH; ++h)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      *reinterpret_cast<floatx4_t*>(&lds.acc[w][n][64 * h + 16 * g + 4 * r]) =
          floatx4_t{acc[h][0][r], acc[h][1][r], acc[h][2][r], acc[h][3][r]};
  if (g == 0) {
    s_m[w][n] = m;
    s_l[w][n] = lt;
  }
  __syncthreads();
  constexpr int kCh = D / 4;
  for (int i = threadIdx.x; i < nrows * kCh; i += 64 * kF32Waves) {
    const int rr = i / kCh, c = i % kCh;
    float mx = -INFINITY;
#pragma unroll
    for (int v = 0; v < kF32Waves; ++v) mx = fmaxf(mx, s_m[v][rr]);
    // A wave that met none of the row's keys holds m = -inf and zero sums. So
    // does one whose scores were all NaN, but for its sums: every wave's are
    // added, whatever its m, so that a NaN reaches the row.
    const float base = mx == -INFINITY ? 0.f : mx;
    floatx4_t num = {0.f, 0.f, 0.f, 0.f};
    float den = 0.f;
#pragma unroll
    for (int v = 0; v < kF32Waves; ++v) {
      const float wgt = __builtin_amdgcn_exp2f(s_m[v][rr] - base);
      den = fmaf(wgt, s_l[v][rr], den);
      const floatx4_t x = *reinterpret_cast<const floatx4_t*>(&lds.acc[v][rr][4 * c]);
#pragma unroll
      for (int e = 0; e < 4; ++e) num[e] = fmaf(wgt, x[e], num[e]);
    }
    const float inv = 1.f / den;
    floatx4_t o;
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = num[e] * inv;
    const int64_t orow = row0 + rr;
    const int ohead = kvh * G + (int)(orow % G);
    if (den == 0.f) {  // no key to attend to: the reference's softmax over nothing is 0 / 0
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = li_quiet_nan<float>();
    }
    if (nparts > 1) {
      const int64_t pr = ((int64_t)seq * a.num_heads + ohead) * a.num_parts + part;
      *reinterpret_cast<floatx4_t*>(a.part_o + pr * D + 4 * c) = o;
      if (c == 0) a.part_lse[pr] = mx + log2f(den);
    } else {
      *reinterpret_cast<floatx4_t*>(static_cast<float*>(a.out) + (first_tok + orow / G) * a.o_s0 +
                                    (int64_t)ohead * a.o_s1 + 4 * c) = o;
    }
  }
  if (!a.qsl) break;  // a decode step's grid has a work-group for every unit
  __syncthreads();    // the states are read before the next unit's stages overwrite them
  }  // units
}

bool rows_aligned(const void* p, int64_t s0, int64_t s1) {
  return aligned16(p) && s0 % 4 == 0 && s1 % 4 == 0;
}

}  // namespace

bool attend_f32_applies(const AttnArgs& a, int dtype) {
  // A decode step has a work-group for every unit, and a launch fewer than
  // 2^32 threads: past that the general kernel's smaller work-groups still fit.
  // (A packed pass's grid is capped.)
  const int64_t units = (int64_t)a.batch * a.num_parts * a.num_kv_heads * cdiv(a.groups, kF32Rows);
  if (!a.qsl && units >= (1LL << 32) / (64 * kF32Waves)) return false;
  return dtype == LI_F32 && !a.kv_fp8 && (a.head_dim == 64 || a.head_dim == 128) && rows_aligned(a.q, a.q_s0, a.q_s1) &&
         rows_aligned(a.out, a.o_s0, a.o_s1) && rows_aligned(a.kp, a.p_s0, a.p_s1) &&
         rows_aligned(a.vp, a.p_s0, a.p_s1) && a.p_s0 >= 0 && a.p_s0 < (1LL << 30);
}

int launch_attend_f32(AttnArgs a, hipStream_t s) {
  a.num_qblocks = (int)std::min<int64_t>(cdiv64((int64_t)std::max(a.max_query_len, 1) * a.groups, kF32Rows), 0x7fffffff);
  const int64_t most = (int64_t)a.batch * a.num_qblocks * a.num_parts;
  if (most == 0) return LI_OK;
  int64_t per_head = most;
  if (a.qsl) {
    // About twice what the CUs hold at once (two or three each): the first
    // round is then dealt by the hardware as work-groups end (against just
    // what they hold: 106 -> 98 us, at head_dim 128 234 -> 221 us; twice
    // this again: 109 and 220 us).
    per_head = std::min<int64_t>(most, cdiv(device_cu_count() * 6, a.num_kv_heads));
  }
  const dim3 grid((unsigned)(per_head * a.num_kv_heads)), block(64 * kF32Waves);
  if (a.head_dim == 128) hipLaunchKernelGGL(attend_f32<128>, grid, block, 0, s, a);
  else hipLaunchKernelGGL(attend_f32<64>, grid, block, 0, s, a);
  return check_launch("attend_f32");
}

}  // namespace li
