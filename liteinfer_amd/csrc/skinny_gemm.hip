// out = x W^T for the rows of a decode step's batch: the engine's
// projections, q/k/v, output, gate/up with the SiLU gate, down and head
// (liteinfer/models/llama.py:101-161, nn.Linear in the reference).
//
// At a decode step's batch a projection reads its weights once and does
// little else, so its bound is HBM: x is a few hundred KB and stays in L2.
// A work-group of NW waves takes a tile of 16 NW weight rows (N) and a run
// of K, all BM rows of x beside it. Both operands go straight into LDS
// (global_load_lds_dwordx4) in a ring of stages of 128 k: rows of 256 bytes,
// 16-byte chunk c of row r at c ^ (r % 16), so that the 16 rows an operand
// read spans lie in 16 different bank groups. R - 1 stages are in flight, one
// barrier a stage; up to 32 rows two work-groups of four waves share a CU
// (96 .. 120 KiB in flight on it; 27 GB/s a CU times ~2 us of loaded latency
// needs ~54), past that one of eight. Wave w owns weight rows 16 w .. + 15:
//   D (16 n x 16 m) += A = W rows (16 n x 32 k), B = x^T (32 k x 16 m)
// and lane (m, g) = (lane % 16, lane / 16) ends with outputs n = 4g .. 4g + 3
// of row m. Sums are fp32, rounded once.
//
// Few tiles are cut along K into `splits` runs so that the grid fills the GPU;
// each run then writes its fp32 sums and the op that follows (add_rms_norm,
// silu_mul or skinny_reduce) adds them before it rounds.
//
// Where a work-group starts its run of K matters: rows of a power-of-two
// stride read at one k at a time by every work-group of an XCD meet on a few
// HBM channels. The stages are taken in a rotated order, five further for
// each work-group an XCD holds (gate/up of the 8B architecture, one row: 44.8
// us unrotated, 36.9 rotated, 39 .. 42 rotated by the tile itself).
//
// Measured (MI355X, graph replay over weights larger than the caches), rows 1
// and 32, us (TB/s of weights at one row), against hipBLASLt's:
//   6144 x 4096    10.1 (5.0)  11.3      14.5  15.3
//   4096 x 4096     7.6 (4.4)   8.5      15.4  13.1
//   28672 x 4096   39.0 (6.0)  40.7      66.3  57.8   (the gate included)
//   4096 x 14336   20.5 (5.7)  22.4      27.2  31.5
//   16032 x 4096   22.3 (5.9)  23.7      29.4  27.5
//   2048 x 2048     3.6 (2.3)   4.8      11.0  11.2
// The small ones are a launch and one loaded latency.
#include "li_mfma.h"

namespace {

using namespace li;

constexpr int kStageK = 128;
constexpr int kRotate = 5;
constexpr int kRowBytes = kStageK * 2;

struct GemmArgs {
  const char* x;
  const char* w;
  char* out;       // T rows (splits == 1)
  float* part;     // [splits][m][n] fp32 (splits > 1)
  int64_t x_s, w_s, o_s;  // row strides in bytes (x, w), in elements (out)
  int m, n, k;
  int splits;
  int gate;  // W holds [gate | up] rows, n / 2 each; out = silu(gate) * up, n / 2 wide
};

// Rows of x up to which skinny_gemm runs its small work-groups, and up to
// which it runs at all (batch_gemm past them).
constexpr int kFewRows = 32, kSkinnyRows = 64;

// How a projection is cut: weight rows of a tile, runs of K (0: it is left to
// the caller's own GEMM).
struct Cut {
  int tile, splits;
};

// Up to 64 rows the projections of the 8B and 1B architectures measured faster
// here than through hipBLASLt (1.0 .. 3.0 times; what does not: uneven_rounds,
// and the sums of 33 .. 64 rows that nothing adds, `linear` in engine/ops.py).
// K is cut into
// as many runs as fill the GPU once, of at least two stages (of one, the sums
// cost the norm more than the run saves: a step of 4 layers of the 1B
// architecture at 24 rows 322 -> 312 us); not at all where
// the tiles alone are three quarters of a work-group a CU or more (what a
// second run gains is less than adding the sums costs: 16,032 x 4,096 at 8
// rows 21.5 us whole, 26.9 in two).
//
// Past 64 rows a work-group reads x as often as its weights, and the runs'
// sums cost more than they did; what stays faster (us, this against
// hipBLASLt's, the norm that adds the sums included):
//   whole tiles at up to 128 rows, where uneven_rounds allows: 28672 x 4096
//     with its gate 53 / 58 at 128 rows (74 / 61 at 160), 32064 x 2048 30 /
//     34, 128256 x 4096 217 / 233;
//   runs of K no shorter than 768 of a weight no wider than twice its K:
//     4096 x 14336 40 / 79 at 128 rows and 49 / 66 at 256, 6144 x 4096 24 / 25
//     and 30 / 40 (4096 x 4096, runs of 512: 24 / 29 and 28 / 27; 3072 x 2048,
//     runs of 205: 17 / 14; 16032 x 4096, twice as wide: 38 / 35);
//   the same in tiles of 64 rows up to 192 rows, half as many runs: 4096 x
//     4096 22 / 28 at 128 rows, 26 / 31 at 160 (30 / 27 at 256), 2048 x 8192
//     20 / 24 and 25 / 29.
constexpr int kMinRun = 768;

Cut cut_of(int m, int n, int k) {
  const int cus = li::device_cu_count(), stages = k / kStageK;
  auto tiles = [&](int tile) { return (n + tile - 1) / tile; };
  auto runs = [&](int tile, int per_cu) {
    const int t = tiles(tile);
    return t * 4 >= cus * 3 ? 1 : std::max(1, std::min(cus * per_cu / t, stages / 2));
  };
  if (m <= kFewRows) return {64, runs(64, 2)};  // (two work-groups a CU)
  if (m <= kSkinnyRows) return {128, runs(128, 1)};
  if (tiles(128) * 4 >= cus * 3) return {128, m <= 128 ? 1 : 0};
  if (n <= 2 * (int64_t)k) {
    if (k / runs(128, 1) >= kMinRun) return {128, runs(128, 1)};
    if (m <= 192 && k / runs(64, 1) >= kMinRun) return {64, runs(64, 1)};
  }
  return {0, 0};
}

// Past 32 rows a wide weight's 128-row tiles take a CU each, round by round,
// and a last round that is nearly empty costs a whole one: hipBLASLt, whose
// tiles follow the shape, is then the faster one, so the plan leaves those
// to it. The lines, us here / hipBLASLt's (rounds of 256 tiles):
//   65 .. 128 rows, K under 4096, up to two rounds: 33024 x 1024 (1.01) 31 /
//     21, 40960 x 2048 (1.25) 50 / 44, 49152 x 3584 (1.5) 87 / 77, 61440 x
//     2048 (1.9) 58 / 54; from two on 65536 x 2048 61 / 72, 128256 x 2048 123
//     / 123;
//   65 .. 128 rows, longer K, up to one and a half: 33024 x 4096 87 / 69,
//     40960 x 4096 89 / 80; from there 49152 x 4096 92 / 101, 128256 x 4096
//     217 / 233;
//   33 .. 64 rows, up to one and a half: 40960 x 1024 23 / 21, 33024 x 3584 63
//     / 56 (and 36864 x 4096 69 / 73); from there 57344 x 3584 74 / 77.
// What is left on the wrong side: 65536 x 3072 at 128 rows 89 / 84, 98304 x
// 1024 56 / 49. At 32 rows and fewer (64-row tiles, two a CU) every width was
// faster here. Under K of 512 both are mostly a launch, and whichever is
// ahead changes with the row count.
bool uneven_rounds(int m, int n, int k) {
  const int cus = li::device_cu_count(), t = (n + 127) / 128;
  if (m <= kFewRows || k < 512 || t <= cus) return false;
  return t < (m > kSkinnyRows && k < 4096 ? 2 * cus : cus * 3 / 2);
}

// Stores lane (m, g)'s four sums of a group of 16 outputs: 16 group + 4g ..
// of row m, or with kGate (rows 0-7 of the group: gate outputs 8 group ..,
// rows 8-15 the up outputs of the same) the gated outputs. Every lane of the
// wave takes part.
template <typename T, bool kGate>
__device__ __forceinline__ void store_outputs(const GemmArgs& a, const floatx4_t& acc, int split, int m, int group,
                                              int g) {
  if constexpr (kGate) {
    // Lanes 0-31 hold gate outputs 0-7, lanes 32-63 the up outputs.
    const int col = 8 * group + 4 * (g & 1);
    if (a.splits > 1) {
      if (m < a.m && col < a.n / 2)
        *reinterpret_cast<floatx4_t*>(a.part + ((int64_t)split * a.m + m) * a.n + (g < 2 ? 0 : a.n / 2) + col) = acc;
      return;
    }
    float o[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float up = __shfl_xor(acc[r], 32, 64);
      const float gf = li_to_float(li_from_float<T>(acc[r]));
      const float s = li_to_float(li_from_float<T>(gf / (1.f + expf(-gf))));
      o[r] = s * li_to_float(li_from_float<T>(up));
    }
    if (g < 2 && m < a.m && col < a.n / 2)
      *reinterpret_cast<uint2*>(a.out + (m * a.o_s + col) * 2) = uint2{li_pack2<T>(o[0], o[1]), li_pack2<T>(o[2], o[3])};
  } else {
    const int col = 16 * group + 4 * g;
    if (m >= a.m || col >= a.n) return;
    if (a.splits == 1)
      *reinterpret_cast<uint2*>(a.out + (m * a.o_s + col) * 2) = uint2{li_pack2<T>(acc[0], acc[1]), li_pack2<T>(acc[2], acc[3])};
    else
      *reinterpret_cast<floatx4_t*>(a.part + ((int64_t)split * a.m + m) * a.n + col) = acc;
  }
}

// BM: rows of x a work-group holds (m <= BM). R: ring stages.
template <typename T, int BM, int R, int NW, bool kGate>
__global__ __launch_bounds__(64 * NW) void skinny_gemm(GemmArgs a) {
  using M = Mfma<T>;
  using Frag = typename M::Frag;
  constexpr int kMt = BM / 16;
  constexpr int kTileN = 16 * NW;
  constexpr int kXPer = BM / 4 / NW;  // x loads of a wave per stage
  static_assert(kXPer >= 1 && kXPer * 4 * NW == BM, "the waves split x's loads evenly");
  constexpr int kPer = 4 + kXPer;
  constexpr int kStage = (kTileN + BM) * kRowBytes;
  static_assert(R == 3 || R == 4, "the waits below count up to two newer stages");
  static_assert((R - 2) * kPer < 64, "vmcnt range");
  __shared__ __attribute__((aligned(1024))) char ring[R][kStage];
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n16 = lane & 15, g = lane >> 4;
  const int tile = (int)(blockIdx.x / (unsigned)a.splits), split = (int)(blockIdx.x % (unsigned)a.splits);
  const int total = a.k / kStageK;
  const int s0 = (int)((int64_t)total * split / a.splits), s1 = (int)((int64_t)total * (split + 1) / a.splits);
  const int ns = s1 - s0;

  // This lane's chunk of the rows it loads: load i of the wave covers four
  // rows, 16 lanes side by side on each. (Rows past the last repeat it.)
  const char* wrow[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int t = 4 * i + g;  // row of the wave's 16
    int64_t row;
    if (kGate) {  // rows 0-7: gate, 8-15: the up rows of the same outputs
      const int col = min(tile * (kTileN / 2) + 8 * w + (t & 7), a.n / 2 - 1);
      row = (t < 8 ? 0 : a.n / 2) + col;
    } else {
      row = min(tile * kTileN + 16 * w + t, a.n - 1);
    }
    wrow[i] = a.w + row * a.w_s + (int64_t)s0 * kRowBytes + 16 * (n16 ^ t);
  }
  const char* xrow[kXPer];
  int xat[kXPer];
#pragma unroll
  for (int i = 0; i < kXPer; ++i) {
    const int p = w * kXPer + i;  // four-row group of x
    const int t = 4 * p + g;
    xrow[i] = a.x + (int64_t)min(t, a.m - 1) * a.x_s + (int64_t)s0 * kRowBytes + 16 * (n16 ^ (t & 15));
    xat[i] = kTileN * kRowBytes + 1024 * p;
  }
  const uint32_t base = lds_addr(&ring[0][0]);
  const unsigned rotated = (unsigned)(tile >> 3) * kRotate;
  auto issue = [&](int st) {
    const uint32_t dst = base + (uint32_t)(st % R) * kStage;
    const int64_t at = (int64_t)((rotated + (unsigned)st) % (unsigned)ns) * kRowBytes;
#pragma unroll
    for (int i = 0; i < 4; ++i) dma16<true>(wrow[i] + at, dst + 4096 * w + 1024 * i);
#pragma unroll
    for (int i = 0; i < kXPer; ++i) dma16<false>(xrow[i] + at, dst + xat[i]);
  };

  floatx4_t acc[kMt];
#pragma unroll
  for (int i = 0; i < kMt; ++i) acc[i] = floatx4_t{0.f, 0.f, 0.f, 0.f};
  uint32_t off[kStageK / 32];
#pragma unroll
  for (int j = 0; j < kStageK / 32; ++j) off[j] = (uint32_t)(n16 * kRowBytes + 16 * ((4 * j + g) ^ n16));

#pragma unroll
  for (int st = 0; st < R - 1; ++st)
    if (st < ns) issue(st);
  for (int st = 0; st < ns; ++st) {
    // Stage st has landed once only the stages issued after it are in flight.
    const int newer = min(R - 2, ns - 1 - st);
    if (newer == 2) li_wait_vm<(R > 3 ? 2 : 1) * kPer>();
    else if (newer == 1) li_wait_vm<kPer>();
    else li_wait_vm<0>();
    lds_barrier();  // every wave's part of it; and all are done with stage st - 1, whose place the next loads take
    if (st + R - 1 < ns) issue(st + R - 1);
    const uint32_t cur = base + (uint32_t)(st % R) * kStage;
#pragma unroll
    for (int j = 0; j < kStageK / 32; ++j) {
      const Frag wf = lds_read_frag<Frag>(cur + 4096 * w + off[j]);
#pragma unroll
      for (int i = 0; i < kMt; ++i)
        acc[i] = M::mma(wf, lds_read_frag<Frag>(cur + kTileN * kRowBytes + 4096 * i + off[j]), acc[i]);
    }
    // The stage's reads are complete before the next stage's barrier is reached.
    __builtin_amdgcn_sched_barrier(0);
  }

#pragma unroll
  for (int i = 0; i < kMt; ++i) store_outputs<T, kGate>(a, acc[i], split, 16 * i + n16, tile * NW + w, g);
}

// The same for 65 .. 256 rows, where x is too large to stream beside the
// weights at their depth: x [BM rows] and W [BN rows] have rings of their own
// (RX and RW stages of 64 k, rows of 128 bytes, 16-byte chunk c of row r at
// c ^ (r / 2 % 8): rows two apart share a bank row, so 16 rows' chunks lie in
// 16 different bank groups). Eight waves, BM / 64 of them along x's rows and
// the rest along N, each 64 rows by BN / 16 / kWn groups of 16 outputs.
//
// Its loads set its pace: 28672 x 4096 at 256 rows takes 71 us with the loads
// alone (3.1 MB a CU, 44 GB/s; 66 without those of x, 63 without those of W),
// 55 with the LDS reads and products alone, 78 whole; hence the rule in
// cut_of. That is with the wait below, which holds the 256-row kernels to 32
// KB in flight a CU where their rings would allow 64 (48 in 64-row tiles): not
// what a CU can load.
template <typename T, int BM, int BN, int RX, int RW, bool kGate>
__global__ __launch_bounds__(512) void batch_gemm(GemmArgs a) {
  using M = Mfma<T>;
  using Frag = typename M::Frag;
  constexpr int kRow = 128;             // bytes of a row's 64 k
  constexpr int kWm = BM / 64, kWn = 8 / kWm;
  constexpr int kNf = BN / 16 / kWn;    // output groups of a wave
  constexpr int kXi = BM / 64, kWi = BN / 64;  // loads of a wave per stage: eight rows each
  static_assert(kNf >= 1 && RX == 3 && RW >= 4, "ring depths");
  __shared__ __attribute__((aligned(1024))) char xring[RX][BM * kRow];
  __shared__ __attribute__((aligned(1024))) char wring[RW][BN * kRow];
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n16 = lane & 15, g = lane >> 4;
  const int tile = (int)(blockIdx.x / (unsigned)a.splits), split = (int)(blockIdx.x % (unsigned)a.splits);
  const int total = a.k / 64;
  const int s0 = (int)((int64_t)total * split / a.splits), s1 = (int)((int64_t)total * (split + 1) / a.splits);
  const int ns = s1 - s0;

  // Output (weight) row of tile row t.
  auto weight_row = [&](int t) -> int64_t {
    if (kGate) {  // of each 16: eight gate rows, then the up rows of the same outputs
      const int col = min(tile * (BN / 2) + t / 16 * 8 + (t & 7), a.n / 2 - 1);
      return ((t & 8) ? a.n / 2 : 0) + col;
    }
    return min(tile * BN + t, a.n - 1);
  };
  const int lr = lane >> 3, lc = lane & 7;
  const char* wrow[kWi];
  const char* xrow[kXi];
#pragma unroll
  for (int i = 0; i < kWi; ++i) {
    const int t = 8 * (w * kWi + i) + lr;
    wrow[i] = a.w + weight_row(t) * a.w_s + (int64_t)s0 * kRow + 16 * (lc ^ ((t >> 1) & 7));
  }
#pragma unroll
  for (int i = 0; i < kXi; ++i) {
    const int t = 8 * (w * kXi + i) + lr;
    xrow[i] = a.x + (int64_t)min(t, a.m - 1) * a.x_s + (int64_t)s0 * kRow + 16 * (lc ^ ((t >> 1) & 7));
  }
  const uint32_t xbase = lds_addr(&xring[0][0]), wbase = lds_addr(&wring[0][0]);
  const unsigned rotated = (unsigned)(tile >> 3) * kRotate;
  auto at = [&](int st) -> int64_t { return (int64_t)((rotated + (unsigned)st) % (unsigned)ns) * kRow; };
  auto issue_w = [&](int st) {
    const uint32_t dst = wbase + (uint32_t)(st % RW) * (BN * kRow) + 1024 * kWi * w;
    const int64_t o = at(st);
#pragma unroll
    for (int i = 0; i < kWi; ++i) dma16<true>(wrow[i] + o, dst + 1024 * i);
  };
  auto issue_x = [&](int st) {
    const uint32_t dst = xbase + (uint32_t)(st % RX) * (BM * kRow) + 1024 * kXi * w;
    const int64_t o = at(st);
#pragma unroll
    for (int i = 0; i < kXi; ++i) dma16<false>(xrow[i] + o, dst + 1024 * i);
  };

  const int wm = w % kWm, wn = w / kWm;
  floatx4_t acc[4][kNf];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int f = 0; f < kNf; ++f) acc[i][f] = floatx4_t{0.f, 0.f, 0.f, 0.f};
  uint32_t off[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) off[j] = (uint32_t)(n16 * kRow + 16 * ((4 * j + g) ^ ((n16 >> 1) & 7)));

  Frag w0[kNf], x0[4], w1[kNf] = {}, x1[4] = {};
  auto read = [&](uint32_t wc, uint32_t xc, int j, Frag (&wf)[kNf], Frag (&xf)[4]) __attribute__((always_inline)) {
#pragma unroll
    for (int f = 0; f < kNf; ++f) wf[f] = lds_read_frag<Frag>(wc + f * 16 * kRow + off[j]);
#pragma unroll
    for (int i = 0; i < 4; ++i) xf[i] = lds_read_frag<Frag>(xc + i * 16 * kRow + off[j]);
  };
  auto multiply = [&](const Frag (&wf)[kNf], const Frag (&xf)[4]) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int f = 0; f < kNf; ++f) acc[i][f] = M::mma(wf[f], xf[i], acc[i][f]);
  };
  auto interleave = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 4 + kNf; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // an LDS read
      __builtin_amdgcn_sched_group_barrier(0x008, (5 * kNf + 3) / (4 + kNf), 0);
    }
  };

  // Weights run RW - 1 stages ahead, x two. In order of issue: x 0, x 1 and W
  // 0 .. RW - 2 first, then x st + 2, W st + RW - 1 in stage st.
  issue_x(0);
  if (1 < ns) issue_x(1);
#pragma unroll
  for (int st = 0; st < RW - 1; ++st)
    if (st < ns) issue_w(st);
  for (int st = 0; st < ns; ++st) {
    // Loads newer than both W st and x st: in the first two stages those of W
    // st + 1 .. st + RW - 2 (x 0 and x 1 are older); later W st + RW - 3, x st
    // + 1 and W st + RW - 2; near the end at least x st + 1. One count serves
    // both: with 256 rows it is the first two stages', stricter than the
    // others need (4 against 8, in 64-row tiles 4 against 6).
    constexpr int kNewer = (RW - 2) * kWi < 2 * kWi + kXi ? (RW - 2) * kWi : 2 * kWi + kXi;
    if (st + RW - 1 < ns) li_wait_vm<kNewer>();
    else if (st >= 2 && st + 1 < ns) li_wait_vm<kXi>();
    else li_wait_vm<0>();
    lds_barrier();
    if (st + 2 < ns) issue_x(st + 2);
    if (st + RW - 1 < ns) issue_w(st + RW - 1);
    const uint32_t xc = xbase + (uint32_t)(st % RX) * (BM * kRow) + (uint32_t)wm * 64 * kRow;
    const uint32_t wc = wbase + (uint32_t)(st % RW) * (BN * kRow) + (uint32_t)wn * kNf * 16 * kRow;
    // A half stage's operands are read while the half before is multiplied
    // (across the barrier: the second half of stage st - 1 under the reads of
    // the first half of st), one read with every few products.
    read(wc, xc, 0, w0, x0);
    multiply(w1, x1);
    interleave();
    read(wc, xc, 1, w1, x1);
    multiply(w0, x0);
    interleave();
    __builtin_amdgcn_sched_barrier(0);
  }
  multiply(w1, x1);
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int f = 0; f < kNf; ++f)
      store_outputs<T, kGate>(a, acc[i][f], split, 64 * wm + 16 * i + n16, tile * (BN / 16) + wn * kNf + f, g);
}

// out = the sum of the splits' fp32 sums, rounded.
template <typename T>
__global__ __launch_bounds__(256) void skinny_reduce(const float* part, char* out, int64_t o_s, int m, int n, int splits) {
  const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
  if (i >= (int64_t)m * n) return;
  floatx4_t s = {0.f, 0.f, 0.f, 0.f};
  for (int p0 = 0; p0 < splits; p0 += 8) {
    floatx4_t v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u)
      v[u] = p0 + u < splits ? *reinterpret_cast<const floatx4_t*>(part + (int64_t)(p0 + u) * m * n + i)
                             : floatx4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < 8; ++u)
#pragma unroll
      for (int e = 0; e < 4; ++e) s[e] += v[u][e];
  }
  const int64_t row = i / n, col = i - row * n;
  *reinterpret_cast<uint2*>(out + (row * o_s + col) * 2) = uint2{li_pack2<T>(s[0], s[1]), li_pack2<T>(s[2], s[3])};
}

template <typename T, int BM, int R, int NW>
void launch_skinny(const GemmArgs& a, hipStream_t s) {
  const dim3 grid((unsigned)((a.n + 16 * NW - 1) / (16 * NW) * a.splits)), block(64 * NW);
  if (a.gate) hipLaunchKernelGGL((skinny_gemm<T, BM, R, NW, true>), grid, block, 0, s, a);
  else hipLaunchKernelGGL((skinny_gemm<T, BM, R, NW, false>), grid, block, 0, s, a);
}

template <typename T, int BM, int BN, int RW>
void launch_batch(const GemmArgs& a, hipStream_t s) {
  const dim3 grid((unsigned)((a.n + BN - 1) / BN * a.splits)), block(512);
  if (a.gate) hipLaunchKernelGGL((batch_gemm<T, BM, BN, 3, RW, true>), grid, block, 0, s, a);
  else hipLaunchKernelGGL((batch_gemm<T, BM, BN, 3, RW, false>), grid, block, 0, s, a);
}

template <typename T>
void launch_rows(const GemmArgs& a, hipStream_t s) {
  const bool wide = cut_of(a.m, a.n, a.k).tile == 128;
  if (a.m <= 16) launch_skinny<T, 16, 4, 4>(a, s);
  else if (a.m <= kFewRows) launch_skinny<T, 32, 3, 4>(a, s);
  else if (a.m <= kSkinnyRows) launch_skinny<T, 64, 3, 8>(a, s);
  else if (a.m <= 128 && wide) launch_batch<T, 128, 128, 6>(a, s);
  else if (a.m <= 128) launch_batch<T, 128, 64, 8>(a, s);
  else if (wide) launch_batch<T, 256, 128, 4>(a, s);
  else launch_batch<T, 256, 64, 6>(a, s);
}

}  // namespace

static int check_extents(int m, int n, int k) {
  if (m < 0 || n <= 0 || k <= 0) return li::fail(LI_EINVAL, "li_skinny_gemm_plan: bad extents (%d, %d, %d)", m, n, k);
  if (m > LI_SKINNY_MAX_ROWS || n % 8 || k % kStageK)
    return li::fail(LI_EUNSUPPORTED, "li_skinny_gemm: up to %d rows, n a multiple of 8, k of %d; got %d, %d, %d",
                    LI_SKINNY_MAX_ROWS, kStageK, m, n, k);
  if (cut_of(m, n, k).splits == 0)
    return li::fail(LI_EUNSUPPORTED, "li_skinny_gemm: %d rows of %d x %d are a general GEMM's", m, n, k);
  return LI_OK;
}

extern "C" int li_skinny_gemm_plan(int m, int n, int k, int* splits) {
  li::clear_error();
  if (int rc = check_extents(m, n, k)) return rc;
  if (uneven_rounds(m, n, k))
    return li::fail(LI_EUNSUPPORTED, "li_skinny_gemm: %d rows of %d x %d run faster as a general GEMM", m, n, k);
  if (splits) *splits = cut_of(m, n, k).splits;
  return LI_OK;
}

extern "C" int li_skinny_gemm(const void* x, int64_t x_stride, const void* w, int64_t w_stride, void* out,
                              int64_t out_stride, float* partials, int m, int n, int k, int splits, int gate_up,
                              int dtype, void* stream) {
  li::clear_error();
  if (dtype != LI_BF16 && dtype != LI_F16) return li::fail(LI_EUNSUPPORTED, "li_skinny_gemm: bf16 or f16 only");
  if (int rc = check_extents(m, n, k)) return rc;
  if (splits < 1 || splits > k / kStageK) return li::fail(LI_EINVAL, "li_skinny_gemm: %d splits of %d", splits, k);
  if (gate_up && n % 16) return li::fail(LI_EUNSUPPORTED, "li_skinny_gemm: gate / up halves must be multiples of 8");
  if (m == 0) return LI_OK;
  if (!x || !w || (splits == 1 ? !out : !partials)) return li::fail(LI_EINVAL, "li_skinny_gemm: null pointer");
  if (!li::aligned16(x) || !li::aligned16(w) || (x_stride * 2) % 16 || (w_stride * 2) % 16 || x_stride < 0 || w_stride < k ||
      (splits == 1 ? (reinterpret_cast<uintptr_t>(out) % 8 || out_stride % 4) : !li::aligned16(partials)))
    return li::fail(LI_EINVAL, "li_skinny_gemm: rows must be 16-byte aligned with the last axis contiguous");
  const GemmArgs a{static_cast<const char*>(x), static_cast<const char*>(w), static_cast<char*>(out), partials,
                   x_stride * 2, w_stride * 2, out_stride, m, n, k, splits, gate_up};
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (dtype == LI_BF16) launch_rows<li_bf16>(a, s);
  else launch_rows<li_f16>(a, s);
  return li::check_launch("li_skinny_gemm");
}

extern "C" int li_skinny_reduce(const float* partials, void* out, int64_t out_stride, int m, int n, int splits,
                                int dtype, void* stream) {
  li::clear_error();
  if (dtype != LI_BF16 && dtype != LI_F16) return li::fail(LI_EUNSUPPORTED, "li_skinny_reduce: bf16 or f16 only");
  if (m < 0 || n <= 0 || n % 8 || splits < 1) return li::fail(LI_EINVAL, "li_skinny_reduce: bad extents");
  if (m == 0) return LI_OK;
  if (!partials || !out || !li::aligned16(partials) || reinterpret_cast<uintptr_t>(out) % 8 || out_stride % 4)
    return li::fail(LI_EINVAL, "li_skinny_reduce: null or unaligned pointer");
  const int64_t work = (int64_t)m * n / 4;
  const dim3 grid((unsigned)li::cdiv64(work, 256)), block(256);
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (dtype == LI_BF16) hipLaunchKernelGGL(skinny_reduce<li_bf16>, grid, block, 0, s, partials, static_cast<char*>(out), out_stride, m, n, splits);
  else hipLaunchKernelGGL(skinny_reduce<li_f16>, grid, block, 0, s, partials, static_cast<char*>(out), out_stride, m, n, splits);
  return li::check_launch("li_skinny_reduce");
}
