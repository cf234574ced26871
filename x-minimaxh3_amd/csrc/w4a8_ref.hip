// Few-row GEMM on the reference's grouped int4 weights, decoded in registers (gfx950).
//
// y = out(fp32(sum_k a[m, k] * w8[n, k]) * (xs[m] * s_channel[n])) (+ bias), w8 the decoded int8 grid
// (the reference's w4a8_int8.py:344-363). Decoding to memory moves 1.5 bytes per weight before the GEMM
// reads another; a problem of few rows is bound by that traffic. Here each packed weight is read
// once and decoded where its MFMA needs it.
//
// A workgroup of eight waves owns 32 kBI rows x 256 columns of one K slice, wave w columns 32 w .. 32 w + 31
// of every row, as v_mfma_i32_32x32x32_i8 blocks with the weights first. K advances 256 per stage: A as two
// 128-byte halves, the packed weights (128 bytes per column) and the stage's scales are fetched with
// direct-to-LDS loads, kStages - 1 stages ahead (40 to 64 KB in flight per CU: HBM's latency times a CU's share of its
// rate is about 41 KB). Lane half h consumes k in [128 h, 128 h + 128) of the stage, step s the 16 k from
// 128 h + 16 s on both operands. e4m3 scales have 256 values, so the workgroup forms the 16 int8 levels of each
// once (4 KB of LDS) and a group's levels are one 16-byte LDS read; fp32 scales form them per group in registers.
// Bound by the arrival of the weights (128-byte pieces of 256 rows per stage): 20 x 5376 -> 21504 at group 16
// 20.8 us for 65 MB, 17.3 us with the decode taken out.
// The int32 sums of a slice go to the workspace; the summing kernel of the INT8 GEMM's split adds the slices and
// applies the epilogue. int32 sums do not depend on the order: the outputs are those of the decode + GEMM route.

#include <algorithm>

#include "w4a8_common.h"

namespace mxq {
namespace {

constexpr int kRefWaves = 8, kRefThreads = kRefWaves * kWave, kRefBN = 256, kRefBK = 256;

template <int kBI, bool kE4M3, int kG>
struct RefCfg {
  static constexpr int kRows = 32 * kBI;
  static constexpr int kScaleRow = kRefBK / kG * (kE4M3 ? 1 : 4);   // scale bytes per column and stage
  static constexpr int kPiece = kScaleRow >= 16 ? 16 : 4;           // bytes per lane of a scale load
  static constexpr int kPieces = kScaleRow / kPiece;                // per column
  static constexpr int kScaleLoads = (32 * kPieces + 63) / 64;      // per wave
  static constexpr int kA = 2 * kRows * 128, kB = kRefBN * 128, kS = kRefBN * kScaleRow;
  static constexpr int kStage = kA + kB + kS;
  static constexpr int kTable = kE4M3 ? 4096 : 0;
  static constexpr int kStages = 3 * kStage + kTable <= 160 * 1024 ? 3 : 2;  // LDS ring
  static constexpr int kLds = kStages * kStage + kTable;
  static constexpr int kLoads = kBI + 4 + kScaleLoads;              // per wave and stage
  static_assert(kLds <= 160 * 1024 && kScaleRow % kPiece == 0 && (kStages - 1) * kLoads < 64, "stage split");
};

MXQ_DEVICE int ref_swz(int r) { return (r >> 1) & 7; }  // 16-byte chunk c of 128-byte row r sits at c ^ ref_swz(r)

MXQ_DEVICE v2u lds_read_b64_at(uint32_t addr) {
  v2u r;
  __asm__ volatile("ds_read_b64 %0, %1" : "=v"(r) : "v"(addr));
  return r;
}

// (The body is a device function: a kernel that names the load builtins itself gets no host-side launch stub.)
template <int kBI, bool kE4M3, int kG>
MXQ_DEVICE void ref_slice(const W4RefArgs& p, const W4RefPlan& plan, int32_t* part, char* lds) {
  typedef RefCfg<kBI, kE4M3, kG> C;
  // m fastest, then columns, then slices, in contiguous ranges per XCD (workgroup ids are dealt to the XCDs in
  // turn): the row tiles that share a weight panel run on one XCD.
  int t;
  {
    const int num = plan.tiles_m * plan.tiles_n * plan.splits, per = num / 8, bid = blockIdx.x;
    t = bid < per * 8 ? (bid % 8) * per + bid / 8 : bid;
  }
  const int tm = t % plan.tiles_m;
  t /= plan.tiles_m;
  const int tn = t % plan.tiles_n, slice = t / plan.tiles_n;
  const int64_t m0 = (int64_t)tm * C::kRows, n0 = (int64_t)tn * kRefBN;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, lr = lane & 31, lh = lane >> 5;
  const int wv = __builtin_amdgcn_readfirstlane(wave);
  const int64_t groups = p.K / kG, k_first = (int64_t)slice * plan.stages * kRefBK;
  const int stages = (int)min<int64_t>(plan.stages, p.K / kRefBK - (int64_t)slice * plan.stages);

  // ---- load sources, at the slice's first stage ----
  const int8_t* a_src[kBI];
  const uint8_t* b_src[4];
  const uint8_t* s_src[C::kScaleLoads];
#pragma unroll
  for (int i = 0; i < kBI; ++i) {
    const int b = wave * kBI + i, half = b / (C::kRows / 8), r = (b % (C::kRows / 8)) * 8 + (lane >> 3);
    a_src[i] = p.a + min(m0 + r, p.M - 1) * p.K + k_first + half * 128 + ((lane & 7) ^ ref_swz(r)) * 16;
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = wave * 32 + i * 8 + (lane >> 3);
    b_src[i] = p.w + min(n0 + r, p.N - 1) * (p.K / 2) + k_first / 2 + ((lane & 7) ^ ref_swz(r)) * 16;
  }
#pragma unroll
  for (int i = 0; i < C::kScaleLoads; ++i) {
    const int piece = i * 2 + lh;
    s_src[i] = reinterpret_cast<const uint8_t*>(p.s_rel) +
               (min(n0 + wave * 32 + lr, p.N - 1) * groups + k_first / kG) * (kE4M3 ? 1 : 4) + (piece % C::kPieces) * C::kPiece;
  }
  auto issue = [&](int kt, int slot) {
    char* st = lds + slot * C::kStage;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      __builtin_amdgcn_global_load_lds((gptr_t)(b_src[i] + (int64_t)kt * 128), (lptr_t)(st + C::kA + (wv * 4 + i) * 1024), 16, 0, 0);
#pragma unroll
    for (int i = 0; i < C::kScaleLoads; ++i)
      if (i * 64 + lane < 32 * C::kPieces)
        __builtin_amdgcn_global_load_lds((gptr_t)(s_src[i] + (int64_t)kt * C::kScaleRow),
                                         (lptr_t)(st + C::kA + C::kB + wv * 32 * C::kScaleRow + i * 64 * C::kPiece), C::kPiece, 0, 0);
#pragma unroll
    for (int i = 0; i < kBI; ++i)
      __builtin_amdgcn_global_load_lds((gptr_t)(a_src[i] + (int64_t)kt * kRefBK), (lptr_t)(st + (wv * kBI + i) * 1024), 16, 0, 0);
  };
  const Levels levels = load_levels(p.codebook);
  const uint32_t lds0 = lds_addr(lds), table = lds0 + C::kStages * C::kStage;
  if constexpr (kE4M3) {
    if (threadIdx.x < 256) lds_write_b128(table + threadIdx.x * 16, level_values(levels, e4m3fn_to_f32(threadIdx.x)));
  }
  issue(0, 0);
  if (C::kStages == 3 && stages > 1) issue(1, 1);

  v16i acc[kBI];
#pragma unroll
  for (int i = 0; i < kBI; ++i) acc[i] = v16i{};
  const uint32_t a_row = (uint32_t)(lh * C::kRows + lr) * 128;  // (rows 32 apart share their swizzle)
  const uint32_t b_row = (uint32_t)(C::kA + (wave * 32 + lr) * 128);
  const int fz = ref_swz(lr);

  int slot = 0;
  for (int kt = 0; kt < stages; ++kt) {
    // Stage kt has landed (its own loads, then everyone's); the slot of stage kt - 1 is free.
    if (C::kStages == 3 && kt + 1 < stages)
      wait_vm_lgkm0<(C::kStages - 2) * C::kLoads>();
    else
      wait_all();
    __builtin_amdgcn_sched_barrier(0);
    barrier_no_drain();
    if (kt + C::kStages - 1 < stages) issue(kt + C::kStages - 1, slot == 0 ? C::kStages - 1 : slot - 1);
    const uint32_t st = lds0 + (uint32_t)(slot * C::kStage);
    slot = slot == C::kStages - 1 ? 0 : slot + 1;
    v4i bq[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) bq[j] = lds_read_b128<0>(st + b_row + (uint32_t)(((lh * 4 + j) ^ fz) << 4));
    // the lane's 128 / kG scales of the stage
    constexpr int kScales = 128 / kG;
    uint32_t sb[kE4M3 ? 2 : kScales];
    const uint32_t sc = st + (uint32_t)(C::kA + C::kB + wave * 32 * C::kScaleRow);
    if constexpr (kE4M3) {
      if constexpr (kG == 16) {
        const v2u r = lds_read_b64_at(sc + lr * 16 + lh * 8);
        sb[0] = r[0];
        sb[1] = r[1];
      } else if constexpr (kG == 32) {
        sb[0] = lds_read_b32(sc + (lh * 32 + lr) * 4);
      } else {
        sb[0] = lds_read_b32(sc + lr * 4);
      }
    } else {
      if constexpr (kG == 16) {
        const v4i r0 = lds_read_b128<0>(sc + lh * 1024 + lr * 16), r1 = lds_read_b128<512>(sc + lh * 1024 + lr * 16);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          sb[j] = (uint32_t)r0[j];
          sb[4 + j] = (uint32_t)r1[j];
        }
      } else if constexpr (kG == 32) {
        const v4i r = lds_read_b128<0>(sc + (lh * 32 + lr) * 16);
#pragma unroll
        for (int j = 0; j < 4; ++j) sb[j] = (uint32_t)r[j];
      } else {
        const v2u r = lds_read_b64_at(sc + lr * 16 + lh * 8);
        sb[0] = r[0];
        sb[1] = r[1];
      }
    }
    wait_lgkm<0>();
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (kE4M3 && kG == 64) sb[0] >>= 16 * lh;
    // Steps of 16 k per lane, each step's levels and A fragments read behind the previous step's MFMAs.
    v4i lv[2], fa[2][kBI];
    v4u cur = {};
    auto read_step = [&](auto S) {
      constexpr int s = decltype(S)::value;
      if constexpr (kE4M3 && s * 16 % kG == 0) {
        constexpr int g = s * 16 / kG;
        lv[s & 1] = lds_read_b128<0>(table + ((sb[g >> 2] >> (8 * (g & 3))) & 0xFFu) * 16);
      }
      static_for<kBI>([&](auto I) {
        fa[s & 1][decltype(I)::value] = lds_read_b128<decltype(I)::value * 32 * 128>(st + a_row + (uint32_t)((s ^ fz) << 4));
      });
    };
    read_step(std::integral_constant<int, 0>{});
    static_for<8>([&](auto S) {
      constexpr int s = decltype(S)::value;
      if constexpr (s < 7) {
        read_step(std::integral_constant<int, s + 1>{});
        wait_lgkm<kBI + (kE4M3 && (s + 1) * 16 % kG == 0 ? 1 : 0)>();
      } else {
        wait_lgkm<0>();
      }
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (s * 16 % kG == 0) {
        if constexpr (kE4M3)
          cur = __builtin_bit_cast(v4u, lv[s & 1]);
        else
          cur = level_values(levels, __uint_as_float(sb[s * 16 / kG]));
      }
      uint32_t o0, o1, o2, o3;
      decode8((uint32_t)bq[s >> 1][(s & 1) * 2], cur, o0, o1);
      decode8((uint32_t)bq[s >> 1][(s & 1) * 2 + 1], cur, o2, o3);
      const v4i fb = {(int)o0, (int)o1, (int)o2, (int)o3};
#pragma unroll
      for (int i = 0; i < kBI; ++i) acc[i] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fb, fa[s & 1][i], acc[i], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    });
  }

  // Lane l holds output row l % 32 of each block and the column runs q * 8 + (l / 32) * 4 + {0..3}.
  int32_t* out = part + (int64_t)slice * p.M * plan.ldp;
#pragma unroll
  for (int i = 0; i < kBI; ++i) {
    const int64_t row = m0 + i * 32 + lr;
    if (row >= p.M) continue;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int64_t col = n0 + wave * 32 + q * 8 + lh * 4;
      if (col < plan.ldp)  // (ldp is a multiple of 4)
        *reinterpret_cast<v4i*>(out + row * plan.ldp + col) =
            v4i{acc[i][q * 4], acc[i][q * 4 + 1], acc[i][q * 4 + 2], acc[i][q * 4 + 3]};
    }
  }
}

template <int kBI, bool kE4M3, int kG>
__global__ __launch_bounds__(kRefThreads, 1) void w4a8_ref_kernel(W4RefArgs p, W4RefPlan plan, int32_t* part) {
  __shared__ __attribute__((aligned(16))) char lds[RefCfg<kBI, kE4M3, kG>::kLds];
  ref_slice<kBI, kE4M3, kG>(p, plan, part, lds);
}

template <int kBI, bool kE4M3>
void launch_ref_g(const W4RefArgs& p, const W4RefPlan& plan, int32_t* part, hipStream_t st) {
  const unsigned grid = (unsigned)(plan.tiles_m * plan.tiles_n * plan.splits);
  if (p.group == 16)
    w4a8_ref_kernel<kBI, kE4M3, 16><<<grid, kRefThreads, 0, st>>>(p, plan, part);
  else if (p.group == 32)
    w4a8_ref_kernel<kBI, kE4M3, 32><<<grid, kRefThreads, 0, st>>>(p, plan, part);
  else
    w4a8_ref_kernel<kBI, kE4M3, 64><<<grid, kRefThreads, 0, st>>>(p, plan, part);
}

template <int kBI>
void launch_ref_t(const W4RefArgs& p, const W4RefPlan& plan, int32_t* part, hipStream_t st) {
  if (p.e4m3)
    launch_ref_g<kBI, true>(p, plan, part, st);
  else
    launch_ref_g<kBI, false>(p, plan, part, st);
}

}  // namespace

// Up to 128 rows always (us per call, decode + GEMM and here, ConvRot quantizer included, weights from HBM: 20 x 5376 ->
// 21504 group 16 e4m3 92 and 30, 64 x 7168 -> 5376 53 and 28, 128 x 20480 -> 5120 123 and 50, 128 x 5376 -> 21504
// fp32 scales 87 and 59). Past that the weights are decoded once per 128-row tile: worth it while all tiles
// run at once and the levels are cheap (333 x 5376 -> 21504 93 and 87, 512 rows 111 and 146; fp32 scales
// of group 16, 200 rows 86 and 111; both against the decode of decode_levels_kernel). K is cut so that
// the tiles fill the CUs, as far as `room` bytes hold the sums.
W4RefPlan plan_w4_ref(const W4RefArgs& p, int64_t room) {
  W4RefPlan g{};
  if (p.K % kRefBK != 0 || (p.group != 16 && p.group != 32 && p.group != 64)) return g;
  if ((uintptr_t)p.a % 16 || (uintptr_t)p.w % 16 || (uintptr_t)p.s_rel % 16) return g;
  const int rows = p.M <= 32 ? 1 : p.M <= 64 ? 2 : 4;
  const int64_t tiles_m = (p.M + 32 * rows - 1) / (32 * rows), tiles_n = (p.N + kRefBN - 1) / kRefBN;
  if (p.M > 128 && (p.M > 384 || tiles_m * tiles_n > 256 || (!p.e4m3 && p.group == 16))) return g;
  const int64_t tiles = tiles_m * tiles_n, stages = p.K / kRefBK, ldp = (p.N + 3) / 4 * 4;
  int64_t splits = std::min({stages, std::max<int64_t>(1, std::min(mxq_cu_count(), 256) / tiles), room / (p.M * ldp * 4)});
  if (splits < 1 || tiles * splits > INT32_MAX) return g;
  const int64_t per = (stages + splits - 1) / splits;
  splits = (stages + per - 1) / per;
  return W4RefPlan{rows, (int)tiles_m, (int)tiles_n, (int)splits, (int)per, ldp, splits * p.M * ldp * 4};
}

int launch_w4_ref(const W4RefArgs& p, const W4RefPlan& plan, int32_t* part, hipStream_t st) {
  if (plan.rows == 1)
    launch_ref_t<1>(p, plan, part, st);
  else if (plan.rows == 2)
    launch_ref_t<2>(p, plan, part, st);
  else
    launch_ref_t<4>(p, plan, part, st);
  return mxq_check_launch("w4a8_ref_kernel");
}

}  // namespace mxq
