// W8A16 GEMM, block tiles: wavefronts of up to 64 weight rows x 128 activation rows, and K groups
// inside the workgroup. Included by w8a16.hip.
#pragma once

namespace ts {

// A workgroup of WN x WM x KG wavefronts computes a (32 IN WN) x (32 JM WM) tile of Y^T on
// v_mfma_f32_32x32x16_f16. Each K step is 64 SUB columns, staged by LDS DMA into a ring of S
// stages; the step's 4 SUB MFMA K slices are shared by the KG wavefront groups (a group keeps
// its own accumulators; they meet in LDS after the last step), so a small tile still has enough
// wavefronts with large operand blocks.
//
// Why this split: the 128-row tiles of w8a16_wide_kernel stack four wavefronts of 32 weight rows,
// each of which reads the whole activation tile from LDS, 18 KB of LDS per 16 MFMAs (128 x 128
// tile); 64 x 96 per wavefront reads 16 KB per 24 MFMAs and 64 x 64 reads 12 KB per 16, and a
// 256 x 192 workgroup tile takes half the DMA bytes per MFMA. Stage layouts (swizzles) and operand
// layouts are w8a16_wide_kernel's: within a 64-column sub-step, lane (h, r) of MFMA slice q uses
// weight bytes 32 h + 8 q .. + 7 of its row and activation chunk 4 h + q.
//
// The DMAs are issued from inline assembly, outside the compiler's wait bookkeeping, with their
// waits written out: at the barrier in the middle of step t the batches of steps t + 1 .. t + S - 1
// may be in flight, and step t + 1's must have landed, so all but S - 2 batches are waited for
// (all of them once step t + 1 is the last). Step t + S is issued into step t's stage right after
// that barrier, which every wavefront passes with its reads of the stage complete (lgkmcnt 0).
template <int IN, int JM, int WN, int WM, int KG, int SUB, int S>
struct TileShape {
  static constexpr int kThreads = 64 * WN * WM * KG, kGroups = KG;
  static constexpr int kTN = 32 * IN * WN, kTM = 32 * JM * WM, kBK = 64 * SUB;
  static constexpr int kWBytes = kTN * kBK, kXBytes = kTM * kBK * 2;
  static constexpr int kStage = kWBytes + kXBytes;
  static constexpr int kPitch = kTN + 8;                  // halves per row of the epilogue tile
  static constexpr int kOut = kTM * kPitch * 2;
  static constexpr int kReduce = KG > 1 ? (KG / 2) * kTN * kTM * 4 : 0;
  static constexpr int kMax2 = kOut > kReduce ? kOut : kReduce;
  static constexpr int kLds = S * kStage > kMax2 ? S * kStage : kMax2;
};

// Order of one phase: NDS LDS reads, then NM MFMAs, the NV VALU instructions spread over those
// from the HOLD-th on (widening that waits for reads of the same phase starts late).
template <int NM, int NV, int NDS, int HOLD>
__device__ __forceinline__ void phase_schedule() {
  constexpr int per = NV > 0 ? (NV + NM - HOLD - 1) / (NM - HOLD) : 0;
  if constexpr (NDS > 0) __builtin_amdgcn_sched_group_barrier(0x100, NDS, 0);
#pragma unroll
  for (int m = 0; m < NM; ++m) {
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    if constexpr (per > 0)
      if (m >= HOLD) __builtin_amdgcn_sched_group_barrier(0x002, per, 0);
  }
  __builtin_amdgcn_sched_barrier(0);
}

template <int IN, int JM, int WN, int WM, int KG, int SUB, int S>
__global__ void __launch_bounds__(64 * WN * WM * KG) w8a16_tile_kernel(
    const half_t* __restrict__ x, int64_t ldx, const int8_t* __restrict__ wq,
    const void* __restrict__ scale, int scale_is_fp16, const half_t* __restrict__ bias,
    half_t* __restrict__ y, int64_t ldy, int M, int N, int K, GemmIo io) {
  using T = TileShape<IN, JM, WN, WM, KG, SUB, S>;
  constexpr int NT = T::kThreads, TN = T::kTN, TM = T::kTM, BK = T::kBK;
  constexpr int XD = TM * 8 * SUB / NT, WD = TN * 4 * SUB / NT;   // DMAs per thread per step
  constexpr int BATCH = XD + WD;
  constexpr int QW = 4 * SUB / KG;                        // K slices per wavefront and step
  static_assert(XD * NT == TM * 8 * SUB && WD * NT == TN * 4 * SUB, "tiles split over the threads");
  static_assert(QW == 2 || QW == 4, "a group's slices stay inside one 64-column sub-step");
  static_assert((S - 1) * BATCH < 64, "vmcnt holds 6 bits; the first wait leaves S - 1 batches");
  static_assert(S >= 2 && T::kLds + 8 * TN <= 160 * 1024, "LDS of one CU");
  __shared__ __align__(16) char smem[T::kLds];
  __shared__ float s_sc[TN], s_bs[TN];
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kg = w / (WN * WM), wn = (w % (WN * WM)) % WN, wm = (w % (WN * WM)) / WN;
  const int r = lane & 31, h = lane >> 5;
  const int n_tile = blockIdx.x * TN, m_base = blockIdx.y * TM;
  const int glu = io.glu;                                 // gate rows, then up rows, as the wide kernel
  const int g0 = blockIdx.x * (TN / 2);
  auto weight_row = [&](int nl) {
    if (glu) {
      const int i = g0 + nl % (TN / 2);
      return (nl >= TN / 2 ? glu : 0) + (i < glu ? i : glu - 1);
    }
    const int n = n_tile + nl;
    return n < N ? n : N - 1;
  };
  const int nk = K / BK;                                  // the host sends whole steps only

  float sc_r = 1.f, bs_r = 0.f;                           // of column tid, used in the epilogue
  if (tid < TN) {
    const int nc = weight_row(tid);
    sc_r = load_scale(scale, scale_is_fp16, nc);
    if (bias) bs_r = (float)bias[nc];
  }
  const half_t* xp[XD];
  const int8_t* wp[WD];
#pragma unroll
  for (int i = 0; i < XD; ++i) {
    const int c = i * NT + tid, sub = c / (TM * 8), row = (c / 8) % TM, pos = c % 8;
    const int mm = m_base + row;
    xp[i] = x + x_row(io, mm < M ? mm : M - 1) * ldx + 64 * sub + 8 * (pos ^ ((row >> 1) & 7));
  }
#pragma unroll
  for (int i = 0; i < WD; ++i) {
    const int c = i * NT + tid, sub = c / (TN * 4), row = (c / 4) % TN, pos = c % 4;
    wp[i] = wq + (int64_t)weight_row(row) * K + 64 * sub + 16 * (pos ^ ((row >> 2) & 3));
  }
  const unsigned lds0 = (unsigned)(size_t)(__attribute__((address_space(3))) char*)smem + 1024 * w;
  auto issue = [&](int stage) {                           // the next step's tiles into a stage
    const unsigned base = lds0 + stage * T::kStage;
#pragma unroll
    for (int i = 0; i < XD; ++i) {
      asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, off"
                   :: "v"(xp[i]), "{m0}"(base + T::kWBytes + 16 * NT * i) : "memory");
      xp[i] += BK;
    }
#pragma unroll
    for (int i = 0; i < WD; ++i) {
      asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, off"
                   :: "v"(wp[i]), "{m0}"(base + 16 * NT * i) : "memory");
      wp[i] += BK;
    }
  };

  float16_t acc[IN][JM];
#pragma unroll
  for (int i = 0; i < IN; ++i)
#pragma unroll
    for (int j = 0; j < JM; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

  // This wavefront's slices of a step: slices q0 .. q0 + QW - 1 of sub-step `sub`.
  const int sub = kg * QW / 4, q0 = kg * QW % 4;
  const int wrow = 32 * IN * wn + r, xrow = 32 * JM * wm + r;    // rows of subtile 0
  int aoff[QW / 2], boff[QW];
#pragma unroll
  for (int p = 0; p < QW / 2; ++p)
    aoff[p] = sub * TN * 64 + wrow * 64 + 16 * ((2 * h + q0 / 2 + p) ^ ((r >> 2) & 3));
#pragma unroll
  for (int q = 0; q < QW; ++q)
    boff[q] = T::kWBytes + sub * TM * 128 + xrow * 128 + 16 * ((4 * h + q0 + q) ^ ((r >> 1) & 7));
  int4_t araw[IN][QW / 2];                                // the step's weight pieces
  half8_t a[QW][IN], b[QW][JM];                           // operands of its slices
  auto read_a = [&](int so) {
#pragma unroll
    for (int p = 0; p < QW / 2; ++p)
#pragma unroll
      for (int i = 0; i < IN; ++i) araw[i][p] = ld<int4_t>(smem + so + aoff[p] + 32 * 64 * i);
  };
  auto read_b = [&](int so, int q) {
#pragma unroll
    for (int j = 0; j < JM; ++j) b[q][j] = ld<half8_t>(smem + so + boff[q] + 32 * 128 * j);
  };
  auto convert = [&](int q) {
#pragma unroll
    for (int i = 0; i < IN; ++i) {
      const int4_t v = araw[i][q >> 1];
      const int lo = (q & 1) * 2;
      a[q][i] = i8x8_to_half8(int2_t{v[lo], v[lo + 1]});
    }
  };
  auto mma = [&](int q) {
#pragma unroll
    for (int i = 0; i < IN; ++i)
#pragma unroll
      for (int j = 0; j < JM; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[q][i], b[q][j], acc[i][j], 0, 0, 0);
  };
  // One phase is the IN x JM MFMAs of one slice, with the LDS reads and the widening that later
  // phases need issued between them: NDS reads first, then VALU instructions behind each MFMA
  // from the HOLD-th on.
  constexpr int NM = IN * JM;
  int stage = 0;
  // Slices 0 .. QW/2 - 1, while the rest of the step's operands are read and widened.
  auto first_half = [&]() {
    const int so = stage * T::kStage;
    if constexpr (QW == 4) {
      read_b(so, 2);
      read_b(so, 3);
      convert(1);
      mma(0);
      phase_schedule<NM, 10 * IN, 2 * JM, 0>();
      convert(2);
      convert(3);
      mma(1);
      phase_schedule<NM, 20 * IN, 0, 0>();
    } else {
      read_b(so, 1);
      convert(1);
      mma(0);
      phase_schedule<NM, 10 * IN, JM, 0>();
    }
  };
  // The other slices, while the next step's first operands are read (its stage is `stage` now).
  auto second_half = [&]() {
    const int so = stage * T::kStage;
    read_a(so);
    read_b(so, 0);
    if constexpr (QW == 4) {
      mma(2);
      phase_schedule<NM, 0, IN * 2 + JM, 0>();
      read_b(so, 1);
      convert(0);
      mma(3);
      phase_schedule<NM, 10 * IN, JM, 0>();
    } else {
      mma(1);
      convert(0);
      phase_schedule<NM, 10 * IN, IN + JM, NM / 2>();
    }
  };

#pragma unroll
  for (int u = 0; u < S; ++u)
    if (u < nk) issue(u);
  if (nk >= S)
    wait_vmem_below_lds_done<(S - 1) * BATCH>();
  else
    wait_vmem_below_lds_done<0>();
  workgroup_barrier();
  read_a(0);
  read_b(0, 0);
  if constexpr (QW == 4) read_b(0, 1);
  convert(0);
  __builtin_amdgcn_sched_barrier(0);
  int kt = 0;
  for (; kt + S < nk; ++kt) {                             // steps whose successors fill the ring
    first_half();
    wait_vmem_below_lds_done<(S - 2) * BATCH>();
    workgroup_barrier();
    issue(stage);
    stage = stage + 1 == S ? 0 : stage + 1;
    second_half();
  }
  for (; kt + 1 < nk; ++kt) {                             // the ring drains
    first_half();
    wait_vmem_below_lds_done<0>();
    workgroup_barrier();
    stage = stage + 1 == S ? 0 : stage + 1;
    second_half();
  }
  first_half();
#pragma unroll
  for (int q = QW / 2; q < QW; ++q) mma(q);
  __syncthreads();                                        // the stages are free

  // The K groups' sums meet in LDS, pairwise (group g adds group g + KG / 2, ...).
#pragma unroll
  for (int half = KG / 2; half >= 1; half /= 2) {
    float4_t* red = reinterpret_cast<float4_t*>(smem);
    const int wi = (kg % half) * WN * WM + w % (WN * WM);
    if (kg >= half && kg < 2 * half) {
#pragma unroll
      for (int i = 0; i < IN; ++i)
#pragma unroll
        for (int j = 0; j < JM; ++j)
#pragma unroll
          for (int a4 = 0; a4 < 4; ++a4)
            red[((wi * IN + i) * JM + j) * 256 + a4 * 64 + lane] =
                float4_t{acc[i][j][4 * a4], acc[i][j][4 * a4 + 1], acc[i][j][4 * a4 + 2],
                         acc[i][j][4 * a4 + 3]};
    }
    __syncthreads();
    if (kg < half) {
#pragma unroll
      for (int i = 0; i < IN; ++i)
#pragma unroll
        for (int j = 0; j < JM; ++j)
#pragma unroll
          for (int a4 = 0; a4 < 4; ++a4) {
            const float4_t v = red[((wi * IN + i) * JM + j) * 256 + a4 * 64 + lane];
#pragma unroll
            for (int c = 0; c < 4; ++c) acc[i][j][4 * a4 + c] += v[c];
          }
    }
    __syncthreads();
  }

  // Lane (h, r) of subtile (i, j), element 4 a4 + c: column nl = 32 IN wn + 32 i + 8 a4 + 4 h + c
  // of tile row 32 JM wm + 32 j + r.
  if (tid < TN) {
    s_sc[tid] = sc_r;
    s_bs[tid] = bs_r;
  }
  __syncthreads();
  half_t* tile = reinterpret_cast<half_t*>(smem);          // fp16 results, [TM][kPitch]
  if (kg == 0) {
#pragma unroll
    for (int i = 0; i < IN; ++i)
#pragma unroll
      for (int a4 = 0; a4 < 4; ++a4) {
        const int nl = 32 * (IN * wn + i) + 8 * a4 + 4 * h;
        const float4_t sc = *reinterpret_cast<const float4_t*>(&s_sc[nl]);
        const float4_t bs = *reinterpret_cast<const float4_t*>(&s_bs[nl]);
#pragma unroll
        for (int j = 0; j < JM; ++j) {
          const float o[4] = {acc[i][j][4 * a4] * sc[0] + bs[0], acc[i][j][4 * a4 + 1] * sc[1] + bs[1],
                              acc[i][j][4 * a4 + 2] * sc[2] + bs[2],
                              acc[i][j][4 * a4 + 3] * sc[3] + bs[3]};
          *reinterpret_cast<half4_t*>(tile + (32 * (JM * wm + j) + r) * T::kPitch + nl) =
              half4_t{(half_t)o[0], (half_t)o[1], (half_t)o[2], (half_t)o[3]};
        }
      }
  }
  __syncthreads();
  if (io.rope_cos != nullptr) {
    // RoPE and the K/V cache write, as w8a16_wide_kernel's epilogue: every 128 columns are a head.
    const int H = io.rope_heads, KVH = io.rope_kv_heads;
    for (int it = tid; it < TM * (TN / 128) * 8; it += NT) {
      const int m = it / (TN / 16), hl = (it / 8) % (TN / 128), g = it & 7;
      const int mm = m_base + m, hd = blockIdx.x * (TN / 128) + hl;
      if (mm >= M || hd >= H + 2 * KVH) continue;
      const half_t* src = tile + m * T::kPitch + 128 * hl + 8 * g;
      half8_t y1 = *reinterpret_cast<const half8_t*>(src);
      half8_t y2 = *reinterpret_cast<const half8_t*>(src + 64);
      if (hd < H + KVH) {
        const int64_t prow = rope_row(io.positions[mm], io.rope_max_pos) * 64 + 8 * g;
        half4_t a1, a2, c1, c2;
        rope4(lo4(y1), lo4(y2), ld<float4_t>(io.rope_cos + prow), ld<float4_t>(io.rope_sin + prow),
              a1, a2);
        rope4(hi4(y1), hi4(y2), ld<float4_t>(io.rope_cos + prow + 4),
              ld<float4_t>(io.rope_sin + prow + 4), c1, c2);
        y1 = half8_t{a1[0], a1[1], a1[2], a1[3], c1[0], c1[1], c1[2], c1[3]};
        y2 = half8_t{a2[0], a2[1], a2[2], a2[3], c2[0], c2[1], c2[2], c2[3]};
      }
      half_t* dst = y + (int64_t)mm * ldy + 128 * hd + 8 * g;
      st<half8_t>(dst, y1);
      st<half8_t>(dst + 64, y2);
      if (hd >= H) {
        const int64_t slot = io.slots[mm];
        if (slot >= 0 && slot < io.num_slots) {            // -1 = padding row
          const int kvh = hd < H + KVH ? hd - H : hd - H - KVH;
          half_t* crow = (hd < H + KVH ? io.kc : io.vc) +
                         (((slot >> 4) * KVH + kvh) * kBlockSize + (slot & 15)) * 128 + 8 * g;
          st<half8_t>(crow, y1);
          st<half8_t>(crow + 64, y2);
        }
      }
    }
    return;
  }
  // Rows of the tile as 16-byte pieces, 8 columns per thread (8-byte stores where the rows of y
  // are only 8-byte aligned).
  const bool wide_rows = ldy % 8 == 0 && (reinterpret_cast<uintptr_t>(y) & 15) == 0;
  const int cols = glu ? TN / 2 : TN, first = glu ? g0 : n_tile, end = glu ? glu : N;
  for (int it = tid; it < TM * (cols / 8); it += NT) {
    const int m = it / (cols / 8), cc = 8 * (it % (cols / 8));
    const int mm = m_base + m, nn = first + cc;
    if (mm >= M || nn >= end) continue;
    half8_t v = *reinterpret_cast<const half8_t*>(tile + m * T::kPitch + cc);
    if (glu) {
      const half8_t u = *reinterpret_cast<const half8_t*>(tile + m * T::kPitch + TN / 2 + cc);
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = silu_mul_h(v[e], u[e]);
    }
    if (io.yf) {
      float* dst = io.yf + (int64_t)mm * io.ldyf + nn;
      if (nn + 7 < end) {
        st<float4_t>(dst, float4_t{(float)v[0], (float)v[1], (float)v[2], (float)v[3]});
        st<float4_t>(dst + 4, float4_t{(float)v[4], (float)v[5], (float)v[6], (float)v[7]});
      } else {
        for (int e = 0; e < 8; ++e)
          if (nn + e < end) dst[e] = (float)v[e];
      }
      continue;
    }
    half_t* dst = y + (int64_t)mm * ldy + nn;
    if (nn + 7 < end) {
      if (wide_rows) {
        st<half8_t>(dst, v);
      } else {
        st<half4_t>(dst, lo4(v));
        st<half4_t>(dst + 4, hi4(v));
      }
    } else {
      for (int e = 0; e < 8; ++e)
        if (nn + e < end) dst[e] = v[e];
    }
  }
}

}  // namespace ts
