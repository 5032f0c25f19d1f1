// Few-row matmul on int8 MFMA: up to 32 activation rows (16 for Q5_K and the 32-value types) against a weight matrix streamed once from
// HBM.  Serves the decode matvec from a few rows on (the reference's tensor-core matvec, mmvq_tc_k.cuh,
// fast_mmvq.rs:1897-2126, and its plain launcher at b <= 8), its fused GLU form, and the expert-grouped matmul when the
// experts receive few rows each.
//
// What bounds it: HBM, once the texture addresser is out of the way.  The addresser takes a load's lanes four at a
// time and one cache line a cycle, so the MFMA operand layout, in which neighbouring lanes hold different rows, costs
// 64 cycles for each 1 KB load when it is loaded straight into registers: 830 cycles per 32 weight rows and superblock
// with the activations, 23 k cycles per CU at 14336x4096, 11 of that form's 16 us.  Here both operands go by DMA into
// LDS as contiguous 16-byte pieces (17 to 20 cycles per KB) and the waves read their operands from there.
//
// A workgroup owns 16 TC weight rows (TC tiles) and all activation rows; its NW waves split the superblocks of K.  A
// wave walks its superblocks, and for each the TC tiles: one unit is 16 weight rows x 256 values.  Everything a wave
// stages it reads itself, so no barrier is needed until the partial sums meet: the DMA of the unit after next is issued
// as soon as a unit's bytes are in registers, and a counted s_waitcnt covers the one that is read.  The activations of
// a superblock are kept in registers over its TC tiles while those of the next one are on their way.
//
// Each wave's lane (kg, r) builds the two int8 weight planes of row r (planes.h) as the MFMA B column, with activation
// row r as the A row; one 16x16x64 MFMA per plane per 64 values, the Q4_K min term through one f16 MFMA per superblock,
// and the per-superblock f32 scaling of the reference (k_quants.rs:1848-1928, 2145-2232, 2518-2575).  Weights of 32-value
// blocks (Q8_0, Q4_0, Q5_0) against Q8_0 activations stage superblocks of eight blocks the same way and take one 16x16x32
// MFMA a block, whose sums are scaled by both blocks' scales (432-449, 615-637, 982-999): 4 conversions, 4 products and 4
// fused adds a lane and block, which the loads cover.  11008x4096 Q8_0 at 5 / 16 rows 12.5 / 13.1 us, 3.8 TB/s (the matvec
// 21 / 53); 32768x4096 27.1 / 28.4, 5.3 TB/s (44 / 101).
#include "common.h"
#include "inferencequant.h"
#include "planes.h"
#include "skinny.h"
#include "units.h"

namespace {

// Where the activations of row m, superblock sb lie: 256 int8 values at q0 + m qrow + sb qsb, the f32 scale at d0 + m
// drow + sb dsb (byte offsets from base)
struct act_rows {
  const uint8_t *base;
  int64_t bytes;
  uint32_t q0, qrow, qsb, d0, drow, dsb;
};

template <int N>
__device__ __forceinline__ void wait_vm() {
  static_assert(N >= 0 && N < 64, "vmcnt field");
  __asm__ volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
__device__ __forceinline__ void wait_lds() { __asm__ volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

// 16 (4) bytes per lane from off + soff of the resource to lds + 16 (4) lane.  soff is uniform and outside the range
// check, which the vector part alone passes or fails.
__device__ __forceinline__ void dma16(rsrc_t r, uint8_t *lds, uint32_t off, uint32_t soff) {
#if defined(__HIP_DEVICE_COMPILE__)
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void *)lds, 16, off, soff, 0, 0);
#endif
}
__device__ __forceinline__ void dma4(rsrc_t r, uint8_t *lds, uint32_t off, uint32_t soff) {
#if defined(__HIP_DEVICE_COMPILE__)
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void *)lds, 4, off, soff, 0, 0);
#endif
}

constexpr uint32_t kNowhere = 0x80000000u;  // past every resource's end: reads zeros with no memory traffic

template <class WT, int NW, int TC, int MT, int D>
struct RowsLds {
  static constexpr int kUnit = 256 * WT::kPieces;            // a unit's window: 16 rows x kPieces 16-byte pieces
  // a superblock's activations: 16 MT rows of 256 values (chunk c of row m at c ^ (m % 16)), then their scales; for the
  // 32-value types 16 rows of eight 34-byte Q8_0 blocks
  static constexpr int kAct = WT::kB32 ? 272 * 16 * MT : 256 * 16 * MT + 4 * 16 * MT;
  static constexpr int kWave = kAct + D * kUnit;
  static constexpr int kSums = NW * TC * MT * 1024;          // the partial sums, in the same memory afterwards
  static constexpr int kBytes = NW * kWave > kSums ? NW * kWave : kSums;
};

// A superblock's activations in registers: operand rows, f32 scales of the four output rows, the Q4_K / Q5_K min operand
template <bool B32, int MT>
struct ActRegs {
  struct T {
    v4i q[MT][4];
    v4f d[MT];
    v4h m[MT];
  };
};
template <int MT>
struct ActRegs<true, MT> {
  static_assert(MT == 1, "32-value types take 16 rows");
  struct T {
    u32x2 q[8];  // per block
    v4f d[8];
  };
};
template <class WT>
constexpr bool has_min() {
  if constexpr (WT::kB32)
    return false;
  else
    return WT::kMin;
}

// One pass: the workgroup's 16 TN weight rows from n0 against activation rows [m0, m0 + mr), mr <= 16 MT.
// MT: 16-row activation tiles (1 or 2).  GLU: tiles [0, TC / 2) are gate rows (W), [TC / 2, TC) the up rows (W2) at the
// same places.  Row m is stored to destination row ids[m] when ids is given, else m.
template <class WT, class Out, int NW, int TC, int MT, int D, bool GLU>
__device__ __forceinline__ void rows_pass(uint8_t *lds, const uint8_t *__restrict__ W, const uint8_t *__restrict__ W2,
                                          int64_t nrows_w, int64_t w_row_bytes, const act_rows &ap, int m0, int mr,
                                          int nsb, typename Out::T *__restrict__ dst, int64_t ldd, int activation,
                                          const int32_t *__restrict__ ids) {
  typedef RowsLds<WT, NW, TC, MT, D> L;
  constexpr int MR = 16 * MT;            // activation rows
  constexpr int TN = GLU ? TC / 2 : TC;  // tiles of output columns
  constexpr int P = WT::kPieces, UB = L::kUnit;
  constexpr int LW = (16 * P + 63) / 64, LA = WT::kB32 ? (17 * MR + 63) / 64 : MR / 4 + 1;  // DMA loads of a unit and of a superblock's activations

  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, kg = lane >> 4,
            r = lane & 15;
  uint8_t *const abuf = lds + wave * L::kWave, *const wbuf = abuf + L::kAct;
  const int64_t n0 = (int64_t)blockIdx.x * (16 * TN);
  const int64_t rows_here = nrows_w - n0 < 16 * TN ? nrows_w - n0 : 16 * TN;
  // resources over the workgroup's rows, from the dword that holds the first byte to the end of the dword that holds
  // the last (superblocks of 210 bytes start and end inside dwords); rows past the end read as zeros
  const uintptr_t wt = (uintptr_t)(W + n0 * w_row_bytes), wt2 = (uintptr_t)((GLU ? W2 : W) + n0 * w_row_bytes);
  const uint32_t dl = (uint32_t)(wt & 3), dl2 = (uint32_t)(wt2 & 3);
  const uint32_t tile_bytes = (uint32_t)(16 * w_row_bytes);

  // this lane's pieces of a unit: piece 64 i + lane is row C / P, 16-byte piece C % P
  uint32_t wpc[LW];
#pragma unroll
  for (int i = 0; i < LW; i++) {
    const int C = 64 * i + lane, row = C / P;
    wpc[i] = (uint32_t)(row * w_row_bytes) + 16 * (uint32_t)(C - row * P);
  }
  // Tile t of superblock sb into slot `slot`.  Superblocks of whole dwords are their own pieces: the superblock's offset
  // is uniform, and a row past the end fails the range check by its own offset.  Others start at the dword that holds
  // their first byte, and their last piece ends past them, so the whole offset is checked.  skip: nothing is left to
  // load; the loads are issued from an empty resource so that the wait counts hold.
  constexpr bool kWhole = WT::kBytes % 16 == 0;
  auto issue_w = [&](int t, int sb, uint8_t *slot, bool skip) {
    const bool up = GLU && t >= TN;
    const int rn = (int)(rows_here * w_row_bytes) + (up ? dl2 : dl);
    const rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void *)((up ? wt2 - dl2 : wt - dl)), (short)0,
                                                        skip ? 0 : (rn + 3) & ~3, 0x00020000);
    const uint32_t ot = (uint32_t)(up ? t - TN : t) * tile_bytes + (up ? dl2 : dl), os = (uint32_t)sb * WT::kBytes;
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < LW; i++)
      if (64 * i + 64 <= 16 * P || lane < 16 * P - 64 * i)
        dma16(rs, slot + 1024 * i, kWhole ? wpc[i] + ot : (wpc[i] + ot + os) & ~3u, kWhole ? os : 0u);
    __builtin_amdgcn_sched_barrier(0);
  };

  // wave w takes superblocks w, w + NW, ...: what the waves have in flight at a time is one run of each row
  const int s0 = wave, s1 = nsb;
  uint32_t aoff[LA];
#pragma unroll
  for (int i = 0; i < LA; i++) {
    // row and 16-byte chunk of this lane's i-th load (the last one of the K-quants: the scales, dwords)
    const int C = 64 * i + lane, row = WT::kB32 ? C / 17 : i < MR / 4 ? C / 16 : lane;
    const uint32_t in_row = WT::kB32 ? 16 * (C - 17 * row) : i < MR / 4 ? 16 * (r ^ (row & 15)) : 0;
    aoff[i] = row < mr ? (WT::kB32 || i < MR / 4 ? ap.q0 + (uint32_t)(m0 + row) * ap.qrow
                                                : ap.d0 + (uint32_t)(m0 + row) * ap.drow) + in_row
                       : kNowhere;
  }
  auto issue_a = [&](int sb, bool skip) {
    const rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc((void *)ap.base, (short)0, skip ? 0 : (int)ap.bytes, 0x00020000);
    const uint32_t oq = (uint32_t)sb * ap.qsb, od = (uint32_t)sb * ap.dsb;
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < LA; i++) {
      if (!WT::kB32 && i == MR / 4) {
        if (lane < MR) dma4(ra, abuf + 256 * MR, aoff[i], od);
      } else if (!WT::kB32 || 64 * i + 64 <= 17 * MR || lane < 17 * MR - 64 * i) {
        dma16(ra, abuf + 1024 * i, aoff[i], oq);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  };

  v4f fa[TC][MT];
#pragma unroll
  for (int t = 0; t < TC; t++)
#pragma unroll
    for (int x = 0; x < MT; x++) fa[t][x] = (v4f){};

  if (s0 < s1) {
    issue_a(s0, false);
#pragma unroll
    for (int u = 0; u < D; u++) issue_w(u % TC, s0 + u / TC * NW, wbuf + UB * u, s0 + u / TC * NW >= s1);
    int slot = 0;
    for (int sb = s0; sb < s1; sb += NW) {
      // the activations of sb have landed once at most the weight loads issued after them are outstanding
      wait_vm<(TC < D ? TC : D) * LW>();
      typename ActRegs<WT::kB32, MT>::T act;
      if constexpr (WT::kB32) {
#pragma unroll
        for (int j = 0; j < 8; j++) {
          act.q[j] = (u32x2){lds_dw(abuf + 272 * r, 34 * j + 2, kg), lds_dw(abuf + 272 * r, 34 * j + 18, kg)};
#pragma unroll
          for (int i = 0; i < 4; i++) {
            const _Float16 h = __builtin_bit_cast(_Float16, *(const uint16_t *)(abuf + 272 * (4 * kg + i) + 34 * j));
            act.d[j][i] = (float)h;
          }
        }
      } else {
#pragma unroll
        for (int x = 0; x < MT; x++) {
#pragma unroll
          for (int t = 0; t < 4; t++)
            act.q[x][t] = *(const v4i *)(abuf + 256 * (16 * x + r) + 16 * ((WT::act_offset(t, kg) / 16) ^ r));
          act.d[x] = *(const v4f *)(abuf + 256 * MR + 4 * (16 * x + 4 * kg));
        }
      }
      wait_lds();
      issue_a(sb + NW, sb + NW >= s1);
      if constexpr (has_min<WT>()) {
        // the 32-value sums of the two sub-blocks this lane's min operand carries: its own halves plus its
        // partner's (lane ^ 16), split as planes.h min_frag does
#pragma unroll
        for (int x = 0; x < MT; x++) {
          uint32_t s[4];
#pragma unroll
          for (int t = 0; t < 4; t++) {
            int acc = 0;
#pragma unroll
            for (int i = 0; i < 4; i++) acc = sdot4(act.q[x][t][i], 0x01010101, acc);
            s[t] = (uint32_t)acc;
          }
          swap_lane_rows(s[0], s[2]);
          swap_lane_rows(s[1], s[3]);
          uint32_t hp, lp;
          s32_split(((s[0] + s[2]) & 0xffffu) | ((s[1] + s[3]) << 16), hp, lp);
          act.m[x] = __builtin_bit_cast(v4h, (u32x2){hp, lp});
        }
      }
#pragma unroll
      for (int t = 0; t < TC; t++) {
        // newer than this unit's loads: those of the D - 1 units after it, and the next superblock's activations while
        // fewer than D units were issued after them
        if (t < D)
          wait_vm<(D - 1) * LW + LA>();
        else
          wait_vm<(D - 1) * LW>();
        uint8_t *const wslot = wbuf + UB * slot;
        auto next_unit = [&]() {  // the unit's bytes are in registers: its slot is free
          const int tn = (t + D) % TC, sn = sb + (t + D) / TC * NW;
          wait_lds();
          issue_w(tn, sn, wslot, sn >= s1);
        };
        if constexpr (WT::kB32) {
          u32x2 wv[8];
          uint32_t wd[8];
#pragma unroll
          for (int j = 0; j < 8; j++) wv[j] = WT::block(wslot + 16 * P * r, j, kg, wd[j]);
          next_unit();
#pragma unroll
          for (int j = 0; j < 8; j++) {
            const v4i iv = mfma16x32_i8(act.q[j], wv[j]);
            const float d = (float)__builtin_bit_cast(_Float16, (uint16_t)wd[j]) * (1.0f / (1 << WT::kUp));
#pragma unroll
            for (int i = 0; i < 4; i++) fa[t][0][i] = __builtin_fmaf(act.d[j][i], d * (float)iv[i], fa[t][0][i]);
          }
        } else {
          typename WT::Raw raw;
          const uint32_t o = (uint32_t)(r * w_row_bytes) + (uint32_t)sb * WT::kBytes + (GLU && t >= TN ? dl2 : dl) +
                             (WT::kBytes % 4 ? (uint32_t)(GLU && t >= TN ? t - TN : t) * tile_bytes : 0u);
          WT::load_lds(wslot + 16 * P * r, o & 3, kg, raw);
          next_unit();
          typename WT::Prep p;
          WT::prepare(raw, kg, p);
          v4i acc1[MT], acc2[MT];
#pragma unroll
          for (int x = 0; x < MT; x++) acc1[x] = acc2[x] = (v4i){};
#pragma unroll
          for (int q = 0; q < 4; q++) {
            v4i b1, b2;
            WT::planes(raw, p, q, b1, b2, kg);
#pragma unroll
            for (int x = 0; x < MT; x++) {
              acc1[x] = mfma16_i8(act.q[x][q], b1, acc1[x]);
              acc2[x] = mfma16_i8(act.q[x][q], b2, acc2[x]);
            }
          }
#pragma unroll
          for (int x = 0; x < MT; x++) {
            v4f fmin = (v4f){};
            if (WT::kMin) fmin = mfma16_f16(act.m[x], p.bmin, fmin);
#pragma unroll
            for (int i = 0; i < 4; i++) {
              const int iv = (acc1[x][i] << WT::kShift) + acc2[x][i];
              float v = p.d * (float)iv;
              if (WT::kMin) v = __builtin_fmaf(-p.dmin, fmin[i], v);
              fa[t][x][i] = __builtin_fmaf(act.d[x][i], v, fa[t][x][i]);
            }
          }
        }
        slot = slot + 1 == D ? 0 : slot + 1;
        // (the sums are formed here: left alone, the compiler sinks every tile's scaling to the loop's end and keeps their
        // MFMA results in registers until then, up to 75 more)
#pragma unroll
        for (int x = 0; x < MT; x++) __asm__ volatile("" : "+v"(fa[t][x]));
      }
    }
  }

  // the waves' partial sums, added in wave order: value (t, x, i) of lane l is output column n0 + 16 t + l % 16,
  // activation row m0 + 16 x + 4 (l / 16) + i
  wait_vm<0>();  // (the empty loads still write LDS)
  __syncthreads();
  float *const red = (float *)lds;
  constexpr int V = TC * MT * 4;  // values per lane
#pragma unroll
  for (int t = 0; t < TC; t++)
#pragma unroll
    for (int x = 0; x < MT; x++)
#pragma unroll
      for (int i = 0; i < 4; i++) red[(wave * V + (t * MT + x) * 4 + i) * 64 + lane] = fa[t][x][i];
  __syncthreads();
  for (int v = wave; v < TN * MT * 4; v += NW) {
    float a = 0.0f;
#pragma unroll
    for (int w = 0; w < NW; w++) a += red[(w * V + v) * 64 + lane];
    if (GLU) {
      float u = 0.0f;
#pragma unroll
      for (int w = 0; w < NW; w++) u += red[(w * V + TN * MT * 4 + v) * 64 + lane];
      a = glu_act(activation, a) * u;
    }
    const int t = v / (4 * MT), m = 16 * ((v >> 2) % MT) + 4 * kg + (v & 3);
    const int c = 16 * t + r;
    if (m < mr && c < rows_here) Out::store(dst, (ids ? (int64_t)ids[m0 + m] : (int64_t)(m0 + m)) * ldd + n0 + c, a);
  }
}

// Up to 16 MT activation rows
template <class WT, class Out, int NW, int TC, int MT, int D, int WPE, bool GLU>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(WPE))) void k_rows(
    const uint8_t *__restrict__ W, const uint8_t *__restrict__ W2, int64_t nrows_w, int64_t w_row_bytes, act_rows ap,
    int mrows, int nsb, typename Out::T *__restrict__ dst, int64_t ldd, int activation) {
  __shared__ __attribute__((aligned(16))) uint8_t lds[RowsLds<WT, NW, TC, MT, D>::kBytes];
  rows_pass<WT, Out, NW, TC, MT, D, GLU>(lds, W, W2, nrows_w, w_row_bytes, ap, 0, mrows, nsb, dst, ldd, activation,
                                         nullptr);
}

// Expert-grouped: expert e = blockIdx.z owns activation rows [bounds[e], bounds[e + 1]) and weights W + e *
// expert_bytes (GLU: gate W, up W2); row m is stored to destination row ids_dst[m] (m itself when ids_dst is null).
// Workgroup (x, y) takes the 32-row chunks y, y + gridDim.y, ... of its expert, so every row is covered whatever the
// grid's height.
template <class WT, int NW, int TC, int D, int WPE, bool GLU>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(WPE))) void k_rows_moe(
    const uint8_t *__restrict__ W, const uint8_t *__restrict__ W2, int64_t expert_bytes, int64_t nrows_w,
    int64_t w_row_bytes, act_rows ap, const int32_t *__restrict__ bounds, const int32_t *__restrict__ ids_dst, int nsb,
    float *__restrict__ dst, int64_t ldd, int activation) {
  __shared__ __attribute__((aligned(16))) uint8_t lds[RowsLds<WT, NW, TC, 2, D>::kBytes];
  const int64_t e = blockIdx.z;
  const int m1 = bounds[e + 1];
  W += e * expert_bytes;
  if (GLU) W2 += e * expert_bytes;
  for (int m0 = bounds[e] + 32 * (int)blockIdx.y; m0 < m1; m0 += 32 * (int)gridDim.y) {  // uniform over the workgroup
    const int mr = m1 - m0;
    if (mr <= 16)
      rows_pass<WT, out_f32, NW, TC, 1, D, GLU>(lds, W, W2, nrows_w, w_row_bytes, ap, m0, mr, nsb, dst, ldd, activation,
                                                ids_dst);
    else
      rows_pass<WT, out_f32, NW, TC, 2, D, GLU>(lds, W, W2, nrows_w, w_row_bytes, ap, m0, mr < 32 ? mr : 32, nsb, dst,
                                                ldd, activation, ids_dst);
    __syncthreads();  // the next pass stages over the partial sums
  }
}

template <class WT, class Out, int NW, int TC, int MT, bool GLU>
void launch_k(const void *w, const void *w2, int64_t nrows, int64_t wrb, const act_rows &ap, int mrows, int64_t nsb,
              void *dst, int64_t ldd, int activation, hipStream_t s) {
  constexpr int cols = 16 * (GLU ? TC / 2 : TC);
  k_rows<WT, Out, NW, TC, MT, 2, (WT::kB32 || MT > 1 ? 3 : 4), GLU><<<(unsigned)qmm_ceil_div(nrows, cols), 64 * NW, 0, s>>>(
      (const uint8_t *)w, (const uint8_t *)w2, nrows, wrb, ap, mrows, (int)nsb, (typename Out::T *)dst, ldd, activation);
}

template <class WT, class Out, int MT>
void launch_mt(const void *w, const void *w2, int64_t nrows, int64_t wrb, const act_rows &ap, int mrows, int64_t nsb,
               void *dst, int64_t ldd, int activation, hipStream_t s) {
#define QMM_L(NW, TC, GLU) launch_k<WT, Out, NW, TC, MT, GLU>(w, w2, nrows, wrb, ap, mrows, nsb, dst, ldd, activation, s)
  const int64_t tiles = qmm_ceil_div(nrows, 16), cus = qmm_device_cus();
  // A workgroup's tiles share its activations, so more of them mean fewer activation bytes; too many leave CUs without
  // work, or each wave with a long chain of units.  MI355X, us at 4 / 16 / 24 rows, Q4_K with K = 4096 unless said
  // otherwise, as (waves, tiles):
  //   N = 4096   (8, 1) 5.0 / 5.4 / 6.7     (4, 2) 6.2 / 6.2 / 7.7     N = 1024  (8, 1) 4.3 / 4.4   (4, 2) 6.0 / 6.0
  //   N = 8192   (4, 2) 6.8 / 6.9 / 8.7     (8, 1) 8.0 / 8.5 / 12.3    (8, 4) 8.9 / 9.1 / 11.4
  //   N = 14336  (8, 4) 9.8 / 10.3 / 12.4   (4, 4) 10.9 / 10.0 / 12.1  (4, 2) 10.1 / 10.9 / 13.7
  //   N = 17408  (4, 6) 13.9 / 12.8 / 15.8  (4, 4) 14.2 / 15.5 / 19.2  (4, 8) 16.2 / 15.6 / 19.8
  //   N = 65536  (4, 8) 29.9 / 31.8 / 37.5  (4, 4) 31.0 / 34.4 / 41.3  (8, 4) 31.8 / 34.7 / 47.5
  //   Q6_K 4096x14336 (8, 1) 14.5 / 16.0 / 19.3, (4, 2) 22.5 / 22.7 / 26.0; 14336x4096 (8, 4) 14.6 / 14.7 / 16.9, (4, 2)
  //   14.7 / 15.2 / 17.3
  //   GLU 2 x 14336 (4, 4) 15.6 / 17.4 / 21.0, (4, 2) 16.7 / 19.3 / 23.3; 2 x 8960x3072 (4, 2) 10.6 / 11.8 / 14.7, (4, 4)
  //   11.5 / 12.8 / 15.9; Q6_K 2 x 11008 (4, 2) 19.1 / 20.3 / 23.9, (4, 4) 22.2 / 23.1 / 26.5
  // and at 3 / 16 rows, K = 4096, the types that take 16 rows:
  //   Q8_0 N = 8192 (4, 2) 9.1 / 9.5, (8, 2) 9.6 / 9.9; Q4_0 (8, 2) 7.6 / 8.0, (4, 2) 8.4 / 8.5; Q5_0 (8, 2) 9.1 / 9.4, (4, 2)
  //   9.8 / 9.6; Q5_K (4, 2) 8.9 / 8.7, (8, 2) 9.0 / 9.4; N = 14336 Q8_0 (8, 4) 14.2 / 14.7, (4, 4) 13.9 / 14.9, (4, 6)
  //   34 / 34, Q4_0 (8, 4) 10.4 / 10.7, (4, 4) 12.6 / 12.0; N = 32768 Q8_0 (4, 4) 27.1 / 28.4, (8, 4) 28.8 / 29.8, (4, 6)
  //   41.5 / 42.1, Q5_K (4, 4) 22.4 / 22.8, (8, 4) 22.2 / 24.4, (4, 6) 29 / 30 (more tiles spill)
  // (the 32x32x32 and 16x16x64 kernels with register-loaded operands before this one: N = 14336 14.5 / 17.0 / 18.5, N =
  // 4096 5.5 / 6.7 / 9.3, Q6_K 4096x14336 22.9 / 26.1 / 31.4, GLU 2 x 14336 28.3 / 33.5 / 37.0)
  if (w2) {
    if (WT::kBytes == 144 && tiles > 3 * cus)
      QMM_L(4, 4, true);
    else
      QMM_L(4, 2, true);
  } else if (tiles <= cus) {
    QMM_L(8, 1, false);
  } else if (tiles <= 2 * cus) {
    if constexpr (WT::kB32 && WT::kBytes < 272)
      QMM_L(8, 2, false);
    else
      QMM_L(4, 2, false);
  } else if (tiles <= 4 * cus) {
    QMM_L(8, 4, false);
  } else if constexpr (WT::kB32 || WT::kRows == 16) {
    QMM_L(4, 4, false);
  } else if (tiles <= 6 * cus) {
    QMM_L(4, 6, false);
  } else {
    QMM_L(4, 8, false);
  }
#undef QMM_L
}

template <class WT, class Out>
void launch_decode(const void *vx, const void *vx2, const act_rows &ap, void *dst, int ncols_x, int nrows_x,
                   int stride_col_dst, int b, int activation, hipStream_t s) {
  const int64_t nsb = ncols_x / 256, wrb = nsb * WT::kBytes;
  if constexpr (WT::kRows > 16) {
    if (b > 16) return launch_mt<WT, Out, 2>(vx, vx2, nrows_x, wrb, ap, b, nsb, dst, stride_col_dst, activation, s);
  }
  launch_mt<WT, Out, 1>(vx, vx2, nrows_x, wrb, ap, b, nsb, dst, stride_col_dst, activation, s);
}

template <class WT>
bool dispatch_out(int out_type, const void *vx, const void *vx2, const act_rows &ap, void *dst, int ncols_x, int nrows_x,
                  int stride_col_dst, int b, int activation, hipStream_t s) {
  // a workgroup's rows (128 at most) are addressed with 31 bits
  if (b > WT::kRows || 128 * ((int64_t)ncols_x / 256 * WT::kBytes + 16) > 0x7ffffff0) return false;
  switch (out_type) {
    case QMM_TYPE_F16:
      launch_decode<WT, out_f16>(vx, vx2, ap, dst, ncols_x, nrows_x, stride_col_dst, b, activation, s);
      break;
    case QMM_TYPE_BF16:
      launch_decode<WT, out_bf16>(vx, vx2, ap, dst, ncols_x, nrows_x, stride_col_dst, b, activation, s);
      break;
    default: launch_decode<WT, out_f32>(vx, vx2, ap, dst, ncols_x, nrows_x, stride_col_dst, b, activation, s);
  }
  return true;
}

#define QMM_SK(WT) \
  return dispatch_out<WT>(out_type, vx, vx2, ap, dst, ncols_x, nrows_x, stride_col_dst, b, activation, s)
bool dispatch_kq(int type, int out_type, const void *vx, const void *vx2, const act_rows &ap, void *dst, int ncols_x,
                 int nrows_x, int stride_col_dst, int b, int activation, hipStream_t s) {
  switch (type) {
    case QMM_TYPE_Q4K: QMM_SK(wq4k16);
    case QMM_TYPE_Q5K: QMM_SK(wq5k16);
    case QMM_TYPE_Q6K: QMM_SK(wq6k16);
    default: return false;
  }
}
bool dispatch_b32(int type, int out_type, const void *vx, const void *vx2, const act_rows &ap, void *dst, int ncols_x,
                  int nrows_x, int stride_col_dst, int b, int activation, hipStream_t s) {
  switch (type) {
    case QMM_TYPE_Q8_0: QMM_SK(wb16_q8_0);
    case QMM_TYPE_Q4_0: QMM_SK(wb16_q4_0);
    case QMM_TYPE_Q5_0: QMM_SK(wb16_q5_0);
    default: return false;
  }
}
#undef QMM_SK

// Q8_1 slots (units.h): rows of 288-byte slots {f32 d; int8 qs[256]; int16 s32[8]; pad}
bool slot_rows(const void *vy, int ncols_x, int stride_col_y, int b, act_rows &ap) {
  if (b < 1 || b > 32 || ncols_x % 256 != 0 || stride_col_y % 8 != 0 || (int64_t)b * stride_col_y * 36 > 0x7ffffff0)
    return false;
  const uint32_t rb = (uint32_t)stride_col_y * 36;
  ap = {(const uint8_t *)vy, (int64_t)b * rb, 4, rb, 288, 0, rb, 288};
  return true;
}

}  // namespace

bool qmm_skinny_decode(int type, int out_type, const void *vx, const void *vy, void *dst, int ncols_x, int nrows_x,
                       int stride_col_y, int stride_col_dst, int b, hipStream_t s) {
  act_rows ap;
  return slot_rows(vy, ncols_x, stride_col_y, b, ap) &&
         dispatch_kq(type, out_type, vx, nullptr, ap, dst, ncols_x, nrows_x, stride_col_dst, b, 0, s);
}

bool qmm_skinny_glu(int type, int out_type, const void *vx_gate, const void *vx_up, const void *vy, void *dst,
                    int ncols_x, int nrows_x, int stride_col_y, int stride_col_dst, int b, int activation,
                    hipStream_t s) {
  act_rows ap;
  return slot_rows(vy, ncols_x, stride_col_y, b, ap) &&
         dispatch_kq(type, out_type, vx_gate, vx_up, ap, dst, ncols_x, nrows_x, stride_col_dst, b, activation, s);
}

bool qmm_skinny_b32(int type, int out_type, const void *vx, const void *vx2, const void *vy, void *dst, int ncols_x,
                    int nrows_x, int stride_col_y, int stride_col_dst, int b, int activation, hipStream_t s) {
  // whole superblocks of eight blocks, and rows that start on dwords
  if (b < 1 || ncols_x % 256 != 0 || stride_col_y % 2 != 0 || ((uintptr_t)vx | (uintptr_t)vx2 | (uintptr_t)vy) % 4 != 0 ||
      (int64_t)b * stride_col_y * 34 > 0x7ffffff0)
    return false;
  const uint32_t rb = (uint32_t)stride_col_y * 34;
  const act_rows ap{(const uint8_t *)vy, (int64_t)b * rb, 0, rb, 272, 0, 0, 0};
  return dispatch_b32(type, out_type, vx, vx2, ap, dst, ncols_x, nrows_x, stride_col_dst, b, activation, s);
}

// rows of K / 256 blocks of 260 bytes {f32 d; int8 qs[256]}
bool qmm_skinny_tc(int type, int out_type, const void *vx, const void *vy, void *dst, int ncols_x, int nrows_x,
                   int stride_col_dst, int b, hipStream_t s) {
  const int64_t rb = (int64_t)(ncols_x / 256) * 260;
  if (b < 1 || b > 32 || ncols_x % 256 != 0 || b * rb > 0x7ffffff0) return false;
  const act_rows ap{(const uint8_t *)vy, b * rb, 4, (uint32_t)rb, 260, 0, (uint32_t)rb, 260};
  return dispatch_kq(type, out_type, vx, nullptr, ap, dst, ncols_x, nrows_x, stride_col_dst, b, 0, s);
}

// Prefill tiles of one channel: qs[nsb][rows][256] int8, then d[nsb][rows] f32
static bool moe_rows(int64_t ncols_x, int64_t w_row_bytes, const void *y, int64_t ncols_dst, int64_t num_experts,
                     act_rows &ap) {
  if (ncols_x % 256 != 0 || ncols_dst <= 0 || num_experts <= 0 || num_experts > 65535) return false;
  if (ncols_dst > QMM_SKINNY_MOE_ROWS * num_experts) return false;
  const int64_t nsb = ncols_x / 256;
  if (nsb * ncols_dst * 276 > 0x7ffffff0 || 128 * (w_row_bytes + 16) > 0x7ffffff0) return false;
  ap = {(const uint8_t *)y, nsb * ncols_dst * 260, 0, 256, (uint32_t)(256 * ncols_dst),
        (uint32_t)(nsb * ncols_dst * 256), 4, (uint32_t)(4 * ncols_dst)};
  return true;
}

template <class WT, int TC, bool GLU>
static void launch_moe(const void *x, const void *x2, const act_rows &ap, const int32_t *ids_dst, const int32_t *bounds,
                       float *dst, int64_t nsb, int64_t nrows_x, int64_t w_row_bytes, int64_t ncols_dst, int64_t ldd,
                       int64_t num_experts, int activation, hipStream_t s) {
  // enough 32-row passes for an expert of average size; larger experts loop over theirs
  const unsigned chunks = (unsigned)qmm_ceil_div(qmm_ceil_div(ncols_dst, num_experts), 32);
  const unsigned cols = 16 * (GLU ? TC / 2 : TC);
  k_rows_moe<WT, 4, TC, 2, 2, GLU>
      <<<dim3((unsigned)qmm_ceil_div(nrows_x, cols), chunks, (unsigned)num_experts), 256, 0, s>>>(
          (const uint8_t *)x, (const uint8_t *)x2, nrows_x * w_row_bytes, nrows_x, w_row_bytes, ap, bounds, ids_dst,
          (int)nsb, dst, ldd, activation);
}

bool qmm_skinny_moe(int type, const void *x, const void *y, const int32_t *ids_dst, const int32_t *bounds, float *dst,
                    int64_t ncols_x, int64_t nrows_x, int64_t w_row_bytes, int64_t ncols_dst, int64_t ldd,
                    int64_t num_experts, hipStream_t s) {
  act_rows ap;
  if (!moe_rows(ncols_x, w_row_bytes, y, ncols_dst, num_experts, ap)) return false;
  // (4 waves, 4 tiles; MI355X, 8 x Q4_K experts of 4096x14336 at 4 / 16 / 32 rows each on average: 41 / 52 / 78 us, 5.1
  // TB/s of weights at 16 rows; 2 tiles 45 / 52 / 77, 8 tiles 45 / 60 / 100)
  if (type == QMM_TYPE_Q4K)
    launch_moe<wq4k16, 4, false>(x, nullptr, ap, ids_dst, bounds, dst, ncols_x / 256, nrows_x, w_row_bytes, ncols_dst,
                                 ldd, num_experts, 0, s);
  else if (type == QMM_TYPE_Q6K)
    launch_moe<wq6k16, 4, false>(x, nullptr, ap, ids_dst, bounds, dst, ncols_x / 256, nrows_x, w_row_bytes, ncols_dst,
                                 ldd, num_experts, 0, s);
  else
    return false;
  return true;
}

bool qmm_skinny_moe_glu(int type, const void *gate, const void *up, const void *y, const int32_t *bounds, float *dst,
                        int64_t ncols_x, int64_t nrows_x, int64_t w_row_bytes, int64_t ncols_dst, int64_t ldd,
                        int64_t num_experts, int activation, hipStream_t s) {
  act_rows ap;
  if (!moe_rows(ncols_x, w_row_bytes, y, ncols_dst, num_experts, ap)) return false;
  // (4 waves; 2 x 8 Q4_K experts of 14336x4096 at 4 / 16 / 32 rows each on average: 4 gate and 4 up tiles 92 / 109 / 160
  // us, 4.8 TB/s of weights at 16 rows; 2 and 2 tiles 88 / 118 / 161; gate and up as two launches 2 x 53 / 65 / 92)
  const bool few = ncols_dst <= 8 * num_experts;
#define QMM_M(WT, TC)                                                                                               \
  launch_moe<WT, TC, true>(gate, up, ap, nullptr, bounds, dst, ncols_x / 256, nrows_x, w_row_bytes, ncols_dst, ldd, \
                           num_experts, activation, s)
  if (type == QMM_TYPE_Q4K && few)
    QMM_M(wq4k16, 4);
  else if (type == QMM_TYPE_Q4K)
    QMM_M(wq4k16, 8);
  else if (type == QMM_TYPE_Q6K)
    QMM_M(wq6k16, 4);
  else
    return false;
#undef QMM_M
  return true;
}
