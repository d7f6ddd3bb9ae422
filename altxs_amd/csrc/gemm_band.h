// Row-band GEMM for launches with many rows (encode windows, chunk scoring,
// batched products) on tensors with K = 256 or 512.
//
// A workgroup of four waves keeps a band of 16*MB rows of A (bf16 or fp16) in
// LDS for the whole launch and walks column tiles ct = cx, cx + gridDim.x, ...;
// each wave owns 16*NBW columns of a tile and applies every weight operand to
// the band's MB row blocks.  The stages with a prologue (QKV, MLP up, LM head)
// normalise the band's rows themselves, with the 16-row tasks' arithmetic.
//
// The MFMA operands are swapped against gemm_task: the weights are the A
// operand and the activations the B operand, so D is the output's transpose
// (the same products in the same order: v_mfma_f32_16x16x32 gives the same
// bits for A x B and (B^T x A^T)^T) and lane l holds row l % 16 and four
// consecutive columns 4 (l / 16) .. +3 of a 16 x 16 block.  Every epilogue
// therefore works on whole 16-byte runs of a row straight from the
// accumulators: no strip through LDS, no barrier after the band is staged, so
// one wave's epilogue runs under the other waves' MFMAs.
//
// Bit-identical to gemm_task for the same K-split: every 16 x 16 block sees its
// MFMA sequence (k-steps in order, two per group from zero, acc += scale * t,
// each K-slice of K/KS from zero, slices added in order).
#pragma once
#include "gemm.h"

namespace altxs {

// Loads of 16 bytes at 8-byte aligned addresses (group scales).
typedef u32x4 __attribute__((aligned(8))) u32x4_a8;

// Epilogues with a per-band LDS table (kBandLds(): bytes per row) fill it in
// band_setup(); others have none.
template <class E, class = void> struct epi_band_lds : std::false_type {};
template <class E>
struct epi_band_lds<E, std::void_t<decltype(&E::band_lds_per_row)>> : std::true_type {};
// Epilogues that take some column tiles unswapped (lane l: column l % 16, rows
// 4 (l / 16) .. +3) say which.
template <class E, class = void> struct epi_has_unswapped : std::false_type {};
template <class E>
struct epi_has_unswapped<E, std::void_t<decltype(&E::unswapped)>> : std::true_type {};

template <int K, int MB>
__host__ __device__ constexpr size_t band_a_bytes() { return (size_t)16 * MB * (K + 8) * 2; }

// Group-scaled accumulation of one 16 x 16 block: acc += scale * t, one FMA per element.
__device__ __forceinline__ void fma4(f32x4& acc, const float (&s)[4], const f32x4& t) {
#pragma unroll
  for (int i = 0; i < 4; ++i) acc[i] = __builtin_fmaf(s[i], t[i], acc[i]);
}

template <int BITS, int K, int MB, int NBW, int KS, class Epi, int AM, class Pro>
__global__ __launch_bounds__(256, 2) void gemm_band_kernel(QT w, int R, const uint16_t* __restrict__ A, Epi epi,
                                                           int64_t codes_stride, int64_t scales_stride, Pro pro) {
  static_assert(AM == A_BF16 || AM == A_F16, "16-bit A rows");
  static_assert(K == 256 || K == 512, "band widths");
  constexpr int KB = K / 256, KBS = KB / KS, GPT = K / 64, AST = K + 8;
  static_assert(KB % KS == 0, "K-slices of the band");
  constexpr bool EXP = BITS == kExpBits;
  static_assert(!EXP || AM == A_BF16, "expanded codes are bf16 values");
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  uint16_t* As = (uint16_t*)smem;
  unsigned char* elds = smem + band_a_bytes<K, MB>();
  const int batch = blockIdx.z;
  w.codes += batch * codes_stride;
  w.scales += batch * scales_stride;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, lg = lane >> 4, col = lane & 15;
  // Workgroups are dealt to the 8 XCDs round-robin by linear id: every column
  // group of a row band runs on one XCD, consecutively, so the band enters
  // that XCD's L2 once.
  int cx = blockIdx.x, ry = blockIdx.y;
  if (gridDim.y % 8 == 0) {
    const int bid = blockIdx.x + gridDim.x * blockIdx.y;
    const int j = bid / 8;
    ry = bid % 8 + 8 * (j / gridDim.x);
    cx = j % gridDim.x;
  }
  constexpr int TCOL = 64 * NBW;  // columns of a workgroup's tile
  const int m0 = ry * 16 * MB, NT = (w.N + TCOL - 1) / TCOL, GX = gridDim.x;
  auto nblk = [&](int ct) { return ct * (TCOL / 16) + NBW * wave; };  // this wave's first 16-column block

  // Weight operands.  Expanded codes stream from memory PF groups ahead
  // through a ring of register slots (group q in slot q % NSLOT), across tile
  // boundaries; packed codes of the next tile load behind this one's last use.
  constexpr int NSLOT = NBW == 4 ? 2 : 4, PF = NSLOT - 1;
  static_assert(GPT % NSLOT == 0, "ring slots are compile-time indices");
  using WBlk = Blk<EXP ? 4 : BITS, A_BF16, false>;
  u32x4 eb[EXP ? NSLOT : 1][NBW][2];
  WBlk wt[EXP ? 1 : KB][EXP ? 1 : NBW];
  auto load_grp = [&](int slot, int nb, int q) {
    if constexpr (EXP) {
      const int kb = q / 4, g = q % 4;
#pragma unroll
      for (int j = 0; j < NBW; ++j) {
        const u32x4* p = (const u32x4*)(w.codes + ((size_t)(nb + j) * KB + kb) * 8192) + lane;
        eb[slot][j][0] = p[64 * (2 * g)];
        eb[slot][j][1] = p[64 * (2 * g + 1)];
      }
    }
  };
  auto load_packed = [&](int nb, int kb) {
    if constexpr (!EXP) {
#pragma unroll
      for (int j = 0; j < NBW; ++j) load_w(wt[kb][j], w, nb + j, kb, lane);
    }
  };
  auto valid = [&](int ct) { return ct < NT && nblk(ct) * 16 < w.N; };  // N % (16 NBW) == 0 (host)
  if (valid(cx)) {
#pragma unroll
    for (int q = 0; q < PF; ++q) load_grp(q, nblk(cx), q);
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) load_packed(nblk(cx), kb);
  }

  if constexpr (epi_band_lds<Epi>::value) epi.template band_setup<16 * MB>(elds, m0, R);
  if constexpr (Pro::kStage) {
    static_assert(Pro::kScratch == 0, "no prologue scratch in the band's LDS");
    static_assert(AST == lds_stride(K, A_BF16), "stage() row stride");
    pro.template stage_band<AM, MB>(As, m0, R, K, cx == 0);
  } else {
    // one wave instruction moves a whole K = 512 row (lane l: k = 8 l .. +7),
    // or two K = 256 rows, by global->LDS DMA
    constexpr int RPI = 512 / K;
    if constexpr (RPI == 1) {
#pragma unroll 4
      for (int i = 0; i < 4 * MB; ++i) {
        const int r = wave * (4 * MB) + i;
        if (m0 + r < R)
          __builtin_amdgcn_global_load_lds(
              (const __attribute__((address_space(1))) void*)(A + (int64_t)(m0 + r) * K + lane * 8),
              (__attribute__((address_space(3))) void*)(As + r * AST), 16, 0, 0);
      }
      __builtin_amdgcn_s_waitcnt(0);
    } else {
#pragma unroll 4
      for (int i = 0; i < 2 * MB; ++i) {
        const int r = wave * (4 * MB) + 2 * i + (lane >> 5);
        if (m0 + r < R)
          *(u32x4*)(As + r * AST + (lane & 31) * 8) = *(const u32x4*)(A + (int64_t)(m0 + r) * K + (lane & 31) * 8);
      }
    }
  }
  __syncthreads();

  using Op = std::conditional_t<AM == A_F16, f16x8, bf16x8>;
  auto mfma = [](Op a, Op b, f32x4 c) {
    if constexpr (AM == A_F16) return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
    else return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  };
  for (int ct = cx; ct < NT; ct += GX) {
    if (!valid(ct)) break;
    const int nb = nblk(ct);
    const int nbn = valid(ct + GX) ? nblk(ct + GX) : nb;  // the last tile re-reads its own first groups
    const FragAt at{m0, nb * 16, R, lane, batch, elds};
    // this lane's first A operand; opaque, or the compiler keeps the whole band
    // (loop-invariant LDS reads) in registers and spills
    int aoff = col * AST + 8 * lg;
    asm volatile("" : "+v"(aoff));
    const auto pre = epi.template frag_prefetch<NBW, MB>(at);
    f32x4 acc[NBW][MB], tot[KS > 1 ? NBW : 1][KS > 1 ? MB : 1];
#pragma unroll
    for (int j = 0; j < NBW; ++j)
#pragma unroll
      for (int m = 0; m < MB; ++m) acc[j][m] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto kloop = [&](auto swapped) {
      constexpr bool SW = decltype(swapped)::value;
      // swapped: a lane's four columns' scales of the k-block's four groups
      // (half 4 i + g); unswapped: its one column's (half g)
      constexpr int SCW = SW ? 8 : 2;
      uint32_t sc[NBW][SCW];
      auto load_sc = [&](int kb) {
#pragma unroll
        for (int j = 0; j < NBW; ++j) {
          const uint16_t* p = w.scales + ((size_t)(nb + j) * KB + kb) * 64;
          if constexpr (SW) {
            const u32x4 x = *(const u32x4_a8*)(p + 16 * lg), y = *(const u32x4_a8*)(p + 16 * lg + 8);
#pragma unroll
            for (int i = 0; i < 4; ++i) { sc[j][i] = x[i]; sc[j][4 + i] = y[i]; }
          } else {
            const u32x2 x = *(const u32x2*)(p + 4 * col);
            sc[j][0] = x[0]; sc[j][1] = x[1];
          }
        }
      };
#pragma unroll
      for (int q = 0; q < GPT; ++q) {
        const int kb = q / 4, g = q % 4;
        if (g == 0) load_sc(kb);
        Op wo[NBW][2];
        if constexpr (EXP) {
          const int qn = q + PF;
          if (qn < GPT) load_grp(qn % NSLOT, nb, qn);
          else load_grp(qn % NSLOT, nbn, qn - GPT);
#pragma unroll
          for (int j = 0; j < NBW; ++j)
#pragma unroll
            for (int ss = 0; ss < 2; ++ss) wo[j][ss] = __builtin_bit_cast(Op, eb[q % NSLOT][j][ss]);
        } else {
#pragma unroll
          for (int j = 0; j < NBW; ++j)
#pragma unroll
            for (int ss = 0; ss < 2; ++ss) {
              if constexpr (AM == A_F16) wo[j][ss] = b_op_f16<BITS>(wt[kb][j].p0, wt[kb][j].p1, 2 * g + ss, BITS);
              else wo[j][ss] = b_op_bf16<BITS>(wt[kb][j].p0, wt[kb][j].p1, 2 * g + ss, BITS);
            }
        }
#pragma unroll
        for (int m = 0; m < MB; ++m) {
          const uint16_t* ap = As + aoff + 16 * m * AST + 64 * q;
          const Op a0 = __builtin_bit_cast(Op, *(const u32x4*)ap);
          const Op a1 = __builtin_bit_cast(Op, *(const u32x4*)(ap + 32));
          f32x4 t[NBW];
#pragma unroll
          for (int j = 0; j < NBW; ++j)
            t[j] = SW ? mfma(wo[j][0], a0, f32x4{0.f, 0.f, 0.f, 0.f}) : mfma(a0, wo[j][0], f32x4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
          for (int j = 0; j < NBW; ++j) t[j] = SW ? mfma(wo[j][1], a1, t[j]) : mfma(a1, wo[j][1], t[j]);
#pragma unroll
          for (int j = 0; j < NBW; ++j) {
            float s[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const int h = SW ? 4 * i + g : g;
              const uint32_t v = sc[j][h >> 1];
              s[i] = (h & 1) ? half_hi(v) : half_lo(v);
            }
            fma4(acc[j][m], s, t[j]);
          }
        }
        if (KS > 1 && g == 3 && (kb + 1) % KBS == 0) {  // end of a K-slice: slices added in order
          const bool first = kb + 1 == KBS;
#pragma unroll
          for (int j = 0; j < NBW; ++j)
#pragma unroll
            for (int m = 0; m < MB; ++m) {
              f32x4& o = tot[KS > 1 ? j : 0][KS > 1 ? m : 0];
#pragma unroll
              for (int i = 0; i < 4; ++i) o[i] = first ? acc[j][m][i] : o[i] + acc[j][m][i];
              acc[j][m] = f32x4{0.f, 0.f, 0.f, 0.f};
            }
        }
        if (!EXP && g == 3) load_packed(nbn, kb);
        // groups stay apart: moved up, the loads of all of them at once would spill
        __builtin_amdgcn_sched_barrier(0);
      }
      // the results exist here: an epilogue that stores them under a row
      // bound would otherwise draw the products into its branches
#pragma unroll
      for (int j = 0; j < NBW; ++j)
#pragma unroll
        for (int m = 0; m < MB; ++m) {
          if constexpr (KS > 1) asm volatile("" : "+v"(tot[j][m]));
          else asm volatile("" : "+v"(acc[j][m]));
        }
    };
    bool plain = true;
    if constexpr (epi_has_unswapped<Epi>::value) {
      if (epi.unswapped(nb * 16)) {  // uniform
        kloop(std::false_type{});
        epi.template frag_unswapped<NBW, MB>(acc, at);
        plain = false;
      }
    }
    if (plain) {
      kloop(std::true_type{});
      if constexpr (KS > 1) epi.template frag<NBW, MB>(tot, pre, at);
      else epi.template frag<NBW, MB>(acc, pre, at);
    }
  }
}

// Column groups per row band: about `want` workgroups in all, at most one per column tile.
inline int band_col_groups(int64_t bands, int nt, int want) {
  const int64_t g = (want + bands - 1) / bands;
  return g < 1 ? 1 : (g > nt ? nt : (int)g);
}

template <int BITS, int K, int MB, int NBW, int KS, class Epi, int AM, class Pro>
hipError_t launch_gemm_band_m(const QT& w, int R, const uint16_t* A, const Epi& epi, hipStream_t s, int batch,
                              int64_t codes_stride, int64_t scales_stride, const Pro& pro) {
  auto kfn = gemm_band_kernel<BITS, K, MB, NBW, KS, Epi, AM, Pro>;
  size_t lds = band_a_bytes<K, MB>();
  if constexpr (epi_band_lds<Epi>::value) lds += (size_t)16 * MB * epi.band_lds_per_row();
  static size_t configured = 0;
  if (lds > 65536 && lds > configured) {
    hipError_t e = hipFuncSetAttribute((const void*)kfn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
    configured = lds;
  }
  const int bands = (R + 16 * MB - 1) / (16 * MB), nt = (w.N + 64 * NBW - 1) / (64 * NBW);
  const dim3 grid((unsigned)band_col_groups((int64_t)bands * batch, nt, 1024), (unsigned)bands, (unsigned)batch);
  hipLaunchKernelGGL(kfn, grid, dim3(256), lds, s, w, R, A, epi, codes_stride, scales_stride, pro);
  return hipGetLastError();
}

// Rows from which bands are 64 rows high (below: 32, which gives a small launch
// twice the workgroups and half the rows to stage before its first MFMA).
constexpr int kBandTallRows = 4096;

template <int BITS, int K, int KS, class Epi, int AM, class Pro>
hipError_t launch_gemm_band_k(const QT& w, int R, const uint16_t* A, const Epi& epi, hipStream_t s, int batch,
                              int64_t codes_stride, int64_t scales_stride, const Pro& pro) {
  constexpr int NBW = Epi::kFragBlocks;
  if ((int64_t)R * batch >= kBandTallRows)
    return launch_gemm_band_m<BITS, K, 4, NBW, KS, Epi, AM, Pro>(w, R, A, epi, s, batch, codes_stride, scales_stride, pro);
  return launch_gemm_band_m<BITS, K, 2, NBW, KS, Epi, AM, Pro>(w, R, A, epi, s, batch, codes_stride, scales_stride, pro);
}

// Shapes the row-band kernel takes.
inline bool band_fits(const QT& w) {
  return (w.bits <= 6 || w.bits == kExpBits) && w.N % 64 == 0 && (w.K == 256 || w.K == 512);
}

// KS: the 16-row path's K-split of the tensor (pick_ks; K = 256 allows one slice).
template <int BITS, int KS, class Epi, int AM = A_BF16, class Pro = ProNone>
hipError_t launch_gemm_band_t(const QT& w, int R, const uint16_t* A, const Epi& epi, hipStream_t s, int batch = 1,
                              int64_t codes_stride = 0, int64_t scales_stride = 0, const Pro& pro = Pro{}) {
  // A rows come by 16-byte DMA: 16-byte aligned rows only
  if (!band_fits(w) || ((uintptr_t)A & 15) != 0) return hipErrorInvalidValue;
  if (w.K == 512)
    return launch_gemm_band_k<BITS, 512, KS, Epi, AM, Pro>(w, R, A, epi, s, batch, codes_stride, scales_stride, pro);
  if constexpr (KS == 1)
    return launch_gemm_band_k<BITS, 256, 1, Epi, AM, Pro>(w, R, A, epi, s, batch, codes_stride, scales_stride, pro);
  return hipErrorInvalidValue;
}

template <int KS, class Pro, class Epi>
hipError_t launch_gemm_band(int bits, const QT& w, int R, const uint16_t* A, const Pro& pro, const Epi& epi,
                            hipStream_t s) {
  switch (bits) {
    case 2: return launch_gemm_band_t<2, KS, Epi, A_BF16, Pro>(w, R, A, epi, s, 1, 0, 0, pro);
    case 3: return launch_gemm_band_t<3, KS, Epi, A_BF16, Pro>(w, R, A, epi, s, 1, 0, 0, pro);
    case 4: return launch_gemm_band_t<4, KS, Epi, A_BF16, Pro>(w, R, A, epi, s, 1, 0, 0, pro);
    case 6: return launch_gemm_band_t<6, KS, Epi, A_BF16, Pro>(w, R, A, epi, s, 1, 0, 0, pro);
    case kExpBits: return launch_gemm_band_t<kExpBits, KS, Epi, A_BF16, Pro>(w, R, A, epi, s, 1, 0, 0, pro);
    default: return hipErrorInvalidValue;
  }
}
// ks_max: the stage's preferred K-split (pick_ks).
template <class Pro, class Epi>
hipError_t launch_gemm_band4(int ks_max, int bits, const QT& w, int R, const uint16_t* A, const Pro& pro,
                             const Epi& epi, hipStream_t s) {
  switch (pick_ks(w.K, ks_max)) {
    case 2: return launch_gemm_band<2>(bits, w, R, A, pro, epi, s);
    case 1: return launch_gemm_band<1>(bits, w, R, A, pro, epi, s);
    default: return hipErrorInvalidValue;  // K <= 512 allows at most two K-slices
  }
}

}  // namespace altxs
