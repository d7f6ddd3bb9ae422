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

// Epilogues with a per-band LDS table (band_lds(rows) bytes) fill it in
// band_setup(); others have none.
template <class E, class = void> struct epi_band_lds : std::false_type {};
template <class E>
struct epi_band_lds<E, std::void_t<decltype(&E::band_lds)>> : std::true_type {};
// Epilogues that take some column tiles unswapped (lane l: column l % 16, rows
// 4 (l / 16) .. +3) say which.
template <class E, class = void> struct epi_has_unswapped : std::false_type {};
template <class E>
struct epi_has_unswapped<E, std::void_t<decltype(&E::unswapped)>> : std::true_type {};

// Epilogues of stages whose weights are never expanded say so.
template <class E, class = void> struct epi_packed_only : std::false_type {};
template <class E>
struct epi_packed_only<E, std::void_t<decltype(&E::kPackedOnly)>> : std::true_type {};

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
  constexpr bool EXP = BITS == kExpBits, DENSE = BITS == 16;
  static_assert(!(EXP || DENSE) || AM == A_BF16, "expanded codes and dense weights are bf16 values");
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  uint16_t* As = (uint16_t*)smem;
  unsigned char* elds = smem + band_a_bytes<K, MB>();
  const int batch = blockIdx.z;
  w.codes += batch * codes_stride;
  w.scales += batch * scales_stride;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, lg = lane >> 4, col = lane & 15;
  // Workgroups are dealt to the 8 XCDs round-robin by linear id: every column
  // group of a row band runs on one XCD, consecutively, so the band enters
  // that XCD's L2 once.
  const int bid = blockIdx.x + gridDim.x * blockIdx.y;
  int cx = blockIdx.x, ry = blockIdx.y;
  if (gridDim.y % 8 == 0) {
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
  // What bounds the forms with NBW = 4 (QKV, LM head) is registers: accumulators,
  // products, scales and operands take 144 of 256 in a band of 64 rows.  There a
  // packed tile's k-blocks pass through one set of registers (with both at once up
  // to 250 spilled; steps of 4 layers with 3-bit QKV, K = 512: 1024 rows 381 -> 371
  // us, 32768 rows 4577 -> 4318), and dense values, 32 registers a k-block, come
  // half a block at a time where they are used (a lane's 128 bytes are one line;
  // dense student, 8192 rows: 3735 -> 3459 us).
  constexpr bool HALF = DENSE && NBW == 4;
  constexpr int NWT = EXP || DENSE || NBW == 4 ? 1 : KB;
  WBlk wt[NWT][EXP || HALF ? 1 : NBW];
  u32x4 dh[HALF ? NBW : 1][4];  // dense: groups 2 q', 2 q' + 1
  auto load_half = [&](int nb, int q) {
    if constexpr (HALF) {
#pragma unroll
      for (int j = 0; j < NBW; ++j) {
        const u32x4* p = (const u32x4*)(w.codes + ((size_t)(nb + j) * KB + q / 4) * 8192) + 8 * lane + 2 * (q % 4);
#pragma unroll
        for (int i = 0; i < 4; ++i) dh[j][i] = p[i];
      }
    }
  };
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
    if constexpr (!EXP && !HALF) {
#pragma unroll
      for (int j = 0; j < NBW; ++j) load_w(wt[kb % NWT][j], w, nb + j, kb, lane);
    }
  };
  // This workgroup's column tiles cx, cx + GX, ..., from a start of its own:
  // workgroups in step would all write the same columns of their rows at once,
  // addresses a row apart, which are few channels of L2 and memory.
  const int nk = (NT - cx + GX - 1) / GX, rot = (bid / 8) % nk;
  auto tile = [&](int k) { return cx + GX * (k + rot < nk ? k + rot : k + rot - nk); };
  auto valid = [&](int k) { return k < nk && nblk(tile(k)) * 16 < w.N; };  // N % (16 NBW) == 0 (host)
  {
    const int nb = valid(0) ? nblk(tile(0)) : 0;
#pragma unroll
    for (int q = 0; q < PF; ++q) load_grp(q, nb, q);
    if constexpr (!DENSE) {
#pragma unroll
      for (int kb = 0; kb < NWT; ++kb) load_packed(nb, kb);
    }
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
  for (int k = 0; k < nk; ++k) {
    const int nb = valid(k) ? nblk(tile(k)) : 0;
    const int nbn = valid(k + 1) ? nblk(tile(k + 1)) : 0;  // (nothing more: block 0's first groups, unused)
    if (!valid(k)) {
#pragma unroll
      for (int q = 0; q < PF; ++q) load_grp(q, nbn, q);
      if constexpr (!DENSE) {
#pragma unroll
        for (int kb = 0; kb < NWT; ++kb) load_packed(nbn, kb);
      }
      continue;
    }
    // Opaque per tile: this lane's first A operand (or the compiler keeps the
    // whole band, loop-invariant LDS reads, in registers) and the epilogue's
    // lane and row (or it keeps every tile's addresses); either spills.
    int aoff = col * AST + 8 * lg, fl = lane, fm = m0;
    asm volatile("" : "+v"(aoff), "+v"(fl), "+v"(fm));
    fm = __builtin_amdgcn_readfirstlane(fm);
    const FragAt at{fm, nb * 16, R, fl, batch, elds};
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
        if (HALF && g % 2 == 0) load_half(nb, q);
        if (g == 0) {
          if constexpr (DENSE) load_packed(nb, kb);
          else load_sc(kb);
          if constexpr (!EXP && !DENSE) {
            // opaque: decoding that both forms of the loop share would otherwise move
            // above their branch, a tile's worth of it, and spill
#pragma unroll
            for (int j = 0; j < NBW; ++j) {
#pragma unroll
              for (uint32_t& x : wt[kb % NWT][j].p0) asm volatile("" : "+v"(x));
              if constexpr (Planes<BITS>::P1 > 0) {
#pragma unroll
                for (uint32_t& x : wt[kb % NWT][j].p1) asm volatile("" : "+v"(x));
              }
            }
          }
        }
        Op wo[NBW][2];
        if constexpr (HALF) {
#pragma unroll
          for (int j = 0; j < NBW; ++j)
#pragma unroll
            for (int ss = 0; ss < 2; ++ss) wo[j][ss] = __builtin_bit_cast(Op, dh[j][2 * (g % 2) + ss]);
        } else if constexpr (EXP) {
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
              if constexpr (AM == A_F16) wo[j][ss] = b_op_f16<BITS>(wt[kb % NWT][j].p0, wt[kb % NWT][j].p1, 2 * g + ss, BITS);
              else wo[j][ss] = b_op_bf16<BITS>(wt[kb % NWT][j].p0, wt[kb % NWT][j].p1, 2 * g + ss, BITS);
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
              s[i] = DENSE ? 1.f : (h & 1) ? half_hi(v) : half_lo(v);  // dense: acc += t
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
        if (!EXP && !DENSE && g == 3) {  // the next k-block into these registers: this tile's, or the next tile's
          const int kn = kb + NWT;
          load_packed(kn < KB ? nb : nbn, kn % KB);
        }
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

// Column groups per row band: about `want` workgroups in all, at most one per
// column tile, with equal numbers of tiles (13 groups of 16 tiles left three of
// them twice the work: 40 3-bit matrices 512 -> 2048 by 72 rows 28 us, in 8 groups 25).
// Few tiles that would split unevenly, on bands enough for a workgroup per CU or more:
// the groups whose rounds of two workgroups per CU walk the fewest tiles, or one group
// when the bands alone fill a round (256 matrices, 3 bits: 512 -> 384 by 100 rows,
// tiles 2 + 1 33.1 us, 3 25.9; 512 -> 640 46.6 and 39.4, by 40 rows 2 + 2 + 1 27.7, 3 + 2 23.8).
constexpr int band_col_groups(int64_t bands, int nt, int want) {
  const int64_t g = (want + bands - 1) / bands;
  const int per = g < 1 ? nt : (int)((nt + g - 1) / g);
  if (per < 1) return nt;
  if (nt % per == 0 || nt >= 8 || bands < want / 4) return (nt + per - 1) / per;
  int best = 1;
  int64_t cost = nt;
  for (int k = 2; k <= nt && bands < want / 2; ++k) {
    const int64_t c = (bands * k + want / 2 - 1) / (want / 2) * ((nt + k - 1) / k);
    if (c < cost) { cost = c; best = k; }
  }
  return best;
}
static_assert(band_col_groups(80, 16, 1024) == 8 && band_col_groups(64, 16, 1024) == 16 &&
                  band_col_groups(2048, 16, 1024) == 1 && band_col_groups(1, 3, 1024) == 3 &&
                  band_col_groups(200, 3, 1024) == 3 && band_col_groups(512, 3, 1024) == 1 &&
                  band_col_groups(511, 3, 1024) == 3 && band_col_groups(512, 4, 1024) == 2 &&
                  band_col_groups(512, 9, 1024) == 2 && band_col_groups(256, 5, 1024) == 2 &&
                  band_col_groups(255, 5, 1024) == 5 && band_col_groups(400, 5, 1024) == 5, "column groups");

template <int BITS, int K, int MB, int NBW, int KS, class Epi, int AM, class Pro>
hipError_t launch_gemm_band_m(const QT& w, int R, const uint16_t* A, const Epi& epi, hipStream_t s, int batch,
                              int64_t codes_stride, int64_t scales_stride, const Pro& pro) {
  auto kfn = gemm_band_kernel<BITS, K, MB, NBW, KS, Epi, AM, Pro>;
  size_t lds = band_a_bytes<K, MB>();
  if constexpr (epi_band_lds<Epi>::value) lds += epi.band_lds(16 * MB);
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

// Bands are 64 rows high where the launch then still has two workgroups per CU,
// or one from 4096 rows; else 32, which gives a small launch twice the workgroups and
// half the rows to stage before its first MFMA (1024 rows: QKV 18.5 us in bands of
// 32).  The taller band decodes a packed weight, or reads a dense one, half as
// often: LM head (512 -> 16384, 3 bits) at 1024 rows 67 us in bands of 32, 62 of 64;
// a 4096-row step on expanded weights at D = 512, 4 layers (384 QKV workgroups) 737 and
// 717, at D = 256, 2 layers (192) 183 and 199.  Bands never span the matrices of a
// batch: of 32 rows and fewer a taller one would be half empty, of 65 to 96 the second
// one (256 matrices, 3 bits, us in bands of 64 / 32: 512 -> 2048 by 32 rows 55 / 40, by 72
// 108 / 103, by 100 116 / 140; 512 -> 512 by 72 34 / 31, by 100 34 / 39).  33 to 64
// rows, one band either way or two, take the taller from 384 workgroups (40 matrices 512
// -> 1536 by 40 rows, 480: 10.2 us, in bands of 32 12.6).
constexpr int kBandTallRows = 4096, kBandTallWgs = 512, kBandTallWgsOne = 384, kBandTallWgsMin = 256;
constexpr bool band_tall(int64_t R, int64_t batch, int64_t N, int nbw) {
  const int64_t wgs = (R + 63) / 64 * batch * ((N + 64 * nbw - 1) / (64 * nbw));
  if (R <= 32 || (R > 64 && R <= 96)) return false;
  return wgs >= (R <= 64 ? kBandTallWgsOne : kBandTallWgs) || (R * batch >= kBandTallRows && wgs >= kBandTallWgsMin);
}
static_assert(band_tall(4096, 1, 1536, 4) && !band_tall(4096, 1, 768, 4) && !band_tall(4095, 1, 1536, 4) &&
                  band_tall(1024, 1, 16384, 4) && !band_tall(32, 1024, 2048, 2) && band_tall(33, 256, 2048, 2) &&
                  band_tall(64, 256, 2048, 2) && !band_tall(65, 256, 2048, 2) && !band_tall(96, 256, 2048, 2) &&
                  band_tall(97, 256, 2048, 2) && band_tall(64, 64, 896, 2) && !band_tall(63, 63, 768, 2) &&
                  !band_tall(1024, 1, 2048, 2), "band height");

template <int BITS, int K, int KS, class Epi, int AM, class Pro>
hipError_t launch_gemm_band_k(const QT& w, int R, const uint16_t* A, const Epi& epi, hipStream_t s, int batch,
                              int64_t codes_stride, int64_t scales_stride, const Pro& pro) {
  constexpr int NBW = Epi::kFragBlocks;
  if (band_tall(R, batch, w.N, NBW))
    return launch_gemm_band_m<BITS, K, 4, NBW, KS, Epi, AM, Pro>(w, R, A, epi, s, batch, codes_stride, scales_stride, pro);
  return launch_gemm_band_m<BITS, K, 2, NBW, KS, Epi, AM, Pro>(w, R, A, epi, s, batch, codes_stride, scales_stride, pro);
}

// Shapes the row-band kernel takes.  Dense bf16 weights too: on 16-row tasks each
// 16 rows read a stage's weights again (a step of the dense student at 2048
// rows 3437 us, at 8192 12267; in bands and K-splits 1578 and 4041).
inline bool band_fits(const QT& w) {
  return (w.bits <= 6 || w.bits == kExpBits || w.bits == 16) && w.N % 64 == 0 && (w.K == 256 || w.K == 512);
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
    case 16: return launch_gemm_band_t<16, KS, Epi, A_BF16, Pro>(w, R, A, epi, s, 1, 0, 0, pro);
    case kExpBits:
      if constexpr (!epi_packed_only<Epi>::value)
        return launch_gemm_band_t<kExpBits, KS, Epi, A_BF16, Pro>(w, R, A, epi, s, 1, 0, 0, pro);
      [[fallthrough]];
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

// ---------------------------------------------------------------------------
// K-split GEMM for launches with many rows on expanded tensors whose stage has
// four K-slices (the MLP down-projection): wave w of a workgroup computes K-slice
// w of a 16*MB x 16*NBW tile, its operands straight from memory into registers
// (A in operand order, op_tile; weights expanded: 1 KB per load), so the k-loop
// has no barrier and the four dependent slices of gemm_task run side by side.
// The slices' tiles then meet in LDS and are added in slice order; the epilogue
// works on four consecutive columns per thread.  Swapped operands and the MFMA
// sequence as in the row-band kernel: the same bits as gemm_task.
// ---------------------------------------------------------------------------
template <int MB, int NBW>
__host__ __device__ constexpr size_t ksplit_lds_bytes() { return (size_t)4 * 16 * MB * (16 * NBW + 4) * 4; }

// DENSE: bits-16 weights (a lane's eight k-steps of a block in one 128-byte line,
// no scales).
template <int MB, int NBW, bool DENSE, class Epi>
__global__ __launch_bounds__(256, 2) void gemm_ksplit_kernel(QT w, int R, const uint16_t* __restrict__ A, Epi epi) {
  constexpr int ROWS = 16 * MB, COLS = 16 * NBW, CS = COLS + 4;
  constexpr int NSLOT = 4, PF = 2;  // operand ring: group q's loads are issued PF groups ahead
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  float* Cp = (float*)smem;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, lg = lane >> 4, col = lane & 15;
  int cx = blockIdx.x, ry = blockIdx.y;
  if (gridDim.y % 8 == 0) {  // the column tiles of a row tile on one XCD, consecutively
    const int bid = blockIdx.x + gridDim.x * blockIdx.y;
    const int j = bid / 8;
    ry = bid % 8 + 8 * (j / gridDim.x);
    cx = j % gridDim.x;
  }
  const int m0 = ry * ROWS, nb0 = cx * NBW;
  const int KB = w.K >> 8, KBS = KB / 4, NG = 4 * KBS;  // 256-blocks, and 64-wide groups of a slice
  const u32x4* ap[MB];
#pragma unroll
  for (int m = 0; m < MB; ++m) {  // row blocks past the last: it again, never stored
    const int rb = min(m0 / 16 + m, (R - 1) / 16);
    ap[m] = (const u32x4*)A + ((int64_t)rb * (w.K >> 5) + wave * KBS * 8) * 64 + lane;
  }
  const u32x4* wp[NBW];
  const uint16_t* sp[NBW];
#pragma unroll
  for (int j = 0; j < NBW; ++j) {
    const size_t blk = (size_t)(nb0 + j) * KB + wave * KBS;
    wp[j] = (const u32x4*)(w.codes + blk * 8192) + (DENSE ? 8 * lane : lane);
    sp[j] = DENSE ? nullptr : w.scales + blk * 64 + 16 * lg;
  }
  u32x4 ar[NSLOT][MB][2], wr[NSLOT][NBW][2];
  auto load = [&](int slot, int q) {
#pragma unroll
    for (int j = 0; j < NBW; ++j) {
      const u32x4* p = wp[j] + (DENSE ? 512 * (q >> 2) + 2 * (q & 3) : 128 * q);
      wr[slot][j][0] = p[0];
      wr[slot][j][1] = p[DENSE ? 1 : 64];
    }
#pragma unroll
    for (int m = 0; m < MB; ++m) {
      ar[slot][m][0] = ap[m][128 * q];
      ar[slot][m][1] = ap[m][128 * q + 64];
    }
  };
  uint32_t sc[NBW][8];
  auto load_sc = [&](int kb) {
#pragma unroll
    for (int j = 0; j < NBW; ++j) {
      const u32x4 x = *(const u32x4_a8*)(sp[j] + 64 * kb), y = *(const u32x4_a8*)(sp[j] + 64 * kb + 8);
#pragma unroll
      for (int i = 0; i < 4; ++i) { sc[j][i] = x[i]; sc[j][4 + i] = y[i]; }
    }
  };
  f32x4 acc[NBW][MB];
#pragma unroll
  for (int j = 0; j < NBW; ++j)
#pragma unroll
    for (int m = 0; m < MB; ++m) acc[j][m] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int q = 0; q < PF; ++q) load(q, q);
  for (int kb = 0; kb < KBS; ++kb) {
    if constexpr (!DENSE) load_sc(kb);
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int qn = 4 * kb + g + PF;
      load((g + PF) % NSLOT, qn < NG ? qn : NG - 1);  // unconditional: the last groups once more
#pragma unroll
      for (int m = 0; m < MB; ++m) {
        const bf16x8 a0 = __builtin_bit_cast(bf16x8, ar[g % NSLOT][m][0]);
        const bf16x8 a1 = __builtin_bit_cast(bf16x8, ar[g % NSLOT][m][1]);
        f32x4 t[NBW];
#pragma unroll
        for (int j = 0; j < NBW; ++j)
          t[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wr[g % NSLOT][j][0]), a0,
                                                         f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
        for (int j = 0; j < NBW; ++j)
          t[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wr[g % NSLOT][j][1]), a1, t[j], 0, 0, 0);
#pragma unroll
        for (int j = 0; j < NBW; ++j) {
          float s[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int h = 4 * i + g;
            s[i] = DENSE ? 1.f : (h & 1) ? half_hi(sc[j][h >> 1]) : half_lo(sc[j][h >> 1]);
          }
          fma4(acc[j][m], s, t[j]);
        }
      }
      __builtin_amdgcn_sched_barrier(0);  // groups stay apart (see the row-band kernel)
    }
  }
  float* C = Cp + (size_t)wave * ROWS * CS;
#pragma unroll
  for (int j = 0; j < NBW; ++j)
#pragma unroll
    for (int m = 0; m < MB; ++m) *(f32x4*)(C + (16 * m + col) * CS + 16 * j + 4 * lg) = acc[j][m];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < ROWS * COLS / 4 / 256; ++i) {
    const int e = threadIdx.x + 256 * i, rr = e / (COLS / 4), c4 = e % (COLS / 4) * 4;
    if (m0 + rr >= R) continue;
    const float* p = Cp + rr * CS + c4;
    f32x4 v = *(const f32x4*)p;
#pragma unroll
    for (int k = 1; k < 4; ++k) {
      const f32x4 x = *(const f32x4*)(p + (size_t)k * ROWS * CS);
#pragma unroll
      for (int u = 0; u < 4; ++u) v[u] += x[u];
    }
    epi.put4(v, (int64_t)(m0 + rr) * w.N + nb0 * 16 + c4, nb0 * 16 + c4);
  }
}

// The K-split kernel's shapes: four K-slices of whole 256-blocks.  Its operands
// are shared by nothing but the XCD's L2, so from about 8192 rows the 64 x 128
// tiles of gemm_big_kernel, which share A rows through LDS, are ahead (K = 2048,
// N = 512: 1024 rows 11.9 us against 27.5, 32768 rows 213 against 160; steps of 4 layers,
// 3 bits: 4096 rows 825 / 837, 6144 1199 / 1211, 8192 1478 / 1449, 16384 2665 / 2619; 64 x
// 64 tiles here spill: 287).
constexpr int kKsplitMaxRows = 8192;
inline bool ksplit_fits(const QT& w, int R, int ks) {
  return ks == 4 && (w.K >> 8) % 4 == 0 && w.N % 32 == 0 &&
         (w.bits == 16 || (w.bits == kExpBits && R < kKsplitMaxRows));
}

template <class Epi>
hipError_t launch_gemm_ksplit(const QT& w, int R, const uint16_t* A, const Epi& epi, hipStream_t s) {
  if (!ksplit_fits(w, R, 4) || ((uintptr_t)A & 15) != 0) return hipErrorInvalidValue;
  constexpr int MB = 4, NBW = 2;
  auto kfn = w.bits == 16 ? gemm_ksplit_kernel<MB, NBW, true, Epi> : gemm_ksplit_kernel<MB, NBW, false, Epi>;
  const dim3 grid((unsigned)(w.N / (16 * NBW)), (unsigned)((R + 16 * MB - 1) / (16 * MB)));
  hipLaunchKernelGGL(kfn, grid, dim3(256), (ksplit_lds_bytes<MB, NBW>()), s, w, R, A, epi);
  return hipGetLastError();
}

}  // namespace altxs
