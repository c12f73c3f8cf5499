// Grouped GEMMs of the expert FFN for calls with few tokens per expert (decode and small
// batches), all four weight x activation formats. Such a call is bound by reading the used
// experts' weights once from HBM; the large-tile kernels (afd_gemm_mx.hip, afd_gemm_fp8.hip,
// afd_gemm_a16.hip) then leave CUs idle (8 column tiles of 512 per expert: 14 experts of a
// decode step occupy 112 of 256 CUs, 38 experts take two rounds) and pay a barrier every half
// stage.
//
// Split: a workgroup of 4 wavefronts owns a row group (at most 32 R = 32 or 64 rows of one
// expert) x the 256 weight rows of one image column; wavefront w streams its 64 rows (gate_up: 32 gate and the
// matching 32 up rows; 4 KiB of each image) over the whole K from HBM into registers, several K
// stages of 128 ahead (depth()), so 256-column items fill the chip and 2 or 3 workgroups a CU keep
// 104-209 KB of weights in flight. A stage passes through LDS on its way to the matrix instructions: the
// weights through the wavefront's own area, which lets the loads be contiguous kilobytes (read in
// fragment order, half a line a load, non-temporal loads reach 5.3 TB/s here and default ones
// 6.1; contiguous non-temporal ones 7.0), the activations through a block the four wavefronts fill
// a quarter each and share (each wavefront reading its own copy from L2 was as fast at 1 to 16
// rows per expert and 20 to 35% slower at 32 to 64).
//
// Measured against the large-tile kernels (whole expert call, cold caches, with the router's one
// launch for few pairs, which gives about 5 to 10 us of it): hidden 4096, inter 2048, 64 of 256
// MXFP4 experts local, top-8, Zipf(1.2): 8 tokens 75 -> 42 us, 64 tokens 151 -> 100, 300 tokens
// 188 -> 160 (fp8 activations); 128 tokens 233 -> 125 (bf16 activations). Hidden 4096, inter 1536,
// 64 FP8-block experts, top-8, uniform routing: 8 tokens 226 -> 135 us, 128 tokens 275 -> 203. The
// reads then run at 5.0 to 5.5 TB/s.
//
// Every accumulator sees the MFMAs of the large-tile kernels, in their order, with their scale
// arithmetic, and the epilogues are theirs, so a token's result does not depend on which kernel
// ran (bit for bit; the batch, job and subset tests rest on it). K is therefore not split.
#include <type_traits>

#include "afd_common.h"
#include "afd_gemm_dev.h"
#include "afd_internal.h"

namespace afd {

namespace {

enum { kGateUp = 0, kDown = 1, kGateUpParam = 2 };
// weight x activation formats: MXFP4 x MXFP8, FP8 block x FP8 1x128, MXFP4 x bf16, FP8 x bf16
enum { kMx8 = 0, kF8 = 1, kMx16 = 2, kF16 = 3 };

struct RowsArgs {
  const uint8_t* a;          // gate_up: token rows [n][K] (e4m3 or bf16); down: the h images
  const uint8_t* as;         // their scales (MXFP8 gate_up, FP8 1x128); else unused
  const afd_job* rows_desc;  // gate_up: if set, a / as are its x or xq / xs
  uint32_t topk_magic;       // div_magic(topk)
  const uint8_t* b;          // weight images [E][N/256][K/128 or K/64]
  const float* bs;           // FP8: block scales [E][N/128][K/128] (gate blocks, then up)
  const int32_t* sorted_pairs;
  const int32_t* counts;
  RowsGate gate;
  int num_local;
  int K, N;
  uint32_t ntn_magic;  // div_magic(N / 256)
  ActParams act;
  uint8_t* hq;   // gate_up out: the down GEMM's h images
  float* hs;     // gate_up out (FP8 1x128): their scales [row tiles][N/2/128][256]
  uint16_t* y;   // down out: bf16 [np][N]
};

template <int FMT>
struct Fmt {
  static constexpr bool kMxW = FMT == kMx8 || FMT == kMx16;
  static constexpr bool kA16 = FMT == kMx16 || FMT == kF16;
  static constexpr int kBM = FMT == kF8 ? kFp8BlockM : kBlockM;  // rows of a row tile
  static constexpr int kImgs = kMxW ? 1 : 2;                     // weight images per 128 K
  static constexpr int kImgBytes = kMxW ? kImgB : kImgF8B;
  // bytes of a row tile's h images per 128 K
  static constexpr int kHStage = FMT == kMx8 ? kImgA : FMT == kMx16 ? kImgA16 : 2 * (kA16 ? kImgData : kImgF8B);
  static constexpr int kABlock = kA16 ? 8192 : 4096;  // bytes of 32 activation rows x 128 K
  static constexpr int kALoads = kABlock / 4096;      // 16-byte loads of a lane per block (4 wavefronts)
};

// Global-memory pointers by type: read through a generic one (a row pointer may come from the job
// descriptor) the compiler would issue flat loads, whose waits also count LDS operations.
typedef const __attribute__((address_space(1))) uint8_t* GPtr;
__device__ __forceinline__ GPtr global_ptr(const void* p) {
  return (GPtr)(reinterpret_cast<uintptr_t>(p));
}
// A uniform pointer, opaque to the optimizer, so loads at it plus a lane offset take the scalar
// base form instead of 64-bit lane pointers stepped through the K loop.
__device__ __forceinline__ GPtr scalar_base(GPtr p) {
  uint64_t v = (uint64_t)p;
  asm volatile("" : "+s"(v));
  return (GPtr)v;
}
template <typename T>
__device__ __forceinline__ T load_global(GPtr base, uint32_t off) {
  return *(const __attribute__((address_space(1))) T*)(base + off);
}
// Weights. kOnce: the expert has one row group, so they are read once: non-temporal, full-line reads
// reach 7.0 TB/s here against 6.2 TB/s with the default policy. An expert with several groups is
// read by each of them, at about the same time and (column counts a multiple of 8) on one XCD: the
// default policy leaves the lines to the other groups. Non-temporal for all (-> this rule), whole
// calls: hidden 4096, inter 2048, 256 FP8 experts, 510 tokens that all go to 32 of them 464 -> 303 us
// (large tiles: 213); 64 MXFP4 experts, 320 tokens to 32 of them 175 -> 152 (large tiles: 159);
// Zipf(1.2) 300 tokens 209 -> 198, uniform routing the same.
template <bool kOnce, typename T>
__device__ __forceinline__ T load_weight(GPtr base, uint32_t off) {
  if constexpr (kOnce)
    return __builtin_nontemporal_load((const __attribute__((address_space(1))) T*)(base + off));
  else
    return load_global<T>(base, off);
}
__device__ __forceinline__ v8i join(v4i lo, v4i hi) {
  return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
}

// K stages in flight for NB 32-row blocks in groups of R: as many as the registers (256, or 168 for
// three workgroups a CU with R = 1) hold beside the 32 NB accumulators (17 or 32 registers of
// weights and 5 or 8 per row block of activations a stage)
template <int FMT, int NB, int R>
constexpr int depth() {
  if (R == 1) return FMT == kMx8 ? 4 : FMT == kMx16 ? 3 : 2;
  return FMT == kMx8 ? 4 : FMT == kMx16 ? (NB == 1 ? 4 : 3) : NB == 1 ? 3 : 2;
}

template <int FMT, int MODE, int R>
__global__ __launch_bounds__(256, R == 1 ? 3 : 2) void rows_gemm_kernel(RowsArgs p) {
  using F = Fmt<FMT>;
  constexpr bool kGU = MODE != kDown;
  constexpr int kBM = F::kBM;
  constexpr int kRows = 32 * R;
  if (p.gate.few_skips()) return;
  const int ntn = p.N / kImgBRows;
  const int t = threadIdx.x, lane = t & 63, lr = lane & 31, lk = lane >> 5;
  const int w = __builtin_amdgcn_readfirstlane(t >> 6);
  const uint32_t sub = div_by_magic(blockIdx.x, p.ntn_magic);
  const int nt = static_cast<int>(blockIdx.x - sub * ntn);
  // Row group `sub` of the call: expert e's rows are cut into ceil(count / kRows) groups, in
  // expert order. Every wavefront finds it from the counts by itself (4 experts a lane, one
  // load and a scan), together with the expert's first row tile of the padded layout.
  int cnt[4], first_group = 0, first_tile = 0;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    cnt[i] = 4 * lane + i < p.num_local ? p.counts[4 * lane + i] : 0;
    first_group += (cnt[i] + kRows - 1) / kRows;
    first_tile += (cnt[i] + kBM - 1) / kBM;
  }
  const int lane_groups = first_group, lane_tiles = first_tile;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int vg = __shfl_up(first_group, d), vt = __shfl_up(first_tile, d);
    if (lane >= d) {
      first_group += vg;
      first_tile += vt;
    }
  }
  const uint64_t past = __ballot(first_group > static_cast<int>(sub));
  if (past == 0) return;
  const int at = __builtin_ctzll(past);  // the lane whose experts hold the group
  int e = 4 * at, group = static_cast<int>(sub) - __builtin_amdgcn_readlane(first_group - lane_groups, at);
  int tile = __builtin_amdgcn_readlane(first_tile - lane_tiles, at), rows = 0;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int c = __builtin_amdgcn_readlane(cnt[i], at);
    const int g = (c + kRows - 1) / kRows;
    if (rows == 0) {  // not found yet
      if (group < g) {
        rows = c;
      } else {
        group -= g;
        tile += (c + kBM - 1) / kBM;
        ++e;
      }
    }
  }
  const int mt = tile + group * kRows / kBM;
  const int r0 = group * kRows % kBM;                // the group's first row in its row tile
  const int live = min(rows - group * kRows, kRows) + r0;  // and the end of its rows
  const int KT = p.K / 128;
  const int kb_n = KT;  // scale blocks along K

  GPtr a_rows = global_ptr(p.a), a_scales = global_ptr(p.as);
  if (kGU && p.rows_desc != nullptr) {
    a_rows = F::kA16 ? global_ptr(p.rows_desc->x) : global_ptr(p.rows_desc->xq);
    a_scales = global_ptr(p.rows_desc->xs);
  }
  // this wavefront's 64 weight rows: rows 64 w + 32 j + lr of image column nt. The lane's two
  // 16-byte chunks of a row (img_b_off; the swizzle depends on lr alone): for the scaled MFMA
  // logical chunks lk and lk + 2 (e2m1: the two k-steps; e4m3: the operand's two halves), for
  // W8A16 chunks 2 lk and 2 lk + 1.
  const GPtr wbase = global_ptr(p.b) + (int64_t(e) * ntn + nt) * (KT * F::kImgs) * int64_t(F::kImgBytes) + w * 4096;
  const uint32_t wo0 = static_cast<uint32_t>(img_b_off(lr, FMT == kF16 ? 2 * lk : lk));
  const uint32_t wo1 = wo0 ^ (FMT == kF16 ? 16u : 32u);
  // FP8: the block-scale rows of its gate (tiles j = 0) and up (j = 1) weight rows, or (down) of
  // its 64 rows
  const float* s_blk[2] = {nullptr, nullptr};
  if constexpr (!F::kMxW) {
    const float* se = p.bs + int64_t(e) * (p.N / 128) * kb_n;
    s_blk[0] = se + (kGU ? nt : 2 * nt + (w >> 1)) * kb_n;
    s_blk[1] = kGU ? se + (ntn + nt) * kb_n : s_blk[0];
  }
  __shared__ __attribute__((aligned(16))) uint8_t lds_all[4 * F::kImgs * 4096];
  uint8_t* lds_w = lds_all + w * (F::kImgs * 4096);
  __shared__ __attribute__((aligned(16))) uint8_t lds_a[2 * R * F::kABlock];
  __shared__ float amax_l[FMT == kF8 && kGU ? R * 4 * 32 : 1];

  // rows [r0, live) of the tile as NB blocks of 32
  auto pass = [&](auto nb_c, auto once_c) __attribute__((always_inline)) {
    constexpr int NB = decltype(nb_c)::value;
    constexpr bool kOnce = decltype(once_c)::value;
    constexpr int D = depth<FMT, NB, R>();
    struct Stage {
      v4i w[F::kImgs][4];  // the wavefront's 4 KiB of each image, 1 KiB a load
      uint32_t sw;         // MXFP4: the scale word of weight row 64 w + lane
      v4i a[NB][F::kALoads];  // the wavefront's quarter of the activation blocks
      uint32_t sa[NB];  // MXFP8: the half-word of this lane half; FP8 1x128: the fp32 scale
    };
    // Lane offsets of the activation loads (ao, kALoads per 32-row block) and of the scales of
    // rows 32 i + lr (so), and where the loaded chunks go in the LDS block (al). gate_up gathers
    // token rows: 8 or 16 chunks of 16 bytes a row, 8 or 4 rows a load; down copies its block of
    // the h images, which already have the block's layout. Rows past the last real one repeat it
    // (gate_up) or are whatever the image holds (down); their results are not stored.
    uint32_t ao[NB][F::kALoads], al[NB][F::kALoads], so[NB];
    auto token = [&](int r) {
      return div_by_magic(static_cast<uint32_t>(p.sorted_pairs[mt * kBM + min(r, live - 1)]), p.topk_magic);
    };
#pragma unroll
    for (int i = 0; i < NB; ++i) {
#pragma unroll
      for (int h = 0; h < F::kALoads; ++h) {
        const int q = w * F::kALoads + h;  // 1 KiB piece of the block
        if constexpr (kGU) {
          constexpr int kPer = F::kA16 ? 16 : 8;  // chunks per row
          const int r = r0 + 32 * i + q * (64 / kPer) + lane / kPer, c = lane % kPer;
          ao[i][h] = token(r) * static_cast<uint32_t>(p.K) * (F::kA16 ? 2u : 1u) + 16u * c;
          al[i][h] = F::kA16 ? (r - r0) * 256 + ((c ^ (r & 15)) << 4) : img_a_off(r, c) - r0 * 128;
        } else {
          const uint32_t l = 16u * lane;
          ao[i][h] = FMT == kMx8   ? r0 * 128 + i * 4096 + q * 1024 + l
                     : FMT == kF8  ? (q >> 1) * kImgF8B + r0 * 64 + i * 2048 + (q & 1) * 1024 + l
                     : FMT == kMx16 ? r0 * 256 + i * 8192 + q * 1024 + l
                                    : (q >> 2) * kImgData + r0 * 128 + i * 4096 + (q & 3) * 1024 + l;
          al[i][h] = i * F::kABlock + q * 1024 + l;
        }
      }
      const int r = r0 + 32 * i + lr;
      so[i] = FMT == kMx8 ? (kGU ? token(r) * static_cast<uint32_t>(p.K / 32) : kImgData + r * 4) + 2u * lk
              : FMT == kF8 ? (kGU ? token(r) * static_cast<uint32_t>(kb_n) : static_cast<uint32_t>(r)) * 4u
                           : 0u;
    }
    auto load = [&](Stage& f, int kt) __attribute__((always_inline)) {
#pragma unroll
      for (int m = 0; m < F::kImgs; ++m) {
        const GPtr img = scalar_base(wbase + int64_t(kt * F::kImgs + m) * F::kImgBytes);
#pragma unroll
        for (int c = 0; c < 4; ++c) f.w[m][c] = load_weight<kOnce, v4i>(img + 1024 * c, 16u * lane);
        if constexpr (F::kMxW) f.sw = load_weight<kOnce, uint32_t>(img + (kImgData - w * 4096 + w * 256), 4u * lane);
      }
#pragma unroll
      for (int i = 0; i < NB; ++i) {
        GPtr base;
        if constexpr (kGU)
          base = scalar_base(a_rows + int64_t(kt) * (F::kA16 ? 256 : 128));
        else
          base = scalar_base(a_rows + (int64_t(mt) * KT + kt) * Fmt<FMT>::kHStage);
#pragma unroll
        for (int h = 0; h < F::kALoads; ++h) f.a[i][h] = load_global<v4i>(base, ao[i][h]);
        if constexpr (FMT == kMx8)
          f.sa[i] = load_global<uint16_t>(kGU ? scalar_base(a_scales + int64_t(kt) * 4) : base, so[i]);
        else if constexpr (FMT == kF8)
          f.sa[i] = load_global<uint32_t>(
              scalar_base(a_scales + (kGU ? int64_t(kt) * 4 : (int64_t(mt) * kb_n + kt) * (kBM * 4))), so[i]);
      }
    };
    v16f acc[NB][2];
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int q = 0; q < 16; ++q) acc[i][j][q] = 0.0f;
    // FP8: the scales the accumulators are relative to (weights: sw0 / sw1; activations: sx) and
    // the next K block's weight scales, as in afd_gemm_fp8.hip and afd_gemm_a16.hip
    float sw0 = 1.0f, sw1 = 1.0f, swn0 = 1.0f, swn1 = 1.0f, sx[NB];
#pragma unroll
    for (int i = 0; i < NB; ++i) sx[i] = 1.0f;
    if constexpr (!F::kMxW) {
      swn0 = sw0 = load_uniform(s_blk[0]);
      swn1 = sw1 = load_uniform(s_blk[1]);
    }
    auto mma = [&](const Stage& f, int kt) __attribute__((always_inline)) {
      // The stage through LDS: the weights in the wavefront's own area, from load order to fragment
      // order; the activations in a block the four wavefronts fill and share, one of two (a
      // wavefront that writes stage kt + 2 has passed the barrier of kt + 1, which every wavefront
      // reaches after its reads of kt). Own writes done, then the barrier; loads stay in flight.
#pragma unroll
      for (int m = 0; m < F::kImgs; ++m)
#pragma unroll
        for (int c = 0; c < 4; ++c) *reinterpret_cast<v4i*>(lds_w + m * 4096 + c * 1024 + 16 * lane) = f.w[m][c];
      uint8_t* block = lds_a + (kt & 1) * (R * F::kABlock);
#pragma unroll
      for (int i = 0; i < NB; ++i)
#pragma unroll
        for (int h = 0; h < F::kALoads; ++h) *reinterpret_cast<v4i*>(block + al[i][h]) = f.a[i][h];
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      wait_lds();
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      // 16-byte chunk c of the activation operand of row 32 i + lr: fp8 K [16 lk + 32 c, + 16) of
      // the stage, bf16 phase c / 4, K [32 lk + 8 (c % 4), + 8) of its 64
      auto a_chunk = [&](int i, int c) {
        const int r = r0 + 32 * i + lr;
        int off;
        if constexpr (F::kA16 && (kGU || FMT == kMx16))
          off = i * 8192 + lr * 256 + (((8 * (c >> 2) + 4 * lk + (c & 3)) ^ (lr & 15)) << 4);
        else if constexpr (F::kA16)
          off = i * 8192 + (c >> 2) * 4096 + img_a_off(r, 4 * lk + (c & 3)) - (r - lr) * 128;
        else if constexpr (kGU || FMT == kMx8)
          off = img_a_off(r, 2 * c + lk) - r0 * 128;
        else
          off = i * 4096 + (c >> 1) * 2048 + img_b_off(lr, lk + 2 * (c & 1));
        return *reinterpret_cast<const v4i*>(block + off);
      };
      v4i w4[2][2];  // MXFP4: [j][chunk]
      v8i w8[2][2];  // FP8: [image][j], both chunks
#pragma unroll
      for (int m = 0; m < F::kImgs; ++m)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const v4i c0 = *reinterpret_cast<const v4i*>(lds_w + m * 4096 + wo0 + 2048 * j);
          const v4i c1 = *reinterpret_cast<const v4i*>(lds_w + m * 4096 + wo1 + 2048 * j);
          if constexpr (F::kMxW) {
            w4[j][0] = c0;
            w4[j][1] = c1;
          } else {
            w8[m][j] = join(c0, c1);
          }
        }
      if constexpr (FMT == kMx8) {
        // scale word of row 64 w + lane -> those of rows 32 j + lr in both lane halves, then
        // this half's 16 bits (bytes 0, 1: k-steps 0, 1)
        const auto r = __builtin_amdgcn_permlane32_swap(f.sw, f.sw, false, false);
        const uint32_t sb[2] = {r[0] >> (16 * lk), r[1] >> (16 * lk)};
        static_for<2>([&](auto ksc) {
          constexpr int ks = decltype(ksc)::value;
#pragma unroll
          for (int i = 0; i < NB; ++i) {
            const v8i fa = join(a_chunk(i, 2 * ks), a_chunk(i, 2 * ks + 1));
#pragma unroll
            for (int j = 0; j < 2; ++j)
              acc[i][j] = mfma_scale_f4_f8(w4[j][ks], fa, acc[i][j], 4 /*A e2m1*/, 0 /*B e4m3*/, ks,
                                                static_cast<int>(sb[j]), ks, static_cast<int>(f.sa[i]));
          }
        });
      } else if constexpr (FMT == kF8) {
#pragma unroll
        for (int i = 0; i < NB; ++i) {
          const float x = __uint_as_float(f.sa[i]);
          const float f0 = (sx[i] * sw0) * __builtin_amdgcn_rcpf(x * swn0);
          const float f1 = (sx[i] * sw1) * __builtin_amdgcn_rcpf(x * swn1);
          sx[i] = x;
#pragma unroll
          for (int q = 0; q < 16; ++q) {
            acc[i][0][q] *= f0;
            acc[i][1][q] *= f1;
          }
        }
        sw0 = swn0;
        sw1 = swn1;
        const int kn = min(kt + 1, kb_n - 1);
        swn0 = load_uniform(s_blk[0] + kn);
        swn1 = load_uniform(s_blk[1] + kn);
        static_for<2>([&](auto ksc) {
          constexpr int ks = decltype(ksc)::value;
#pragma unroll
          for (int i = 0; i < NB; ++i) {
            const v8i fa = join(a_chunk(i, 2 * ks), a_chunk(i, 2 * ks + 1));
#pragma unroll
            for (int j = 0; j < 2; ++j) {
              acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(w8[ks][j], fa, acc[i][j], 0, 0, 0,
                                                                          127, 0, 127);
            }
          }
        });
      } else {
        float scale[2][2] = {};  // MXFP4: [phase][j]
        if constexpr (FMT == kMx16) {
          // block 2 c + lk of a row at byte 2 lk + c of its scale word
          const auto r = __builtin_amdgcn_permlane32_swap(f.sw, f.sw, false, false);
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            const uint32_t h = r[j] >> (16 * lk);
            scale[0][j] = __uint_as_float((h & 255u) << 23);
            scale[1][j] = __uint_as_float(((h >> 8) & 255u) << 23);
          }
        } else {
          if (kt > 0) {
            const float f0 = sw0 * __builtin_amdgcn_rcpf(swn0), f1 = sw1 * __builtin_amdgcn_rcpf(swn1);
#pragma unroll
            for (int i = 0; i < NB; ++i)
#pragma unroll
              for (int q = 0; q < 16; ++q) {
                acc[i][0][q] *= f0;
                acc[i][1][q] *= f1;
              }
          }
          sw0 = swn0;
          sw1 = swn1;
          const int kn = min(kt + 1, kb_n - 1);
          swn0 = load_uniform(s_blk[0] + kn);
          swn1 = load_uniform(s_blk[1] + kn);
        }
        static_for<2>([&](auto cc) {
          constexpr int c = decltype(cc)::value;
          static_for<4>([&](auto sc) {
            constexpr int s = decltype(sc)::value;
            v8bf fa[NB];
#pragma unroll
            for (int i = 0; i < NB; ++i) fa[i] = __builtin_bit_cast(v8bf, a_chunk(i, 4 * c + s));
#pragma unroll
            for (int j = 0; j < 2; ++j) {
              v8bf wb;
              if constexpr (FMT == kMx16)
                wb = expand_fp4(static_cast<uint32_t>(w4[j][c][s]), scale[c][j]);
              else
                wb = expand_fp8(static_cast<uint32_t>(w8[c][j][2 * s]), static_cast<uint32_t>(w8[c][j][2 * s + 1]));
#pragma unroll
              for (int i = 0; i < NB; ++i)
                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wb, fa[i], acc[i][j], 0, 0, 0);
            }
          });
        });
      }
    };
    // K loop, D stages in flight: each stage's registers take stage kt + D once its MFMAs are
    // issued (clamped to the last stage, so no load is behind a branch: the compiler's counted
    // waits would assume it away and drain the others)
    const int last = KT - 1;
    Stage st[D];
    static_for<D>([&](auto dc) { load(st[decltype(dc)::value], min(static_cast<int>(decltype(dc)::value), last)); });
    int k0 = 0;
    for (; k0 + D < KT; k0 += D) {
      static_for<D>([&](auto dc) {
        constexpr int d = decltype(dc)::value;
        mma(st[d], k0 + d);
        __builtin_amdgcn_sched_barrier(0);
        load(st[d], min(k0 + d + D, last));
        __builtin_amdgcn_sched_barrier(0);
      });
    }
    static_for<D>([&](auto dc) {
      constexpr int d = decltype(dc)::value;
      if (k0 + d < KT) mma(st[d], k0 + d);
      __builtin_amdgcn_sched_barrier(0);
    });

    // Accumulator q of tile (i, j): activation row r0 + 32 i + lr, weight row 64 w + 32 j +
    // 8 (q / 4) + 4 lk + q % 4 of image column nt. The epilogues are those of the large-tile
    // kernels, with stores of real rows only.
    bool real[NB];
#pragma unroll
    for (int i = 0; i < NB; ++i) real[i] = r0 + 32 * i + lr < live;
    if constexpr (kGU) {
      auto store_h = [&](auto fn) __attribute__((always_inline)) {
        float h[NB][16], m[NB];
#pragma unroll
        for (int i = 0; i < NB; ++i) {
          // the running scales of the two tiles (1 with MX weights)
          const float l0 = FMT == kF8 ? sx[i] * sw0 : sw0, l1 = FMT == kF8 ? sx[i] * sw1 : sw1;
          m[i] = 0.0f;
#pragma unroll
          for (int q = 0; q < 16; ++q) {
            h[i][q] = F::kMxW ? fn(acc[i][0][q], acc[i][1][q]) : fn(acc[i][0][q] * l0, acc[i][1][q] * l1);
            if constexpr (!F::kA16) m[i] = fmaxf(m[i], fabsf(h[i][q]));
          }
          if constexpr (!F::kA16) m[i] = fmaxf(m[i], xor32(m[i], lk));
        }
        if constexpr (FMT == kF8) {
          // the image column's 128 h columns are one 1x128 group: its amax over the 4 wavefronts
#pragma unroll
          for (int i = 0; i < NB; ++i)
            if (lk == 0) amax_l[(w * NB + i) * 32 + lr] = m[i];
          __syncthreads();
#pragma unroll
          for (int i = 0; i < NB; ++i)
#pragma unroll
            for (int v = 0; v < 4; ++v) m[i] = fmaxf(m[i], amax_l[(v * NB + i) * 32 + lr]);
        }
#pragma unroll
        for (int i = 0; i < NB; ++i) {
          const int r = r0 + 32 * i + lr;
          if constexpr (FMT == kMx8) {
            const uint32_t code = mx_scale_code(m[i], 8);
            const float inv = mx_inv_scale(code);
            uint32_t d[4];
#pragma unroll
            for (int q4 = 0; q4 < 4; ++q4)
              d[q4] = pk4_e4m3(h[i][4 * q4] * inv, h[i][4 * q4 + 1] * inv, h[i][4 * q4 + 2] * inv,
                               h[i][4 * q4 + 3] * inv);
            const v4i chunk = e4m3_chunk(d, lk);
            // MX block w of the 4 in K stage nt of the down GEMM
            uint8_t* img = p.hq + (int64_t(mt) * ntn + nt) * kImgA;
            if (real[i]) {
              *reinterpret_cast<v4i*>(img + img_a_off(r, 2 * w + lk)) = chunk;
              if (lk == 0) img[kImgData + r * 4 + scale_byte(w)] = static_cast<uint8_t>(code);
            }
          } else if constexpr (FMT == kF8) {
            const float sc = fmaxf(m[i], kFp8Eps) / kE4m3Max;
            const float rsc = 1.0f / sc;
            uint32_t d[4];
#pragma unroll
            for (int q4 = 0; q4 < 4; ++q4)
              d[q4] = pk4_e4m3_near(div_by(h[i][4 * q4], sc, rsc), div_by(h[i][4 * q4 + 1], sc, rsc),
                                    div_by(h[i][4 * q4 + 2], sc, rsc), div_by(h[i][4 * q4 + 3], sc, rsc));
            const v4i chunk = e4m3_chunk(d, lk);
            uint8_t* img = p.hq + (int64_t(mt) * ntn * 2 + 2 * nt + (w >> 1)) * kImgF8B;
            if (real[i]) {
              *reinterpret_cast<v4i*>(img + img_b_off(r, 2 * (w & 1) + lk)) = chunk;
              if (w == 0 && lk == 0) p.hs[(int64_t(mt) * ntn + nt) * kBM + r] = sc;
            }
          } else {
            v4i chunk[2];
            bf16_chunks(h[i], chunk);
            if (real[i]) {
#pragma unroll
              for (int pr = 0; pr < 2; ++pr) {
                const int c = 2 * pr + lk;  // 16-byte chunk of the wavefront's 32 columns
                if constexpr (FMT == kMx16) {
                  uint8_t* img = p.hq + (int64_t(mt) * ntn + nt) * kImgA16;
                  *reinterpret_cast<v4i*>(img + r * 256 + (((4 * w + c) ^ (r & 15)) << 4)) = chunk[pr];
                } else {
                  uint8_t* img = p.hq + (int64_t(mt) * ntn * 2 + 2 * nt + (w >> 1)) * kImgData;
                  *reinterpret_cast<v4i*>(img + img_a_off(r, 4 * (w & 1) + c)) = chunk[pr];
                }
              }
            }
          }
        }
      };
      if constexpr (MODE == kGateUpParam) {
        if (p.act.act == AFD_ACT_SITU)
          store_h([&](float g, float u) { return act_situ(g, u, p.act.a, p.act.inv_a, p.act.l, p.act.inv_l); });
        else
          store_h([&](float g, float u) { return act_swiglu_limit(g, u, p.act.l); });
      } else {
        store_h([](float g, float u) { return act_swiglu(g, u); });
      }
    } else {
#pragma unroll
      for (int i = 0; i < NB; ++i) {
        const int64_t r = int64_t(mt) * kBM + r0 + 32 * i + lr;
        const float l = FMT == kF8 ? sx[i] * sw0 : sw0;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          float h[16];
#pragma unroll
          for (int q = 0; q < 16; ++q) h[q] = F::kMxW ? acc[i][j][q] : acc[i][j][q] * l;
          v4i chunk[2];
          bf16_chunks(h, chunk);
          if (real[i]) {
            uint16_t* dst = p.y + r * p.N + nt * kImgBRows + 64 * w + 32 * j;
#pragma unroll
            for (int pr = 0; pr < 2; ++pr) *reinterpret_cast<v4i*>(dst + 8 * (2 * pr + lk)) = chunk[pr];
          }
        }
      }
    }
  };
  auto pass_rows = [&](auto once_c) __attribute__((always_inline)) {
    if constexpr (R == 2) {
      if (live - r0 > 32) {
        pass(std::integral_constant<int, 2>{}, once_c);
        return;
      }
    }
    pass(std::integral_constant<int, 1>{}, once_c);
  };
  if (__builtin_expect(rows <= kRows, 1))  // the expert's only group (its code comes first)
    pass_rows(std::true_type{});
  else
    pass_rows(std::false_type{});
}

template <int FMT, int MODE>
int launch_rows(const RowsArgs& p, const RowsPlan& plan, hipStream_t stream) {
  const dim3 grid(static_cast<unsigned>(plan.grid_groups * (p.N / kImgBRows)));
  if (plan.group_shift == 5)
    hipLaunchKernelGGL((rows_gemm_kernel<FMT, MODE, 1>), grid, dim3(256), 0, stream, p);
  else
    hipLaunchKernelGGL((rows_gemm_kernel<FMT, MODE, 2>), grid, dim3(256), 0, stream, p);
  AFD_CHECK_LAUNCH();
  return AFD_OK;
}

template <int MODE>
int launch_fmt(const RowsArgs& p, const afd_moe_cfg& cfg, const RowsPlan& plan, hipStream_t stream) {
  if (cfg.act_fmt == AFD_A_BF16)
    return cfg.weight_fmt == AFD_W_MXFP4 ? launch_rows<kMx16, MODE>(p, plan, stream)
                                         : launch_rows<kF16, MODE>(p, plan, stream);
  return cfg.weight_fmt == AFD_W_MXFP4 ? launch_rows<kMx8, MODE>(p, plan, stream)
                                       : launch_rows<kF8, MODE>(p, plan, stream);
}

RowsArgs rows_args(const afd_moe_cfg& cfg, uint8_t* ws, const afd_ws_layout& L, const RowsPlan& plan) {
  RowsArgs p = {};
  p.gate = rows_gate(plan, ws, L);
  p.topk_magic = div_magic(cfg.topk);
  p.act = act_params(cfg);
  p.sorted_pairs = reinterpret_cast<const int32_t*>(ws + L.sorted_pairs);
  p.num_local = cfg.num_local;
  p.counts = reinterpret_cast<const int32_t*>(ws + L.counts);
  return p;
}

}  // namespace

RowsGate rows_gate(const RowsPlan& plan, uint8_t* ws, const afd_ws_layout& L) {
  if (plan.form != kRowsBoth) return RowsGate{nullptr};
  return RowsGate{reinterpret_cast<const int32_t*>(call_counters(ws, L)) + kRowsFewWord};
}

int launch_rows_gate_up(const afd_moe_cfg& cfg, const afd_expert_weights& wt, uint8_t* ws,
                        const afd_ws_layout& L, const void* x, const void* xs, const afd_job* rows_desc,
                        const RowsPlan& plan, hipStream_t stream) {
  RowsArgs p = rows_args(cfg, ws, L, plan);
  p.a = static_cast<const uint8_t*>(x);
  p.as = static_cast<const uint8_t*>(xs);
  p.rows_desc = rows_desc;
  p.b = static_cast<const uint8_t*>(wt.w13);
  p.bs = static_cast<const float*>(wt.s13);
  p.K = cfg.hidden;
  p.N = 2 * cfg.inter;
  p.ntn_magic = div_magic(p.N / kImgBRows);
  p.hq = ws + L.hq;
  p.hs = reinterpret_cast<float*>(ws + L.hs);
  return cfg.activation != AFD_ACT_SWIGLU ? launch_fmt<kGateUpParam>(p, cfg, plan, stream)
                                         : launch_fmt<kGateUp>(p, cfg, plan, stream);
}

int launch_rows_down(const afd_moe_cfg& cfg, const afd_expert_weights& wt, uint8_t* ws,
                     const afd_ws_layout& L, const RowsPlan& plan, hipStream_t stream) {
  RowsArgs p = rows_args(cfg, ws, L, plan);
  p.a = ws + L.hq;
  p.as = ws + L.hs;
  p.b = static_cast<const uint8_t*>(wt.w2);
  p.bs = static_cast<const float*>(wt.s2);
  p.K = cfg.inter;
  p.N = cfg.hidden;
  p.ntn_magic = div_magic(p.N / kImgBRows);
  p.y = reinterpret_cast<uint16_t*>(ws + L.y);
  return launch_fmt<kDown>(p, cfg, plan, stream);
}

}  // namespace afd
