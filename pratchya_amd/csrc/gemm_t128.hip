// GEMM on 128-row output tiles for products that leave the 256x256 persistent
// kernel (gemm.hip) short of tiles, and for the f32-accurate products of the
// quantized Linear's backward, whose operands it reads as exact bf16 planes.
//
//   C[m][n] = sum over segments s, k of A_s[m][k] * B_s[n][k]
//
// A segment multiplies one plane of A with one plane of B; an operand's planes
// are bf16 matrices of one shape, a fixed stride apart, K-contiguous or K-major.
// An f32 operand is up to three exact planes; one that is exact in a single
// plane is read where it lies, with no packed copy.  With FP8 operands (BF false) there is one segment and a K step
// is one 128-wide block whose e8m0 bytes the MFMA applies.
//
// One workgroup of 4 waves computes a TM x 128 tile (TM 128: waves 2 x 2, each
// 64 x 64; TM 32: each wave 32 x 32 of the tile's 128 columns) over one slice
// of the K steps; two stages of 128 bytes of K per row go HBM -> LDS by DMA,
// one barrier per step, and two workgroups share a CU, so that one's MFMAs run
// under the other's barrier and LDS reads.  Splitting K (splits > 1) fills the
// chip where the tiles alone do not: the slices write f32 partials, which
// k_reduce_slices sums in slice order (deterministic) with the same epilogues.
//
// Bound: a step's LDS traffic (64 KB of fragment reads and 32 KB of DMA writes
// per workgroup) takes about as long as its MFMAs, so the rate tops out near
// half of the matrix peak: 8192^3 bf16 1014 us (1.08 PFLOP/s; the 256x256
// kernel 805).  Short of tiles it wins: [4096, 8192] . [8192, 2048] 124 us
// against 174, [1024, 6144] . [6144, 1024] 26 against 123.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <numeric>
#include <type_traits>

#include "pratchya_fp8.h"
#include "quant_device.h"

int pratchya_set_error(int code, const char* fmt, ...);
int pratchya_quantize_dequantize_sum(const float* part, int parts, int64_t n_groups, void* out, bool out_bf16,
                                     bool fix_nan, uint8_t* sc_fp8, float* sc_fp32, hipStream_t st);

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v8i __attribute__((ext_vector_type(8)));
typedef int v2i __attribute__((ext_vector_type(2)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef short v4s __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) void lds_void;
typedef __attribute__((address_space(3))) v4s lds_v4s;

constexpr int KB = 128;                  // bytes of K per row and step
constexpr int TN = 128;                  // output columns of a tile

// One operand.  Scales (FP8: both operands; bf16: B only): the block of (row,
// step s of the plane) is row / r_div * s_r + (s * sk2 >> 1), its group that
// >> kg_sh.
struct OpArgs {
  const uint8_t* p;
  const uint8_t* e8;
  const float* g32;
  uint32_t ld, bytes;                    // row stride, readable bytes
  uint32_t pstride;                      // bytes from a plane to the next
  uint32_t e8_bytes, g32_bytes;
  uint32_t r_div, s_r, sk2, kg_sh;
  uint32_t planes, planes_alt;           // plane of segment s: 4 bits at 4 s
};

struct T128Args {
  OpArgs a, b;
  void* C;
  float* part;                           // splits > 1: f32 partials [splits][M][N]
  const uint16_t* X;                     // OUT 2
  const uint32_t* flags;                 // bf16 planes, may be null: see k_gemm_t128
  int64_t ldc, ldx;
  int M, N, spp, segs, segs_short, span, splits, tiles_m, tiles_n;
  // independent products of one shape: bytes (A, B) and elements (C, X) from
  // one to the next
  int batch;
  int64_t a_bs, b_bs, c_bs, x_bs;
};

__device__ __forceinline__ int swz(int r) { return (r & 7) ^ ((r >> 3) & 1); }

__device__ __forceinline__ v8i join(v4i lo, v4i hi) { return v8i{lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w}; }

// 1 KB of a stage by LDS DMA (16 bytes per lane); scale loads.  Every offset is
// range-checked: past the operand's end they read zeros.
__device__ __forceinline__ void dma_kb(__amdgpu_buffer_rsrc_t rs, uint8_t* lds, uint32_t off) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_void*)lds, 16, off, 0, 0, 0);
}
__device__ __forceinline__ uint32_t load_word(__amdgpu_buffer_rsrc_t rs, uint32_t off) {
  return __builtin_amdgcn_raw_buffer_load_b32(rs, (int)off, 0, 0);
}
__device__ __forceinline__ uint32_t load_byte(__amdgpu_buffer_rsrc_t rs, uint32_t i) {
  return __builtin_amdgcn_raw_buffer_load_b8(rs, (int)i, 0, 0);
}
__device__ __forceinline__ float load_f32(__amdgpu_buffer_rsrc_t rs, uint32_t i) {
  return u2f(__builtin_amdgcn_raw_buffer_load_b32(rs, (int)(i * 4u), 0, 0));
}

__device__ __forceinline__ v4f load_f32x4(__amdgpu_buffer_rsrc_t rs, uint32_t off) {
  return __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(rs, (int)off, 0, 0));
}

// K-major bf16 fragment of 32 operand rows (see the K-major operand of
// gemm.hip): the stage holds 64 K rows of 256 bytes, 16-byte chunks
// XOR-swizzled by 4 * (k mod 4).
__device__ __forceinline__ v4i tr_pair(const uint8_t* p0, const uint8_t* p1) {
  const v4s a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s*)p0);
  const v4s b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s*)p1);
  const v2i x = __builtin_bit_cast(v2i, a), y = __builtin_bit_cast(v2i, b);
  return v4i{x.x, x.y, y.x, y.y};
}
template <int SECOND>                      // K row of the second MFMA's values
__device__ __forceinline__ v8i read_frag_tn(const uint8_t* base) {
  return join(tr_pair(base, base + 4 * 256), tr_pair(base + SECOND * 256, base + (SECOND + 4) * 256));
}

// The mantissa of a group maximum, in [1, 2) ([0, 1) for a subnormal one): the
// bf16 plane holds the power of two (pratchya_planes, POW2).  0 and
// non-finite maxima count as 1 (their blocks' planes are 0, or already not
// finite).
__device__ __forceinline__ float mantissa_unit(float g) {
  const uint32_t b = f2u(g) & 0x7FFFFFFFu;
  const float normal = u2f((f2u(g) & 0x807FFFFFu) | 0x3F800000u);
  const float unit = b < 0x00800000u ? g * 0x1p126f : normal;
  return b - 1u < 0x7F7FFFFFu ? unit : 1.0f;    // selects: branches here would cut the step into pieces
}

// 1.5 x - 0.5 b on bf16 pairs, each operation rounded (k_ns_combine's bits).
__device__ __forceinline__ uint32_t ns_pair(uint32_t xw, uint32_t bw) {
  const uint32_t xr = pack_bf16x2(1.5f * u2f(xw << 16), 1.5f * u2f(xw & 0xFFFF0000u));
  const uint32_t br = pack_bf16x2(0.5f * u2f(bw << 16), 0.5f * u2f(bw & 0xFFFF0000u));
  return pack_bf16x2(u2f(xr << 16) - u2f(br << 16), u2f(xr & 0xFFFF0000u) - u2f(br & 0xFFFF0000u));
}

#define PINNED_WAITCNT(imm)            \
  do {                                 \
    __builtin_amdgcn_sched_barrier(0); \
    __builtin_amdgcn_s_waitcnt(imm);   \
    __builtin_amdgcn_sched_barrier(0); \
  } while (0)

__device__ __forceinline__ void wg_barrier() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_barrier" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// OUT 0: f32, 1: bf16, 2: bf16 1.5 X - 0.5 C.  SC 0: no scales, 1: FP8, both
// operands' e8m0 bytes and group maxima, 2: bf16, the mantissas of B's group
// maxima, 3 and 4: bf16 power-of-two planes of payloads quantized in blocks of
// 16 or 32 along K, the mantissas of both operands' group maxima per block: an
// MFMA's sums over one block (two MFMAs' over 32) join the total times both.
// The joins (16 multiply-adds per lane and MFMA, 64 clocks beside its 32) run
// as a pipeline with the MFMAs (fine_step), where one after the other they left
// both units waiting: forward of 8192 x [4096, 4096] in blocks of 32 469 -> 426
// us, four fifths of it the product (400 us by itself at a trace's lower clocks;
// the six-pair f32 product took 1585).  flags (bf16): flags[0] == 0 says that the
// planes of the segments past segs_short are all zero (the segments are left
// out); flags[1] != 0 that B's plane 0 holds non-finite values, which may take
// part in the first segment only (0 * inf): the others then read planes_alt, a
// copy without.
template <bool BF, int TM, bool TNA, bool TNB, int SC, int OUT>
__global__ __launch_bounds__(256, 2) void k_gemm_t128(T128Args p) {
  static_assert(BF || (!TNA && !TNB), "K-major operands are bf16");
  static_assert(TM == 128 || (TM == 32 && !TNA), "a K-major A stage holds 128 rows");
  constexpr int MI = TM == 128 ? 2 : 1, NI = MI;
  constexpr int WN = NI * 32;                            // columns of a wave
  constexpr int A_BYTES = TM * KB, STAGE = A_BYTES + TN * KB;
  constexpr int NA = TM / 32;                            // A DMA instructions per wave and stage
  constexpr bool FINE = SC >= 3;
  constexpr int FB = SC == 3 ? 16 : 32, KBS = 64 / FB;   // block size, blocks of a step
  __shared__ __attribute__((aligned(1024))) uint8_t lds[2 * STAGE];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = TM == 128 ? (wave & 1) : 0, wn = TM == 128 ? (wave >> 1) : wave;
  const int l32 = lane & 31, lhi = lane >> 5;

  // workgroup -> (slice, tile): each XCD (workgroups are dealt to the 8 in
  // turn) takes consecutive numbers, which walk bands of up to 8 tile rows of
  // one slice, so that it shares few panels in its L2
  const int tiles = p.tiles_m * p.tiles_n, total = tiles * p.splits * p.batch;
  int L = blockIdx.x;
  if (total % 8 == 0) L = (L & 7) * (total >> 3) + (L >> 3);
  const int unit = L / tiles;
  L -= unit * tiles;
  const int slice = unit % p.splits, bi = unit / p.splits;
  const int gm = p.tiles_m < 8 ? p.tiles_m : 8;
  const int band = L / (gm * p.tiles_n);
  const int in_band = min(p.tiles_m - band * gm, gm);
  const int w = L - band * gm * p.tiles_n;
  const int m0 = (band * gm + w % in_band) * TM, n0 = (w / in_band) * TN;

  uint32_t planes_a = p.a.planes, planes_b = p.b.planes;
  int segs = p.segs;
  if (BF && p.flags) {
    if (__builtin_amdgcn_readfirstlane(p.flags[0]) == 0u) segs = p.segs_short;
    if (__builtin_amdgcn_readfirstlane(p.flags[1]) != 0u) planes_b = p.b.planes_alt;
  }
  const int steps = segs * p.spp;
  const int k_begin = (int)((uint32_t)slice * (uint32_t)steps / (uint32_t)p.splits);
  const int k_end = (int)((uint32_t)(slice + 1) * (uint32_t)steps / (uint32_t)p.splits);

  constexpr int kFlags = 0x00020000;
  const __amdgpu_buffer_rsrc_t rs_a = __builtin_amdgcn_make_buffer_rsrc((void*)(p.a.p + bi * p.a_bs), 0, (int)p.a.bytes, kFlags);
  const __amdgpu_buffer_rsrc_t rs_b = __builtin_amdgcn_make_buffer_rsrc((void*)(p.b.p + bi * p.b_bs), 0, (int)p.b.bytes, kFlags);
  const __amdgpu_buffer_rsrc_t rs_ea = __builtin_amdgcn_make_buffer_rsrc((void*)p.a.e8, 0, (int)p.a.e8_bytes, kFlags);
  const __amdgpu_buffer_rsrc_t rs_eb = __builtin_amdgcn_make_buffer_rsrc((void*)p.b.e8, 0, (int)p.b.e8_bytes, kFlags);
  const __amdgpu_buffer_rsrc_t rs_ga = __builtin_amdgcn_make_buffer_rsrc((void*)p.a.g32, 0, (int)p.a.g32_bytes, kFlags);
  const __amdgpu_buffer_rsrc_t rs_gb = __builtin_amdgcn_make_buffer_rsrc((void*)p.b.g32, 0, (int)p.b.g32_bytes, kFlags);

  // Per-lane byte offsets of the stage's DMA instructions at K step 0 (the
  // whole offset goes through the range check: rows past the end read zeros).
  // K-contiguous: instruction i loads rows 8 i .. 8 i + 7 of the wave's, 128
  // bytes each; K-major: K rows 4 i .. 4 i + 3 of the wave's 16, 256 bytes.
  uint32_t oa[NA], ob[4];
#pragma unroll
  for (int i = 0; i < NA; ++i) {
    if constexpr (TNA) oa[i] = (uint32_t)(wave * 16 + i * 4 + (lane >> 4)) * p.a.ld +
                               (uint32_t)(m0 * 2 + (((lane & 15) ^ ((lane >> 4) << 2)) << 4));
    else oa[i] = (uint32_t)(m0 + wave * 8 * NA + i * 8 + (lane >> 3)) * p.a.ld +
                 (uint32_t)(((lane & 7) ^ (lane >> 3) ^ ((wave * NA + i) & 1)) << 4);
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if constexpr (TNB) ob[i] = (uint32_t)(wave * 16 + i * 4 + (lane >> 4)) * p.b.ld +
                               (uint32_t)(n0 * 2 + (((lane & 15) ^ ((lane >> 4) << 2)) << 4));
    else ob[i] = (uint32_t)(n0 + wave * 32 + i * 8 + (lane >> 3)) * p.b.ld +
                 (uint32_t)(((lane & 7) ^ (lane >> 3) ^ (i & 1)) << 4);
  }
  const uint32_t step_a = TNA ? 64u * p.a.ld : (uint32_t)KB, step_b = TNB ? 64u * p.b.ld : (uint32_t)KB;

  // row block indices of the lane's scale entries
  uint32_t ra[MI], rb[NI], rg[NI][4];
  if constexpr (SC == 1) {
#pragma unroll
    for (int i = 0; i < MI; ++i) ra[i] = (uint32_t)(m0 + wm * 64 + i * 32 + l32) / p.a.r_div * p.a.s_r;
#pragma unroll
    for (int i = 0; i < NI; ++i) rb[i] = (uint32_t)(n0 + wn * WN + i * 32 + l32) / p.b.r_div * p.b.s_r;
  }
  // Fine blocks: A's mantissas of a step are one row's KBS (16) or one (32: two
  // blocks share a group) consecutive group maxima; the wave's of B, one per
  // block of K and of its columns, are loaded one per lane and handed out as
  // scalars.
  uint32_t fa_row[MI];
  const int fq_k = lane / (WN / FB) % KBS, fq_n = lane % (WN / FB);
  uint32_t fb_n = 0;
  if constexpr (FINE) {
#pragma unroll
    for (int i = 0; i < MI; ++i) fa_row[i] = (uint32_t)(m0 + wm * 64 + i * 32 + l32) * (uint32_t)p.spp * (SC == 3 ? 16u : 4u);
    fb_n = (uint32_t)(n0 + wn * WN) / FB + (uint32_t)fq_n;
  }
  if constexpr (SC == 1 || SC == 2) {
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        rg[i][j] = (uint32_t)(n0 + wn * WN + i * 32 + 8 * j + 4 * lhi) / p.b.r_div * p.b.s_r;
  }

  // next step's e8m0 bytes and, at a span's start, group maxima
  uint32_t ea_n[MI], eb_n[NI];
  v4f fa_n[MI];
  float fb_g = 1.0f;
  // (a last word that the array holds in part would be out of range: zeros)
  const bool a_words = SC == 1 && p.a.sk2 == 2 && p.a.s_r % 4 == 0 && p.a.e8_bytes % 4 == 0 &&
                       (reinterpret_cast<uintptr_t>(p.a.e8) & 3) == 0;
  int a_shift = 0;
  float ga_n[MI], gb_n[NI][4];
  int seg = k_begin / p.spp, s = k_begin - seg * p.spp;
  int in_span = s % p.span;                // of the next step to load
  bool start_n = true;                     // the loaded step starts a span (or the slice)
  uint8_t* dma_st = lds;
  uint32_t dma_ka = 0, dma_kb_ = 0;
  auto dma = [&](int i) {                  // instruction i of the stage's load
    if (i < NA) dma_kb(rs_a, dma_st + (wave * NA + i) * 1024, oa[i] + dma_ka);
    else dma_kb(rs_b, dma_st + A_BYTES + (wave * 4 + i - NA) * 1024, ob[i - NA] + dma_kb_);
  };
  auto load_stage = [&](uint8_t* st, bool first) {
    const uint32_t ka = ((planes_a >> (4 * seg)) & 15u) * p.a.pstride + (uint32_t)s * step_a;
    const uint32_t kb = ((planes_b >> (4 * seg)) & 15u) * p.b.pstride + (uint32_t)s * step_b;
    dma_st = st;
    dma_ka = ka;
    dma_kb_ = kb;
    if constexpr (SC == 1) {
      const uint32_t ta = (uint32_t)s * p.a.sk2 >> 1, tb = (uint32_t)s * p.b.sk2 >> 1;
      // A's bytes of consecutive steps lie side by side: one aligned word holds
      // four steps' where every row starts on a word
      if (!a_words) {
#pragma unroll
        for (int i = 0; i < MI; ++i) ea_n[i] = load_byte(rs_ea, ra[i] + ta);
      } else if (first || (s & 3) == 0) {
#pragma unroll
        for (int i = 0; i < MI; ++i) ea_n[i] = load_word(rs_ea, (ra[i] + ta) & ~3u);
      }
      a_shift = a_words ? (s & 3) * 8 : 0;
#pragma unroll
      for (int i = 0; i < NI; ++i) eb_n[i] = load_byte(rs_eb, rb[i] + tb);
    }
    if constexpr (FINE) {
#pragma unroll
      for (int i = 0; i < MI; ++i) {
        if constexpr (SC == 3) fa_n[i] = load_f32x4(rs_ga, fa_row[i] + (uint32_t)s * 16u);
        else fa_n[i].x = load_f32(rs_ga, (fa_row[i] >> 2) + (uint32_t)s);
      }
      fb_g = load_f32(rs_gb, (((uint32_t)s * KBS + (uint32_t)fq_k) * p.b.s_r + fb_n) >> p.b.kg_sh);
    }
    if constexpr (SC == 1 || SC == 2) {
      start_n = first || in_span == 0;
      if (start_n) {
        const uint32_t ta = (uint32_t)s * p.a.sk2 >> 1, tb = (uint32_t)s * p.b.sk2 >> 1;
        if constexpr (SC == 1) {
#pragma unroll
          for (int i = 0; i < MI; ++i)
            ga_n[i] = load_f32(rs_ga, (ra[i] + ta) >> p.a.kg_sh);
        }
#pragma unroll
        for (int i = 0; i < NI; ++i)
#pragma unroll
          for (int j = 0; j < 4; ++j)
            gb_n[i][j] = load_f32(rs_gb, (rg[i][j] + tb) >> p.b.kg_sh);
      }
    }
    if (++in_span == p.span) in_span = 0;
    if (++s == p.spp) {
      s = 0;
      in_span = 0;
      ++seg;
    }
  };

  v16f acc[MI][NI], tot[SC != 0 ? MI : 1][SC != 0 ? NI : 1];
#pragma unroll
  for (int mi = 0; mi < MI; ++mi)
#pragma unroll
    for (int ni = 0; ni < NI; ++ni) {
      acc[mi][ni] = v16f{0};
      if constexpr (SC != 0) tot[mi][ni] = v16f{0};
    }
  // units of the span being accumulated; a span's sums join the total scaled
  // by them (FP8: the group maxima over 128 each; a maximum of 0 has zero
  // payloads)
  float ua[MI], ub[NI][4];
  auto flush = [&]() {
    if constexpr (SC == 1 || SC == 2) {
#pragma unroll
      for (int mi = 0; mi < MI; ++mi)
#pragma unroll
        for (int ni = 0; ni < NI; ++ni)
#pragma unroll
          for (int v = 0; v < 16; ++v) {
            const float u = SC == 1 ? ua[mi] * ub[ni][v >> 2] : ub[ni][v >> 2];
            tot[mi][ni][v] += acc[mi][ni][v] * u;
            acc[mi][ni][v] = 0.0f;
          }
    }
  };

  int ch[2][2];
  {
    const int sw = swz(l32);
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int h = 0; h < 2; ++h) ch[ks][h] = ((ks * 4 + (FINE ? h * 2 + lhi : lhi * 2 + h)) ^ sw) << 4;
  }
  const int g16 = lane >> 4, j16 = lane & 15;
  // (fine blocks: an MFMA's 16 K values are consecutive, so that they are one
  // block's: lanes 32-63 hold its upper 8)
  const int tn_kc = ((FINE ? 8 : 16) * (g16 >> 1) + (j16 >> 2)) * 256 + (2 * (g16 & 1) + ((j16 & 3) >> 1)) * 16 + (j16 & 1) * 8;
  const int tn_s = j16 >> 2;
  // a 32-row block of 128-byte rows keeps a row's swizzle (it depends on l32)
  auto frag = [&](const uint8_t* base, auto tn, int blk, int ks) {
    if constexpr (decltype(tn)::value)
      return read_frag_tn<FINE ? 16 : 8>(base + tn_kc + ks * 32 * 256 + ((blk ^ tn_s) << 6));
    else {
      const uint8_t* r = base + (blk * 32 + l32) * KB;
      return join(*reinterpret_cast<const v4i*>(r + ch[ks][0]), *reinterpret_cast<const v4i*>(r + ch[ks][1]));
    }
  };

  // Fine blocks: a step's units (a 32x32 output tile, half a step of K) run as a
  // pipeline, unit u's MFMAs issued ahead of the multiply-adds that join unit
  // u - 1's sums to the totals; the last unit's join carries over to the next
  // step, under its fragment reads.  The next stage's DMA goes out without a
  // branch, also in the last step (range-checked bytes that nobody reads).
  v16f pc[SC == 3 ? 2 : 1];
  float pu[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  if constexpr (FINE) {
#pragma unroll
    for (int h = 0; h < (SC == 3 ? 2 : 1); ++h) pc[h] = v16f{0};
  }
  auto fine_join = [&](int mi, int ni) {
    if constexpr (SC == 3) {
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int v = 0; v < 16; ++v) tot[mi][ni][v] += pc[h][v] * pu[h * 2 + (v >> 3)];
    } else if constexpr (SC == 4) {
#pragma unroll
      for (int v = 0; v < 16; ++v) tot[mi][ni][v] += pc[0][v] * pu[0];
    }
  };
  auto fine_step = [&](const uint8_t* st, const float (&um)[MI][4], const float* un) {
    if constexpr (FINE) {
      constexpr int UNITS = MI * NI;                       // per half step
      constexpr int PER = (NA + 4 + UNITS - 1) / UNITS;    // DMA instructions beside each unit of the first half
      v8i fa[2][MI], fb[2][NI];
      auto reads = [&](int ks) {
#pragma unroll
        for (int i = 0; i < MI; ++i) fa[ks][i] = frag(st, std::bool_constant<TNA>{}, wm * 2 + i, ks);
#pragma unroll
        for (int i = 0; i < NI; ++i) fb[ks][i] = frag(st + A_BYTES, std::bool_constant<TNB>{}, wn * NI + i, ks);
      };
      reads(0);
      __builtin_amdgcn_sched_barrier(0);
      fine_join(MI - 1, NI - 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < 2 * UNITS; ++u) {
        const int ks = u / UNITS, mi = u % UNITS / NI, ni = u % NI;
        const v8i a = fb[ks][ni], b = fa[ks][mi];
        const bf16x8_t a0 = __builtin_bit_cast(bf16x8_t, v4i{a.s0, a.s1, a.s2, a.s3});
        const bf16x8_t b0 = __builtin_bit_cast(bf16x8_t, v4i{b.s0, b.s1, b.s2, b.s3});
        const bf16x8_t a1 = __builtin_bit_cast(bf16x8_t, v4i{a.s4, a.s5, a.s6, a.s7});
        const bf16x8_t b1 = __builtin_bit_cast(bf16x8_t, v4i{b.s4, b.s5, b.s6, b.s7});
        v16f c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a0, b0, v16f{0}, 0, 0, 0), d;
        if constexpr (SC == 3) d = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a1, b1, v16f{0}, 0, 0, 0);
        else c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a1, b1, c, 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        if (u == 0) reads(1);
        if (ks == 0) {
#pragma unroll
          for (int i = u * PER; i < (u + 1) * PER && i < NA + 4; ++i) dma(i);
        }
        if (u > 0) fine_join((u - 1) % UNITS / NI, (u - 1) % NI);
        pc[0] = c;
        if constexpr (SC == 3) {
          pc[1] = d;
#pragma unroll
          for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int q = 0; q < 2; ++q)
              pu[h * 2 + q] = um[mi][ks * 2 + h] * un[(ks * 2 + h) * (WN / FB) + ni * 2 + q];
        } else {
          pu[0] = um[mi][0] * un[ks * (WN / FB) + ni];
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };

  // bf16.  Row-contiguous operands: the next stage's DMA goes out first, for the
  // longest lead ([4096, 2048] . [2048, 8192] 130 us, behind the reads 138).  A
  // K-major operand takes four times the reads: the second half's go out under
  // the first half's MFMAs and the DMA behind the step's last read, since a read
  // after it would wait for the DMA, which the compiler takes to write what it
  // reads ([2048, 8192] . [8192, 8192], both K-major: 289 -> 264 us).
  auto bf16_step = [&](const uint8_t* st, bool more, uint8_t* next) {
    if constexpr (BF && !FINE) {
      constexpr int UNITS = MI * NI;
      constexpr bool EARLY = !TNA && !TNB;
      v8i fa[2][MI], fb[2][NI];
      auto reads = [&](int ks) {
#pragma unroll
        for (int i = 0; i < MI; ++i) fa[ks][i] = frag(st, std::bool_constant<TNA>{}, wm * 2 + i, ks);
#pragma unroll
        for (int i = 0; i < NI; ++i) fb[ks][i] = frag(st + A_BYTES, std::bool_constant<TNB>{}, wn * NI + i, ks);
      };
      auto stage_dma = [&]() {
        __builtin_amdgcn_sched_barrier(0);
        if (more) {
#pragma unroll
          for (int i = 0; i < NA + 4; ++i) dma(i);
        }
        __builtin_amdgcn_sched_barrier(0);
      };
      if (more) load_stage(next, false);
      if (EARLY) stage_dma();
      reads(0);
      if (!EARLY) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < 2 * UNITS; ++u) {
        const int ks = u / UNITS, mi = u % UNITS / NI, ni = u % NI;
        if (EARLY && u == UNITS) reads(1);
        const v8i a = fb[ks][ni], b = fa[ks][mi];
        acc[mi][ni] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
            __builtin_bit_cast(bf16x8_t, v4i{a.s0, a.s1, a.s2, a.s3}),
            __builtin_bit_cast(bf16x8_t, v4i{b.s0, b.s1, b.s2, b.s3}), acc[mi][ni], 0, 0, 0);
        acc[mi][ni] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
            __builtin_bit_cast(bf16x8_t, v4i{a.s4, a.s5, a.s6, a.s7}),
            __builtin_bit_cast(bf16x8_t, v4i{b.s4, b.s5, b.s6, b.s7}), acc[mi][ni], 0, 0, 0);
        if (!EARLY && u == 0) {
          __builtin_amdgcn_sched_barrier(0);
          reads(1);
          stage_dma();
        }
      }
    }
  };

  // FP8: as with a K-major operand (1000 x [2176, 2944] 24.8 -> 24.0 us); the DMA
  // of the last step goes out too (range-checked bytes that nobody reads).
  auto fp8_step = [&](const uint8_t* st, const uint32_t* ea, const uint32_t* eb) {
    if constexpr (!BF) {
      constexpr int UNITS = MI * NI;
      v8i fa[2][MI], fb[2][NI];
      auto reads = [&](int ks) {
#pragma unroll
        for (int i = 0; i < MI; ++i) fa[ks][i] = frag(st, std::bool_constant<TNA>{}, wm * 2 + i, ks);
#pragma unroll
        for (int i = 0; i < NI; ++i) fb[ks][i] = frag(st + A_BYTES, std::bool_constant<TNB>{}, wn * NI + i, ks);
      };
      reads(0);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < 2 * UNITS; ++u) {
        const int ks = u / UNITS, mi = u % UNITS / NI, ni = u % NI;
        acc[mi][ni] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(fb[ks][ni], fa[ks][mi], acc[mi][ni], 0, 0, 0,
                                                                     (int)eb[ni], 0, (int)ea[mi]);
        if (u == 0) {
          __builtin_amdgcn_sched_barrier(0);
          reads(1);
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int i = 0; i < NA + 4; ++i) dma(i);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
  };

  if (k_begin < k_end) {
    load_stage(lds, true);
#pragma unroll
    for (int i = 0; i < NA + 4; ++i) dma(i);
    for (int k = k_begin; k < k_end; ++k) {
      uint8_t* st = lds + ((k - k_begin) & 1) * STAGE;
      PINNED_WAITCNT(0);                   // this wave's share of stage k (and its reads of stage k - 1) is done
      wg_barrier();
      uint32_t ea[MI], eb[NI];
      if constexpr (SC == 1) {
#pragma unroll
        for (int i = 0; i < MI; ++i) ea[i] = ea_n[i] >> a_shift;
#pragma unroll
        for (int i = 0; i < NI; ++i) eb[i] = eb_n[i];
      }
      float um[MI][4], un[FINE ? KBS * (WN / FB) : 1];
      if constexpr (FINE) {
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
          for (int j = 0; j < (SC == 3 ? 4 : 1); ++j) um[i][j] = mantissa_unit(fa_n[i][j]);
        const float b = mantissa_unit(fb_g);
#pragma unroll
        for (int i = 0; i < KBS * (WN / FB); ++i) un[i] = u2f(readlane_u32(f2u(b), i));
      }
      if constexpr (SC == 1 || SC == 2) {
        if (start_n) {
          if (k != k_begin) flush();
#pragma unroll
          for (int i = 0; i < MI; ++i)
            if constexpr (SC == 1) ua[i] = ga_n[i] * 0.0078125f;
#pragma unroll
          for (int i = 0; i < NI; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) ub[i][j] = SC == 1 ? gb_n[i][j] * 0.0078125f : mantissa_unit(gb_n[i][j]);
        }
      }
      uint8_t* next = lds + ((k - k_begin + 1) & 1) * STAGE;
      if constexpr (BF && !FINE) {
        bf16_step(st, k + 1 < k_end, next);
      } else {
        load_stage(next, false);
        if constexpr (FINE) fine_step(st, um, un);
        else fp8_step(st, ea, eb);
      }
    }
    flush();
    if constexpr (FINE) fine_join(MI - 1, NI - 1);
    if constexpr (FINE || !BF) PINNED_WAITCNT(0);          // the last step's DMA
  }

  // Epilogue: 32 rows of the wave's columns at a time through the wave's part
  // of the LDS (free once every wave has read its last stage), then whole row
  // pieces to C or the slice's partial.
  constexpr int PITCH = WN * 4 + 16;
  static_assert(4 * 32 * PITCH <= 2 * STAGE, "staging fits the stages");
  __syncthreads();
  uint8_t* stg = lds + wave * (32 * PITCH);
  const int col0 = n0 + wn * WN;
#pragma unroll
  for (int mi = 0; mi < MI; ++mi) {
#pragma unroll
    for (int ni = 0; ni < NI; ++ni)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        v4f c;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if constexpr (SC != 0) c[i] = tot[mi][ni][4 * j + i];
          else c[i] = acc[mi][ni][4 * j + i];
        }
        *reinterpret_cast<v4f*>(stg + l32 * PITCH + (ni * 32 + 8 * j + 4 * lhi) * 4) = c;
      }
    __builtin_amdgcn_s_waitcnt(0xC07F);
    __builtin_amdgcn_wave_barrier();
    const int row0 = m0 + wm * 64 + mi * 32;
    if (OUT == 0 || p.splits > 1) {
      float* out = p.splits > 1 ? p.part + (int64_t)unit * p.M * p.N : static_cast<float*>(p.C) + bi * p.c_bs;
      const int64_t ld = p.splits > 1 ? (int64_t)p.N : p.ldc;
#pragma unroll
      for (int it = 0; it < WN / 8; ++it) {
        const int q = it * 64 + lane, r = q / (WN / 4), c = (q % (WN / 4)) * 4;
        const v4f v = *reinterpret_cast<const v4f*>(stg + r * PITCH + c * 4);
        if (row0 + r < p.M && col0 + c < p.N) *reinterpret_cast<v4f*>(out + (row0 + r) * ld + col0 + c) = v;
      }
    } else {
      uint16_t* out = static_cast<uint16_t*>(p.C) + bi * p.c_bs;
#pragma unroll
      for (int it = 0; it < WN / 16; ++it) {
        const int q = it * 64 + lane, r = q / (WN / 8), c = (q % (WN / 8)) * 8;
        const v4f v = *reinterpret_cast<const v4f*>(stg + r * PITCH + c * 4);
        const v4f x = *reinterpret_cast<const v4f*>(stg + r * PITCH + c * 4 + 16);
        v4i o = {(int)pack_bf16x2(v.x, v.y), (int)pack_bf16x2(v.z, v.w), (int)pack_bf16x2(x.x, x.y),
                 (int)pack_bf16x2(x.z, x.w)};
        if (row0 + r < p.M && col0 + c < p.N) {
          if constexpr (OUT == 2) {
            const v4i xv = *reinterpret_cast<const v4i*>(p.X + bi * p.x_bs + (row0 + r) * p.ldx + col0 + c);
#pragma unroll
            for (int i = 0; i < 4; ++i) o[i] = (int)ns_pair((uint32_t)xv[i], (uint32_t)o[i]);
          }
          *reinterpret_cast<v4i*>(out + (row0 + r) * p.ldc + col0 + c) = o;
        }
      }
    }
    __builtin_amdgcn_s_waitcnt(0xC07F);
    __builtin_amdgcn_wave_barrier();
  }
}

// C = the slices' sum, in slice order, with k_gemm_t128's epilogues.
template <int OUT>
__global__ __launch_bounds__(256) void k_reduce_slices(const float* part, int splits, int M, int N,
                                                       void* C, int64_t ldc,
                                                       const uint16_t* X, int64_t ldx, int64_t c_bs,
                                                       int64_t x_bs) {
  part += (int64_t)blockIdx.y * splits * M * N;
  C = static_cast<uint8_t*>(C) + (int64_t)blockIdx.y * c_bs * (OUT == 0 ? 4 : 2);
  if constexpr (OUT == 2) X += (int64_t)blockIdx.y * x_bs;
  constexpr int CH = OUT == 0 ? 4 : 8;
  const int per_row = N / CH;
  const int64_t n = (int64_t)M * per_row, stride = (int64_t)M * N;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
    const int64_t r = i / per_row;
    const int c = (int)(i - r * per_row) * CH;
    const float* src = part + r * N + c;
    v4f v[CH / 4];
#pragma unroll
    for (int h = 0; h < CH / 4; ++h) v[h] = *reinterpret_cast<const v4f*>(src + 4 * h);
#pragma unroll 4
    for (int s = 1; s < splits; ++s)
#pragma unroll
      for (int h = 0; h < CH / 4; ++h) v[h] += *reinterpret_cast<const v4f*>(src + s * stride + 4 * h);
    if constexpr (OUT == 0) {
      *reinterpret_cast<v4f*>(static_cast<float*>(C) + r * ldc + c) = v[0];
    } else {
      v4i o = {(int)pack_bf16x2(v[0].x, v[0].y), (int)pack_bf16x2(v[0].z, v[0].w), (int)pack_bf16x2(v[1].x, v[1].y),
               (int)pack_bf16x2(v[1].z, v[1].w)};
      if constexpr (OUT == 2) {
        const v4i xv = *reinterpret_cast<const v4i*>(X + r * ldx + c);
#pragma unroll
        for (int h = 0; h < 4; ++h) o[h] = (int)ns_pair((uint32_t)xv[h], (uint32_t)o[h]);
      }
      *reinterpret_cast<v4i*>(static_cast<uint16_t*>(C) + r * ldc + c) = o;
    }
  }
}

}  // namespace

extern "C" int64_t pratchya_gemm_span(int64_t rows, int64_t K, int64_t r_div, int64_t s_r, int64_t s_k, int64_t kg);

namespace {

constexpr int kMaxSplits = 32;

int t128_rows(int64_t M) { return M <= 32 ? 32 : 128; }

int t128_cus() {
  static int cached[64] = {0};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  if (!cached[dev]) {
    int v = 0;
    if (hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || v < 8) v = 256;
    cached[dev] = v;
  }
  return cached[dev];
}

// Slices of the K steps: as many as fill two workgroups per CU, each at least
// min_steps long (below that a slice's start and its partial cost more than
// the steps it takes off the others).
int t128_splits(int64_t M, int64_t N, int64_t steps, int64_t batch) {
  const int rows = t128_rows(M);
  const int64_t tiles = batch * ((M + rows - 1) / rows) * ((N + TN - 1) / TN);
  const int64_t min_steps = rows == 32 ? 2 : 4;
  int64_t s = 2 * t128_cus() / tiles;
  if (s > steps / min_steps) s = steps / min_steps;
  if (s > kMaxSplits) s = kMaxSplits;
  return s < 1 ? 1 : (int)s;
}

template <bool BF, int TM, bool TNA, bool TNB, int SC, int OUT>
void t128_launch(const T128Args& p, hipStream_t stream, bool reduce = true) {
  hipLaunchKernelGGL((k_gemm_t128<BF, TM, TNA, TNB, SC, OUT>), dim3((unsigned)(p.tiles_m * p.tiles_n * p.splits * p.batch)),
                     dim3(256), 0, stream, p);
  if (p.splits > 1 && reduce) {
    const int64_t n = (int64_t)p.M * (p.N / (OUT == 0 ? 4 : 8));
    const int64_t blocks = (n + 255) / 256;
    hipLaunchKernelGGL((k_reduce_slices<OUT>), dim3((unsigned)(blocks < 2048 ? blocks : 2048), (unsigned)p.batch),
                       dim3(256), 0, stream, p.part, p.splits, p.M, p.N, p.C, p.ldc, p.X, p.ldx, p.c_bs, p.x_bs);
  }
}

int t128_status(const char* who) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return pratchya_set_error(PRATCHYA_EHIP, "%s: launch failed: %s", who, hipGetErrorString(e));
  return PRATCHYA_OK;
}

int ilog2_exact(int64_t v) {
  for (int i = 0; i < 32; ++i)
    if (((int64_t)1 << i) == v) return i;
  return -1;
}

// Tiles, slices and the partials' workspace of one call.
int t128_shape(const char* who, T128Args* p, int64_t M, int64_t N, int64_t steps, void* ws, int64_t ws_bytes,
               int64_t batch = 1) {
  const int rows = t128_rows(M);
  p->M = (int)M;
  p->N = (int)N;
  p->tiles_m = (int)((M + rows - 1) / rows);
  p->tiles_n = (int)((N + TN - 1) / TN);
  p->splits = t128_splits(M, N, steps, batch);
  p->batch = (int)batch;
  if ((int64_t)p->tiles_m * p->tiles_n * p->splits * batch > INT32_MAX / 2)
    return pratchya_set_error(PRATCHYA_EUNSUPPORTED, "%s: too many tiles", who);
  const int64_t need = batch * p->splits * M * N * 4;
  if (p->splits > 1 && (!ws || ws_bytes < need || (reinterpret_cast<uintptr_t>(ws) & 15)))
    return pratchya_set_error(PRATCHYA_EINVAL, "%s: workspace of %lld bytes (16-byte aligned) needed", who, (long long)need);
  p->part = static_cast<float*>(ws);
  return PRATCHYA_OK;
}

constexpr int64_t kMaxOffset = (int64_t)UINT32_MAX;

}  // namespace

extern "C" int64_t pratchya_gemm_t128_workspace_bytes(int64_t M, int64_t N, int64_t steps, int64_t batch) {
  if (M < 1 || N < 1 || steps < 1 || M > INT32_MAX || N > INT32_MAX || batch < 1 || batch > 65535) return 0;
  const int s = t128_splits(M, N, steps, batch);
  return s > 1 ? batch * s * M * N * 4 : 0;
}

namespace {

// `reduce` false: the f32 slices (their count in *splits) stay in ws, C unused
// with more than one.
int bs_t128(const char* who, const uint8_t* A, int64_t lda, const uint8_t* a_sc8, const float* a_sc32,
            int64_t a_rdiv, int64_t a_sr, int64_t a_sk, int64_t a_kg, const uint8_t* B,
            int64_t ldb, const uint8_t* b_sc8, const float* b_sc32, int64_t b_rdiv,
            int64_t b_sr, int64_t b_sk, int64_t b_kg, int64_t M, int64_t N, int64_t K,
            void* C, int64_t ldc, int c_dtype, void* ws, int64_t ws_bytes,
            hipStream_t stream, bool reduce, int* splits) {
  if (M <= 0 || N <= 0 || K <= 0) {
    if (M < 0 || N < 0 || K < 0) return pratchya_set_error(PRATCHYA_EINVAL, "%s: negative size", who);
    return PRATCHYA_OK;
  }
  if (c_dtype != PRATCHYA_DT_F32 && c_dtype != PRATCHYA_DT_BF16)
    return pratchya_set_error(PRATCHYA_EINVAL, "%s: unsupported output dtype %d", who, c_dtype);
  const int chunk = c_dtype == PRATCHYA_DT_BF16 ? 8 : 4;
  if (K % KB || N % chunk)
    return pratchya_set_error(PRATCHYA_EUNSUPPORTED, "%s: K a multiple of 128 and N of %d (got %lld, %lld)", who, chunk,
                              (long long)K, (long long)N);
  if (!A || !B || !a_sc8 || !a_sc32 || !b_sc8 || !b_sc32 || !C)
    return pratchya_set_error(PRATCHYA_EINVAL, "%s: null buffer", who);
  if (lda < K || ldb < K || ldc < N || lda % 16 || ldb % 16 || ldc % chunk ||
      (reinterpret_cast<uintptr_t>(A) | reinterpret_cast<uintptr_t>(B) | reinterpret_cast<uintptr_t>(C)) % 16)
    return pratchya_set_error(PRATCHYA_EINVAL, "%s: leading dimensions / alignment not supported", who);
  if (a_rdiv < 1 || b_rdiv < 1 || a_kg < 1 || b_kg < 1 || a_sr < 0 || a_sk < 0 || b_sr < 0 || b_sk < 0)
    return pratchya_set_error(PRATCHYA_EINVAL, "%s: bad scale layout", who);
  const int ash = ilog2_exact(a_kg), bsh = ilog2_exact(b_kg);
  // B's group maxima are read per 4 rows
  const bool rows4 = b_rdiv % 4 == 0 || (b_rdiv == 1 && b_kg % (4 * b_sr) == 0 && b_sk % (4 * b_sr) == 0 && b_sr > 0);
  if (ash < 0 || bsh < 0 || !rows4)
    return pratchya_set_error(PRATCHYA_EUNSUPPORTED, "%s: groups of a power of two of blocks, shared by 4 rows of B", who);
  const int64_t nk = K / KB;
  const int64_t last_a = ((M - 1) / a_rdiv) * a_sr + (nk - 1) * a_sk, last_b = ((N - 1) / b_rdiv) * b_sr + (nk - 1) * b_sk;
  const int64_t Mr = (M + 127) / 128 * 128, Nr = (N + 127) / 128 * 128;
  if (Mr * lda + K > kMaxOffset || Nr * ldb + K > kMaxOffset || (Mr / a_rdiv + 1) * a_sr + nk * a_sk > INT32_MAX ||
      (Nr / b_rdiv + 1) * b_sr + nk * b_sk > INT32_MAX || M > INT32_MAX / 2 || N > INT32_MAX / 2 ||
      nk * a_sk > INT32_MAX / 2 || nk * b_sk > INT32_MAX / 2 || nk > (1 << 26))
    return pratchya_set_error(PRATCHYA_EUNSUPPORTED, "%s: operands beyond 32-bit offsets", who);
  T128Args p{};
  p.a = OpArgs{A, a_sc8, a_sc32, (uint32_t)lda, (uint32_t)((M - 1) * lda + K), 0, (uint32_t)(last_a + 1),
               (uint32_t)((last_a / a_kg + 1) * 4), (uint32_t)a_rdiv, (uint32_t)a_sr, (uint32_t)(2 * a_sk), (uint32_t)ash,
               0, 0};
  p.b = OpArgs{B, b_sc8, b_sc32, (uint32_t)ldb, (uint32_t)((N - 1) * ldb + K), 0, (uint32_t)(last_b + 1),
               (uint32_t)((last_b / b_kg + 1) * 4), (uint32_t)b_rdiv, (uint32_t)b_sr, (uint32_t)(2 * b_sk), (uint32_t)bsh,
               0, 0};
  p.C = C;
  p.ldc = ldc;
  p.spp = (int)nk;
  p.segs = p.segs_short = 1;
  p.span = (int)std::gcd(pratchya_gemm_span(M, K, a_rdiv, a_sr, a_sk, a_kg), pratchya_gemm_span(N, K, b_rdiv, b_sr, b_sk, b_kg));
  const int rc = t128_shape(who, &p, M, N, nk, ws, ws_bytes);
  if (rc) return rc;
  if (splits) *splits = p.splits;
  const bool bf = c_dtype == PRATCHYA_DT_BF16;
  if (t128_rows(M) == 32) {
    if (bf) t128_launch<false, 32, false, false, 1, 1>(p, stream);
    else t128_launch<false, 32, false, false, 1, 0>(p, stream, reduce);
  } else {
    if (bf) t128_launch<false, 128, false, false, 1, 1>(p, stream);
    else t128_launch<false, 128, false, false, 1, 0>(p, stream, reduce);
  }
  return t128_status(who);
}

}  // namespace

extern "C" int pratchya_gemm_bs_t128(const uint8_t* A, int64_t lda, const uint8_t* a_sc8, const float* a_sc32,
                                     int64_t a_rdiv, int64_t a_sr, int64_t a_sk, int64_t a_kg, const uint8_t* B,
                                     int64_t ldb, const uint8_t* b_sc8, const float* b_sc32, int64_t b_rdiv,
                                     int64_t b_sr, int64_t b_sk, int64_t b_kg, int64_t M, int64_t N, int64_t K,
                                     void* C, int64_t ldc, int c_dtype, void* ws, int64_t ws_bytes,
                                     hipStream_t stream) {
  return bs_t128("gemm_t128", A, lda, a_sc8, a_sc32, a_rdiv, a_sr, a_sk, a_kg, B, ldb, b_sc8, b_sc32, b_rdiv, b_sr,
                 b_sk, b_kg, M, N, K, C, ldc, c_dtype, ws, ws_bytes, stream, true, nullptr);
}

extern "C" int64_t pratchya_gemm_t128_fq_workspace_bytes(int64_t M, int64_t N, int64_t steps) {
  if (M < 1 || N < 1 || steps < 1 || M > INT32_MAX || N > INT32_MAX) return 0;
  return (int64_t)t128_splits(M, N, steps, 1) * M * N * 4;
}

// The slices' sum is requantized as it is read, in one launch of 6.3 us for 4 x
// [4096, 4096] where a reduction and the requantization took 7.9 and a second
// call from the host: the Linear 48 -> 35 us.
extern "C" int pratchya_gemm_bs_t128_fq(const uint8_t* A, int64_t lda, const uint8_t* a_sc8, const float* a_sc32,
                                        int64_t a_rdiv, int64_t a_sr, int64_t a_sk, int64_t a_kg, const uint8_t* B,
                                        int64_t ldb, const uint8_t* b_sc8, const float* b_sc32, int64_t b_rdiv,
                                        int64_t b_sr, int64_t b_sk, int64_t b_kg, int64_t M, int64_t N, int64_t K,
                                        void* y, int y_dtype, int fix_nan, uint8_t* sc_fp8, float* sc_fp32, void* ws,
                                        int64_t ws_bytes, hipStream_t stream) {
  const char* who = "gemm_t128_fq";
  if (M <= 0 || N <= 0 || K <= 0) {
    if (M < 0 || N < 0 || K < 0) return pratchya_set_error(PRATCHYA_EINVAL, "%s: negative size", who);
    return PRATCHYA_OK;
  }
  if (y_dtype != PRATCHYA_DT_F32 && y_dtype != PRATCHYA_DT_BF16)
    return pratchya_set_error(PRATCHYA_EINVAL, "%s: unsupported output dtype %d", who, y_dtype);
  if (M > INT32_MAX / 2 || N > INT32_MAX / 2 || N % 128 || M * N % 1024 || M * N / 1024 * 8 > (int64_t)UINT32_MAX - 16)
    return pratchya_set_error(PRATCHYA_EUNSUPPORTED, "%s: groups of 8 blocks of 128 columns (got %lld x %lld)", who,
                              (long long)M, (long long)N);
  if (!y || (!sc_fp8) != (!sc_fp32)) return pratchya_set_error(PRATCHYA_EINVAL, "%s: null buffer", who);
  if (reinterpret_cast<uintptr_t>(y) % 16 || reinterpret_cast<uintptr_t>(sc_fp8) % 8 ||
      reinterpret_cast<uintptr_t>(sc_fp32) % 4)
    return pratchya_set_error(PRATCHYA_EINVAL, "%s: alignment not supported", who);
  const int64_t need = K % KB ? 0 : pratchya_gemm_t128_fq_workspace_bytes(M, N, K / KB);
  if (!ws || ws_bytes < need) return pratchya_set_error(PRATCHYA_EINVAL, "%s: workspace of %lld bytes needed", who, (long long)need);
  int splits = 1;
  const int rc = bs_t128(who, A, lda, a_sc8, a_sc32, a_rdiv, a_sr, a_sk, a_kg, B, ldb, b_sc8, b_sc32, b_rdiv, b_sr,
                         b_sk, b_kg, M, N, K, ws, N, PRATCHYA_DT_F32, ws, ws_bytes, stream, false, &splits);
  if (rc) return rc;
  return pratchya_quantize_dequantize_sum(static_cast<const float*>(ws), splits, M * N / 1024, y,
                                          y_dtype == PRATCHYA_DT_BF16, fix_nan != 0, sc_fp8, sc_fp32, stream);
}

extern "C" int pratchya_gemm_bf16_planes(const void* A, int64_t lda, int64_t a_stride, int a_kmajor, int a_held,
                                         uint32_t a_planes, const void* B, int64_t ldb, int64_t b_stride, int b_kmajor,
                                         int b_held, uint32_t b_planes, uint32_t b_planes_alt, int64_t M, int64_t N,
                                         int64_t K, int segs, int segs_short, const uint32_t* flags,
                                         const float* b_sc32, int64_t b_brow, int64_t b_bcol, int64_t b_kg, void* C,
                                         int64_t ldc, int c_dtype, const void* X, int64_t ldx, int64_t batch,
                                         int64_t a_batch, int64_t b_batch, int64_t c_batch, int64_t x_batch, void* ws,
                                         int64_t ws_bytes, hipStream_t stream) {
  const char* who = "gemm_bf16_planes";
  if (M <= 0 || N <= 0 || K <= 0 || batch <= 0) {
    if (M < 0 || N < 0 || K < 0 || batch < 0) return pratchya_set_error(PRATCHYA_EINVAL, "%s: negative size", who);
    return PRATCHYA_OK;
  }
  if (batch > 1 && (batch > 65535 || a_batch % 8 || b_batch % 8 || c_batch % 8 || x_batch % 8 || flags || b_sc32))
    return pratchya_set_error(PRATCHYA_EUNSUPPORTED, "%s: batches of plain products, strides multiples of 8", who);
  if (c_dtype != PRATCHYA_DT_F32 && c_dtype != PRATCHYA_DT_BF16)
    return pratchya_set_error(PRATCHYA_EINVAL, "%s: unsupported output dtype %d", who, c_dtype);
  const int chunk = c_dtype == PRATCHYA_DT_BF16 ? 8 : 4;
  if (K % 64 || N % chunk || (a_kmajor && M % 8) || (b_kmajor && N % 8))
    return pratchya_set_error(PRATCHYA_EUNSUPPORTED, "%s: K a multiple of 64, N of %d, rows of a K-major operand of 8",
                              who, chunk);
  if (!A || !B || !C) return pratchya_set_error(PRATCHYA_EINVAL, "%s: null buffer", who);
  if (segs < 1 || segs > 8 || segs_short < 1 || segs_short > segs || a_held < 1 || b_held < 1 || a_held > 8 || b_held > 8)
    return pratchya_set_error(PRATCHYA_EINVAL, "%s: bad segments", who);
  for (int s = 0; s < segs; ++s)
    if ((int)((a_planes >> (4 * s)) & 15u) >= a_held || (int)((b_planes >> (4 * s)) & 15u) >= b_held ||
        (int)((b_planes_alt >> (4 * s)) & 15u) >= b_held)
      return pratchya_set_error(PRATCHYA_EINVAL, "%s: a segment names a plane that is not held", who);
  const int64_t wa = a_kmajor ? M : K, wb = b_kmajor ? N : K;      // a plane's row length, and its rows
  const int64_t ha = a_kmajor ? K : M, hb = b_kmajor ? K : N;
  if (lda < wa || ldb < wb || ldc < N || lda % 8 || ldb % 8 || ldc % chunk || a_stride % 8 || b_stride % 8 ||
      (a_held > 1 && a_stride < wa) || (b_held > 1 && b_stride < wb) ||
      (reinterpret_cast<uintptr_t>(A) | reinterpret_cast<uintptr_t>(B) | reinterpret_cast<uintptr_t>(C)) % 16 ||
      (X && (c_dtype != PRATCHYA_DT_BF16 || ldx < N || ldx % 8 || reinterpret_cast<uintptr_t>(X) % 16)))
    return pratchya_set_error(PRATCHYA_EINVAL, "%s: leading dimensions / alignment not supported", who);
  const int64_t Mr = (M + 127) / 128 * 128, Nr = (N + 127) / 128 * 128;
  const int64_t pa = a_held > 1 ? (a_held - 1) * a_stride : 0, pb = b_held > 1 ? (b_held - 1) * b_stride : 0;
  if (2 * (pa + (a_kmajor ? K + 1 : Mr) * lda + Mr) > kMaxOffset || 2 * (pb + (b_kmajor ? K + 1 : Nr) * ldb + Nr) > kMaxOffset ||
      M > INT32_MAX / 2 || N > INT32_MAX / 2 || segs * (K / 64) > (1 << 24))
    return pratchya_set_error(PRATCHYA_EUNSUPPORTED, "%s: operands beyond 32-bit offsets", who);
  T128Args p{};
  p.a.p = static_cast<const uint8_t*>(A);
  p.a.ld = (uint32_t)(2 * lda);
  p.a.bytes = (uint32_t)(2 * (pa + (ha - 1) * lda + wa));
  p.a.pstride = (uint32_t)(2 * a_stride);
  p.a.planes = p.a.planes_alt = a_planes;
  p.a.r_div = p.b.r_div = 1;
  p.b.p = static_cast<const uint8_t*>(B);
  p.b.ld = (uint32_t)(2 * ldb);
  p.b.bytes = (uint32_t)(2 * (pb + (hb - 1) * ldb + wb));
  p.b.pstride = (uint32_t)(2 * b_stride);
  p.b.planes = b_planes;
  p.b.planes_alt = b_planes_alt;
  p.C = C;
  p.ldc = ldc;
  p.X = static_cast<const uint16_t*>(X);
  p.ldx = ldx;
  p.flags = flags;
  p.spp = (int)(K / 64);
  p.segs = segs;
  p.segs_short = segs_short;
  p.span = p.spp;
  if (b_sc32) {
    // B: the power-of-two plane of a [N, K] matrix quantized (b_brow, b_bcol),
    // its group maxima constant over aligned 64 columns and 4 rows
    const int sh = ilog2_exact(b_kg);
    if (b_kmajor || a_kmajor || X || c_dtype != PRATCHYA_DT_F32 || sh < 0 || b_brow < 1 || b_brow % 4 || b_bcol < 1 ||
        128 % b_bcol || K % b_bcol || N % b_brow)
      return pratchya_set_error(PRATCHYA_EUNSUPPORTED, "%s: scale layout of B not supported", who);
    const int64_t nb = K / b_bcol, blocks = pratchya_gemm_span(N, nb * 128, b_brow, nb, 1, b_kg);
    if (blocks != nb && (blocks * b_bcol) % 64)
      return pratchya_set_error(PRATCHYA_EUNSUPPORTED, "%s: B's groups change inside 64 columns", who);
    if ((Nr / b_brow + 1) * nb > INT32_MAX / 2)
      return pratchya_set_error(PRATCHYA_EUNSUPPORTED, "%s: operands beyond 32-bit offsets", who);
    p.span = blocks == nb ? p.spp : (int)(blocks * b_bcol / 64);
    p.b.g32 = b_sc32;
    p.b.g32_bytes = (uint32_t)((((N / b_brow) * nb - 1) / b_kg + 1) * 4);
    p.b.r_div = (uint32_t)b_brow;
    p.b.s_r = (uint32_t)nb;
    p.b.sk2 = (uint32_t)(128 / b_bcol);
    p.b.kg_sh = (uint32_t)sh;
  }
  p.a_bs = 2 * a_batch;
  p.b_bs = 2 * b_batch;
  p.c_bs = c_batch;
  p.x_bs = x_batch;
  const int rc = t128_shape(who, &p, M, N, (int64_t)segs_short * p.spp, ws, ws_bytes, batch);
  if (rc) return rc;
  const bool bf = c_dtype == PRATCHYA_DT_BF16, small = t128_rows(M) == 32;
  if (b_sc32) {
    if (small) t128_launch<true, 32, false, false, 2, 0>(p, stream);
    else t128_launch<true, 128, false, false, 2, 0>(p, stream);
  } else if (X) {
    if (small || a_kmajor) return pratchya_set_error(PRATCHYA_EUNSUPPORTED, "%s: the combination needs a K-contiguous A of over 32 rows", who);
    if (b_kmajor) t128_launch<true, 128, false, true, 0, 2>(p, stream);
    else t128_launch<true, 128, false, false, 0, 2>(p, stream);
  } else if (a_kmajor && small) {
    return pratchya_set_error(PRATCHYA_EUNSUPPORTED, "%s: a K-major A needs over 32 rows", who);
  } else if (a_kmajor != b_kmajor) {
    if (bf) return pratchya_set_error(PRATCHYA_EUNSUPPORTED, "%s: one K-major operand is supported with f32 output", who);
    if (a_kmajor) t128_launch<true, 128, true, false, 0, 0>(p, stream);
    else if (small) t128_launch<true, 32, false, true, 0, 0>(p, stream);
    else t128_launch<true, 128, false, true, 0, 0>(p, stream);
  } else if (a_kmajor) {
    if (bf) t128_launch<true, 128, true, true, 0, 1>(p, stream);
    else t128_launch<true, 128, true, true, 0, 0>(p, stream);
  } else if (small) {
    if (bf) t128_launch<true, 32, false, false, 0, 1>(p, stream);
    else t128_launch<true, 32, false, false, 0, 0>(p, stream);
  } else {
    if (bf) t128_launch<true, 128, false, false, 0, 1>(p, stream);
    else t128_launch<true, 128, false, false, 0, 0>(p, stream);
  }
  return t128_status(who);
}

extern "C" int pratchya_gemm_fine(const void* A, int64_t lda, const float* a_sc32, const void* B, int64_t ldb,
                                  const float* b_sc32, int64_t b_kg, int64_t blk, int64_t M, int64_t N, int64_t K,
                                  float* C, int64_t ldc, void* ws, int64_t ws_bytes, hipStream_t stream) {
  const char* who = "gemm_fine";
  if (M <= 0 || N <= 0 || K <= 0) {
    if (M < 0 || N < 0 || K < 0) return pratchya_set_error(PRATCHYA_EINVAL, "%s: negative size", who);
    return PRATCHYA_OK;
  }
  const int sh = ilog2_exact(b_kg);
  if ((blk != 16 && blk != 32) || K % 64 || N % blk || sh < 0)
    return pratchya_set_error(PRATCHYA_EUNSUPPORTED, "%s: blocks of 16 or 32, K a multiple of 64, groups of a power of two "
                              "of blocks", who);
  if (!A || !B || !a_sc32 || !b_sc32 || !C) return pratchya_set_error(PRATCHYA_EINVAL, "%s: null buffer", who);
  if (lda < K || ldb < N || ldc < N || lda % 8 || ldb % 8 || ldc % 4 ||
      (reinterpret_cast<uintptr_t>(A) | reinterpret_cast<uintptr_t>(B) | reinterpret_cast<uintptr_t>(C) |
       reinterpret_cast<uintptr_t>(a_sc32)) % 16)
    return pratchya_set_error(PRATCHYA_EINVAL, "%s: leading dimensions / alignment not supported", who);
  const int64_t Mr = (M + 127) / 128 * 128, Nr = (N + 127) / 128 * 128, nbn = N / blk;
  if (2 * (Mr * lda + K) > kMaxOffset || 2 * ((K + 1) * ldb + Nr) > kMaxOffset || Mr * (K / 4) > kMaxOffset ||
      (K / blk + 1) * nbn > INT32_MAX / 4 || M > INT32_MAX / 2 || N > INT32_MAX / 2 || K > (1 << 26))
    return pratchya_set_error(PRATCHYA_EUNSUPPORTED, "%s: operands beyond 32-bit offsets", who);
  T128Args p{};
  p.a.p = static_cast<const uint8_t*>(A);
  p.a.ld = (uint32_t)(2 * lda);
  p.a.bytes = (uint32_t)(2 * ((M - 1) * lda + K));
  p.a.g32 = a_sc32;
  p.a.g32_bytes = (uint32_t)(M * (K / (blk == 16 ? 16 : 64)) * 4);
  p.a.r_div = p.b.r_div = 1;
  p.b.p = static_cast<const uint8_t*>(B);
  p.b.ld = (uint32_t)(2 * ldb);
  p.b.bytes = (uint32_t)(2 * ((K - 1) * ldb + N));
  p.b.g32 = b_sc32;
  p.b.g32_bytes = (uint32_t)((((K / blk) * nbn - 1) / b_kg + 1) * 4);
  p.b.s_r = (uint32_t)nbn;
  p.b.kg_sh = (uint32_t)sh;
  p.C = C;
  p.ldc = ldc;
  p.spp = p.span = (int)(K / 64);
  p.segs = p.segs_short = 1;
  const int rc = t128_shape(who, &p, M, N, p.spp, ws, ws_bytes);
  if (rc) return rc;
  const bool small = t128_rows(M) == 32;
  if (blk == 16) {
    if (small) t128_launch<true, 32, false, true, 3, 0>(p, stream);
    else t128_launch<true, 128, false, true, 3, 0>(p, stream);
  } else {
    if (small) t128_launch<true, 32, false, true, 4, 0>(p, stream);
    else t128_launch<true, 128, false, true, 4, 0>(p, stream);
  }
  return t128_status(who);
}

// --------------------------------------------------------------------------
// Planes: the bf16 operands of pratchya_gemm_bf16_planes, from a quantized
// payload, an f32 or a bf16 matrix [T, W] (row-major, 8 values per thread; the
// planes keep the layout, rows T .. T_pad are zeros).
//   POW2    payload with its scales -> one plane, f32(q) * (2^(e-127) * G') / 128
//           with G' the group maximum's power of two: 4 significant bits, exact.
//           (A value whose dequantization is not finite is that value; with flags,
//           flags[1] and the second plane as for BF16.)
//   SPLIT3  payload with its scales -> the three pieces of the dequantized f32
//           value (k_split_pack's: the top 8 significant bits, the next 8, the
//           rest; their sum is the value).  A payload quantized from bf16 has
//           bf16 group maxima, its values 12 significant bits and no third
//           piece; flags[0] is set where one is not zero.
//   SPLIT4  f32, times its block's scale if given (dequantize_impl_bwd of a
//           cotangent): the three pieces and, fourth, the first piece with
//           non-finite values as 0.
//   SPLIT4Q payload with its scales -> SPLIT4's planes of the dequantized value.
//   BF16    bf16, times its block's scale if given: the rounded value; flags[1]
//           is set where one is not finite, and the second plane then written
//           (by k_plane_finite) with those as 0.
// --------------------------------------------------------------------------
namespace {

enum { PL_POW2 = 0, PL_SPLIT3 = 1, PL_SPLIT4 = 2, PL_BF16 = 3, PL_SPLIT4Q = 4 };

struct PlanesArgs {
  const uint8_t* src;
  const uint8_t* e8;
  const float* g32;
  uint16_t* dst;
  uint32_t* flags;
  uint32_t n, T, per_row;                // chunks, rows, chunks per row
  uint32_t a, lb, nbc, lk;               // block rows, log2 block columns, blocks per block row, log2 blocks per group
  int64_t pstride;
};

__device__ __forceinline__ float top8(float v) { return u2f(f2u(v) & 0xFFFF0000u); }

template <int MODE>
__global__ __launch_bounds__(256) void k_planes(PlanesArgs p) {
  const uint32_t i = blockIdx.x * 256u + threadIdx.x;
  if (i >= p.n) return;
  const uint32_t r = i / p.per_row, c = (i - r * p.per_row) * 8u;
  uint16_t* dst = p.dst + (int64_t)i * 8;
  constexpr int NP = MODE == PL_SPLIT3 ? 3 : (MODE == PL_SPLIT4 || MODE == PL_SPLIT4Q ? 4 : 1);
  if (r >= p.T) {
#pragma unroll
    for (int k = 0; k < NP; ++k) *reinterpret_cast<uint4*>(dst + k * p.pstride) = make_uint4(0, 0, 0, 0);
    return;
  }
  float sc = 0.0f, sp = 0.0f;              // scale, and with the maximum's power of two
  if (p.e8) {
    const uint32_t blk = r / p.a * p.nbc + (c >> p.lb);
    const float G = p.g32[blk >> p.lk], s = e8m0_decode(p.e8[blk]);
    sc = s * G;
    if constexpr (MODE == PL_POW2) {
      const uint32_t gb = f2u(G) & 0x7FFFFFFFu;
      sp = s * (gb == 0u ? 0.0f : gb < 0x00800000u ? 0x1p-126f : u2f(gb & 0x7F800000u));
    }
  }
  float v[8];
  if constexpr (MODE == PL_POW2 || MODE == PL_SPLIT3 || MODE == PL_SPLIT4Q) {
    const uint2 w = *reinterpret_cast<const uint2*>(p.src + (int64_t)i * 8);
    fp8_word(w.x, v[0], v[1], v[2], v[3]);
    fp8_word(w.y, v[4], v[5], v[6], v[7]);
  } else if constexpr (MODE == PL_SPLIT4) {
    const float4* f = reinterpret_cast<const float4*>(p.src) + (int64_t)i * 2;
    const float4 x = f[0], y = f[1];
    v[0] = x.x; v[1] = x.y; v[2] = x.z; v[3] = x.w;
    v[4] = y.x; v[5] = y.y; v[6] = y.z; v[7] = y.w;
  } else {
    const uint4 w = *(reinterpret_cast<const uint4*>(p.src) + i);
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = elem_f32<true>(w, k);
  }
  uint32_t o[NP][4], third = 0, odd = 0;
  if constexpr (MODE == PL_POW2) {
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const float full = v[k] * sc;
      v[k] = is_finite_f(full) ? (v[k] * sp) * 0.0078125f : full;
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      o[0][k] = pack_bf16x2(v[2 * k], v[2 * k + 1]);
      odd |= (uint32_t)((o[0][k] & 0x7F80u) == 0x7F80u) | (uint32_t)((o[0][k] & 0x7F800000u) == 0x7F800000u);
    }
  } else {
    if (p.e8) {
#pragma unroll
      for (int k = 0; k < 8; ++k) v[k] = (v[k] * sc) * 0.0078125f;
    }
    if constexpr (MODE == PL_BF16) {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        o[0][k] = pack_bf16x2(v[2 * k], v[2 * k + 1]);
        odd |= (uint32_t)((o[0][k] & 0x7F80u) == 0x7F80u) | (uint32_t)((o[0][k] & 0x7F800000u) == 0x7F800000u);
      }
    } else {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        float q[NP][2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const float x = v[2 * k + h];
          const bool fin = is_finite_f(x);
          const float p0 = top8(x), r0 = x - p0, p1 = top8(r0), p2 = r0 - p1;
          q[0][h] = fin ? p0 : x;
          q[1][h] = fin ? p1 : 0.0f;
          q[2][h] = fin ? p2 : 0.0f;
          if constexpr (NP == 4) q[3][h] = fin ? p0 : 0.0f;
        }
#pragma unroll
        for (int j = 0; j < NP; ++j) o[j][k] = pack_bf16x2(q[j][0], q[j][1]);
        third |= o[2][k] & 0x7FFF7FFFu;
      }
    }
  }
#pragma unroll
  for (int j = 0; j < NP; ++j)
    *reinterpret_cast<uint4*>(dst + j * p.pstride) = make_uint4(o[j][0], o[j][1], o[j][2], o[j][3]);
  // one store per wave at most, and none once the flag is seen set
  if constexpr (MODE == PL_SPLIT3 || MODE == PL_BF16 || MODE == PL_POW2) {
    uint32_t* f = p.flags + (MODE == PL_SPLIT3 ? 0 : 1);
    const uint64_t any = __ballot((MODE == PL_SPLIT3 ? third : odd) != 0u);
    if (p.flags && any != 0u && (threadIdx.x & 63) == (uint32_t)__builtin_ctzll(any) &&
        __hip_atomic_load(f, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0u)
      __hip_atomic_fetch_or(f, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

// plane 1 = plane 0 with non-finite values as 0, where flags[1] says that it
// holds any.
__global__ __launch_bounds__(256) void k_plane_finite(uint16_t* __restrict__ dst, int64_t pstride, int64_t n,
                                                      const uint32_t* __restrict__ flags) {
  if (flags[1] == 0u) return;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
    uint4 w = *reinterpret_cast<const uint4*>(dst + i * 8);
    uint32_t* q = &w.x;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      if ((q[k] & 0x7F80u) == 0x7F80u) q[k] &= 0xFFFF0000u;
      if ((q[k] & 0x7F800000u) == 0x7F800000u) q[k] &= 0x0000FFFFu;
    }
    *reinterpret_cast<uint4*>(dst + pstride + i * 8) = w;
  }
}

}  // namespace

extern "C" int pratchya_planes(int mode, const void* src, const uint8_t* sc8, const float* sc32, int64_t T, int64_t W,
                               int64_t a, int64_t b, int64_t T_pad, void* dst, uint32_t* flags, hipStream_t stream) {
  const char* who = "planes";
  if (T < 0 || W < 0 || mode < PL_POW2 || mode > PL_SPLIT4Q)
    return pratchya_set_error(PRATCHYA_EINVAL, "%s: negative size or unknown mode %d", who, mode);
  if (T == 0 || W == 0) return PRATCHYA_OK;
  const bool scaled = sc8 != nullptr;
  const int lb = ilog2_exact(b);
  if (T_pad < T || W % 8 || (scaled && (a < 1 || T % a || lb < 3 || W % b)))
    return pratchya_set_error(PRATCHYA_EUNSUPPORTED, "%s: W a multiple of 8, blocks of a power of two of at least 8 columns", who);
  const int64_t nbc = scaled ? W / b : 1, nblk = scaled ? (T / a) * nbc : 1;
  const int64_t kg = scaled ? std::gcd(a * b / 16 > 1 ? a * b / 16 : 1, nblk) : 1;
  const int lk = ilog2_exact(kg);
  if (lk < 0) return pratchya_set_error(PRATCHYA_EUNSUPPORTED, "%s: groups of a power of two of blocks", who);
  const int64_t n = T_pad * (W / 8);
  if (n > INT32_MAX || nblk > INT32_MAX) return pratchya_set_error(PRATCHYA_EUNSUPPORTED, "%s: too large", who);
  const bool payload = mode == PL_POW2 || mode == PL_SPLIT3 || mode == PL_SPLIT4Q;
  if (!src || !dst || (scaled && !sc32) || (payload && !scaled) || ((mode == PL_SPLIT3 || mode == PL_BF16) && !flags) ||
      reinterpret_cast<uintptr_t>(dst) % 16 || reinterpret_cast<uintptr_t>(src) % (payload ? 8 : 16))
    return pratchya_set_error(PRATCHYA_EINVAL, "%s: null or misaligned buffer", who);
  PlanesArgs p{static_cast<const uint8_t*>(src), sc8, sc32, static_cast<uint16_t*>(dst), flags, (uint32_t)n, (uint32_t)T,
               (uint32_t)(W / 8), (uint32_t)a, (uint32_t)(lb < 0 ? 0 : lb), (uint32_t)nbc, (uint32_t)lk, T_pad * W};
  const dim3 grid((unsigned)((n + 255) / 256)), block(256);
  switch (mode) {
    case PL_SPLIT3: hipLaunchKernelGGL(k_planes<PL_SPLIT3>, grid, block, 0, stream, p); break;
    case PL_SPLIT4Q: hipLaunchKernelGGL(k_planes<PL_SPLIT4Q>, grid, block, 0, stream, p); break;
    case PL_SPLIT4: hipLaunchKernelGGL(k_planes<PL_SPLIT4>, grid, block, 0, stream, p); break;
    default: {
      if (mode == PL_POW2) hipLaunchKernelGGL(k_planes<PL_POW2>, grid, block, 0, stream, p);
      else hipLaunchKernelGGL(k_planes<PL_BF16>, grid, block, 0, stream, p);
      if (!flags) break;
      const int64_t blocks = (n + 255) / 256;
      hipLaunchKernelGGL(k_plane_finite, dim3((unsigned)(blocks < 1024 ? blocks : 1024)), block, 0, stream, p.dst,
                         p.pstride, n, flags);
    }
  }
  return t128_status(who);
}
