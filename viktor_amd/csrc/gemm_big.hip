// Large-M GEMMs of the prefill / scoring forward: y[M, N] = x[M, K] @ w[N, K]^T, bf16 in, fp32 accumulate.
//
// MI355X design (M = tokens or frames x N = 512..4096 x K = 512..3072):
//   * 128 x 128 output tile per workgroup of 4 wavefronts, each 64 x 64 (16 fp32 MFMA tiles, 64 accumulator
//     registers), two workgroups per CU: one workgroup's barriers and epilogue overlap the other's MFMAs, and a
//     packed batch of a few thousand rows still fills the chip (smaller ones take 64 x 128 and 64 x 64 tiles).
//   * What bounds the K loop: with the MFMAs and LDS reads alone it runs at 1820 TFLOP/s (MFMAs alone 2080), with the
//     loads alone at the rate of the global->LDS stream. That stream is issued as direct loads (buffer_load .. lds,
//     16 bytes a lane, no registers) of 64-wide K slabs: 8 lanes take a row's whole 128-byte line, 24-29 TB/s over
//     the chip; 32-wide slabs (64-byte rows) reached 16 TB/s. With real operands the clock then falls with the power
//     drawn: the loop without an epilogue runs at 1100-1240 TFLOP/s (zero operands: 1490) for every tile shape tried.
//   * Against 256 x 128 tiles with 32-wide slabs in a three-stage ring (same box, us): N = 512, K = 512 / 1536 + bf16
//     residual at M = 4099: 18.5 / 35.1 -> 11.2 / 20.4, M = 45057: 46.0 / 92.5 -> 40.7 / 77.7, M = 131136: 122 / 278
//     -> 111 / 269; SwiGLU N = 1536, K = 512: 20.5 -> 17.8, 154 -> 146, 427 -> 417; Wqkv N = 768: M = 45057 62 -> 53,
//     M = 131136 see launch_big_shape.
//   * Tiles are ordered XCD-aware: workgroup p runs on XCD p % 8, so each XCD gets a contiguous range of
//     tiles and the N-tiles that share a block of x rows share that XCD's L2.
//   * The product is formed transposed, C^T = W X^T (the weight fragment is the MFMA A operand), so each
//     lane ends with 4 consecutive output columns of one row; the epilogue stages each wavefront's block
//     through LDS and stores whole rows in 16-byte chunks.
//   * SwiGLU: the tile's W rows are 64 gate rows and the matching 64 up rows; both land in the same lane,
//     and the epilogue stores bf16(bf16(silu(bf16(g))) * bf16(u)) over 64 output columns.
//   * Every row of y is computed by the same code whatever M is (no split of K; every tile shape adds the same
//     32-wide MFMA steps in the same order), so a row's result does not depend on the other rows of the product.
#include <type_traits>

#include "common.h"
#include "slab_loads.h"

namespace vk {

constexpr int GB_BK = 64;           // K per stage
constexpr int GB_ROWB = GB_BK * 2;  // bytes per LDS row

// A workgroup of RW x GW wavefronts, each 16 FX rows of x by 64 weight rows.
template <int RW_, int GW_, int FX_>
struct GbShape {
  static constexpr int RW = RW_, GW = GW_, FX = FX_;
  static constexpr int WAVES = RW * GW;
  static constexpr int WROWS = 16 * FX;                                // rows of x per wavefront
  static constexpr int BM = RW * WROWS;                                // rows of x per workgroup
  static constexpr int BW = 64 * GW;                                   // rows of w per workgroup
  static constexpr int XTILEB = BM * GB_ROWB, WTILEB = BW * GB_ROWB;
  static constexpr int STAGEB = XTILEB + WTILEB;
  static constexpr size_t SMEM = 2 * static_cast<size_t>(STAGEB);
  static constexpr int RPL = 1024 / GB_ROWB;                           // rows per direct-load instruction
  static constexpr int XLOADS = BM / RPL / WAVES;                      // x instructions per wave per stage
  static constexpr int WLOADS = BW / RPL / WAVES;
  static constexpr int LOADS = XLOADS + WLOADS;
  static constexpr int WG_PER_CU = SMEM > 81920 ? 1 : SMEM > 53248 ? 2 : 3;
  static constexpr int WAVES_PER_SIMD = WG_PER_CU * WAVES / 4 > 0 ? WG_PER_CU * WAVES / 4 : 1;
};
using GbWide = GbShape<2, 4, 8>;    // 256 x 256, 128 KB: one workgroup of 8 wavefronts per CU
using GbFlat = GbShape<2, 2, 2>;    // 64 x 128, 48 KB: up to three workgroups per CU
using GbSmall = GbShape<2, 1, 2>;   // 64 x 64, 32 KB, two wavefronts
using GbSquare = GbShape<2, 2, 4>;  // 128 x 128, 64 KB: two workgroups per CU

typedef __attribute__((address_space(3))) void lds_void;

// A buffer descriptor over `bytes` bytes from p (raw, unstrided), and one 16-byte direct buffer->LDS load per lane:
// lane l reads p + vo + so into dst + 16 l (zero if that is past the end; slab_loads.h: for either reading of the range
// check). Plain device functions: written in a kernel template
// with arguments that depend on its parameters, the builtin makes the host pass drop the kernel's launch stub.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t gb_rsrc(const bf16_t *p, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t *>(p), 0, bytes, 0x00020000);
}
__device__ __forceinline__ void gb_buf_lds(__amdgpu_buffer_rsrc_t r, char *dst, uint32_t vo, uint32_t so) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void *)dst, 16, vo, so, 0, 0);
}

// s_waitcnt immediate that waits for vmcnt <= n and leaves expcnt / lgkmcnt unconstrained (gfx9 encoding:
// vmcnt[3:0] in bits 3:0, vmcnt[5:4] in bits 15:14, expcnt in 6:4, lgkmcnt in 11:8)
constexpr int vmcnt_imm(int n) { return (n & 0xF) | (0x7 << 4) | (0xF << 8) | (((n >> 4) & 3) << 14); }

// Epilogues: bf16 out, fp32 out, SwiGLU, or the attention input stage of a Wqkv product (GB_QKV): the
// product's 64-column heads (H q heads, HKV k heads, HKV v heads) are rounded to bf16 as the unfused product
// stores them; q and k heads then get the per-head RMSNorm (when qw / kw are given: bf16(x / rms * w)) and
// the half-split rotary embedding at the row's position (bf16(y1 c - y2 s), bf16(y1 s + y2 c), with the
// table entries as stored), the rounding points of vk_qkv_rope_cache; then every head goes to its
// destination -- q rows, the KV cache and / or k / v rows.
//
// GB_RESID: y is a bf16 residual stream updated in place, y = bf16(bf16(acc + bias) + bf16(alpha y)) (alpha = 1,
// no bias: add_rmsnorm's x += bf16(delta); the encoder's DeepNorm sum with its out_proj bias and alpha), and
// ss_out[row, col / 64] receives the fp32 sum of squares of the row's new bf16 values over each 64-column block
// (the RMSNorm that follows reads them instead of a pass of its own over the row).
// GB_QKV reads fp32 rotary tables, GB_QKV_BF16 bf16 ones (the table type is a compile-time choice, so the epilogue's
// prefetched table registers are not merged across two load shapes); both take bf16 QK-norm weights. GB_QKV_W32 is
// GB_QKV with fp32 QK-norm weights: nn.RMSNorm under torch.autocast bf16 with fp32 master weights, which returns
// bf16(x / rms * w) for a bf16 head (the multiply by w in fp32, one rounding), before the fp32 rotation.
//
// GB_RESID_F32: y is an fp32 residual stream updated in place, y = alpha y + bf16(acc + bias): the autocast residual
// add x + sublayer(x) of an fp32 stream and a bf16 product (viktor/decoder.py:118-120 under torch.autocast bf16);
// ss_out as GB_RESID, over the new fp32 values.
// Both residual forms read the old residual from resid_in instead when it is given (out of place: y is then only
// written, and resid_in keeps the previous layer's stream, as a backward pass needs it).
enum GbEpi { GB_BF16 = 0, GB_F32 = 1, GB_SWIGLU = 2, GB_QKV = 3, GB_RESID = 4, GB_QKV_BF16 = 5, GB_RESID_F32 = 6,
             GB_QKV_W32 = 7 };

struct GbQkv {
  const void *qw, *kw;  // per-head RMSNorm weights [64], bf16 (fp32 for GB_QKV_W32); both NULL: no norm
  float eps;
  const void *cos_t, *sin_t;  // [table_rows, 32], fp32 (table_f32) or bf16
  int table_f32;
  int64_t table_rows;
  const int32_t *pos, *rope_pos, *seq;  // per row: cache position, rotary position (NULL: pos), cache row
  bf16_t *q;                            // q head h of row t at q + t q_ld + 64 h
  int64_t q_ld;
  bf16_t *kc, *vc;  // cache row (seq, pos) head h at kc + seq stride_cb + pos stride_cs + 64 h (NULL: none)
  int64_t stride_cb, stride_cs, cache_rows, cache_len;
  bf16_t *ko, *vo;  // k / v head h of row t at ko + t kv_ld + 64 h (NULL: none)
  int64_t kv_ld;
  bf16_t *raw;      // the product itself, rounded to bf16, rows [M, N] before the QK-norm and rotation (NULL: none)
  int H, HKV;
  // GB_RESID
  const float *bias;  // [N] or NULL
  float alpha;
  float *ss_out;         // [M, N / 64]
  const void *resid_in;  // the old residual rows [M, N] (NULL: the output itself, updated in place)
};

template <int EPI, class SH>
__global__ __launch_bounds__(64 * SH::WAVES, SH::WAVES_PER_SIMD) void gemm_big_kernel(
    const bf16_t *__restrict__ x, const bf16_t *__restrict__ w, void *__restrict__ y, int64_t M, int N, int K,
    int tiles_n, int tiles_total, int group_m, const GbQkv qa) {
  constexpr int GB_STAGEB = SH::STAGEB, GB_LOADS = SH::LOADS, NWAVES = SH::WAVES, GW = SH::GW, FX = SH::FX;
  constexpr int GB_BM = SH::BM, GB_XTILEB = SH::XTILEB, WROWS = SH::WROWS;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  constexpr bool SWIGLU = EPI == GB_SWIGLU, OUT_F32 = EPI == GB_F32, RESID = EPI == GB_RESID;
  constexpr bool RESID32 = EPI == GB_RESID_F32;
  constexpr bool QKV = EPI == GB_QKV || EPI == GB_QKV_BF16 || EPI == GB_QKV_W32;
  constexpr bool TAB_F32 = EPI == GB_QKV || EPI == GB_QKV_W32, W32 = EPI == GB_QKV_W32;
  // wid through readfirstlane: wave-uniform for the compiler, so branches on the wavefront's quadrant or head are scalar
  const int tid = threadIdx.x, lane = tid & 63, wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wid / GW, wn = wid % GW;
  constexpr int OUT_COLS = SWIGLU ? 32 * GW : 64 * GW;

  // XCD-aware tile order: physical workgroup p runs on XCD p % 8; XCD x owns the contiguous logical
  // range [x q + min(x, r), ...) of q + (x < r) tiles (q = total / 8, r = total % 8) -- a bijection
  const int p = blockIdx.x;
  const int xcd = p & 7, idx = p >> 3;
  const int q8 = tiles_total >> 3, r8 = tiles_total & 7;
  const int tile = xcd * q8 + min(xcd, r8) + idx;
  // logical order: groups of group_m row blocks, each walked column block by column block (group_m row blocks
  // per column block), so an XCD's resident workgroups share group_m A blocks and a few weight blocks in its
  // L2 instead of every weight block (a bijection: the last group has the remaining row blocks)
  const int tiles_m = tiles_total / tiles_n;
  const int grp = tile / (group_m * tiles_n), first_m = grp * group_m;
  const int gm = min(tiles_m - first_m, group_m), in_grp = tile - grp * group_m * tiles_n;
  const int mt = first_m + in_grp % gm, nt = in_grp / gm;
  const int64_t m0 = static_cast<int64_t>(mt) * GB_BM;
  const int n0 = nt * OUT_COLS;

  f32x4 acc[4][FX];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < FX; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  const int fr = lane & 15, fg = lane >> 4;
  auto mfmas = [&](const bf16x8(&xf)[FX], const bf16x8(&wf)[4]) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < FX; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[i], xf[j], acc[i][j], 0, 0, 0);
  };
  // one LDS read of the next slice between the MFMAs of this one, then the MFMAs left over
#define GB_INTERLEAVE()                                                        \
  do {                                                                         \
    constexpr int per_ = 4 * FX / (FX + 4);                                    \
    _Pragma("unroll") for (int r_ = 0; r_ < FX + 4; ++r_) {                    \
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);                       \
      __builtin_amdgcn_sched_group_barrier(0x008, per_, 0);                    \
    }                                                                          \
    __builtin_amdgcn_sched_group_barrier(0x008, 4 * FX - per_ * (FX + 4), 0);  \
  } while (0)
  // Two stages of 64-wide K slabs (LDS rows of 128 bytes: a direct load's 8 lanes of a row take one whole
  // cache line; with 64-byte rows the same stream ran at 16 instead of 24 TB/s). The stage holds a slab's
  // two 32-wide slices; a wavefront reads the next slice's fragments while this one's MFMAs run, from two
  // register sets. Once every wavefront has its fragments of slab kt in registers (the barrier), slab kt + 2
  // goes into its stage; slab kt + 1 had the time of a whole slab to land. Buffer loads (offsets: slab_loads.h): rows
  // past M or N are past the descriptor's end and read as zero (they only reach outputs that are not stored), and the K
  // offset rides in the scalar offset, so a source takes one 32-bit register.
  // LDS slot of K chunk c (16 bytes) in row r: c ^ ((r >> 1) & 7), so 16 consecutive rows of a chunk cover all
  // 64 banks.
  const int64_t xrows = M - m0 < GB_BM ? M - m0 : GB_BM;
  const auto xr = gb_rsrc(x + m0 * K, slab_bytes(static_cast<uint32_t>(xrows), K));
  constexpr int HALVES = SWIGLU ? 2 : 1;  // SwiGLU: gate rows n0.. of w, then the matching up rows N + n0..
  const uint32_t wrows = N - n0 < SH::BW / HALVES ? N - n0 : SH::BW / HALVES;
  const auto wr = gb_rsrc(w + static_cast<int64_t>(n0) * K, slab_bytes(wrows, K));
  const auto wr2 = gb_rsrc(w + static_cast<int64_t>(SWIGLU ? N + n0 : n0) * K, slab_bytes(wrows, K));
  static_assert(SH::RPL == SLAB_ROWS && GB_ROWB == SLAB_BYTES, "a direct load covers 8 rows of a slab");
  auto issue = [&](int stage, int kt) {
    char *base = smem + stage * GB_STAGEB;
    const uint32_t so = slab_scalar_offset(kt);
#pragma unroll
    for (int i = 0; i < SH::XLOADS; ++i)
      gb_buf_lds(xr, base + (wid + NWAVES * i) * 1024, slab_vector_offset(wid, NWAVES, i, lane, K), so);
#pragma unroll
    for (int i = 0; i < SH::WLOADS; ++i) {
      constexpr int HL = SH::WLOADS / HALVES;
      gb_buf_lds(i >= HL ? wr2 : wr, base + GB_XTILEB + (wid + NWAVES * i) * 1024,
                 slab_vector_offset(wid, NWAVES, i >= HL ? i - HL : i, lane, K), so);
    }
  };
  const int sw = 16 * (fg ^ ((fr >> 1) & 7));
  const int xo = (wm * WROWS + fr) * 128 + sw;
  int wo[2];  // fragments 0, 1 and 2, 3 (SwiGLU: gate and up rows)
  wo[0] = GB_XTILEB + ((SWIGLU ? wn * 32 : wn * 64) + fr) * 128 + sw;
  wo[1] = SWIGLU ? wo[0] + 32 * GW * 128 : wo[0] + 32 * 128;
  auto read_frags = [&](int stage, int kk, bf16x8(&xf)[FX], bf16x8(&wf)[4]) {
    const char *base = smem + stage * GB_STAGEB;
#pragma unroll
    for (int j = 0; j < FX; ++j) xf[j] = *reinterpret_cast<const bf16x8 *>(base + (xo ^ (64 * kk)) + j * 2048);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      wf[i] = *reinterpret_cast<const bf16x8 *>(base + (wo[i >> 1] ^ (64 * kk)) + (i & 1) * 2048);
  };
  const int nk = K / 64;
  constexpr std::integral_constant<int, 0> even{};
  constexpr std::integral_constant<int, 1> odd{};
  const int first = nk & 1;  // slab 0's stage
  issue(first, 0);
  if (nk > 1) {
    issue(first ^ 1, 1);
    __builtin_amdgcn_s_waitcnt(vmcnt_imm(GB_LOADS));
  } else {
    __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
  }
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  bf16x8 xa[FX], wa[4], xb[FX], wb[4];
  if (FX != 8) read_frags(first, 0, xa, wa);
  // The residual epilogues' operands (old rows, bias) are loaded in the last slab but one, behind the last direct loads,
  // so their round trips pass under its MFMAs (M = 131136, N = 512: 115 -> 111 us at K = 512, 290 -> 269 at K = 1536).
  // The QKV epilogues' (QK-norm weights, every row's rotary position; the table rows, which depend on the positions,
  // go one row group ahead) measured the same there or after the loop, and are loaded after it.
  u32x2 res_old[RESID ? FX : 1][4];
  f32x4 r32_old[RESID32 ? FX : 1][4];
  f32x4 res_b4[(RESID || RESID32) ? 4 : 1];
  using NwT = typename std::conditional<W32, f32x4, u32x2>::type;
  NwT qk_nw[QKV ? 4 : 1];
  int qk_rp[QKV ? FX : 1];
  const int qk_hd = (n0 + wn * 64) >> 6;  // GB_QKV: this wavefront's head (64 columns, wave-uniform)
  const bool qk_rot = QKV && qk_hd < qa.H + qa.HKV;
  const void *qk_w = QKV ? (qk_hd < qa.H ? qa.qw : qa.kw) : nullptr;
  auto prefetch = [&]() {
    if constexpr (RESID || RESID32) {
#pragma unroll
      for (int j = 0; j < FX; ++j) {
        int64_t rrow = m0 + wm * WROWS + 16 * j + fr;
        rrow = rrow < M ? rrow : M - 1;
        const void *old = qa.resid_in ? qa.resid_in : y;
        const int64_t at = rrow * N + n0 + wn * 64 + 4 * fg;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if constexpr (RESID)
            res_old[j][i] = *reinterpret_cast<const u32x2 *>(static_cast<const bf16_t *>(old) + at + 16 * i);
          else
            r32_old[j][i] = *reinterpret_cast<const f32x4 *>(static_cast<const float *>(old) + at + 16 * i);
        }
      }
#pragma unroll
      for (int i = 0; i < 4; ++i)
        res_b4[i] = qa.bias != nullptr ? *reinterpret_cast<const f32x4 *>(qa.bias + n0 + wn * 64 + 16 * i + 4 * fg)
                                       : f32x4{0.f, 0.f, 0.f, 0.f};
    }
  };
  auto load_qkv = [&]() {
    if constexpr (QKV) {
      if (qk_w != nullptr) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if constexpr (W32)
            qk_nw[i] = *reinterpret_cast<const f32x4 *>(static_cast<const float *>(qk_w) + 16 * i + 4 * fg);
          else
            qk_nw[i] = *reinterpret_cast<const u32x2 *>(static_cast<const bf16_t *>(qk_w) + 16 * i + 4 * fg);
        }
      }
#pragma unroll
      for (int j = 0; j < FX; ++j) {
        int64_t rrow = m0 + wm * WROWS + 16 * j + fr;
        rrow = rrow < M ? rrow : M - 1;
        int64_t rp = qa.rope_pos != nullptr ? qa.rope_pos[rrow] : qa.pos[rrow];
        qk_rp[j] = static_cast<int>(rp < 0 ? 0 : (rp >= qa.table_rows ? qa.table_rows - 1 : rp));
      }
    }
  };

  // Slab kt: its second slice's fragments are read under its first slice's MFMAs; once every wavefront has them in
  // registers and slab kt + 1 is whole in LDS (the waits and the barrier), slab kt + 2 is issued into this stage and
  // the next slab's first fragments are read under the second slice's MFMAs. A bare s_barrier: __syncthreads()
  // would also wait for the epilogue's operands, which go out in the last slab but one.
  auto landed = [&](bool loads) {
    if (loads) __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  // (the stage is a compile-time parity: its LDS offsets are then immediates; with a run-time stage the loop ran 3-15%
  // slower)
  auto slab = [&](auto stage, int kt) {
    read_frags(stage, 1, xb, wb);
    mfmas(xa, wa);
    GB_INTERLEAVE();
    landed(true);
    issue(stage, kt + 2);
    read_frags(stage ^ 1, 0, xa, wa);
    mfmas(xb, wb);
    GB_INTERLEAVE();
  };
  auto last_but_one = [&](auto stage) {
    read_frags(stage, 1, xb, wb);
    mfmas(xa, wa);
    GB_INTERLEAVE();
    landed(true);
    prefetch();
    read_frags(stage ^ 1, 0, xa, wa);
    mfmas(xb, wb);
    GB_INTERLEAVE();
  };
  auto last = [&](auto stage) {
    read_frags(stage, 1, xb, wb);
    mfmas(xa, wa);
    GB_INTERLEAVE();
    landed(false);  // every wavefront has finished reading the ring: the epilogue stages through it
    mfmas(xb, wb);
  };
  if constexpr (FX == 8) {
    // no registers for a second set of fragments beside 128 accumulators: a slab's 24 fragments are read, its stage is
    // refilled once every wavefront has them, and the next slab is waited for after the MFMAs
    auto step = [&](auto stage, int kt) {
      read_frags(stage, 0, xa, wa);
      read_frags(stage, 1, xb, wb);
      mfmas(xa, wa);
      landed(false);
      if (kt + 2 < nk) issue(stage, kt + 2);
      mfmas(xb, wb);
      if (kt + 2 < nk)
        __builtin_amdgcn_s_waitcnt(vmcnt_imm(GB_LOADS));
      else
        __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
      asm volatile("" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
    };
    int kt = 0;
    if (nk & 1) step(odd, kt++);
    for (; kt < nk; kt += 2) {
      step(even, kt);
      step(odd, kt + 1);
    }
    prefetch();
  } else {
    // the last slab is always in stage 1, so an odd count has a step of its own in front
    int kt = 0;
    if (nk & 1) {
      if (nk > 1) slab(odd, kt++);
    }
    for (; kt + 3 < nk; kt += 2) {
      slab(even, kt);
      slab(odd, kt + 1);
    }
    if (nk > 1)
      last_but_one(even);
    else
      prefetch();
    last(odd);
  }
#undef GB_INTERLEAVE

  // Epilogue through LDS: a lane holds 4 consecutive columns of one row per (i, j), so direct stores would
  // write 16 rows x 16-32 B per instruction. Each wavefront instead stages its block of rows in its own
  // quarter of the (now idle) ring, a pass of rows at a time (row pitch + 16 B against bank conflicts), and
  // stores 16-byte chunks whose lanes cover whole rows.
  // GB_QKV: the rotary table entries of 16-row group j (lane: its row's 4 consecutive entries at 16 i + 4 fg,
  // i = 0, 1): four fp32 values (GB_QKV) or four bf16 values in two words (GB_QKV_BF16) per table and i
  using TabT = typename std::conditional<TAB_F32, f32x4, u32x2>::type;
  auto qk_tables = [&](int j, TabT (&c)[2], TabT (&sn)[2]) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int64_t ti = static_cast<int64_t>(qk_rp[j]) * 32 + 16 * i + 4 * fg;
      if constexpr (TAB_F32) {
        c[i] = *reinterpret_cast<const f32x4 *>(static_cast<const float *>(qa.cos_t) + ti);
        sn[i] = *reinterpret_cast<const f32x4 *>(static_cast<const float *>(qa.sin_t) + ti);
      } else {
        c[i] = *reinterpret_cast<const u32x2 *>(static_cast<const bf16_t *>(qa.cos_t) + ti);
        sn[i] = *reinterpret_cast<const u32x2 *>(static_cast<const bf16_t *>(qa.sin_t) + ti);
      }
    }
  };
  TabT qk_c[2][2], qk_s[2][2];  // two row groups' table entries: the current one and the next
  if (qk_rot) {
    load_qkv();
    qk_tables(0, qk_c[0], qk_s[0]);
  }
  constexpr int ESZ = (OUT_F32 || RESID32) ? 4 : 2;   // output element bytes
  constexpr int QCOLS = SWIGLU ? 32 : 64;             // output columns of a wavefront
  constexpr int RB = QCOLS * ESZ;                     // bytes of one quadrant row
  constexpr int PITCH = RB + 16;
  // rows staged per pass: what fits this wavefront's share of the ring (a power of two, 32..128)
  constexpr int STG_BYTES = static_cast<int>(SH::SMEM / NWAVES);
  constexpr int PASS_ROWS = WROWS * PITCH <= STG_BYTES ? WROWS : (WROWS > 64 && 64 * PITCH <= STG_BYTES ? 64 : 32);
  constexpr int CPR = RB / 16;                        // 16-byte chunks per row
  static_assert(PASS_ROWS * PITCH <= STG_BYTES, "epilogue staging exceeds the wavefront's share of LDS");
  char *stg = smem + wid * STG_BYTES;
  const int64_t qrow0 = m0 + wm * WROWS;
  const int qcol0 = n0 + wn * QCOLS;
#pragma unroll
  for (int pass = 0; pass < WROWS / PASS_ROWS; ++pass) {
#pragma unroll
    for (int jj = 0; jj < PASS_ROWS / 16; ++jj) {
      const int j = pass * (PASS_ROWS / 16) + jj;
      char *rowp = stg + (16 * jj + fr) * PITCH;
      if (RESID) {
        // lane: row 16 j + fr, columns qcol0 + 16 i + 4 fg + e (the same elements prefetch read for it)
        int64_t rrow = qrow0 + 16 * j + fr;
        const bool live = rrow < M;
        rrow = live ? rrow : M - 1;
        float ss = 0.f;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const u32x2 old = res_old[j][i];
          const f32x4 b4 = res_b4[i];
          float o[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float xo = (e & 1) ? hi_bf(old[e >> 1]) : lo_bf(old[e >> 1]);
            o[e] = round_bf(round_bf(acc[i][j][e] + b4[e]) + round_bf(qa.alpha * xo));
            ss += o[e] * o[e];
          }
          *reinterpret_cast<u32x2 *>(rowp + (16 * i + 4 * fg) * 2) = u32x2{pack_bf(o[0], o[1]), pack_bf(o[2], o[3])};
        }
        ss += __shfl_xor(ss, 16, 64);  // the row's other 48 columns of this block: lanes fr + 16, + 32, + 48
        ss += __shfl_xor(ss, 32, 64);
        if (live && fg == 0) qa.ss_out[rrow * (N >> 6) + (qcol0 >> 6)] = ss;
      } else if (RESID32) {
        // lane: row 16 j + fr, columns qcol0 + 16 i + 4 fg + e (the same elements prefetch read for it)
        const int64_t rrow = qrow0 + 16 * j + fr;
        float ss = 0.f;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const f32x4 old = r32_old[j][i];
          const f32x4 b4 = res_b4[i];
          f32x4 o;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            o[e] = qa.alpha * old[e] + round_bf(acc[i][j][e] + b4[e]);
            ss += o[e] * o[e];
          }
          *reinterpret_cast<f32x4 *>(rowp + (16 * i + 4 * fg) * 4) = o;
        }
        ss += __shfl_xor(ss, 16, 64);
        ss += __shfl_xor(ss, 32, 64);
        if (rrow < M && fg == 0) qa.ss_out[rrow * (N >> 6) + (qcol0 >> 6)] = ss;
      } else if (QKV) {
        // this wavefront's 64 columns are one head (wave-uniform); lane: row 16 j + fr, columns 16 i + 4 fg + e
        const int hd = qcol0 >> 6;
        float v[4][4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int e = 0; e < 4; ++e) v[i][e] = round_bf(acc[i][j][e]);
        if (qa.raw != nullptr && qcol0 < N) {  // the unrotated projection, as the plain product stores it
          const int64_t rrow = qrow0 + 16 * j + fr;
          if (rrow < M)
#pragma unroll
            for (int i = 0; i < 4; ++i)
              *reinterpret_cast<u32x2 *>(qa.raw + rrow * N + qcol0 + 16 * i + 4 * fg) =
                  u32x2{pack_bf(v[i][0], v[i][1]), pack_bf(v[i][2], v[i][3])};
        }
        if (hd < qa.H + qa.HKV) {  // q or k head: QK-norm, then the rotation
          // the next group's table entries go out before this group's arithmetic
          if (j + 1 < FX) qk_tables(j + 1, qk_c[(j + 1) & 1], qk_s[(j + 1) & 1]);
          if (qk_w != nullptr) {
            float ss = 0.f;
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
              for (int e = 0; e < 4; ++e) ss += v[i][e] * v[i][e];
            ss += __shfl_xor(ss, 16, 64);  // the row's other 48 columns: lanes fr + 16, + 32, + 48
            ss += __shfl_xor(ss, 32, 64);
            const float r = rsqrtf(ss * (1.0f / 64.0f) + qa.eps);
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
              for (int e = 0; e < 4; ++e) {
                float wv;
                if constexpr (W32)
                  wv = qk_nw[i][e];
                else
                  wv = (e & 1) ? hi_bf(qk_nw[i][e >> 1]) : lo_bf(qk_nw[i][e >> 1]);
                v[i][e] = round_bf(v[i][e] * r * wv);
              }
          }
#pragma unroll
          for (int i = 0; i < 2; ++i) {
            // the lane's 4 consecutive table entries (loaded one group ahead)
            const TabT c4 = qk_c[j & 1][i], s4 = qk_s[j & 1][i];
            float cs[4], sn[4];
            if constexpr (TAB_F32) {
#pragma unroll
              for (int e = 0; e < 4; ++e) {
                cs[e] = c4[e];
                sn[e] = s4[e];
              }
            } else {
#pragma unroll
              for (int e = 0; e < 4; ++e) {
                cs[e] = (e & 1) ? hi_bf(c4[e >> 1]) : lo_bf(c4[e >> 1]);
                sn[e] = (e & 1) ? hi_bf(s4[e >> 1]) : lo_bf(s4[e >> 1]);
              }
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              // (which product is fused into the sum is written out: with fp32 tables both are inexact, and the compiler
              // chose another one in each tile shape)
              const float y1 = v[i][e], y2 = v[i + 2][e];
              v[i][e] = __builtin_fmaf(y1, cs[e], -(y2 * sn[e]));
              v[i + 2][e] = __builtin_fmaf(y2, cs[e], y1 * sn[e]);
            }
          }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
          *reinterpret_cast<u32x2 *>(rowp + (16 * i + 4 * fg) * 2) =
              u32x2{pack_bf(v[i][0], v[i][1]), pack_bf(v[i][2], v[i][3])};
      } else if (SWIGLU) {
        // silu(g) = g / (1 + e^-g) as g times the hardware reciprocal (1 ulp) instead of the IEEE division: the
        // epilogue's VALU work is on this product's critical path (the product ~5% faster at the prefill shape);
        // 0.007% of the outputs then differ from the division's by one bf16 ulp
        // qa.raw: the gate | up product rows [M, 2 N] as the plain product stores them (the backward's operand)
        const int64_t grow = qrow0 + 16 * j + fr;
        const bool keep = qa.raw != nullptr && grow < M;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          float o[4], gt4[4], up4[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float gt = round_bf(acc[i][j][e]);
            const float up = round_bf(acc[i + 2][j][e]);
            gt4[e] = gt;
            up4[e] = up;
            o[e] = round_bf(gt * __builtin_amdgcn_rcpf(1.0f + __expf(-gt))) * up;
          }
          *reinterpret_cast<u32x2 *>(rowp + (16 * i + 4 * fg) * 2) = u32x2{pack_bf(o[0], o[1]), pack_bf(o[2], o[3])};
          if (keep && qcol0 + 16 * i + 4 * fg < N) {  // (N % 8 == 0: 4 columns are all inside or all outside)
            bf16_t *gr = qa.raw + grow * (2 * static_cast<int64_t>(N)) + qcol0 + 16 * i + 4 * fg;
            *reinterpret_cast<u32x2 *>(gr) = u32x2{pack_bf(gt4[0], gt4[1]), pack_bf(gt4[2], gt4[3])};
            *reinterpret_cast<u32x2 *>(gr + N) = u32x2{pack_bf(up4[0], up4[1]), pack_bf(up4[2], up4[3])};
          }
        }
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if (OUT_F32)
            *reinterpret_cast<f32x4 *>(rowp + (16 * i + 4 * fg) * 4) = acc[i][j];
          else
            *reinterpret_cast<u32x2 *>(rowp + (16 * i + 4 * fg) * 2) =
                u32x2{pack_bf(acc[i][j][0], acc[i][j][1]), pack_bf(acc[i][j][2], acc[i][j][3])};
        }
      }
    }
    // GB_QKV with a cache: the cache row and position of the pass's (up to 128) rows, one pair of rows per lane (rows
    // lane and 64 + lane), handed to the lane that stores a row's chunk by a lane shuffle below
    int cs_lo = 0, cs_hi = 0, cp_lo = 0, cp_hi = 0;
    if (QKV && (qcol0 >> 6) >= qa.H && qa.kc != nullptr) {
      const int64_t r0 = min(qrow0 + pass * PASS_ROWS + lane, M - 1), r1 = min(qrow0 + pass * PASS_ROWS + 64 + lane, M - 1);
      cs_lo = qa.seq[r0];
      cp_lo = qa.pos[r0];
      cs_hi = qa.seq[r1];
      cp_hi = qa.pos[r1];
    }
    // same wavefront reads back (LDS keeps a wavefront's accesses in order): chunk id -> (row, chunk)
#pragma unroll
    for (int it = 0; it < PASS_ROWS * CPR / 64; ++it) {
      const int id = it * 64 + lane;
      const int r = id / CPR, c = id % CPR;
      const u32x4 v = *reinterpret_cast<const u32x4 *>(stg + r * PITCH + c * 16);
      const int64_t row = qrow0 + pass * PASS_ROWS + r;
      const int col = qcol0 + c * (16 / ESZ);
      if (QKV) {
        const int hd = qcol0 >> 6;  // c: the 16-byte chunk (8 columns) of the head
        // (every lane takes part in the shuffles, before any lane leaves the iteration; r < 64 is fixed per it)
        const bool lo_half = it * 64 / CPR < 64;
        const int64_t sq = __shfl(lo_half ? cs_lo : cs_hi, r & 63, 64);
        const int64_t ps = __shfl(lo_half ? cp_lo : cp_hi, r & 63, 64);
        if (row >= M || hd >= qa.H + 2 * qa.HKV) continue;
        if (hd < qa.H) {
          *reinterpret_cast<u32x4 *>(qa.q + row * qa.q_ld + hd * 64 + 8 * c) = v;
          continue;
        }
        const bool is_k = hd < qa.H + qa.HKV;
        const int hk = is_k ? hd - qa.H : hd - qa.H - qa.HKV;
        bf16_t *cdst = is_k ? qa.kc : qa.vc;
        if (cdst != nullptr) {
          if (sq >= 0 && sq < qa.cache_rows && ps >= 0 && ps < qa.cache_len)
            *reinterpret_cast<u32x4 *>(cdst + sq * qa.stride_cb + ps * qa.stride_cs + hk * 64 + 8 * c) = v;
        }
        bf16_t *odst = is_k ? qa.ko : qa.vo;
        if (odst != nullptr) *reinterpret_cast<u32x4 *>(odst + row * qa.kv_ld + hk * 64 + 8 * c) = v;
        continue;
      }
      // non-temporal: the product's rows are read back by a later kernel, not by this one, and stores that
      // allocate in L2 would push out the A blocks the XCD's next column tiles read
      if (row < M && col < N)
        __builtin_nontemporal_store(v, reinterpret_cast<u32x4 *>(static_cast<char *>(y) + (row * N + col) * ESZ));
    }
  }
}

template <int EPI, class SH>
static int launch_big_shape(const bf16_t *x, const bf16_t *w, void *y, int64_t M, int N, int K, const GbQkv &qa,
                            hipStream_t s) {
  VK_RAISE_LDS_ONCE((gemm_big_kernel<EPI, SH>), SH::SMEM, "linear");
  constexpr int OUT_COLS = EPI == GB_SWIGLU ? SH::BW / 2 : SH::BW;
  const int tiles_n = (N + OUT_COLS - 1) / OUT_COLS;
  const int64_t tiles_m = (M + SH::BM - 1) / SH::BM;
  const int64_t total = tiles_m * tiles_n;
  if (total >= (int64_t(1) << 31)) return fail(VK_ERR_ARG, "linear: too many tiles");
  // (the descriptors hold a row block's bytes in 32 bits)
  if (K > (1 << 22)) return fail(VK_ERR_ARG, "linear: K %d too large", K);
  // Row blocks per group of the tile order: an XCD has 64 workgroups resident, 16 x 4 tiles of 128 x 128 for few column
  // blocks, once there is more than one resident round (M = 131136, N = 512, K = 1536: 230 -> 198 us for the loop alone
  // against groups of 8; residual K = 1536 at M = 17000 / 24459 / 36000 / 60000, inputs not in cache: bf16 54.8 / 62.4 /
  // 91.5 / 139.5 -> 50.3 / 60.4 / 86.9 / 135.0, fp32 57.5 / 70.2 / 97.9 / 150.9 -> 53.5 / 65.5 / 96.2 / 147.0, at 45057 1-2%
  // the other way); before, 8 (M = 9000, N = 512, K = 3072: 48 -> 41 us against 16). With more column blocks:
  //   * SwiGLU without kept rows: 16 (N = 1536 as part of an MLP, M = 9000 / 24459 / 45057 36.6 / 90.0 / 160.3 -> 35.8 /
  //     88.1 / 156.2);
  //   * SwiGLU with kept rows: 8 (M = 17000 / 32772 84 / 167, with 16 95 / 179);
  //   * Wqkv: 16 once the rows in and out outgrow the 256 MB last-level cache. M = 131136 with
  //     groups of 8 and 16 (in brackets: 256 x 128 tiles in groups of 8, the same rows as 16 here): N = 1536 310 and 301 us
  //     (305), fp32 weights and the kept product 220 and 214 (214), fp32 tables 166 and 164 (161), bf16 tables and a cache
  //     177 and 176 (172), at M = 90000 112 and 108 (109). Below it 8: M = 45057 97 and 98, 70 and 72, 57 and 59, 56 and
  //     59.
  bool rows16 = false;
  if constexpr (SH::BM == 128) {
    int64_t row_cols = 0;
    if constexpr (EPI == GB_QKV || EPI == GB_QKV_BF16 || EPI == GB_QKV_W32)
      row_cols = K + 64 * qa.H + 128 * qa.HKV * ((qa.ko != nullptr) + (qa.kc != nullptr)) + (qa.raw != nullptr ? N : 0);
    if constexpr (EPI == GB_SWIGLU) rows16 = qa.raw == nullptr && total >= 2048;
    rows16 = rows16 || M * row_cols * 2 > (int64_t(256) << 20) || (tiles_n <= 4 && total > 2 * device_cus_cached());
  }
  const int group_m = rows16 ? 16 : 8;
  gemm_big_kernel<EPI, SH><<<static_cast<unsigned>(total), 64 * SH::WAVES, SH::SMEM, s>>>(
      x, w, y, M, N, K, tiles_n, static_cast<int>(total), group_m, qa);
  return VK_OK;
}

template <class SH>
static int64_t gb_tiles(int64_t M, int N) {
  return (M + SH::BM - 1) / SH::BM * ((N + SH::BW - 1) / SH::BW);
}

template <int EPI>
static int launch_big(const bf16_t *x, const bf16_t *w, void *y, int64_t M, int N, int K, const GbQkv &qa,
                      hipStream_t s) {
  // 256 x 256 tiles read a third fewer bytes into LDS per flop, but one of them fills a CU, so its epilogue runs alone and a
  // round of them takes 1.6-2 rounds of 128 x 128 tiles (two per CU). They are taken where their count fits its rounds the
  // better. Plain epilogues, N = 512, bf16 out, inputs not in cache, us with 128 x 128 and 256 x 256 tiles (rounds):
  //   K = 3072: M = 13000 (1, 1) 50, 81; 16500 (2, 1) 82, 79; 24459 (2, 1) 96, 82; 36000 (3, 2) 144, 153; 45057 (3, 2) 170, 165;
  //   55000 (4, 2) 209, 175; 75000 (5, 3) 275, 252; 131136 (9, 5) 445, 417 (fp32 out and K = 1536 alike): from K = 1024 on
  //   beyond one round of 128 x 128 tiles;
  //   K = 768: 24459 28.6, 26.3; 36000 41.0, 45.7; 55000 56.4, 52.8; 75000 77, 79; 90000 (6, 3) 84.1, 81.0; 131136 124, 126:
  //   where they halve the rounds;
  //   K = 512: 18500 17.1, 16.6; 28000 21.4, 19.5 (fp32 out 24.1, 23.7); 55000 39.4, 39.3 (39.2, 44.8); 131136 74, 84; N =
  //   1536: 18500 (4, 2) 34.0, 35.3; 30000 (6, 3) 52.9, 53.0: for a single round against two.
  // The Wqkv epilogues gain only in a well-filled single round: bf16 tables and a cache, M = 15000 27.1, 28.8; 17000 30.6,
  // 28.9; 21000 33.8, 30.8 (fp32 tables 33.0, 29.5, fp32 weights and the kept product 40.0, 39.1); not at N = 1536, M = 8000
  // 25.7, 28.0 and 10000 29.0, 29.7.
  const int64_t cus = device_cus_cached();
  if constexpr (EPI == GB_BF16 || EPI == GB_F32 || EPI == GB_QKV || EPI == GB_QKV_BF16 || EPI == GB_QKV_W32) {
    const int64_t wide = gb_tiles<GbWide>(M, N), square = gb_tiles<GbSquare>(M, N);
    const int64_t wide_rounds = (wide + cus - 1) / cus, square_rounds = (square + 2 * cus - 1) / (2 * cus);
    const bool fits = EPI == GB_BF16 || EPI == GB_F32
                          ? square_rounds > 1 && (K >= 1024 || (square_rounds >= 2 * wide_rounds &&
                                                                (K >= 768 || wide_rounds == 1)))
                          : N <= 1024 && wide_rounds == 1 && square > 3 * cus;
    if (fits) return launch_big_shape<EPI, GbWide>(x, w, y, M, N, K, qa, s);
  }
  // Batches whose 128 x 128 tiles leave CUs without one take smaller tiles (the same bits): a tile is a chain of slabs,
  // and more, shorter chains run side by side. Residual product N = 512, K = 512 / 1536 / 2048, us with 128 x 128, 64 x
  // 128, 64 x 64 tiles: M = 1324 (44 tiles of 128 x 128) 9.3 / 15.7 / 22.6, 8.1 / 10.5 / 18.6, 8.3 / 9.3 / 10.9; 4099
  // (132) 9.7 / 21.1 / 24.3, 8.5 / 17.0 / 21.4, 8.6 / 17.4 / 21.7; 7500 (236) 10.0 / 21.4 / 25.6, 9.3 / 18.8 / 22.8,
  // 10.6 / 21.1 / 25.6; 9000 (284) 13.7 / 25.4 / 29.4, 11.9 / 26.6 / 30.6, 13.5 / 31.3 / 38.8. The plain and fp32
  // epilogues go the same way (N = 512, bf16 out, K = 512 / 1536 / 3072: M = 4099 6.2 / 17.3 / 32.4, 6.1 / 12.0 / 27.0, 6.1 /
  // 14.7 / 26.7; 7500 6.5 / 18.6 / 33.3, 6.3 / 17.0 / 29.9, 7.1 / 18.9 / 33.9; fp32 out, K = 512: 6.9, 6.6, 6.4 and 7.5, 7.0,
  // 7.6); the SwiGLU product of N = 1536 has more tiles than CUs from M = 1281 on. The Wqkv epilogues
  // keep 128 x 128 ones: 64 x 128 tiles at M = 4099 take 12.5 us with bf16 tables and a cache, 10.5 with fp32 ones, 11.0 with
  // fp32 weights and the kept product, 15.9 at N = 1536 without norm, against 12.4, 10.5, 12.3 and 13.9.
  if constexpr (EPI != GB_QKV && EPI != GB_QKV_BF16 && EPI != GB_QKV_W32) {
    constexpr int OUT_COLS = EPI == GB_SWIGLU ? GbSquare::BW / 2 : GbSquare::BW;
    const int64_t tiles = (M + GbSquare::BM - 1) / GbSquare::BM * ((N + OUT_COLS - 1) / OUT_COLS);
    if (2 * tiles <= cus) return launch_big_shape<EPI, GbSmall>(x, w, y, M, N, K, qa, s);
    if (tiles <= cus) return launch_big_shape<EPI, GbFlat>(x, w, y, M, N, K, qa, s);
  }
  return launch_big_shape<EPI, GbSquare>(x, w, y, M, N, K, qa, s);
}

// Entry used by vk_linear for large M and by vk_gemm_rows (K % 64 == 0: whole slabs, of any count; N % 8 == 0: whole
// 16-byte output chunks).
int gemm_big(const bf16_t *x, const bf16_t *w, void *y, int64_t M, int N, int K, bool swiglu, bool out_f32,
             hipStream_t s) {
  const GbQkv none{};
  if (swiglu) return launch_big<GB_SWIGLU>(x, w, y, M, N, K, none, s);
  if (out_f32) return launch_big<GB_F32>(x, w, y, M, N, K, none, s);
  return launch_big<GB_BF16>(x, w, y, M, N, K, none, s);
}

// The SwiGLU product that also stores its gate | up rows [M, 2 N] to gu (for vk_linear's gu_out).
int gemm_big_swiglu_keep(const bf16_t *x, const bf16_t *w, void *y, bf16_t *gu, int64_t M, int N, int K,
                         hipStream_t s) {
  GbQkv keep{};
  keep.raw = gu;
  return launch_big<GB_SWIGLU>(x, w, y, M, N, K, keep, s);
}

}  // namespace vk

using namespace vk;

extern "C" int vk_linear_qkv_rope(const void *x, const void *w, int64_t M, int32_t K, const void *q_norm_w,
                                  const void *k_norm_w, int32_t norm_w_dtype, float eps, const void *cos_t, const void *sin_t,
                                  int32_t table_dtype, int64_t table_rows, const int32_t *pos, const int32_t *rope_pos,
                                  const int32_t *seq, void *q, int64_t q_ld, void *k_cache, void *v_cache,
                                  int64_t stride_cb, int64_t stride_cs, int64_t cache_rows, int64_t cache_len,
                                  void *k_out, void *v_out, int64_t kv_ld, void *qkv_out, int32_t n_heads,
                                  int32_t n_kv_heads, int32_t head_dim, void *stream) {
  VK_CHECK_ARG(x && w && cos_t && sin_t && q, "linear_qkv_rope: null pointer");
  VK_CHECK_ARG(head_dim == 64, "linear_qkv_rope: built for head_dim 64 (got %d)", head_dim);
  VK_CHECK_ARG(n_heads > 0 && n_kv_heads > 0, "linear_qkv_rope: bad head counts");
  const int N = 64 * (n_heads + 2 * n_kv_heads);
  VK_CHECK_ARG(M >= 0 && K > 0 && K % 64 == 0, "linear_qkv_rope: need K %% 64 == 0");
  VK_CHECK_ARG(M < (int64_t(1) << 31) / 256 * 256, "linear_qkv_rope: M too large");
  VK_CHECK_ARG((q_norm_w == nullptr) == (k_norm_w == nullptr), "linear_qkv_rope: q and k norm weights go together");
  VK_CHECK_ARG(table_dtype == VK_DTYPE_BF16 || table_dtype == VK_DTYPE_F32, "linear_qkv_rope: bad table dtype");
  VK_CHECK_ARG(norm_w_dtype == VK_DTYPE_BF16 || norm_w_dtype == VK_DTYPE_F32, "linear_qkv_rope: bad norm weight dtype");
  VK_CHECK_ARG(norm_w_dtype == VK_DTYPE_BF16 || table_dtype == VK_DTYPE_F32,
               "linear_qkv_rope: fp32 norm weights go with fp32 rotary tables");
  VK_CHECK_ARG(q_norm_w == nullptr || norm_w_dtype == VK_DTYPE_BF16 || (vk_aligned16(q_norm_w) && vk_aligned16(k_norm_w)),
               "linear_qkv_rope: fp32 norm weights must be 16-byte aligned");
  VK_CHECK_ARG(table_rows > 0 && (pos != nullptr || rope_pos != nullptr), "linear_qkv_rope: rotary positions");
  VK_CHECK_ARG((k_cache == nullptr) == (v_cache == nullptr), "linear_qkv_rope: k_cache and v_cache go together");
  VK_CHECK_ARG(k_cache == nullptr || (seq != nullptr && pos != nullptr), "linear_qkv_rope: cache writes need seq and pos");
  VK_CHECK_ARG((k_out == nullptr) == (v_out == nullptr), "linear_qkv_rope: k_out and v_out go together");
  VK_CHECK_ARG(q_ld % 8 == 0 && kv_ld % 8 == 0 && stride_cb % 8 == 0 && stride_cs % 8 == 0,
               "linear_qkv_rope: row strides must be multiples of 8 elements");
  VK_CHECK_ARG(vk_aligned16(cos_t) && vk_aligned16(sin_t), "linear_qkv_rope: rotary tables must be 16-byte aligned");
  VK_CHECK_ARG(qkv_out == nullptr || vk_aligned16(qkv_out), "linear_qkv_rope: qkv_out must be 16-byte aligned");
  VK_CHECK_ARG(vk_aligned16(x) && vk_aligned16(w) && vk_aligned16(q) && (k_cache == nullptr || (vk_aligned16(k_cache) &&
               vk_aligned16(v_cache))) && (k_out == nullptr || (vk_aligned16(k_out) && vk_aligned16(v_out))),
               "linear_qkv_rope: pointers must be 16-byte aligned");
  if (M == 0) return VK_OK;
  GbQkv qa;
  qa.qw = q_norm_w;
  qa.kw = k_norm_w;
  qa.eps = eps;
  qa.cos_t = cos_t;
  qa.sin_t = sin_t;
  qa.table_f32 = table_dtype == VK_DTYPE_F32;
  qa.table_rows = table_rows;
  qa.pos = pos;
  qa.rope_pos = rope_pos;
  qa.seq = seq;
  qa.q = static_cast<bf16_t *>(q);
  qa.q_ld = q_ld;
  qa.kc = static_cast<bf16_t *>(k_cache);
  qa.vc = static_cast<bf16_t *>(v_cache);
  qa.stride_cb = stride_cb;
  qa.stride_cs = stride_cs;
  qa.cache_rows = cache_rows;
  qa.cache_len = cache_len;
  qa.ko = static_cast<bf16_t *>(k_out);
  qa.vo = static_cast<bf16_t *>(v_out);
  qa.kv_ld = kv_ld;
  qa.raw = static_cast<bf16_t *>(qkv_out);
  qa.H = n_heads;
  qa.HKV = n_kv_heads;
  qa.resid_in = nullptr;
  const auto xb = static_cast<const bf16_t *>(x), wb = static_cast<const bf16_t *>(w);
  const int rc = norm_w_dtype == VK_DTYPE_F32 ? launch_big<GB_QKV_W32>(xb, wb, nullptr, M, N, K, qa, VK_STREAM(stream))
                 : qa.table_f32               ? launch_big<GB_QKV>(xb, wb, nullptr, M, N, K, qa, VK_STREAM(stream))
                                              : launch_big<GB_QKV_BF16>(xb, wb, nullptr, M, N, K, qa, VK_STREAM(stream));
  if (rc != VK_OK) return rc;
  return launch_status("linear_qkv_rope");
}

extern "C" int vk_linear_residual_big(const void *a, const void *w, void *x, int32_t x_dtype, int64_t M, int32_t N,
                                      int32_t K, const float *bias, float alpha, float *ss_out, const void *x_in,
                                      void *stream) {
  VK_CHECK_ARG(a && w && x && ss_out, "linear_residual_big: null pointer");
  VK_CHECK_ARG(x_in == nullptr || vk_aligned16(x_in), "linear_residual_big: x_in must be 16-byte aligned");
  VK_CHECK_ARG(x_dtype == VK_DTYPE_BF16 || x_dtype == VK_DTYPE_F32, "linear_residual_big: bad residual dtype");
  VK_CHECK_ARG(M >= 0 && N > 0 && N % 128 == 0 && K > 0 && K % 64 == 0,
               "linear_residual_big: need N %% 128 == 0 and K %% 64 == 0 (N=%d K=%d)", N, K);
  VK_CHECK_ARG(M < (int64_t(1) << 31) / 256 * 256, "linear_residual_big: M too large");
  VK_CHECK_ARG(vk_aligned16(a) && vk_aligned16(w) && vk_aligned16(x) && (bias == nullptr || vk_aligned16(bias)),
               "linear_residual_big: pointers must be 16-byte aligned");
  if (M == 0) return VK_OK;
  GbQkv qa{};
  qa.bias = bias;
  qa.alpha = alpha;
  qa.ss_out = ss_out;
  qa.resid_in = x_in;
  const auto ab = static_cast<const bf16_t *>(a), wb = static_cast<const bf16_t *>(w);
  const int rc = x_dtype == VK_DTYPE_F32 ? launch_big<GB_RESID_F32>(ab, wb, x, M, N, K, qa, VK_STREAM(stream))
                                         : launch_big<GB_RESID>(ab, wb, x, M, N, K, qa, VK_STREAM(stream));
  if (rc != VK_OK) return rc;
  return launch_status("linear_residual_big");
}
