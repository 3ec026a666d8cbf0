// The GSPO reward on the device: strict identity of each call against its window's label
// (scripts/gspo.py:86-89 with ref_errors, scripts/train.py:170-188):
//   empty label: 1 if len(call) <= empty_max else empty_max / len(call);
//   else 1 - (errors of the global (NW) alignment path that fall on scored label bases) / max(len(call), len(label)),
// where a mismatch or a deletion counts at its label base and an insertion at the label base before it
// (the first base for an insertion before any label base).
//
// The reference takes the path edlib's traceback returns (edlib.align(call, label, "NW", "path")). Here the
// path is fixed by a stated preference among the optimal predecessors of each cell -- diagonal (match or
// mismatch), then up (deletion of a label base), then left (insertion of a call base) -- and the count of
// scored errors is carried forward along each cell's chosen predecessor, which is exactly the count along
// the traceback from the last cell with the same preference (no traceback pass, no per-cell storage). The
// edit distance, and the count when every label base is scored, do not depend on the choice of path.
//
// MI355X design: the DP matrix as a systolic array. A wavefront owns 256 label rows, 4 consecutive ones per lane in
// registers, and advances one call base per step: lane l is l columns behind lane 0, takes the row above its 4 (lane
// l - 1's last row of the step before) and the call base through a one-lane DPP shift, and updates its 4 cells. Labels
// past 256 bases take more wavefronts of the same workgroup, each 128 columns behind the one above it; the row between
// two of them goes through a small LDS ring, handed over once per 64 columns at a barrier. A cell is one 32-bit word,
//   distance << 18 | move << 16 | count,
// so one v_min3_u32 over the three predecessors takes the smallest distance and, among equals, the preferred move
// (0 diagonal, 1 deletion, 2 insertion) with the count that belongs to it; the move bits are then cleared.
// Bound by the chain of integer instructions per cell. Steps whose 64 columns lie inside the call run without the
// column test (its branch and the copies it forces), nine unrolled, and the last lane's row is collected by a lane
// shift instead of a store per step; 4 rows per lane put two wavefronts on a SIMD where 8 left one. 512 calls of about
// 850 bases against labels of 700-1000: 353 us with the test in every step and 8 rows per lane, 278 without it, 218
// with 4 rows (labels of 510, one wavefront of 8 rows each: 6% slower with 4). The form before (a lane per cell of an
// anti-diagonal, three diagonals of 16-bit pairs in LDS) took 5.17 ms: every step waited on its LDS reads and a barrier.
#include <type_traits>

#include "common.h"

namespace vk {

constexpr int RW_MAX_REF = 4096;   // label bases: 16 wavefronts of 256 rows
constexpr int RW_MAX_CALL = 8192;  // call bases: distances stay below 2^14, counts below 2^16
constexpr int RW_R = 4;            // label rows per lane
constexpr int RW_ROWS = 64 * RW_R;
constexpr uint32_t RW_ONE = 1u << 18, RW_DEL = 1u << 16, RW_INS = 2u << 16;

// v moved one lane up (lane l gets lane l - 1's), `first` into lane 0
__device__ __forceinline__ uint32_t rw_shift(uint32_t v, uint32_t first) {
  return static_cast<uint32_t>(__builtin_amdgcn_update_dpp(static_cast<int>(first), static_cast<int>(v), 0x138, 0xf, 0xf, false));
}

// q moved one lane down (lane l gets lane l + 1's), the last lane's v into lane 63
__device__ __forceinline__ uint32_t rw_collect(uint32_t q, uint32_t v) {
  return static_cast<uint32_t>(__builtin_amdgcn_update_dpp(static_cast<int>(v), static_cast<int>(q), 0x130, 0xf, 0xf, false));
}

__global__ __launch_bounds__(1024) void strict_identity_kernel(
    const uint8_t *__restrict__ calls, const int64_t *__restrict__ call_off, const int32_t *__restrict__ call_len,
    const uint8_t *__restrict__ refs, const int64_t *__restrict__ ref_off, const int32_t *__restrict__ ref_len,
    const uint8_t *__restrict__ scored, const int32_t *__restrict__ ref_of_call, int n_refs, int max_ref,
    int max_call, float empty_max, float *__restrict__ reward, int32_t *__restrict__ dist_out,
    int32_t *__restrict__ err_out) {
  __shared__ uint32_t ring[RW_MAX_REF / RW_ROWS - 1][4][64];  // last row of wavefront w: 4 blocks of 64 columns
  __shared__ uint32_t sums[RW_MAX_REF / RW_ROWS];
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = blockIdx.x;
  int r = ref_of_call[c];
  r = r < 0 ? 0 : (r >= n_refs ? n_refs - 1 : r);
  int n = call_len[c], m = ref_len[r];
  n = n < 0 ? 0 : (n > max_call ? max_call : n);
  m = m < 0 ? 0 : (m > max_ref ? max_ref : m);
  if (m == 0) {  // a window without DNA
    if (threadIdx.x == 0) {
      reward[c] = n <= empty_max ? 1.0f : empty_max / static_cast<float>(n);
      dist_out[c] = n;
      err_out[c] = 0;
    }
    return;
  }
  const uint8_t *rg = refs + ref_off[r], *sg = scored + ref_off[r], *cg = calls + call_off[c];
  const int waves = (m + RW_ROWS - 1) / RW_ROWS;  // wavefronts with rows of this label (<= the workgroup's)

  // this lane's rows row0 + 1 .. row0 + 4 are label bases row0 .. row0 + 3 (rows past the label: never read by others)
  const int row0 = (wid * 64 + lane) * RW_R;
  uint32_t base[RW_R], cost[RW_R], left[RW_R];
  uint32_t own = 0;
#pragma unroll
  for (int i = 0; i < RW_R; ++i) {
    const bool in = row0 + i < m;
    base[i] = in ? rg[row0 + i] : 256u;
    const uint32_t sc = in && sg[row0 + i] != 0 ? 1u : 0u;
    cost[i] = RW_ONE + sc;
    own += sc;
  }
  // column 0: i deletions, counted at the scored bases above (an exclusive sum over lanes and wavefronts)
  uint32_t incl = own;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t t = __shfl_up(incl, o, 64);
    incl += lane >= o ? t : 0u;
  }
  if (lane == 63) sums[wid] = incl;
  __syncthreads();
  uint32_t before = incl - own;
  for (int w = 0; w < wid; ++w) before += sums[w];
  uint32_t diag = static_cast<uint32_t>(row0) * RW_ONE + before;
#pragma unroll
  for (int i = 0; i < RW_R; ++i) left[i] = (i ? left[i - 1] : diag) + cost[i];
  const uint32_t top_step = RW_ONE + (sg[0] != 0 ? 1u : 0u);  // row 0: j insertions, each counted at label base 0

  // steps t = 1 .. n + 63 in blocks of 64: lane l updates column t - l. Wavefront w runs block p - 2 w in phase p: the
  // 64 columns it reads were finished, with their last lane's lag of 63, two blocks after they began
  const int blocks = n > 0 ? (n + 63 + 63) / 64 : 0;
  uint32_t ch = 0, ring_out = 0;
  for (int p = 0; p < blocks + 2 * (waves - 1); ++p) {
    const int b = p - 2 * wid;
    if (wid < waves && b >= 0 && b < blocks) {
      const uint32_t next_ch = 64 * b + lane < n ? cg[64 * b + lane] : 0u;
      const uint32_t next_top = wid > 0 ? ring[wid - 1][b & 3][lane] : static_cast<uint32_t>(64 * b + lane + 1) * top_step;
      // a step; check: some lane may be outside columns 1 .. n (the first block, and those past column n - 64). The last
      // lane's last row is collected in ring_out, the latest 64 steps' values in lane order: it lags 63 columns, so after
      // step 62 they are the 64 columns of block b - 1
      auto step = [&](auto check, int s) {
        const uint32_t top = rw_shift(left[RW_R - 1], __builtin_amdgcn_readlane(next_top, s));
        ch = rw_shift(ch, __builtin_amdgcn_readlane(next_ch, s));
        const int j = 64 * b + s + 1 - lane;
        if (!check || (j >= 1 && j <= n)) {
          uint32_t d = diag, u = top;
#pragma unroll
          for (int i = 0; i < RW_R; ++i) {
            const uint32_t dd = d + (base[i] != ch ? cost[i] : 0u);
            const uint32_t du = u + (cost[i] + RW_DEL), dl = left[i] + (cost[i] + RW_INS);
            d = left[i];
            u = min(min(dd, du), dl) & ~(RW_DEL | RW_INS);
            left[i] = u;
          }
          diag = top;
        }
        ring_out = rw_collect(ring_out, left[RW_R - 1]);
      };
      constexpr std::true_type checked{};
      constexpr std::false_type unchecked{};
      const bool inside = b > 0 && 64 * (b + 1) <= n;
      if (inside) {
#pragma unroll 1
        for (int s = 0; s < 63; s += 9) {
#pragma unroll
          for (int e = 0; e < 9; ++e) step(unchecked, s + e);
        }
      } else {
#pragma unroll 1
        for (int s = 0; s < 63; ++s) step(checked, s);
      }
      if (wid + 1 < waves) ring[wid][(b - 1) & 3][lane] = ring_out;  // block b - 1 is complete
      if (inside)
        step(unchecked, 63);
      else
        step(checked, 63);
      // the last block's first column is the last one anybody needs (64 blocks >= n + 63)
      if (wid + 1 < waves && b == blocks - 1 && lane == 63) ring[wid][b & 3][0] = left[RW_R - 1];
    }
    if (waves > 1) __syncthreads();
  }

  const int at = m - 1 - row0;
  if (at >= 0 && at < RW_R) {
    uint32_t v = left[0];
#pragma unroll
    for (int i = 1; i < RW_R; ++i) v = at == i ? left[i] : v;
    const int d = static_cast<int>(v >> 18), e = static_cast<int>(v & 0xffffu);
    dist_out[c] = d;
    err_out[c] = e;
    reward[c] = 1.0f - static_cast<float>(e) / static_cast<float>(n > m ? n : m);
  }
}

// The bases of row c of the engine's output tokens (its decode: up to the first EOS, special tokens write nothing)
// to out[c, 0 .. len[c]): table [vocab, k + 1] holds each token's k bytes and, last, how many it writes. A workgroup
// per row, 4 tokens per thread and pass, the byte positions by a workgroup prefix sum.
__global__ __launch_bounds__(256) void tokens_to_bases_kernel(const int64_t *__restrict__ tokens, int T,
                                                              const uint8_t *__restrict__ table, int vocab, int k,
                                                              int eos, uint8_t *__restrict__ out,
                                                              int32_t *__restrict__ len) {
  __shared__ int stop_s[4], sum_s[4];
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int64_t row = blockIdx.x;
  const int64_t *tk = tokens + row * T;
  uint8_t *dst = out + row * T * k;
  int at = 0;
  for (int t0 = 0; t0 < T; t0 += 1024) {
    const int mine = t0 + 4 * tid;
    int id[4], stop = T;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int64_t v = mine + i < T ? tk[mine + i] : 0;
      id[i] = static_cast<int>(v < 0 ? 0 : (v >= vocab ? vocab - 1 : v));
      if (mine + i < T && id[i] == eos && stop == T) stop = mine + i;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) stop = min(stop, __shfl_xor(stop, o, 64));
    if (lane == 0) stop_s[wid] = stop;
    __syncthreads();
    stop = min(min(stop_s[0], stop_s[1]), min(stop_s[2], stop_s[3]));
    int nb[4], sum = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      nb[i] = mine + i < stop ? table[id[i] * (k + 1) + k] : 0;
      sum += nb[i];
    }
    int incl = sum;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int t = __shfl_up(incl, o, 64);
      incl += lane >= o ? t : 0;
    }
    if (lane == 63) sum_s[wid] = incl;
    __syncthreads();
    int pos = at + incl - sum;
    for (int w = 0; w < wid; ++w) pos += sum_s[w];
#pragma unroll
    for (int i = 0; i < 4; ++i)
      for (int e = 0; e < nb[i]; ++e) dst[pos++] = table[id[i] * (k + 1) + e];
    at += sum_s[0] + sum_s[1] + sum_s[2] + sum_s[3];
    if (stop < T) break;  // (the same for every thread)
    __syncthreads();      // the next pass writes stop_s / sum_s again
  }
  if (tid == 0) len[row] = at;
}

}  // namespace vk

using namespace vk;

extern "C" int vk_strict_identity(const uint8_t *calls, const int64_t *call_off, const int32_t *call_len,
                                  const uint8_t *refs, const int64_t *ref_off, const int32_t *ref_len,
                                  const uint8_t *scored, const int32_t *ref_of_call, int32_t n_calls, int32_t n_refs,
                                  int32_t max_ref_len, int32_t max_call_len, float empty_max, float *reward,
                                  int32_t *edit_distance, int32_t *scored_errors, void *stream) {
  VK_CHECK_ARG(call_off && call_len && ref_off && ref_len && ref_of_call && reward && edit_distance && scored_errors,
               "strict_identity: null pointer");
  VK_CHECK_ARG(n_calls >= 0 && n_refs > 0 && max_ref_len >= 0 && max_call_len >= 0, "strict_identity: bad sizes");
  if (max_ref_len > RW_MAX_REF || max_call_len > RW_MAX_CALL)
    return fail(VK_ERR_UNSUPPORTED, "strict_identity: labels up to %d and calls up to %d bases (got %d / %d)",
                RW_MAX_REF, RW_MAX_CALL, max_ref_len, max_call_len);
  VK_CHECK_ARG((max_call_len == 0 || calls) && (max_ref_len == 0 || (refs && scored)), "strict_identity: null data");
  if (n_calls == 0) return VK_OK;
  const int waves = max_ref_len > RW_ROWS ? (max_ref_len + RW_ROWS - 1) / RW_ROWS : 1;
  strict_identity_kernel<<<static_cast<unsigned>(n_calls), 64 * waves, 0, VK_STREAM(stream)>>>(
      calls, call_off, call_len, refs, ref_off, ref_len, scored, ref_of_call, n_refs, max_ref_len, max_call_len,
      empty_max, reward, edit_distance, scored_errors);
  return launch_status("strict_identity");
}

extern "C" int vk_tokens_to_bases(const int64_t *tokens, int32_t n_rows, int32_t T, const uint8_t *table, int32_t vocab,
                                  int32_t k, int32_t eos, uint8_t *out, int32_t *len, void *stream) {
  VK_CHECK_ARG(n_rows >= 0 && T >= 0 && vocab > 0 && k > 0 && k < 256, "tokens_to_bases: bad sizes");
  VK_CHECK_ARG(static_cast<int64_t>(T) * k < (int64_t(1) << 31) - 4096, "tokens_to_bases: rows too long");
  if (n_rows == 0) return VK_OK;
  VK_CHECK_ARG(table && len && (T == 0 || (tokens && out)), "tokens_to_bases: null pointer");
  tokens_to_bases_kernel<<<static_cast<unsigned>(n_rows), 256, 0, VK_STREAM(stream)>>>(tokens, T, table, vocab, k, eos,
                                                                                      out, len);
  return launch_status("tokens_to_bases");
}
