// Paged attention over per-key flat slot ids and an additive mask: the metadata
// contract of the reference seam (PagedContext.gather_slots + mask,
// infrared/cache/paged_kv_cache.py:75-91, infrared/model/triton_attention.py:81-129).
//
// Works for every mask the reference builds: the decode mask of
// infrared/engine/paged_engine.py:630-638, the causal prefix-hit mask of
// infrared/model/inputs.py:33-54 and the packed varlen mask of
// infrared/model/inputs.py:57-85. Query "columns" are (query token, head)
// pairs of one GQA group, 16 per wavefront tile, so a decode step puts the
// group's heads on the MFMA columns exactly like the block-table kernel.
//
// Softmax semantics follow infrared/model/layers.py:116-117: scores are
// q.k*scale + mask and the softmax runs in fp32. Base-2 scores are clamped at
// -FLT_MAX instead of overflowing to -inf, so a row masked entirely with
// finfo.min averages V uniformly over its keys, as the reference softmax does.
#include <algorithm>

#include "attn_tile.hpp"
#include "status.hpp"

namespace ir {
namespace {

constexpr int kWaves = 4;
constexpr int kTileKeys = 64;    // keys per LDS tile of the wide kernel
constexpr int kWideCols = 128;   // (query token, head) columns per wide workgroup
constexpr int kMaskTokens = 27;  // query tokens 128 columns touch at most, 5 or more heads a token

struct MaskedArgs {
  const uint8_t* q;
  int64_t q_b, q_s, q_h;  // elements
  const uint8_t* kc;
  const uint8_t* vc;
  int64_t c_slot, c_head;  // elements
  int64_t num_slots;
  const int64_t* gs;
  int64_t gs_b, gs_t;
  const uint8_t* mask;
  int64_t m_b, m_s, m_t;  // elements
  int mask_dtype;
  uint8_t* out;
  int64_t o_b, o_s, o_h;  // elements
  int batch, seq_q, seq_k, num_q_heads, num_kv_heads, n_rep, n_rt;
  float scale;
  int32_t* err;
  const int32_t* run_if;  // null, or run only when *run_if != 0
  // key-range parts of a call (1: each workgroup writes its output rows); row
  // ((part * batch + b) * H_kv + kv head) * rows + column of ws_o holds a part's
  // D unnormalised fp32 outputs of a column, of ws_ml its (max, sum)
  int parts;
  int serial;  // the workgroup takes every part itself, one after the other
  float* ws_o;
  float* ws_ml;
  // survey of the mask and the keys (vis null: none), see paged_masked_survey_kernel
  uint8_t* vis;      // [batch][128-column block][tile, padded to 64]: any key visible
  uint8_t* tok_vis;  // [batch][128-column block][group of 8 tiles][32 tokens]: a key clearly visible
  int2* walks;       // [batch][KV head][128-column block]: (parts, tiles) of its walk, parts < 0: of all tiles
  float* bounds;     // [batch][KV head][tile]: largest |K|, inf if K or V is not finite or a slot is bad
};

// Bits of one mask element; mask_val converts them. Split so that a load can
// stay in flight until its score is ready.
__device__ __forceinline__ uint32_t mask_bits(const MaskedArgs& a, int64_t off) {
  return a.mask_dtype == IR_DTYPE_F32 ? ((const uint32_t*)a.mask)[off] : (uint32_t)((const uint16_t*)a.mask)[off];
}

__device__ __forceinline__ float mask_val(int mask_dtype, uint32_t w) {
  switch (mask_dtype) {
    case IR_DTYPE_F32: return __uint_as_float(w);
    case IR_DTYPE_BF16: return bf16_to_f32(w);
    default: return f16_to_f32(w);
  }
}

// Running merge of parts in part order, one column's (max, sum) and 4 outputs:
// the one statement of its arithmetic, so a split call and a serial one give
// the same bits. Every part's max is at least -FLT_MAX: no exponent is NaN.
struct PartMerge {
  float M = -__FLT_MAX__, L = 0.f, o[4] = {0.f, 0.f, 0.f, 0.f};
  __device__ __forceinline__ void add(float m, float l, const float (&x)[4]) {
    const float Mn = fmaxf(M, m);
    const float wa = fast_exp2(M - Mn), wb = fast_exp2(m - Mn);
    L = __builtin_fmaf(wa, L, wb * l);
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = __builtin_fmaf(wa, o[e], wb * x[e]);
    M = Mn;
  }
};

// Row of a part's partial results (see MaskedArgs).
__device__ __forceinline__ int64_t part_row(const MaskedArgs& a, int part, int b, int kvh, int row) {
  return (((int64_t)part * a.batch + b) * a.num_kv_heads + kvh) * ((int64_t)a.seq_q * a.n_rep) + row;
}

// ---------------------------------------------------------------- few columns, or fp32
//
// Decode batches and anything else with at most 32 columns per KV head, short
// frames, every fp32 call, and masks whose key stride is not 1: one workgroup of 4 wavefronts
// per (sequence, KV head, 16 columns, part of the keys), a wavefront taking
// 16-key tiles round-robin. What bounds it is latency: a tile's K and V
// addresses come from slots that are loaded first. So a wavefront keeps the slots
// of the next tile in flight behind the tile being computed, each slot loaded once
// per key and handed to the lanes that need it, and the keys are cut into parts
// when the call has too few workgroups for the CUs (two per CU fit). 24 sequences of
// up to 2048 keys, 28/4 heads of 128, bf16: 17.5 + 3.9 us (merge) against 107 us for
// one part, one tile at a time and four slot loads a lane; 4 workgroups per CU: 33.8 us.
// 16-bit calls also keep the next tile's K, V and mask loads in flight, which gives
// what large batches have to gain (64 sequences x 2048 keys: 50.2 against 53.5 us with
// 8 KV heads of 64, 48.5 / 49.3 with 4 of 128) and costs small ones 0.2 us. fp32 calls
// do not: two tiles take 312 registers at head_dim 128, one 164, and with one
// wavefront a SIMD instead of three 256 tokens x 2048 keys took 193 us against 129,
// 64 decodes 127 / 103; at head_dim 64 43.8 us against 44.8.
template <int DT, int D, bool SERIAL>
__global__ __launch_bounds__(kWaves * 64) __attribute__((amdgpu_waves_per_eu(2)))
void paged_masked_kernel(MaskedArgs a) {
  typedef TileShape<DT, D> Sh;
  constexpr int EB = Sh::EB;
  __shared__ MergeSmem<kWaves, D> sm;
  // a gated call (the fallback half of a graph-captured decode-form check)
  // does nothing unless the check failed
  if (a.run_if && *a.run_if == 0) return;

  const int lane = threadIdx.x & 63;
  const int w = threadIdx.x >> 6;
  const int g = lane >> 4;
  const int c = lane & 15;

  int idx = blockIdx.x;
  const int part = SERIAL ? 0 : idx % a.parts;
  if (!SERIAL) idx /= a.parts;
  const int rt = idx % a.n_rt;
  idx /= a.n_rt;
  const int kvh = idx % a.num_kv_heads;
  const int b = idx / a.num_kv_heads;

  const int rows = a.seq_q * a.n_rep;
  const int row = rt * 16 + c;
  const bool col_ok = row < rows;
  const int sq = col_ok ? row / a.n_rep : 0;
  const int qh = kvh * a.n_rep + (col_ok ? row - sq * a.n_rep : 0);

  uint32_t qr[Sh::KDW];
  if (col_ok)
    load_k<DT, D>(a.q + ((int64_t)b * a.q_b + (int64_t)sq * a.q_s + (int64_t)qh * a.q_h) * EB, g, qr);
  else
    zero_dwords(qr);

  const uint8_t* kc = a.kc + (int64_t)kvh * a.c_head * EB;
  const uint8_t* vc = a.vc + (int64_t)kvh * a.c_head * EB;
  const int64_t slot_bytes = a.c_slot * EB;
  const int64_t mrow = (int64_t)b * a.m_b + (int64_t)sq * a.m_s;
  const int64_t* gs = a.gs + (int64_t)b * a.gs_b;
  const int ntiles = (a.seq_k + 15) >> 4;
  int t_hi = 0;
  State<D> st;
  bool bad = false;

  // slot of key 16 ti + c, the same in the four lane groups; -1 past the keys
  auto load_slot = [&](int ti) -> int64_t {
    const int t = ti * 16 + c;
    return ti < t_hi && t < a.seq_k ? gs[(int64_t)t * a.gs_t] : -1;
  };
  struct Loads {
    Tile<DT, D> tl;
    uint32_t mk[4];
    bool vok[4];
  };
  // Loads of tile ti, whose slots are s: a key that may not be read (past the
  // end, or a slot outside the pool, which is flagged) reads slot 0 (a pool of
  // no slots never gets here); its score becomes -inf and its V row zero.
  auto issue = [&](int ti, int64_t s, Loads& x) {
    const bool in = s >= 0 && s < a.num_slots;
    bad |= !in && ti * 16 + c < a.seq_k;
    const int64_t off = in ? s * slot_bytes : -1;
    load_k<DT, D>(kc + (in ? off : 0), g, x.tl.k);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int64_t vo = __shfl(off, 4 * g + r);
      x.vok[r] = vo >= 0;
      load_v<DT, D>(vc + (x.vok[r] ? vo : 0), c, x.tl.v[r]);
      x.mk[r] = col_ok && x.vok[r] ? mask_bits(a, mrow + (int64_t)(ti * 16 + 4 * g + r) * a.m_t) : 0u;
    }
  };
  auto compute = [&](Loads& x) {
    const f32x4 s = qk_tile<DT, D>(x.tl.k, qr);
    float sv[4];
#pragma unroll
    for (int r = 0; r < 4; ++r)
      sv[r] = x.vok[r] ? fmaxf((s[r] * a.scale + mask_val(a.mask_dtype, x.mk[r])) * kLog2e, -__FLT_MAX__) : kNegInf;
    softmax_pv<DT, D, false>(sv, x.tl.v, x.vok, st);
  };

  auto walk = [&](int p) {
    state_init(st);
    t_hi = (int)((int64_t)(p + 1) * ntiles / a.parts);
    int ti = (int)((int64_t)p * ntiles / a.parts) + w;
    if constexpr (DT == IR_DTYPE_F32) {
      if (a.num_slots > 0) {
        int64_t s = load_slot(ti);
        for (; ti < t_hi; ti += kWaves) {
          Loads x;
          issue(ti, s, x);
          s = load_slot(ti + kWaves);
          compute(x);
        }
      }
    } else if (a.num_slots > 0 && ti < t_hi) {
      Loads x, y;
      issue(ti, load_slot(ti), x);
      int64_t s_next = load_slot(ti + kWaves);
      // tile ti is in flight in x; two tiles per trip, so that each keeps its registers
      for (; ti < t_hi; ti += 2 * kWaves) {
        if (ti + kWaves < t_hi) issue(ti + kWaves, s_next, y);
        s_next = load_slot(ti + 2 * kWaves);
        compute(x);
        if (ti + kWaves >= t_hi) break;
        if (ti + 2 * kWaves < t_hi) issue(ti + 2 * kWaves, s_next, x);
        s_next = load_slot(ti + 3 * kWaves);
        compute(y);
      }
    }
    st.l = wave_sum_groups(st.l);
    merge_publish<kWaves, D>(sm, st, w, g, c);
    __syncthreads();
  };
  const int ncol = min(16, rows - rt * 16);
  constexpr int NIT = (16 * (D / 4) + kWaves * 64 - 1) / (kWaves * 64);  // a thread's (column, 4 outputs) items
  PartMerge run[NIT];
  auto column_of = [&](int i, int& hc, int& d0, float& M, float& L, float (&o)[4]) {
    const int it = threadIdx.x + i * kWaves * 64;
    if (it >= ncol * (D / 4)) return false;
    hc = it / (D / 4);
    d0 = (it - hc * (D / 4)) * 4;
    merge_column<kWaves, D>(sm, hc, d0, M, L, o);
    return true;
  };
  walk(part);
  if constexpr (SERIAL) {
    for (int p = 0;;) {
#pragma unroll
      for (int i = 0; i < NIT; ++i) {
        int hc, d0;
        float M, L, o[4];
        if (column_of(i, hc, d0, M, L, o)) run[i].add(M, L, o);
      }
      if (++p >= a.parts) break;
      __syncthreads();
      walk(p);
    }
  }
  if (bad || (a.num_slots <= 0 && a.seq_k > 0)) flag_error(a.err, IR_ERR_GATHER_RANGE);

#pragma unroll
  for (int i = 0; i < NIT; ++i) {
    int hc, d0;
    float M, L, o[4];
    if (!column_of(i, hc, d0, M, L, o)) continue;
    const int r = rt * 16 + hc;
    if (SERIAL) {
      L = run[i].L;
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = run[i].o[e];
    } else if (a.parts > 1) {
      const int64_t pr = part_row(a, part, b, kvh, r);
      *(f32x4*)(a.ws_o + pr * D + d0) = f32x4{o[0], o[1], o[2], o[3]};
      if (d0 == 0) *(f32x2*)(a.ws_ml + pr * 2) = f32x2{M, L};
      continue;
    }
    const int osq = r / a.n_rep;
    const int oh = kvh * a.n_rep + (r - osq * a.n_rep);
    const float inv = L > 0.f ? 1.f / L : 0.f;
    store4<DT>(a.out + ((int64_t)b * a.o_b + (int64_t)osq * a.o_s + (int64_t)oh * a.o_h + d0) * EB, o, inv);
  }
}

// ---------------------------------------------------------------- survey
//
// A packed frame's mask is block-diagonal: most of its 64-key tiles hold nothing
// a 128-column block may see, and what they add is exactly zero -- provided every
// row sees some key clearly, no score is large enough to bring a masked key back,
// and V is finite (0 * inf is NaN). This kernel finds out, so that the wide
// kernel may leave those tiles out; its parts are then cut from the tiles that
// remain, so probabilities are rounded against other running maxima than without
// a survey. It finds per (KV head, tile) the largest |K|, and per (column block,
// tile) whether any mask value is above kMasked, with a flag for each token that
// has one above kClear. One pass over the mask and the frame's keys. 610 tokens x
// 5333 keys (8 sequences), 28/4 heads of 128, bf16: 9 us + 7.5 us for the walks,
// after which the wide kernel takes 35 us instead of 109.
constexpr float kMasked = -6e4f;    // fp16's finfo.min is -65504
constexpr float kClear = -1e3f;
constexpr float kScoreBound = 25e3f;  // 2 x this + kMasked - kClear stays far below any exponent
constexpr int kSurveyTiles = 8;     // tiles of a mask workgroup: 8 keys a lane
constexpr int kPartTiles = 6;       // tiles of a surveyed block worth a part of their own (12: 72 us against 60
                                    // on 5 decodes and 3 chunks of 170, 79 against 87 on 3 chunks of 180 after 2000)
constexpr int kSurveyMin = 16;      // a surveyed call has at least these tiles
constexpr int kSurveyBlocks = 12;   // and 128-column blocks per (sequence, KV head)
constexpr int64_t kSurveyMaxWgs = 1 << 24;  // a launch holds fewer than 2^32 threads

// Workgroups of the survey: a tile of a KV head each, then kSurveyTiles tiles of a
// column block's mask each (n_rtw blocks a sequence).
inline int64_t survey_wgs(int64_t batch, int64_t num_kv_heads, int64_t nt, int64_t n_rtw) {
  return batch * (num_kv_heads * nt + n_rtw * ((nt + kSurveyTiles - 1) / kSurveyTiles));
}

template <int DT, int D>
__global__ __launch_bounds__(256) void paged_masked_survey_kernel(MaskedArgs a, int nt, int n_rtw) {
  using E = Elem<DT>;
  constexpr int PPR = D / 8;
  __shared__ uint32_t red[4][kSurveyTiles];
  if (a.run_if && *a.run_if == 0) return;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int n_key_wgs = a.batch * a.num_kv_heads * nt;
  if ((int)blockIdx.x < n_key_wgs) {
    // keys of one tile of one KV head
    const int t = blockIdx.x % nt, kvh = blockIdx.x / nt % a.num_kv_heads, b = blockIdx.x / nt / a.num_kv_heads;
    const uint16_t* kc = (const uint16_t*)a.kc + (int64_t)kvh * a.c_head;
    const uint16_t* vc = (const uint16_t*)a.vc + (int64_t)kvh * a.c_head;
    constexpr uint32_t kInfBits = DT == IR_DTYPE_BF16 ? 0x7f80u : 0x7c00u;
    uint32_t big = 0;  // largest |element| of K as bits; the infinity's for what disallows a survey
    bool bad = false;
#pragma unroll
    for (int i = 0; i < kTileKeys * PPR / 256; ++i) {
      const int q = tid + 256 * i, key = t * kTileKeys + q / PPR;
      if (key >= a.seq_k) continue;
      const int64_t sl = a.gs[(int64_t)b * a.gs_b + (int64_t)key * a.gs_t];
      if (sl < 0 || sl >= a.num_slots) {
        bad = true;
        big = kInfBits;
        continue;
      }
      const int64_t off = sl * a.c_slot + (q % PPR) * 8;
      const u32x4 k = *(const u32x4*)(kc + off), v = *(const u32x4*)(vc + off);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        big = max(big, max(k[e] & 0x7fffu, k[e] >> 16 & 0x7fffu));
        if ((v[e] & 0x7fffu) >= kInfBits || (v[e] >> 16 & 0x7fffu) >= kInfBits) big = max(big, kInfBits);
      }
    }
    if (bad) flag_error(a.err, IR_ERR_GATHER_RANGE);
#pragma unroll
    for (int o = 32; o; o >>= 1) big = max(big, (uint32_t)__shfl_xor((int)big, o));
    if (lane == 0) red[w][0] = big;
    __syncthreads();
    if (tid == 0) {
      big = max(max(red[0][0], red[1][0]), max(red[2][0], red[3][0]));
      a.bounds[blockIdx.x] = big >= kInfBits ? __builtin_inff() : E::lo(big);
    }
    return;
  }
  // the mask of one column block's tokens over kSurveyTiles tiles: a wavefront
  // per token, 8 keys a lane
  const int n_groups = (nt + kSurveyTiles - 1) / kSurveyTiles;
  const int idx = blockIdx.x - n_key_wgs;
  const int grp = idx % n_groups, rt = idx / n_groups % n_rtw, b = idx / n_groups / n_rtw;
  const int rows = a.seq_q * a.n_rep;
  const int tok0 = rt * kWideCols / a.n_rep;
  const int ntok = min(rt * kWideCols + kWideCols - 1, rows - 1) / a.n_rep - tok0 + 1;
  const int k0 = grp * (kSurveyTiles * kTileKeys) + lane * 8;
  uint8_t* tok_vis = a.tok_vis + (((int64_t)b * n_rtw + rt) * n_groups + grp) * 32;
  bool any = false;
  for (int tok = w; tok < ntok; tok += 4) {
    const uint16_t* row = (const uint16_t*)a.mask + (int64_t)b * a.m_b + (int64_t)(tok0 + tok) * a.m_s;
    bool clear = false;
    if (k0 + 8 <= a.seq_k) {
      uint32_t x[4];
      __builtin_memcpy(x, row + k0, 16);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float lo = E::lo(x[e]), hi = E::hi(x[e]);
        any |= !(lo <= kMasked) || !(hi <= kMasked);
        clear |= lo > kClear || hi > kClear;
      }
    } else {
      for (int t = k0; t < a.seq_k; ++t) {
        const float v = E::lo(row[t]);
        any |= !(v <= kMasked);
        clear |= v > kClear;
      }
    }
    const bool c = __any(clear);
    if (lane == 0) tok_vis[tok] = c;
  }
  const uint64_t bits = __ballot(any);  // 8 lanes a tile
  if (lane < kSurveyTiles) red[w][lane] = (bits >> (8 * lane) & 0xff) != 0;
  __syncthreads();
  if (tid < kSurveyTiles && grp * kSurveyTiles + tid < nt) {
    const int ntp = (nt + 63) / 64 * 64;
    a.vis[((int64_t)b * n_rtw + rt) * ntp + grp * kSurveyTiles + tid] =
        (red[0][tid] | red[1][tid] | red[2][tid] | red[3][tid]) != 0;
  }
}

// The walk of each column block: which tiles (those some token of it sees, or all
// of them when the survey found a reason) and how many parts they are worth. A
// kernel of its own so that the wide kernel's workgroups past a block's parts end
// after one load.
template <int DT, int D>
__global__ __launch_bounds__(256) void paged_masked_walks_kernel(MaskedArgs a, int nt, int n_rtw) {
  using E = Elem<DT>;
  __shared__ float red[8];
  __shared__ int cnt[4];
  if (a.run_if && *a.run_if == 0) return;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int rt = blockIdx.x % n_rtw, kvh = blockIdx.x / n_rtw % a.num_kv_heads;
  const int b = blockIdx.x / n_rtw / a.num_kv_heads;
  const int rows = a.seq_q * a.n_rep, row0 = rt * kWideCols;
  const int tok0 = row0 / a.n_rep;
  const int ntok = min(row0 + kWideCols - 1, rows - 1) / a.n_rep - tok0 + 1;
  float kmax = 0.f;
  for (int t = tid; t < nt; t += 256) kmax = fmaxf(kmax, a.bounds[((int64_t)b * a.num_kv_heads + kvh) * nt + t]);
  uint32_t qbig = 0;
#pragma unroll
  for (int i = 0; i < kWideCols * (D / 8) / 256; ++i) {
    const int q = tid + 256 * i, row = row0 + q / (D / 8);
    if (row >= rows) continue;
    const int sq = row / a.n_rep, head = kvh * a.n_rep + row - sq * a.n_rep;
    const u32x4 x = *(const u32x4*)((const uint16_t*)a.q + (int64_t)b * a.q_b + (int64_t)sq * a.q_s +
                                    (int64_t)head * a.q_h + (q % (D / 8)) * 8);
#pragma unroll
    for (int e = 0; e < 4; ++e) qbig = max(qbig, max(x[e] & 0x7fffu, x[e] >> 16 & 0x7fffu));
  }
  bool clear = true;  // a lane of wavefront 0 per token
  if (tid < ntok) {
    const int n_groups = (nt + kSurveyTiles - 1) / kSurveyTiles;
    const uint8_t* tv = a.tok_vis + ((int64_t)b * n_rtw + rt) * n_groups * 32 + tid;
    uint32_t any = 0;
    for (int i = 0; i < n_groups; ++i) any |= tv[i * 32];
    clear = any != 0;
  }
  const uint8_t* vis = a.vis + ((int64_t)b * n_rtw + rt) * ((nt + 63) / 64 * 64);
  int n = 0;
  for (int t = tid; t < nt; t += 256) n += vis[t] != 0;
#pragma unroll
  for (int o = 32; o; o >>= 1) {
    kmax = fmaxf(kmax, __shfl_xor(kmax, o));
    qbig = max(qbig, (uint32_t)__shfl_xor((int)qbig, o));
    n += __shfl_xor(n, o);
  }
  if (!__all(clear)) kmax = __builtin_inff();
  if (lane == 0) {
    red[w] = kmax;
    red[4 + w] = E::lo(qbig);
    cnt[w] = n;
  }
  __syncthreads();
  if (tid != 0) return;
  const float km = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  bool ok = true;  // (q: a NaN's bits are above the infinity's, and compare false below)
  float qm = 0.f;
  for (int i = 0; i < 4; ++i) {
    ok = ok && red[4 + i] < __builtin_inff();
    qm = fmaxf(qm, red[4 + i]);
  }
  ok = ok && km < __builtin_inff() && km * qm * (D * fabsf(a.scale)) < kScoreBound;
  n = ok ? cnt[0] + cnt[1] + cnt[2] + cnt[3] : nt;
  const int np = min(a.parts, max(1, (n + kPartTiles - 1) / kPartTiles));
  a.walks[blockIdx.x] = make_int2(ok ? np : -np, n);
}

// ---------------------------------------------------------------- many columns, 16-bit
//
// Chunks: a workgroup of 4 wavefronts owns 128 columns of one KV head and one
// part of the keys; wavefront w owns columns 32 w .. 32 w + 31 as two 16-column
// tiles. Keys walk in 64-key tiles staged once per workgroup in LDS, K and V
// row-major with 32 bytes of padding a row (conflict-free operand reads; V^T
// through the transpose read), in a 2-deep ring: tile kb is computed while tile
// kb + 1 goes from registers to the other buffer, tile kb + 2's K and V and
// tile kb + 3's slots are in flight. Two workgroups share a CU (at most 256
// registers; at head_dim 128 81,712 B of LDS with a staged mask, 208 B below half of
// a CU's, 74,384 B without). 610 tokens x 5333 keys, 28/4 heads of 128, bf16: 109 +
// 7.5 us (merge; 420 TFLOP/s over all pairs, masked ones included) against 827 us with
// 16 columns a workgroup and no staging: there every 16 columns read all keys again.
// Bound by the vector pipe's issue and by latency: 8 vector instructions a MFMA, 2.0
// times the matrix pipe's busy cycles, 43% of wavefront time in waits, 21% waiting to
// issue, no LDS bank conflicts (the same frame, surveyed).
//
// MB: bytes of a mask element (2: the dtype of q; 4: fp32). ML: the mask tile goes
// through LDS too, loaded a tile ahead once per token instead of once per column
// (16-bit masks, 5 or more heads a token: what the LDS left beside two workgroups
// per CU holds); else each lane reads its column's, four keys at a time. (The
// mask's key stride is 1 either way.)
template <int DT, int D, int MB, bool ML>
__global__ __launch_bounds__(kWaves * 64) __attribute__((amdgpu_waves_per_eu(2)))
void paged_masked_wide_kernel(MaskedArgs a) {
  constexpr int CT = 2, BN = kTileKeys, NT = kWaves * 64;
  constexpr int KROW = D + 16;         // elements of an LDS row
  constexpr int KPT = BN * D / 8 / NT;  // 16-byte pieces of K (and V) per thread
  constexpr int KS = D / 32, DTL = D / 16;
  constexpr int PPR = D / 8;  // pieces per row
  using E = Elem<DT>;
  __shared__ __attribute__((aligned(16))) uint16_t ks_lds[2][BN * KROW];
  __shared__ __attribute__((aligned(16))) uint16_t vs_lds[2][BN * KROW];
  constexpr int MP = BN + 4;  // elements of a staged mask row
  __shared__ __attribute__((aligned(16))) uint16_t mk_lds[ML ? 2 : 1][ML ? kMaskTokens * MP : 8];
  __shared__ int slot_lds[2][BN];
  __shared__ uint8_t key_ok[2][BN];
  static_assert(sizeof(ks_lds) + sizeof(vs_lds) + sizeof(mk_lds) + sizeof(slot_lds) + sizeof(key_ok) <= 80 * 1024,
                "two workgroups per CU");
  static_assert(!ML || (MB == 2 && kMaskTokens * (BN / 4) <= 2 * NT), "two 4-key mask pieces a thread");
  if (a.run_if && *a.run_if == 0) return;

  const int tid = threadIdx.x;
  const int lane = tid & 63, w = tid >> 6, g = lane >> 4, c = lane & 15;
  // parts outermost: the workgroups of a surveyed block's unused parts come last,
  // and those in use spread evenly over the XCDs (innermost: 49 us instead of 35);
  // with KV heads innermost the blocks that walk a KV head's keys share a few
  // XCDs' L2s
  const int n_rtw = (a.seq_q * a.n_rep + kWideCols - 1) / kWideCols;
  int idx = blockIdx.x;
  const int kvh = idx % a.num_kv_heads;
  idx /= a.num_kv_heads;
  const int rt = idx % n_rtw;
  idx /= n_rtw;
  const int b = idx % a.batch;
  const int part = idx / a.batch;
  const int rows = a.seq_q * a.n_rep;
  const int ntiles = (a.seq_k + BN - 1) / BN;
  // the tiles and parts of this block's walk: the survey's, else all of them
  int n = ntiles, np = a.parts;
  const uint8_t* vis = nullptr;
  if constexpr (ML) {
    if (a.vis) {
      const int2 x = a.walks[((int64_t)b * a.num_kv_heads + kvh) * n_rtw + rt];
      np = abs(x.x);
      if (part >= np) return;  // (the grid has parts for the longest walk)
      n = x.y;
      if (x.x > 0) vis = a.vis + ((int64_t)b * n_rtw + rt) * ((ntiles + 63) / 64 * 64);
    }
  }

  struct Col {
    int row, sq, head;
    bool ok;
  };
  auto column = [&](int ct) {
    const int row = rt * kWideCols + w * (CT * 16) + ct * 16 + c;
    const bool ok = row < rows;
    const int sq = ok ? row / a.n_rep : 0;
    return Col{row, sq, kvh * a.n_rep + (ok ? row - sq * a.n_rep : 0), ok};
  };

  u32x4 qreg[CT][KS];
  const uint8_t* mrow[CT];  // ML: unused
  int mtok[CT];             // ML: the column's staged mask row
  const int tok0 = rt * kWideCols / a.n_rep;
  const int ntok = min(rt * kWideCols + kWideCols - 1, rows - 1) / a.n_rep - tok0 + 1;
#pragma unroll
  for (int ct = 0; ct < CT; ++ct) {
    const Col col = column(ct);
    const uint16_t* qrow =
        (const uint16_t*)a.q + (int64_t)b * a.q_b + (int64_t)col.sq * a.q_s + (int64_t)col.head * a.q_h;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const u32x4 x = *(const u32x4*)(qrow + ks * 32 + 8 * g);  // (a valid row when !col.ok)
      qreg[ct][ks] = col.ok ? x : u32x4{0u, 0u, 0u, 0u};
    }
    mrow[ct] = a.mask + ((int64_t)b * a.m_b + (int64_t)col.sq * a.m_s) * MB;
    mtok[ct] = col.ok ? col.sq - tok0 : 0;
  }

  const uint16_t* kc = (const uint16_t*)a.kc + (int64_t)kvh * a.c_head;
  const uint16_t* vc = (const uint16_t*)a.vc + (int64_t)kvh * a.c_head;
  const int64_t* gs = a.gs + (int64_t)b * a.gs_b;

  // tiles to walk, 64 to a word; this part's share of them
  auto word = [&](int wi) -> uint64_t {
    const int t = wi * 64 + lane;
    return __ballot(t < ntiles && (!vis || vis[t]));
  };
  int skip = (int)((int64_t)part * n / np);
  int left = (int)((int64_t)(part + 1) * n / np) - skip;
  int wi = 0;
  uint64_t wbits = word(0);
  while (skip > 0 && __popcll(wbits) <= skip) {  // whole words before the share
    skip -= __popcll(wbits);
    wbits = word(++wi);
  }
  for (; skip > 0; --skip) wbits &= wbits - 1;
  // the share's next tile, or -1
  auto next = [&]() {
    if (left <= 0) return -1;
    while (!wbits) {
      if (++wi * 64 >= ntiles) {
        left = 0;
        return -1;
      }
      wbits = word(wi);
    }
    --left;
    const int t = wi * 64 + __builtin_ctzll(wbits);
    wbits &= wbits - 1;
    return __builtin_amdgcn_readfirstlane(t);
  };

  bool bad = false;
  u32x4 kreg[KPT], vreg[KPT];
  bool use[KPT];
  // Slots: thread t < 64 loads key t's of a tile and, a step later, hands it to
  // the workgroup (-1: past the keys, or outside the pool, which is flagged).
  int64_t s_raw = -1;
  auto load_slot = [&](int kb) {
    const int t = kb * BN + tid;
    if (tid < BN) s_raw = kb >= 0 && t < a.seq_k ? gs[(int64_t)t * a.gs_t] : -1;
  };
  auto hand_slot = [&](int kb, int buf) {
    if (tid >= BN) return;
    const bool in = s_raw >= 0 && s_raw < a.num_slots;
    bad |= !in && kb >= 0 && kb * BN + tid < a.seq_k;
    slot_lds[buf][tid] = in ? (int)s_raw : -1;
  };
  // mask pieces of tile kb (4 keys of one of the workgroup's tokens each); keys
  // past the end repeat the last one, their scores are -inf
  uint32_t mreg[2][2];
  auto load_mask = [&](int kb) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int q = tid + NT * i;
      const int tok = q / (BN / 4), t0 = kb * BN + (q % (BN / 4)) * 4;
      if (tok >= ntok) continue;
      const uint16_t* row = (const uint16_t*)a.mask + (int64_t)b * a.m_b + (int64_t)(tok0 + tok) * a.m_s;
      if (t0 + 4 <= a.seq_k) {
        __builtin_memcpy(mreg[i], row + t0, 8);
      } else {
        const int e = a.seq_k - 1;
        mreg[i][0] = row[min(t0, e)] | (uint32_t)row[min(t0 + 1, e)] << 16;
        mreg[i][1] = row[min(t0 + 2, e)] | (uint32_t)row[min(t0 + 3, e)] << 16;
      }
    }
  };
  // K and V pieces of tile kb; unusable keys read slot 0 and are zeroed where
  // they are staged
  auto issue = [&](int kb, int buf) {
    if constexpr (ML) load_mask(kb);
#pragma unroll
    for (int i = 0; i < KPT; ++i) {
      const int q = tid + NT * i;
      const int sl = slot_lds[buf][q / PPR];
      use[i] = sl >= 0;
      const int64_t off = (int64_t)(use[i] ? sl : 0) * a.c_slot + (q % PPR) * 8;
      kreg[i] = *(const u32x4*)(kc + off);
      vreg[i] = *(const u32x4*)(vc + off);
    }
  };
  auto stage = [&](int buf) {
    if constexpr (ML) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int q = tid + NT * i;
        if (q / (BN / 4) < ntok)
          *(u32x2*)&mk_lds[buf][q / (BN / 4) * MP + (q % (BN / 4)) * 4] = u32x2{mreg[i][0], mreg[i][1]};
      }
    }
#pragma unroll
    for (int i = 0; i < KPT; ++i) {
      const int q = tid + NT * i;
      const int key = q / PPR, p = q % PPR;
      const u32x4 z = {0u, 0u, 0u, 0u};
      *(u32x4*)&ks_lds[buf][key * KROW + p * 8] = use[i] ? kreg[i] : z;
      *(u32x4*)&vs_lds[buf][key * KROW + p * 8] = use[i] ? vreg[i] : z;
      if (p == 0) key_ok[buf][key] = use[i];
    }
  };

  f32x4 acc[CT][DTL];
  float m[CT], l[CT];
#pragma unroll
  for (int ct = 0; ct < CT; ++ct) {
    m[ct] = -__FLT_MAX__;
    l[ct] = 0.f;
#pragma unroll
    for (int dt = 0; dt < DTL; ++dt) acc[ct][dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  }

  auto tile = [&](int kb, int buf) {
    const int k0 = kb * BN;
    const uint16_t* kl = ks_lds[buf];
    const uint16_t* vl = vs_lds[buf];
    // the mask of keys k0 + 16 kt + 4 g .. + 3 of each column
    uint32_t mk[CT][4][MB];
    if constexpr (ML) {
    } else if (k0 + BN <= a.seq_k) {
#pragma unroll
      for (int ct = 0; ct < CT; ++ct)
#pragma unroll
        for (int kt = 0; kt < 4; ++kt)
          __builtin_memcpy(mk[ct][kt], mrow[ct] + (k0 + 16 * kt + 4 * g) * MB, 4 * MB);
    } else {
#pragma unroll
      for (int ct = 0; ct < CT; ++ct)
#pragma unroll
        for (int kt = 0; kt < 4; ++kt) {
          uint32_t e[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int t = min(k0 + 16 * kt + 4 * g + r, a.seq_k - 1);  // (keys past the end are -inf below)
            e[r] = MB == 2 ? (uint32_t)((const uint16_t*)mrow[ct])[t] : ((const uint32_t*)mrow[ct])[t];
          }
          if constexpr (MB == 2) {
            mk[ct][kt][0] = e[0] | e[1] << 16;
            mk[ct][kt][1] = e[2] | e[3] << 16;
          } else {
#pragma unroll
            for (int r = 0; r < 4; ++r) mk[ct][kt][r] = e[r];
          }
        }
    }
    f32x4 sc[CT][4];
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
      for (int kt = 0; kt < 4; ++kt) sc[ct][kt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int kt = 0; kt < 4; ++kt) {
        const u32x4 ka = *(const u32x4*)&kl[(kt * 16 + c) * KROW + ks * 32 + 8 * g];
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) sc[ct][kt] = mfma_k32<DT>(ka, qreg[ct][ks], sc[ct][kt]);
      }
    if constexpr (ML) {
#pragma unroll
      for (int ct = 0; ct < CT; ++ct)
#pragma unroll
        for (int kt = 0; kt < 4; ++kt) {
          const u32x2 x = *(const u32x2*)&mk_lds[buf][mtok[ct] * MP + 16 * kt + 4 * g];
          mk[ct][kt][0] = x[0];
          mk[ct][kt][1] = x[1];
        }
    }
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
      for (int kt = 0; kt < 4; ++kt)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          float mv;
          if constexpr (MB == 2)
            mv = r & 1 ? E::hi(mk[ct][kt][r >> 1]) : E::lo(mk[ct][kt][r >> 1]);
          else
            mv = __uint_as_float(mk[ct][kt][r]);
          sc[ct][kt][r] = fmaxf((sc[ct][kt][r] * a.scale + mv) * kLog2e, -__FLT_MAX__);
        }
    // keys that may not be read: rare, so one vote over the tile's 64 keys
    const uint64_t okm = __ballot(key_ok[buf][lane] != 0);
    if (okm != ~0ull) {
#pragma unroll
      for (int kt = 0; kt < 4; ++kt)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (!(okm >> (16 * kt + 4 * g + r) & 1)) {
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) sc[ct][kt][r] = kNegInf;
          }
    }
    u32x4 pb[CT][2];
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
      float mx = kNegInf;
#pragma unroll
      for (int kt = 0; kt < 4; ++kt)
        mx = fmaxf(mx, fmaxf(fmaxf(sc[ct][kt][0], sc[ct][kt][1]), fmaxf(sc[ct][kt][2], sc[ct][kt][3])));
      mx = wave_max_groups_swap(mx);
      const bool grow = mx > m[ct] + kRescaleSlack;
      if (__any(grow)) {
        const float m_new = grow ? mx : m[ct];
        const float alpha = fast_exp2(m[ct] - m_new);  // 1 if unchanged, 0 from the start value
        l[ct] *= alpha;
#pragma unroll
        for (int dt = 0; dt < DTL; ++dt) acc[ct][dt] *= alpha;
        m[ct] = m_new;
      }
#pragma unroll
      for (int kt = 0; kt < 4; ++kt) {
#pragma unroll
        for (int r = 0; r < 4; ++r) sc[ct][kt][r] = fast_exp2(sc[ct][kt][r] - m[ct]);
        l[ct] += (sc[ct][kt][0] + sc[ct][kt][1]) + (sc[ct][kt][2] + sc[ct][kt][3]);
      }
      // P rounded to the input dtype, as softmax(...).to(q.dtype) does; k-slots
      // 0..3 = keys 4g.. of 16-key group 2 st, 4..7 = those of group 2 st + 1
#pragma unroll
      for (int st = 0; st < 2; ++st)
        pb[ct][st] = u32x4{E::pack2(sc[ct][2 * st][0], sc[ct][2 * st][1]), E::pack2(sc[ct][2 * st][2], sc[ct][2 * st][3]),
                           E::pack2(sc[ct][2 * st + 1][0], sc[ct][2 * st + 1][1]),
                           E::pack2(sc[ct][2 * st + 1][2], sc[ct][2 * st + 1][3])};
    }
    const int v_lane = (4 * g + (c >> 2)) * KROW + 4 * (c & 3);
#pragma unroll
    for (int t = 0; t < 2 * DTL; ++t) {
      const int dt = t % DTL, st = t / DTL;
      lds_u16* p = (lds_u16*)vl + v_lane + 32 * st * KROW + 16 * dt;
      const u32x2 lo = lds_read_tr16(p);
      const u32x2 hi = lds_read_tr16(p + 16 * KROW);
      const u32x4 va = {lo[0], lo[1], hi[0], hi[1]};
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) acc[ct][dt] = mfma_k32<DT>(va, pb[ct][st], acc[ct][dt]);
    }
  };

  if (a.num_slots <= 0) {
    bad = a.seq_k > 0;
  } else {
    int t0 = next(), t1 = next(), t2 = next(), t3 = next(), t4 = next();
    if (t0 >= 0) {
      load_slot(t0);
      hand_slot(t0, 0);
      load_slot(t1);
      __syncthreads();
      issue(t0, 0);
      hand_slot(t1, 1);
      load_slot(t2);
      stage(0);
      __syncthreads();
      if (t1 >= 0) issue(t1, 1);
      hand_slot(t2, 0);
      load_slot(t3);
      __syncthreads();
    }
    for (int i = 0; t0 >= 0; ++i) {
      tile(t0, i & 1);
      if (t1 >= 0) stage(i + 1 & 1);
      if (t2 >= 0) issue(t2, i & 1);
      hand_slot(t3, i + 1 & 1);
      load_slot(t4);
      __syncthreads();
      t0 = t1;
      t1 = t2;
      t2 = t3;
      t3 = t4;
      t4 = next();
    }
  }
  if (bad) flag_error(a.err, IR_ERR_GATHER_RANGE);

#pragma unroll
  for (int ct = 0; ct < CT; ++ct) {
    const float lsum = wave_sum_groups_swap(l[ct]);
    const Col col = column(ct);
    if (!col.ok) continue;
    if (a.parts > 1) {
      const int64_t pr = part_row(a, part, b, kvh, col.row);
#pragma unroll
      for (int dt = 0; dt < DTL; ++dt) *(f32x4*)(a.ws_o + pr * D + dt * 16 + 4 * g) = acc[ct][dt];
      if (g == 0) *(f32x2*)(a.ws_ml + pr * 2) = f32x2{m[ct], lsum};
      continue;
    }
    const float inv = lsum > 0.f ? 1.f / lsum : 0.f;
    uint8_t* orow = a.out + ((int64_t)b * a.o_b + (int64_t)col.sq * a.o_s + (int64_t)col.head * a.o_h) * 2;
#pragma unroll
    for (int dt = 0; dt < DTL; ++dt) {
      const float o[4] = {acc[ct][dt][0], acc[ct][dt][1], acc[ct][dt][2], acc[ct][dt][3]};
      store4<DT>(orow + (dt * 16 + 4 * g) * 2, o, inv);
    }
  }
}

// Output rows from a split call's parts, in part order: a thread per 4 columns
// of a row. A launch of its own rather than a last-arrival merge, so a split
// call needs no counters that survive it.
template <int DT, int D>
__global__ __launch_bounds__(256) void paged_masked_merge_kernel(MaskedArgs a) {
  if (a.run_if && *a.run_if == 0) return;
  const int64_t per_part = (int64_t)a.batch * a.num_kv_heads * a.seq_q * a.n_rep;
  const int64_t it = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t row = it / (D / 4);
  if (row >= per_part) return;
  const int d0 = (int)(it - row * (D / 4)) * 4;
  const int rows = a.seq_q * a.n_rep;
  const int64_t unit = row / rows;
  const int r = (int)(row - unit * rows);
  const int n_rtw = (rows + kWideCols - 1) / kWideCols;
  const int parts = a.vis ? abs(a.walks[unit * n_rtw + r / kWideCols].x) : a.parts;
  PartMerge run;
#pragma unroll 4
  for (int p = 0; p < parts; ++p) {
    const int64_t pr = p * per_part + row;
    const f32x2 ml = *(const f32x2*)(a.ws_ml + pr * 2);
    const f32x4 v = *(const f32x4*)(a.ws_o + pr * D + d0);
    const float x[4] = {v[0], v[1], v[2], v[3]};
    run.add(ml[0], ml[1], x);
  }
  const int kvh = (int)(unit % a.num_kv_heads), b = (int)(unit / a.num_kv_heads);
  const int sq = r / a.n_rep;
  const int oh = kvh * a.n_rep + (r - sq * a.n_rep);
  store4<DT>(a.out + ((int64_t)b * a.o_b + (int64_t)sq * a.o_s + (int64_t)oh * a.o_h + d0) * TileShape<DT, D>::EB,
             run.o, run.L > 0.f ? 1.f / run.L : 0.f);
}

// ---------------------------------------------------------------- host side

constexpr int kSurveyParts = 12;
constexpr int kFewKeys = 320;          // a frame of at most these keys,
constexpr int64_t kFewKeysAll = 8192;  // and these over all sequences and KV heads, may take the 16-column kernel
constexpr int64_t kMaxPartBytes = 256ll << 20;  // bound of a call's partial rows

struct Split {
  bool wide;
  bool survey;  // the wide kernel may be told which tiles to leave out
  int64_t nwg;  // workgroups of one part
  int parts;    // parts that pay
};

// The kernel a call takes and the parts it would use. The wide kernel needs a
// 16-bit dtype, a mask of q's dtype or fp32 with unit key stride, and slots and
// mask byte offsets that fit 32 bits. Few columns fill little of a 128-column
// workgroup: up to 16 the 16-column kernel is 1.2-1.5x faster (24 sequences x 2048
// keys, 4 KV heads of 128, bf16, 14 columns: 24.8 us against 35.6 wide), 17 to 32
// tie (28 columns: 40.6 / 36.8; one sequence of 4096: 14.1 / 17.1), and from 33 its
// third pass over the keys loses (35 columns, 64 sequences x 2048: 137 / 75.8). With
// few keys, though, that pass costs nothing and the shorter chain of the 16-column
// kernel wins while its workgroups are resident at once (28/4 heads of 128, us on
// 16 columns / wide: 40 tokens x 40 keys 5.7 / 8.8, 100 x 128 7.7 / 11.3, 256 x 256
// 13.9 / 17.9; 320 x 320, 560 workgroups: 23.2 / 21.9; 16 sequences of 5 x 256, 16K
// keys in all: 14.3 / 13.4; 100 x 512: 17.6 / 16.8).
Split split_of(int64_t batch, int64_t seq_q, int64_t seq_k, int num_q_heads, int num_kv_heads, int head_dim,
               int dtype, int mask_dtype, int64_t mask_t_stride, int64_t num_slots) {
  const int n_rep = num_q_heads / num_kv_heads;
  const int64_t rows = seq_q * n_rep;
  Split s;
  const int64_t slots = (int64_t)device_cus() * 2;
  const bool few_keys = seq_k <= kFewKeys && batch * num_kv_heads * seq_k <= kFewKeysAll &&
                        batch * num_kv_heads * ((rows + 15) / 16) <= slots;
  s.wide = rows > IR_MASKED_FEW_COLUMNS && !few_keys && dtype != IR_DTYPE_F32 &&
           (mask_dtype == dtype || mask_dtype == IR_DTYPE_F32) && mask_t_stride == 1 && seq_k <= (1 << 28) &&
           num_slots <= 0x7fffffff;
  const int64_t nt = (seq_k + kTileKeys - 1) / kTileKeys, n_rtw = (rows + kWideCols - 1) / kWideCols;
  s.nwg = batch * num_kv_heads * (s.wide ? n_rtw : (rows + 15) / 16);
  // The survey reads all keys and the mask once, a launch of ~10 us or one column
  // block's walk, whichever is more, and the walks another ~8: it can pay where
  // several blocks walk the same keys, long enough. bf16, 4 KV heads of 128, with
  // it against without: 256 tokens in 4 chunks after 2000 keys each (14 blocks, 131
  // tiles) 60 / 76 us, after 500 (37 tiles) 45 / 39; 512 in 8 after 200 (28, 39) 46 /
  // 54; 1024 in 16 (56, 291) 101 / 522; a 2048-token prompt (112, 32) 118 / 127. Few
  // blocks lose at any length: 73 tokens, 13 of them decodes (4, 257) 70 / 51; 64
  // sequences x 5 tokens (1, 32) 137 / 76. Tiles of 64 channels take less time each, so
  // more of them (2 KV heads: 515 tokens, 29 blocks, 101 tiles 41 / 45; 305, 17, 98 37 /
  // 33). A dense frame loses what the survey costs (512 tokens at the end of 4096 keys:
  // 108 / 78), which sizes alone do not tell.
  const bool worth = n_rtw >= kSurveyBlocks && nt >= kSurveyMin && s.nwg * nt >= slots * (head_dim == 64 ? 11 : 8);
  // (seq_k: its bytes stay small; its workgroups fit one launch)
  s.survey = s.wide && worth && mask_dtype == dtype && n_rep >= 5 && seq_k <= (1 << 20) &&
             survey_wgs(batch, num_kv_heads, nt, n_rtw) < kSurveyMaxWgs;
  const int64_t units = s.wide ? nt / 2 : (seq_k + 15) / 16 / (2 * kWaves);
  s.parts = (int)std::max<int64_t>(1, std::min<int64_t>({s.nwg > 0 ? slots / s.nwg : 1, units, 64}));
  // Surveyed walks differ in length: a block that holds decode rows walks all their
  // histories. More parts than fill the device cut it (13 decodes and 4 chunks after
  // 1000 keys: 178 us against 473 without them; 5 decodes and 3 chunks 60 / 98), and
  // cost a dense frame their merge (512 tokens after 3584: 107 / 89).
  if (s.survey && s.nwg < 2 * slots) s.parts = std::max(s.parts, (int)std::min<int64_t>(units, kSurveyParts));
  return s;
}

// Bytes of a surveyed call's vis, tok_vis, walks and bounds (each 256-byte aligned).
struct SurveyBytes {
  int64_t vis, tok_vis, walks, bounds;
  int64_t total() const { return vis + tok_vis + walks + bounds; }
};
SurveyBytes survey_bytes(const Split& sp, int64_t batch, int64_t seq_k, int num_kv_heads) {
  if (!sp.survey) return {0, 0, 0, 0};
  const int64_t nt = (seq_k + kTileKeys - 1) / kTileKeys, blocks = sp.nwg / num_kv_heads;  // of all sequences
  auto up = [](int64_t x) { return (x + 255) / 256 * 256; };
  return {up(blocks * ((nt + 63) / 64 * 64)), up(blocks * ((nt + kSurveyTiles - 1) / kSurveyTiles) * 32),
          up(sp.nwg * 8), up(batch * num_kv_heads * nt * 4)};
}

int64_t part_bytes(int64_t batch, int64_t seq_q, int num_q_heads, int head_dim) {
  return batch * seq_q * num_q_heads * (head_dim + 2) * 4;
}

template <int DT, int D>
void launch(const MaskedArgs& a, const Split& sp, hipStream_t s) {
  const dim3 grid((unsigned)(a.serial ? sp.nwg : sp.nwg * a.parts)), block(kWaves * 64);
  if constexpr (DT != IR_DTYPE_F32) {
    if (sp.wide) {
      if (a.mask_dtype == IR_DTYPE_F32)
        hipLaunchKernelGGL((paged_masked_wide_kernel<DT, D, 4, false>), grid, block, 0, s, a);
      else if (a.n_rep >= 5) {
        if (a.vis) {
          const int nt = (a.seq_k + kTileKeys - 1) / kTileKeys, n_rtw = (int)(sp.nwg / a.num_kv_heads / a.batch);
          const unsigned wgs = (unsigned)survey_wgs(a.batch, a.num_kv_heads, nt, n_rtw);
          hipLaunchKernelGGL((paged_masked_survey_kernel<DT, D>), dim3(wgs), dim3(256), 0, s, a, nt, n_rtw);
          hipLaunchKernelGGL((paged_masked_walks_kernel<DT, D>), dim3((unsigned)sp.nwg), dim3(256), 0, s, a, nt, n_rtw);
        }
        hipLaunchKernelGGL((paged_masked_wide_kernel<DT, D, 2, true>), grid, block, 0, s, a);
      } else
        hipLaunchKernelGGL((paged_masked_wide_kernel<DT, D, 2, false>), grid, block, 0, s, a);
    }
  }
  if (!sp.wide) {
    if (a.serial)
      hipLaunchKernelGGL((paged_masked_kernel<DT, D, true>), grid, block, 0, s, a);
    else
      hipLaunchKernelGGL((paged_masked_kernel<DT, D, false>), grid, block, 0, s, a);
  }
  if (a.parts > 1 && !a.serial) {
    const int64_t items = (int64_t)a.batch * a.seq_q * a.num_q_heads * (D / 4);
    hipLaunchKernelGGL((paged_masked_merge_kernel<DT, D>), dim3((unsigned)((items + 255) / 256)), dim3(256), 0, s, a);
  }
}

}  // namespace
}  // namespace ir

using namespace ir;

extern "C" int64_t ir_paged_attention_masked_workspace_size(int batch, int seq_q, int seq_k, int num_q_heads,
                                                            int num_kv_heads, int head_dim, int dtype,
                                                            int mask_dtype, int64_t mask_t_stride) {
  if (batch <= 0 || seq_q <= 0 || seq_k <= 0 || num_q_heads <= 0 || num_kv_heads <= 0 ||
      num_q_heads % num_kv_heads != 0 || (head_dim != 64 && head_dim != 128))
    return 0;
  const Split sp = split_of(batch, seq_q, seq_k, num_q_heads, num_kv_heads, head_dim, dtype, mask_dtype,
                            mask_t_stride, 0);
  const int64_t per = part_bytes(batch, seq_q, num_q_heads, head_dim);
  const int64_t parts = std::min<int64_t>(sp.parts, kMaxPartBytes / per);
  return (parts > 1 ? parts * per : 0) + survey_bytes(sp, batch, seq_k, num_kv_heads).total();
}

extern "C" int ir_paged_attention_masked(const void* q, int64_t q_b_stride, int64_t q_s_stride,
                                         int64_t q_h_stride, const void* k_cache, const void* v_cache,
                                         int64_t cache_slot_stride, int64_t cache_head_stride,
                                         int64_t num_slots, const int64_t* gather_slots, int64_t gs_b_stride,
                                         int64_t gs_t_stride, const void* mask, int64_t mask_b_stride,
                                         int64_t mask_s_stride, int64_t mask_t_stride, int mask_dtype,
                                         void* out, int64_t out_b_stride, int64_t out_s_stride,
                                         int64_t out_h_stride, int batch, int seq_q, int seq_k,
                                         int num_q_heads, int num_kv_heads, int head_dim, float scale,
                                         int dtype, int32_t* err_flags, const int32_t* run_if,
                                         ir_stream_t stream) {
  return ir_paged_attention_masked_ws(q, q_b_stride, q_s_stride, q_h_stride, k_cache, v_cache, cache_slot_stride,
                                      cache_head_stride, num_slots, gather_slots, gs_b_stride, gs_t_stride, mask,
                                      mask_b_stride, mask_s_stride, mask_t_stride, mask_dtype, out, out_b_stride,
                                      out_s_stride, out_h_stride, batch, seq_q, seq_k, num_q_heads, num_kv_heads,
                                      head_dim, scale, dtype, err_flags, run_if, nullptr, 0, stream);
}

extern "C" int ir_paged_attention_masked_ws(const void* q, int64_t q_b_stride, int64_t q_s_stride,
                                         int64_t q_h_stride, const void* k_cache, const void* v_cache,
                                         int64_t cache_slot_stride, int64_t cache_head_stride,
                                         int64_t num_slots, const int64_t* gather_slots, int64_t gs_b_stride,
                                         int64_t gs_t_stride, const void* mask, int64_t mask_b_stride,
                                         int64_t mask_s_stride, int64_t mask_t_stride, int mask_dtype,
                                         void* out, int64_t out_b_stride, int64_t out_s_stride,
                                         int64_t out_h_stride, int batch, int seq_q, int seq_k,
                                         int num_q_heads, int num_kv_heads, int head_dim, float scale,
                                         int dtype, int32_t* err_flags, const int32_t* run_if, void* workspace,
                                         int64_t workspace_bytes, ir_stream_t stream) {
  const int eb = dtype_bytes(dtype);
  IR_REQUIRE(eb > 0, "ir_paged_attention_masked: unknown dtype %d", dtype);
  IR_REQUIRE(dtype_bytes(mask_dtype) > 0, "ir_paged_attention_masked: unknown mask dtype %d", mask_dtype);
  IR_REQUIRE(batch >= 0 && seq_q >= 0 && seq_k >= 0 && num_q_heads > 0 && num_kv_heads > 0 && num_slots >= 0,
             "ir_paged_attention_masked: bad sizes");
  IR_REQUIRE(num_q_heads % num_kv_heads == 0,
             "ir_paged_attention_masked: num_q_heads %d not a multiple of num_kv_heads %d", num_q_heads,
             num_kv_heads);
  if (head_dim != 64 && head_dim != 128)
    return fail(IR_EUNSUPPORTED, "ir_paged_attention_masked: head_dim %d not supported (64, 128)", head_dim);
  if ((int64_t)batch * seq_q == 0) return ok();
  IR_REQUIRE(q && k_cache && v_cache && out && (seq_k == 0 || (gather_slots && mask)),
             "ir_paged_attention_masked: null pointer");
  IR_REQUIRE(aligned16(q) && aligned16(k_cache) && aligned16(v_cache) && aligned16(out),
             "ir_paged_attention_masked: q, caches and out must be 16-byte aligned");
  IR_REQUIRE((q_b_stride * eb) % 16 == 0 && (q_s_stride * eb) % 16 == 0 && (q_h_stride * eb) % 16 == 0 &&
                 (cache_slot_stride * eb) % 16 == 0 && (cache_head_stride * eb) % 16 == 0 &&
                 (out_b_stride * eb) % 16 == 0 && (out_s_stride * eb) % 16 == 0 &&
                 (out_h_stride * eb) % 16 == 0,
             "ir_paged_attention_masked: strides must be multiples of 16 bytes");
  MaskedArgs a;
  a.q = (const uint8_t*)q;
  a.q_b = q_b_stride;
  a.q_s = q_s_stride;
  a.q_h = q_h_stride;
  a.kc = (const uint8_t*)k_cache;
  a.vc = (const uint8_t*)v_cache;
  a.c_slot = cache_slot_stride;
  a.c_head = cache_head_stride;
  a.num_slots = num_slots;
  a.gs = gather_slots;
  a.gs_b = gs_b_stride;
  a.gs_t = gs_t_stride;
  a.mask = (const uint8_t*)mask;
  a.m_b = mask_b_stride;
  a.m_s = mask_s_stride;
  a.m_t = mask_t_stride;
  a.mask_dtype = mask_dtype;
  a.out = (uint8_t*)out;
  a.o_b = out_b_stride;
  a.o_s = out_s_stride;
  a.o_h = out_h_stride;
  a.batch = batch;
  a.seq_q = seq_q;
  a.seq_k = seq_k;
  a.num_q_heads = num_q_heads;
  a.num_kv_heads = num_kv_heads;
  a.n_rep = num_q_heads / num_kv_heads;
  a.n_rt = (int)(((int64_t)seq_q * a.n_rep + 15) / 16);
  a.scale = scale;
  a.err = err_flags;
  a.run_if = run_if;
  const Split sp = split_of(batch, seq_q, seq_k, a.num_q_heads, num_kv_heads, head_dim, dtype, mask_dtype,
                            mask_t_stride, num_slots);
  // as many parts as pay and the workspace holds (none: one part)
  const int64_t per = part_bytes(batch, seq_q, num_q_heads, head_dim);
  IR_REQUIRE(workspace_bytes >= 0 && (!workspace || aligned16(workspace)),
             "ir_paged_attention_masked: the workspace must be 16-byte aligned");
  // A gated call of the narrow kernel mostly does nothing (under capture once
  // per layer): it stays one launch, each workgroup taking the parts of the
  // ungated call one after the other, with the same bits.
  a.serial = run_if && !sp.wide;
  // The survey's bytes come first; a workspace too small for them goes without.
  const SurveyBytes sv = survey_bytes(sp, batch, seq_k, num_kv_heads);
  const bool survey = sv.total() > 0 && workspace && workspace_bytes >= sv.total() && num_slots > 0;
  uint8_t* ws = (uint8_t*)workspace;
  a.vis = a.tok_vis = nullptr;
  a.walks = nullptr;
  a.bounds = nullptr;
  if (survey) {
    a.vis = ws;
    a.tok_vis = a.vis + sv.vis;
    a.walks = (int2*)(a.tok_vis + sv.tok_vis);
    a.bounds = (float*)((uint8_t*)a.walks + sv.walks);
    ws += sv.total();
  }
  const int64_t room = a.serial ? kMaxPartBytes : workspace ? workspace_bytes - (survey ? sv.total() : 0) : 0;
  a.parts = (int)std::max<int64_t>(1, std::min<int64_t>(sp.parts, room / per));
  a.ws_o = (float*)ws;
  a.ws_ml = a.ws_o + (int64_t)a.parts * batch * seq_q * num_q_heads * head_dim;
  IR_REQUIRE(sp.nwg * a.parts < (1ll << 31), "ir_paged_attention_masked: grid too large");
  hipStream_t s = (hipStream_t)stream;
  switch (dtype) {
    case IR_DTYPE_BF16:
      if (head_dim == 128)
        launch<IR_DTYPE_BF16, 128>(a, sp, s);
      else
        launch<IR_DTYPE_BF16, 64>(a, sp, s);
      break;
    case IR_DTYPE_F16:
      if (head_dim == 128)
        launch<IR_DTYPE_F16, 128>(a, sp, s);
      else
        launch<IR_DTYPE_F16, 64>(a, sp, s);
      break;
    default:
      if (head_dim == 128)
        launch<IR_DTYPE_F32, 128>(a, sp, s);
      else
        launch<IR_DTYPE_F32, 64>(a, sp, s);
      break;
  }
  return check_launch("ir_paged_attention_masked");
}
