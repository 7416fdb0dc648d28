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
// Decode batches and anything else with at most 32 columns per KV head, every
// fp32 call, and masks whose key stride is not 1: one workgroup of 4 wavefronts
// per (sequence, KV head, 16 columns, part of the keys), a wavefront taking
// 16-key tiles round-robin. What bounds it is latency: a tile's K and V
// addresses come from slots that are loaded first. So a wavefront keeps the
// next tile's K, V and mask loads and the slots of the tile after that in
// flight behind the tile being computed, each slot loaded once per key and
// handed to the lanes that need it, and the keys are cut into parts when the
// call has too few workgroups for the CUs (two per CU fit). 24 sequences of up to
// 2048 keys, 28/4 heads of 128, bf16: 17.5 + 3.9 us (merge) against 107 us for one
// part, one tile at a time and four slot loads a lane; 4 workgroups per CU: 33.8 us.
template <int DT, int D, bool SERIAL>
__global__ __launch_bounds__(kWaves * 64) __attribute__((amdgpu_waves_per_eu(DT == IR_DTYPE_F32 && D == 128 ? 1 : 2)))
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
    if (a.num_slots > 0 && ti < t_hi) {
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

// ---------------------------------------------------------------- many columns, 16-bit
//
// Chunks: a workgroup of 4 wavefronts owns 128 columns of one KV head and one
// part of the keys; wavefront w owns columns 32 w .. 32 w + 31 as two 16-column
// tiles. Keys walk in 64-key tiles staged once per workgroup in LDS, K and V
// row-major with 32 bytes of padding a row (conflict-free operand reads; V^T
// through the transpose read), in a 2-deep ring: tile kb is computed while tile
// kb + 1 goes from registers to the other buffer, tile kb + 2's K and V and
// tile kb + 3's slots are in flight. Two workgroups share a CU (74 KB of LDS,
// at most 256 registers). 610 tokens x 5333 keys, 28/4 heads of 128, bf16: 109 + 7.5
// us (merge; 420 TFLOP/s over all pairs, masked ones included) against 827 us with
// 16 columns a workgroup and no staging: there every 16 columns read all keys
// again. The matrix and vector pipes carry the rest about equally, as in the
// chunked prefill.
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
  static_assert(!ML || (MB == 2 && kMaskTokens * (BN / 4) <= 2 * NT), "two 4-key mask pieces a thread");
  if (a.run_if && *a.run_if == 0) return;

  const int tid = threadIdx.x;
  const int lane = tid & 63, w = tid >> 6, g = lane >> 4, c = lane & 15;
  // workgroups that walk the same keys are a multiple of (KV heads x parts x
  // sequences) apart, so they mostly share an XCD's L2
  const int per_rt = a.num_kv_heads * a.parts * a.batch;
  const int rt = blockIdx.x / per_rt;
  int idx = blockIdx.x - rt * per_rt;
  const int kvh = idx % a.num_kv_heads;
  idx /= a.num_kv_heads;
  const int part = idx % a.parts;
  const int b = idx / a.parts;
  const int rows = a.seq_q * a.n_rep;

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
  const int ntiles = (a.seq_k + BN - 1) / BN;
  const int t_lo = (int)((int64_t)part * ntiles / a.parts);
  const int t_hi = (int)((int64_t)(part + 1) * ntiles / a.parts);

  bool bad = false;
  u32x4 kreg[KPT], vreg[KPT];
  bool use[KPT];
  // Slots: thread t < 64 loads key t's of a tile and, a step later, hands it to
  // the workgroup (-1: past the keys, or outside the pool, which is flagged).
  int64_t s_raw = -1;
  auto load_slot = [&](int kb) {
    const int t = kb * BN + tid;
    if (tid < BN) s_raw = t < a.seq_k ? gs[(int64_t)t * a.gs_t] : -1;
  };
  auto hand_slot = [&](int kb) {
    if (tid >= BN) return;
    const bool in = s_raw >= 0 && s_raw < a.num_slots;
    bad |= !in && kb * BN + tid < a.seq_k;
    slot_lds[kb & 1][tid] = in ? (int)s_raw : -1;
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
  auto issue = [&](int kb) {
    if constexpr (ML) load_mask(kb);
#pragma unroll
    for (int i = 0; i < KPT; ++i) {
      const int q = tid + NT * i;
      const int sl = slot_lds[kb & 1][q / PPR];
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

  auto tile = [&](int kb) {
    const int k0 = kb * BN;
    const uint16_t* kl = ks_lds[kb & 1];
    const uint16_t* vl = vs_lds[kb & 1];
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
          const u32x2 x = *(const u32x2*)&mk_lds[kb & 1][mtok[ct] * MP + 16 * kt + 4 * g];
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
    const uint64_t okm = __ballot(key_ok[kb & 1][lane] != 0);
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
  } else if (t_lo < t_hi) {
    load_slot(t_lo);
    hand_slot(t_lo);
    load_slot(t_lo + 1);
    __syncthreads();
    issue(t_lo);
    hand_slot(t_lo + 1);
    load_slot(t_lo + 2);
    stage(t_lo & 1);
    __syncthreads();
    if (t_lo + 1 < t_hi) issue(t_lo + 1);
    hand_slot(t_lo + 2);
    load_slot(t_lo + 3);
    __syncthreads();
    for (int kb = t_lo; kb < t_hi; ++kb) {
      tile(kb);
      if (kb + 1 < t_hi) stage((kb + 1) & 1);
      if (kb + 2 < t_hi) issue(kb + 2);
      hand_slot(kb + 3);
      load_slot(kb + 4);
      __syncthreads();
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
  PartMerge run;
#pragma unroll 4
  for (int p = 0; p < a.parts; ++p) {
    const int64_t pr = p * per_part + row;
    const f32x2 ml = *(const f32x2*)(a.ws_ml + pr * 2);
    const f32x4 v = *(const f32x4*)(a.ws_o + pr * D + d0);
    const float x[4] = {v[0], v[1], v[2], v[3]};
    run.add(ml[0], ml[1], x);
  }
  const int rows = a.seq_q * a.n_rep;
  const int64_t unit = row / rows;
  const int r = (int)(row - unit * rows);
  const int kvh = (int)(unit % a.num_kv_heads), b = (int)(unit / a.num_kv_heads);
  const int sq = r / a.n_rep;
  const int oh = kvh * a.n_rep + (r - sq * a.n_rep);
  store4<DT>(a.out + ((int64_t)b * a.o_b + (int64_t)sq * a.o_s + (int64_t)oh * a.o_h + d0) * TileShape<DT, D>::EB,
             run.o, run.L > 0.f ? 1.f / run.L : 0.f);
}

// ---------------------------------------------------------------- host side

constexpr int64_t kMaxPartBytes = 256ll << 20;  // bound of a call's partial rows

struct Split {
  bool wide;
  int64_t nwg;  // workgroups of one part
  int parts;    // parts that pay
};

// The kernel a call takes and the parts it would use. The wide kernel needs a
// 16-bit dtype, a mask of q's dtype or fp32 with unit key stride, and slots and
// mask byte offsets that fit 32 bits.
Split split_of(int64_t batch, int64_t seq_q, int64_t seq_k, int num_q_heads, int num_kv_heads, int dtype,
               int mask_dtype, int64_t mask_t_stride, int64_t num_slots) {
  const int64_t rows = seq_q * (num_q_heads / num_kv_heads);
  Split s;
  s.wide = rows > 32 && dtype != IR_DTYPE_F32 && (mask_dtype == dtype || mask_dtype == IR_DTYPE_F32) &&
           mask_t_stride == 1 && seq_k <= (1 << 28) && num_slots <= 0x7fffffff;
  s.nwg = batch * num_kv_heads * (s.wide ? (rows + kWideCols - 1) / kWideCols : (rows + 15) / 16);
  const int64_t slots = (int64_t)device_cus() * 2;
  const int64_t units = s.wide ? (seq_k + kTileKeys - 1) / kTileKeys / 2 : (seq_k + 15) / 16 / (2 * kWaves);
  s.parts = (int)std::max<int64_t>(1, std::min<int64_t>({s.nwg > 0 ? slots / s.nwg : 1, units, 64}));
  return s;
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
      else if (a.n_rep >= 5)
        hipLaunchKernelGGL((paged_masked_wide_kernel<DT, D, 2, true>), grid, block, 0, s, a);
      else
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
  const Split sp = split_of(batch, seq_q, seq_k, num_q_heads, num_kv_heads, dtype, mask_dtype, mask_t_stride, 0);
  const int64_t per = part_bytes(batch, seq_q, num_q_heads, head_dim);
  const int64_t parts = std::min<int64_t>(sp.parts, kMaxPartBytes / per);
  return parts > 1 ? parts * per : 0;
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
  const Split sp = split_of(batch, seq_q, seq_k, a.num_q_heads, num_kv_heads, dtype, mask_dtype, mask_t_stride,
                            num_slots);
  // as many parts as pay and the workspace holds (none: one part)
  const int64_t per = part_bytes(batch, seq_q, num_q_heads, head_dim);
  IR_REQUIRE(workspace_bytes >= 0 && (!workspace || aligned16(workspace)),
             "ir_paged_attention_masked: the workspace must be 16-byte aligned");
  // A gated call of the narrow kernel mostly does nothing (under capture once
  // per layer): it stays one launch, each workgroup taking the parts of the
  // ungated call one after the other, with the same bits.
  a.serial = run_if && !sp.wide;
  const int64_t room = a.serial ? kMaxPartBytes : workspace ? workspace_bytes : 0;
  a.parts = (int)std::max<int64_t>(1, std::min<int64_t>(sp.parts, room / per));
  a.ws_o = (float*)workspace;
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
