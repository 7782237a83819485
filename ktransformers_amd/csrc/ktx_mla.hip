// ktx_mla.hip — MLA compressed-KV paged attention (absorbed form) for gfx950.  C ABI in include/ktx_mla.h.
//
// All Hq query heads share one latent K = [ckv(512) | k_pe(64)] and V = ckv, so decode attention is two skinny GEMMs per
// KV tile:  S[heads, tokens] = Q[heads, 576] K^T  and  O[heads, 512] += P[heads, tokens] V[tokens, 512], both on
// v_mfma_f32_16x16x32_bf16 with fp32 softmax statistics (flash-decoding: the KV range is split across workgroups and
// the partial (m, l, O) triples are merged by a second launch).
//
// Workgroup = NWV waves; each wave owns 16 heads (Q fragments and the 16x512 fp32 output tile live in registers), all
// waves share one staged 32-token KV tile in LDS:
//   Kt [32][576+8]  bf16 row-major (pad 16 B), ckv rows land by LDS-DMA (global_load_lds, 1 KiB per wave-instruction)
//        -> B operand of S = Q K^T   : ds_read_b128, token = lane&15
//        -> B operand of O += P V    : ds_read_b64_tr_b16 x2 (hardware transpose: 8 tokens of one dim per lane)
//   Pt [NWV][16][32] bf16            : P re-laid from the MFMA C layout to the A layout (wave-private)
#include <hip/hip_runtime.h>

#include <algorithm>
#include <string>

#include "../../include/ktx_mla.h"
#include "ktx_common.h"

extern "C" int ktx_debug_get(int idx);   // ktx_moe.hip (include/ktx_moe.h)

typedef __bf16 v8bf __attribute__((ext_vector_type(8)));

#define MLA_TILE 32
#define MLA_DC 512
#define MLA_DR 64
#define MLA_KROW (MLA_DC + MLA_DR + 8)   // 584 elements = 1168 B (73 x 16 B: rows rotate through the 16-B bank slots)

struct MlaParams {
  const bf16_t *q_nope, *q_pe, *ckv, *k_pe;
  long long ckv_ts, kpe_ts;
  const int32_t *qo_indptr, *kv_indptr, *kv_indices, *kv_len, *d_bsz;
  int batch, total_q, Hq, page_size, nsplit;
  int tiles_shift;   // log2(page_size / 32) when the page size is a power of two (the reference's 64 and 256), else -1: tile -> page without a division
  float sm_scale;
  float* part_o;   // [total_q][Hq][nsplit][512]
  float* part_ml;  // [total_q][Hq][nsplit][2]
  int jobs;        // > 0 (mla_decode_wide_kernel): workgroups per head block that share the tokens' tiles; nsplit is a token's most splits then
  int* njobs;      // [total_q]: how many it takes
  bf16_t* out1;    // nsplit == 1: the split-KV kernel normalises and stores the result itself (no partials, no merge launch)
  float* lse1;
  // optional fused cache append for decode (one new token per request): latent rows [batch][512], [batch][64]
  const bf16_t *app_ckv, *app_kpe;
  bf16_t *ckv_w, *kpe_w;
  long long* dbg;   // tuning aid (scripts/mla_sweep.py): 16 wall-clock stamps per workgroup, NULL in normal use
};
#define MLA_TS(k)                                                                                             \
  do {                                                                                                        \
    if (p.dbg && threadIdx.x == 0)                                                                            \
      p.dbg[(((size_t)blockIdx.z * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x) * 16 + (k)] = wall_clock64(); \
  } while (0)

// the three stamps INSIDE the tile loop (first tile: landed, S done, tile done) cost every tile a compare, an exec save and a branch
// each — compiled in only for the stamp pass of scripts/mla_sweep.py (build with -DKTX_MLA_LOOP_STAMPS)
#ifdef KTX_MLA_LOOP_STAMPS
#define MLA_TS_LOOP(k) do { if (tile == t_begin) MLA_TS(k); } while (0)
#else
#define MLA_TS_LOOP(k) do { } while (0)
#endif

typedef short v4s16 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ v8bf as_v8bf(const uint4& u) {
  union { uint4 u; v8bf v; } c;
  c.u = u;
  return c.v;
}

// B operand of O += P V straight from the row-major K tile: two hardware-transposed LDS reads (ds_read_b64_tr_b16).
// Within a 16-lane group, lane i supplies the address of a 4-element chunk (row i/4, cols (i%4)*4..+3) of a
// [4 tokens][16 dims] block and receives column i of it, i.e. 4 consecutive tokens of one dim (probed on gfx950:
// scripts/tr_probe.hip).  base points at [token (lane>>4)*8 + ((lane&15)>>2)][dim0 + (lane&3)*4].
__device__ __forceinline__ v8bf load_v_frag(const bf16_t* base) {
  typedef __attribute__((address_space(3))) v4s16 lds_v4;
  const v4s16 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4*)(base));
  const v4s16 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4*)(base + 4 * MLA_KROW));
  union { v4s16 h[2]; v8bf v; } c;
  c.h[0] = lo;
  c.h[1] = hi;
  return c.v;
}

// One LDS-DMA wave-instruction: lane l's 16 bytes at gsrc_lane land at LDS byte address lds_addr + 16 l (M0 carries the
// wave-uniform LDS base).  Issued through inline asm ON PURPOSE: for an LDS-DMA it knows about, the compiler drains every
// pending DMA (s_waitcnt vmcnt(0)) in front of any LDS read it cannot prove disjoint from the destination — here the K / V
// fragment reads of the CURRENT tile while the NEXT tile's rows are in flight to the other buffer — which serialised the
// prefetch with the compute: 3.4 us per tile and workgroup, measured, i.e. one HBM round trip per tile.  Unseen by the
// compiler, completion is waited for explicitly in front of the per-tile barrier; the compiler's own waits for ITS loads can
// only wait longer than needed, never shorter (loads retire in order).
// The LDS destination is a BYTE ADDRESS off the dynamic region's base: a generic pointer costs a run-time address-space cast per use
// (a null check and a select), which this compiler also mis-selects in some code shapes (V_CMP_NE_U32 on src_shared_base: a build error).
__device__ __forceinline__ void mla_dma_row_a(const bf16_t* gsrc_lane, uint32_t lds_byte_addr) {
  const uint32_t lds_addr = __builtin_amdgcn_readfirstlane(lds_byte_addr);
  unsigned keep;
  asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off\n\ts_mov_b32 m0, %0"
               : "=&s"(keep)
               : "v"(gsrc_lane), "s"(lds_addr)
               : "memory");
}
// The same with the row's address as a SCALAR base + a 32-bit per-lane byte offset (the saddr form): a staged ckv row is one wave-uniform
// pointer, so its arithmetic (page, row, append override) runs on the scalar unit — as 64-bit per-lane pointers it was ~45 of the tile
// loop's ~260 VALU instructions, and the loop is VALU-issue bound (profiles/r06_W_mla_valu_diet_ab.txt).
__device__ __forceinline__ void mla_dma_row_sa(const bf16_t* gsrc_row, uint32_t lane_byte_off, uint32_t lds_addr) {
  unsigned keep;
  asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2\n\ts_mov_b32 m0, %0"
               : "=&s"(keep)
               : "v"(lane_byte_off), "s"(gsrc_row), "s"(lds_addr)
               : "memory");
}

// Staging of one 32-token tile, entirely by LDS-DMA (no VGPR destination, nothing the compiler has to wait for inside the
// loop).  A tile lies inside one page (page_size % 32 == 0 is required by the launcher), whose index is a scalar load.
// ckv: one 1-KiB row per wave-instruction into Kt[row]; k_pe: eight 128-byte rows per wave-instruction into Kp, 16-byte
// piece g of row r at position g ^ (r & 7) (the XOR keeps the fragment reads of 16 rows at most 2-way bank-conflicted
// although the rows are packed).  Rows past the end of the context re-read the last valid row: finite values that the
// softmax weights them with exactly 0 (their scores are masked), and nothing beyond kv_len is ever touched.
template <int NWV>
__device__ __forceinline__ void mla_stage(const MlaParams& p, int req, int kv_end, int app_pos, int tile, int page_v, int wave, int lane,
                                          uint32_t dK, uint32_t dP) {   // LDS byte addresses of the ckv and the k_pe rows
  const int tok0 = tile * MLA_TILE;
  const int page0 = __builtin_amdgcn_readfirstlane(page_v);
  const size_t row0 = (size_t)page0 * p.page_size + (p.tiles_shift >= 0 ? tok0 & (p.page_size - 1) : tok0 % p.page_size);
  const int last = kv_end - 1 - tok0;   // last valid row of the tile (>= 0: the tile holds a visible token)
  // a whole tile without the appended row (all but one or two tiles of a split): one 64-bit product for the tile, then adds — the
  // general form below spends ~25 scalar instructions per row on clamps, the append override and pointer casts (SQ counters of
  // the loop: as many SALU as VALU instructions, profiles/r06_Z_pmc_mla_decode_128k.txt)
  if (last >= MLA_TILE - 1 && (unsigned)(app_pos - tok0) >= (unsigned)MLA_TILE) {
    const bf16_t* src = p.ckv + (row0 + wave) * p.ckv_ts;
    const size_t step = (size_t)NWV * p.ckv_ts;
    uint32_t dst = dK + (uint32_t)wave * (MLA_KROW * 2);
#pragma unroll
    for (int r = wave; r < MLA_TILE; r += NWV, src += step, dst += NWV * MLA_KROW * 2) mla_dma_row_sa(src, (uint32_t)lane * 16u, dst);
    if (wave < 4) {
      const int r = wave * 8 + (lane >> 3), g = (lane & 7) ^ (lane >> 3);
      mla_dma_row_a(p.k_pe + (row0 + r) * p.kpe_ts + g * 8, dP + (uint32_t)wave * (8 * MLA_DR * 2));
    }
    return;
  }
#pragma unroll
  for (int r = wave; r < MLA_TILE; r += NWV) {   // (every term wave-uniform: scalar arithmetic, mla_dma_row_sa)
    const int rr = min(r, last);
    const bf16_t* src = p.ckv + (row0 + rr) * p.ckv_ts;
    if (tok0 + rr == app_pos) src = p.app_ckv + (size_t)req * MLA_DC;
    mla_dma_row_sa(src, (uint32_t)lane * 16u, dK + (uint32_t)r * (MLA_KROW * 2));
  }
  if (wave < 4) {
    const int r = wave * 8 + (lane >> 3), rr = min(r, last);
    const int g = (lane & 7) ^ (lane >> 3);
    const bf16_t* src = p.k_pe + (row0 + rr) * p.kpe_ts;
    if (tok0 + rr == app_pos) src = p.app_kpe + (size_t)req * MLA_DR;
    mla_dma_row_a(src + g * 8, dP + (uint32_t)wave * (8 * MLA_DR * 2));
  }
}

// which request owns query token qt?  Every wavefront resolves it on its own with ONE round of independent loads
// (lane i looks at request i) — the live-request count *d_bsz is fetched in the same round and applied afterwards, not
// waited for first: right after a kernel boundary each dependent load is another 1.5-3 us (measured with the phase stamps)
__device__ __forceinline__ void mla_find_request(const MlaParams& p, int qt, int lane, int& req, int& kv_end, int& page_base, int& app_pos) {
  req = -1; kv_end = 0; page_base = 0; app_pos = -1;
  const int bsz_raw = p.d_bsz ? *p.d_bsz : p.batch;
  for (int b0 = 0; b0 < p.batch && req < 0; b0 += 64) {
    const int i = b0 + lane;
    int q0 = 0x7fffffff, q1 = 0, kl = 0, kp = 0;
    if (i < p.batch) {
      q0 = p.qo_indptr[i]; q1 = p.qo_indptr[i + 1]; kl = p.kv_len[i]; kp = p.kv_indptr[i];
      // never index past the pages the request owns: a sequence that outgrew its cache attends to (and appends within)
      // its last page instead of reading kv_indices / writing HBM out of bounds
      kl = min(kl, (p.kv_indptr[i + 1] - kp) * p.page_size);
    }
    const int B = min(max(bsz_raw, 0), p.batch);
    const unsigned long long hit = __ballot(i < B && qt >= q0 && qt < q1);
    if (hit) {
      const int src = __ffsll((long long)hit) - 1;
      q0 = __builtin_amdgcn_readlane(q0, src); q1 = __builtin_amdgcn_readlane(q1, src);
      kl = __builtin_amdgcn_readlane(kl, src); kp = __builtin_amdgcn_readlane(kp, src);
      req = b0 + src;
      const int qo_len = q1 - q0;
      kv_end = max(kl - qo_len + (qt - q0) + 1, 0);   // causal: positions < kv_end are visible
      page_base = kp;
      // fused cache append (decode: one new token per request): the newest position is taken from the append buffers
      if (p.app_ckv && qo_len == 1) app_pos = kl - 1;
    }
  }
}

// The appended token (decode: one new row per request) is taken from the append buffers wherever its position is staged;
// the workgroup (hb 0) whose split owns its tile also writes it into the cache (StaticCache.update, custom_cache.py:189-195)
__device__ __forceinline__ void mla_store_appended(const MlaParams& p, int req, int page_base, int app_pos, int tid) {
  if (tid >= 72) return;
  const int page = p.kv_indices ? p.kv_indices[page_base + app_pos / p.page_size] : page_base + app_pos / p.page_size;
  const size_t trow = (size_t)page * p.page_size + app_pos % p.page_size;
  if (tid < 64) *reinterpret_cast<uint4*>(p.ckv_w + trow * p.ckv_ts + tid * 8) = *reinterpret_cast<const uint4*>(p.app_ckv + (size_t)req * MLA_DC + tid * 8);
  else *reinterpret_cast<uint4*>(p.kpe_w + trow * p.kpe_ts + (tid - 64) * 8) = *reinterpret_cast<const uint4*>(p.app_kpe + (size_t)req * MLA_DR + (tid - 64) * 8);
}

template <int NDT>
__device__ __forceinline__ void mla_store_result(const MlaParams& p, int qt, int head0, int ds, int lane, size_t pidx, bool any, const v4f (&o)[NDT],
                                                 const float (&m_run)[4], const float (&l_run)[4]) {
  if (p.out1) {   // one split holds the whole row: the merge kernel's arithmetic for a single partial (weight 1), in place
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int h = head0 + (lane >> 4) * 4 + r;
      const float l = __shfl(l_run[r], lane & 48), m = __shfl(m_run[r], lane & 48);
      const float inv = l > 0.f ? 1.0f / l : 0.f;
      bf16_t* po = p.out1 + ((size_t)qt * p.Hq + h) * MLA_DC + ds * NDT * 16;
#pragma unroll
      for (int i = 0; i < NDT; i++) po[i * 16 + (lane & 15)] = f32_to_bf16(o[i][r] * inv);
      if (p.lse1 && (lane & 15) == 0 && ds == 0)
        p.lse1[(size_t)qt * p.Hq + h] = l > 0.f ? (m + __logf(l)) * 1.44269504089f : -__builtin_inff();
    }
    return;
  }
  // ---- partial results: un-normalised O plus (m, l) per head ------------------------------------------------------------
#pragma unroll
  for (int r = 0; r < 4; r++) {
    const int hrow = (lane >> 4) * 4 + r;
    if ((lane & 15) == 0 && ds == 0) {
      float* ml = p.part_ml + (pidx + (size_t)hrow * p.nsplit) * 2;
      ml[0] = m_run[r];
      ml[1] = l_run[r];
    }
    if (any) {
      float* po = p.part_o + (pidx + (size_t)hrow * p.nsplit) * MLA_DC + ds * NDT * 16;
#pragma unroll
      for (int i = 0; i < NDT; i++) po[i * 16 + (lane & 15)] = o[i][r];
    }
  }
}

// Workgroup = HBW head blocks (16 heads each) x DSPLIT slices: wave (hbw, ds) computes 512/DSPLIT dims of O += P V (which
// divides the fp32 accumulator registers — the 128-VGPR O tile of the undivided form left one wave per SIMD running a
// serial chain of LDS reads and MFMAs, ~7 us per 32-token tile) and every DSPLIT-th 32-wide k-step of S = Q K^T; the DSPLIT
// partial score tiles of a head block meet in LDS and every wave adds them in the same order, so all of them hold the
// same S bit for bit.  (Round 1 had every wave compute the whole S: 36 MFMAs and 36 KiB of LDS reads per wave and tile
// instead of 10 and 10 — measured 3.5-4 us per tile and workgroup at 128 heads.)
// KV split s owns tiles s, s + nsplit, s + 2 nsplit, ...: balanced to within one tile whatever kv_len turns out to be.
template <int HBW, int DSPLIT>
__global__ __launch_bounds__(HBW * DSPLIT * 64) void mla_decode_kernel(MlaParams p) {
  constexpr int NWV = HBW * DSPLIT;
  constexpr int NDT = 32 / DSPLIT;   // 16-dim output tiles per wave
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  bf16_t* Kt = reinterpret_cast<bf16_t*>(smem);                        // [2][32][584] row-major ckv rows (+ pad)
  bf16_t* Kp = Kt + 2 * MLA_TILE * MLA_KROW;                           // [2][32][64] k_pe rows, 16-byte pieces XOR-swizzled
  bf16_t* Pt = Kp + 2 * MLA_TILE * MLA_DR;                             // [NWV][16][32]
  float* Sx = reinterpret_cast<float*>(Pt + NWV * 16 * MLA_TILE);      // [NWV][8][64] partial score tiles
  constexpr int NQ = (18 + DSPLIT - 1) / DSPLIT;                        // k-steps of S per wave: ds, ds + DSPLIT, ...
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int split = blockIdx.x, hb = blockIdx.y, qt = blockIdx.z;
  MLA_TS(0);

  // ---- Q fragments first: A[m = head (lane&15)][k = (lane>>4)*8 .. +7] for this wave's k-steps of 32 (of 16 nope + 2
  // rope).  Their addresses depend on nothing but the block indices, so they are in flight while the request lookup resolves.
  const int hbw = wave / DSPLIT, ds = wave % DSPLIT;
  const int head0 = (hb * HBW + hbw) * 16;
  v8bf qf[NQ];
  {
    const int h = head0 + (lane & 15);
    const bf16_t* qn = p.q_nope + ((size_t)qt * p.Hq + h) * MLA_DC + (lane >> 4) * 8;
    const bf16_t* qr = p.q_pe + ((size_t)qt * p.Hq + h) * MLA_DR + (lane >> 4) * 8;
#pragma unroll
    for (int j = 0; j < NQ; j++) {
      const int s = ds + j * DSPLIT;   // wave-uniform
      qf[j] = as_v8bf(make_uint4(0, 0, 0, 0));
      if (s < 16) qf[j] = as_v8bf(*reinterpret_cast<const uint4*>(qn + s * 32));
      else if (s < 18) qf[j] = as_v8bf(*reinterpret_cast<const uint4*>(qr + (s - 16) * 32));
    }
  }

  int req, kv_end, page_base, app_pos;
  mla_find_request(p, qt, lane, req, kv_end, page_base, app_pos);
  req = __builtin_amdgcn_readfirstlane(req);
  kv_end = __builtin_amdgcn_readfirstlane(kv_end);
  page_base = __builtin_amdgcn_readfirstlane(page_base);
  app_pos = __builtin_amdgcn_readfirstlane(app_pos);
  const size_t pidx = ((size_t)qt * p.Hq + head0) * p.nsplit + split;  // + head*nsplit per head
  if (req < 0) return;
  MLA_TS(1);

  const int ntiles = (kv_end + MLA_TILE - 1) / MLA_TILE;
  const int t_begin = split, t_end = ntiles, t_step = p.nsplit;   // tiles t_begin, t_begin + t_step, ... < t_end

  v4f o[NDT];
#pragma unroll
  for (int i = 0; i < NDT; i++) o[i] = v4f{0.f, 0.f, 0.f, 0.f};
  float m_run[4], l_run[4];
#pragma unroll
  for (int r = 0; r < 4; r++) { m_run[r] = -__builtin_inff(); l_run[r] = 0.f; }

  if (t_begin < t_end) {
    if (app_pos >= 0 && hb == 0 && (app_pos / MLA_TILE) % p.nsplit == split) mla_store_appended(p, req, page_base, app_pos, tid);

    // (LDS destinations as byte addresses off the dynamic region's base, Kt = smem: see mla_dma_row_a)
    const uint32_t lds0 = (uint32_t)(size_t)(__attribute__((address_space(3))) uint8_t*)smem;
    constexpr uint32_t KT_BYTES = MLA_TILE * MLA_KROW * 2, KP_BYTES = MLA_TILE * MLA_DR * 2;
    // The page of a tile is looked up ONE TILE AHEAD of its staging (page_of: the load is issued behind the previous tile's DMA requests
    // and waited for by the loop's own vmcnt(0) in front of the barrier): looked up inside stage() the index was a dependent load in
    // front of every tile's addresses — one exposed L2 round trip per tile with a real page table (the serving seam; the single-request
    // cache passes kv_indices == NULL).
    auto page_of = [&](int tile) -> int {
      const int pidx_ = __builtin_amdgcn_readfirstlane(page_base + (p.tiles_shift >= 0 ? tile >> p.tiles_shift : tile * MLA_TILE / p.page_size));
      return p.kv_indices ? p.kv_indices[pidx_] : pidx_;
    };
    auto stage = [&](int tile, int page_v, int buf) {   // buf = which of the two staged tiles
      mla_stage<NWV>(p, req, kv_end, app_pos, tile, page_v, wave, lane, lds0 + (uint32_t)buf * KT_BYTES, lds0 + 2 * KT_BYTES + (uint32_t)buf * KP_BYTES);
    };

    stage(t_begin, page_of(t_begin), 0);
    int page_nx = page_of(min(t_begin + t_step, t_end - 1));   // (clamped: always a tile of this request)
    MLA_TS(2);
    bf16_t* Pw = Pt + wave * 16 * MLA_TILE;

    int cur = 0;
    for (int tile = t_begin; tile < t_end; tile += t_step, cur ^= 1) {
      bf16_t* Kc = Kt + cur * MLA_TILE * MLA_KROW;
      const bf16_t* Pc = Kp + cur * MLA_TILE * MLA_DR;
      const int tok0 = tile * MLA_TILE;
      const int ntok = min(MLA_TILE, kv_end - tok0);
      // One barrier per tile: behind the explicit wait for this wave's LDS-DMA rows of this tile it publishes them and
      // proves every wave is done reading the other buffer, which the next tile's DMA may now overwrite.
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      MLA_TS_LOOP(3);
      if (tile + t_step < t_end) {
        stage(tile + t_step, page_nx, cur ^ 1);
        page_nx = page_of(min(tile + 2 * t_step, t_end - 1));
      }

      // ---- S = Q K^T for 2 x 16 tokens: this wave's k-steps -------------------------------------------------------------
      v4f s0 = {0.f, 0.f, 0.f, 0.f}, s1 = {0.f, 0.f, 0.f, 0.f};
      const bf16_t* kb0 = Kc + (lane & 15) * MLA_KROW + (lane >> 4) * 8;
      const bf16_t* kb1 = kb0 + 16 * MLA_KROW;
#pragma unroll
      for (int j = 0; j < NQ; j++) {
        const int s = ds + j * DSPLIT;
        if (s < 16) {   // wave-uniform
          const v8bf b0 = as_v8bf(*reinterpret_cast<const uint4*>(kb0 + s * 32));
          const v8bf b1 = as_v8bf(*reinterpret_cast<const uint4*>(kb1 + s * 32));
          s0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(qf[j], b0, s0, 0, 0, 0);
          s1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(qf[j], b1, s1, 0, 0, 0);
        } else if (s < 18) {   // rope k-step: piece (s-16)*4 + (lane>>4) of row (lane&15) (+16), un-swizzled
          const int row = lane & 15, q = (s - 16) * 4 + (lane >> 4);
          const bf16_t* pr = Pc + row * MLA_DR + ((q ^ (row & 7)) * 8);
          const v8bf b0 = as_v8bf(*reinterpret_cast<const uint4*>(pr));
          const v8bf b1 = as_v8bf(*reinterpret_cast<const uint4*>(pr + 16 * MLA_DR));
          s0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(qf[j], b0, s0, 0, 0, 0);
          s1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(qf[j], b1, s1, 0, 0, 0);
        }
      }
      if constexpr (DSPLIT > 1) {   // the head block's partial score tiles meet in LDS; fixed order -> identical S in every wave
        float* sx = Sx + wave * 512 + lane;
#pragma unroll
        for (int r = 0; r < 4; r++) { sx[r * 64] = s0[r]; sx[(4 + r) * 64] = s1[r]; }
        __syncthreads();
        const float* sr = Sx + hbw * DSPLIT * 512 + lane;
#pragma unroll
        for (int r = 0; r < 4; r++) { s0[r] = sr[r * 64]; s1[r] = sr[(4 + r) * 64]; }
#pragma unroll
        for (int d = 1; d < DSPLIT; d++)
#pragma unroll
          for (int r = 0; r < 4; r++) { s0[r] += sr[d * 512 + r * 64]; s1[r] += sr[d * 512 + (4 + r) * 64]; }
      }
      MLA_TS_LOOP(4);
      // lane holds S[head = (lane>>4)*4 + r][token = tok0 + (lane&15) (+16)]
      const bool v0 = (lane & 15) < ntok, v1 = 16 + (lane & 15) < ntok;
      float alpha[4], sa[4], sb[4], mx[4], ps[4];
#pragma unroll
      for (int r = 0; r < 4; r++) {
        sa[r] = v0 ? s0[r] * p.sm_scale : -__builtin_inff();
        sb[r] = v1 ? s1[r] * p.sm_scale : -__builtin_inff();
        mx[r] = fmaxf(sa[r], sb[r]);
      }
      row16_max4(mx[0], mx[1], mx[2], mx[3]);   // (the four heads' reductions interleaved: ktx_common.h)
      float pav[4], pbv[4], mnew[4];
#pragma unroll
      for (int r = 0; r < 4; r++) {
        mnew[r] = fmaxf(m_run[r], mx[r]);        // finite: every processed tile has >= 1 visible token
        pav[r] = __expf(sa[r] - mnew[r]);
        pbv[r] = __expf(sb[r] - mnew[r]);
        ps[r] = pav[r] + pbv[r];
      }
      row16_sum4(ps[0], ps[1], ps[2], ps[3]);
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const float pa = pav[r], pb = pbv[r], m_new = mnew[r], sum = ps[r];
        alpha[r] = __expf(m_run[r] - m_new);
        l_run[r] = l_run[r] * alpha[r] + sum;
        m_run[r] = m_new;
        // P to LDS in [head][token] order for the A-operand re-read (one v_cvt_pk_bf16_f32 for the pair)
        const int hrow = (lane >> 4) * 4 + r;
        const uint32_t pk = ktx_pk_bf16(pa, pb);
        Pw[hrow * MLA_TILE + (lane & 15)] = (bf16_t)(pk & 0xffffu);
        Pw[hrow * MLA_TILE + 16 + (lane & 15)] = (bf16_t)(pk >> 16);
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      const v8bf pf = as_v8bf(*reinterpret_cast<const uint4*>(Pw + (lane & 15) * MLA_TILE + (lane >> 4) * 8));

      // ---- O = O*alpha + P V ; V fragments by transposed reads of the same K tile ------------------------------------
      const bf16_t* vb = Kc + ((lane >> 4) * 8 + ((lane & 15) >> 2)) * MLA_KROW + (lane & 3) * 4 + ds * NDT * 16;
      // the rescale only where some head's running maximum moved (wave-uniform branch; alpha == 1 exactly otherwise, and o * 1 is o:
      // same bits) — past the first tiles of a long context that is rare, and the 4 * NDT multiplies were a sixth of the loop's VALU
      const bool moved = alpha[0] != 1.f || alpha[1] != 1.f || alpha[2] != 1.f || alpha[3] != 1.f;
      if (__builtin_amdgcn_ballot_w64(moved) != 0ull) {
#pragma unroll
        for (int i = 0; i < NDT; i++)
#pragma unroll
          for (int r = 0; r < 4; r++) o[i][r] *= alpha[r];
      }
#pragma unroll
      for (int i = 0; i < NDT; i++) {
        const v8bf b = load_v_frag(vb + i * 16);
        o[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pf, b, o[i], 0, 0, 0);
      }
      MLA_TS_LOOP(5);
    }
  }
  MLA_TS(6);

  mla_store_result<NDT>(p, qt, head0, ds, lane, pidx, t_begin < t_end, o, m_run, l_run);
  MLA_TS(7);
}

// ---- 64 heads per workgroup: batches, long contexts, prompts ------------------------------------------------------------------------
// Which query token and which of its KV splits a workgroup of the jobs form works on.  p.jobs workgroups (per head block) are shared out by
// what the requests hold: D, the tiles per job, is the smallest for which sum_t ceil(tiles_t / D) <= jobs (and no token takes more than
// nsplit, the workspace's slots); every wavefront finds it alone, lane = query token, from one round of loads.
struct MlaWork { int qt, split, nsp, req, kv_end, page_base, app_pos; };
__device__ __forceinline__ MlaWork mla_pick_job(const MlaParams& p, int job, int lane) {
  int q0 = 0x7fffffff, q1 = 0x7fffffff, kl = 0, kp = 0;
  const int bsz_raw = p.d_bsz ? *p.d_bsz : p.batch;
  if (lane < p.batch) {
    q0 = p.qo_indptr[lane]; q1 = p.qo_indptr[lane + 1]; kl = p.kv_len[lane]; kp = p.kv_indptr[lane];
    kl = min(kl, (p.kv_indptr[lane + 1] - kp) * p.page_size);   // never past the pages the request owns
  }
  const int B = min(max(bsz_raw, 0), p.batch);
  int r = 0;
  for (int i = 0; i < B; i++) r += __builtin_amdgcn_readlane(q1, i) <= lane ? 1 : 0;
  const int src = min(r, 63);
  const int tq0 = __shfl(q0, src, 64), tq1 = __shfl(q1, src, 64), tkl = __shfl(kl, src, 64), tkp = __shfl(kp, src, 64);
  const bool live = lane < p.total_q && r < B && lane >= tq0;
  const int vis = live ? max(tkl - (tq1 - tq0) + (lane - tq0) + 1, 0) : 0;   // causal: positions < vis are visible
  const int tiles = (vis + 2 * MLA_TILE - 1) / (2 * MLA_TILE);   // steps of 64 tokens
  const int sum = (int)wave_sum((float)tiles), most = (int)wave_max((float)tiles), nlive = (int)wave_sum(live ? 1.f : 0.f);
  auto jobs_of = [&](int d) { return live ? max(1, (tiles + d - 1) / d) : 0; };
  // at D = ceil(sum / (jobs - live tokens)) every token's rounding up is paid for (the launcher gives two jobs a token and more)
  int lo = max(1, max((sum + p.jobs - 1) / p.jobs, (most + p.nsplit - 1) / p.nsplit));
  int hi = max(lo, (sum + p.jobs - nlive - 1) / max(1, p.jobs - nlive));
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if ((int)wave_sum((float)jobs_of(mid)) <= p.jobs) hi = mid;
    else lo = mid + 1;
  }
  const int n = jobs_of(lo);
  int inc = n;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int a = __shfl_up(inc, o, 64);
    if (lane >= o) inc += a;
  }
  const unsigned long long later = __ballot(inc > job);
  MlaWork w;
  if (!later) { w.req = -1; return w; }
  const int t = __ffsll((long long)later) - 1;
  w.qt = t;
  w.nsp = __builtin_amdgcn_readlane(n, t);
  w.split = job - (__builtin_amdgcn_readlane(inc, t) - w.nsp);
  w.req = __builtin_amdgcn_readlane(r, t);
  w.kv_end = __builtin_amdgcn_readlane(vis, t);
  w.page_base = __builtin_amdgcn_readlane(tkp, t);
  // fused cache append (decode: one new token per request): the newest position is taken from the append buffers
  w.app_pos = p.app_ckv && __builtin_amdgcn_readlane(tq1 - tq0, t) == 1 ? __builtin_amdgcn_readlane(tkl, t) - 1 : -1;
  return w;
}

// Reductions over the four 16-lane rows of a wavefront (lanes l, l ^ 16, l ^ 32, l ^ 48): gfx950's row swaps — v_permlane32_swap
// exchanges the upper 32 lanes of one register with the lower 32 of another, v_permlane16_swap the odd rows with the even rows — are
// plain VALU instructions; the ds_bpermute shuffles they replace are LDS-crossbar round trips, four of them in a dependent chain per
// query tile and key tile.  Sum: (x_l + x_{l^32}) + (that of l ^ 16) — fp32 addition is commutative, so every lane of a query gets the
// same bits, and they are the bits the shuffle version produced ((x + shfl16) + shfl32 groups the rows as (r0 + r1) + (r2 + r3) for
// rows 0 / 1 and likewise here after the 32-swap first: see pf_sum_rows).
typedef unsigned pf_v2u __attribute__((ext_vector_type(2)));
typedef uint32_t pf_u4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ float pf_max_rows(float x) {
  pf_v2u r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
  r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float pf_sum_rows(float x) {
  // the shuffle version computed (x + x^16) first, then + the same of l ^ 32: keep that association — rows (r0 + r1) and (r2 + r3)
  // first (16-swap), then across the halves (32-swap)
  pf_v2u r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// Workgroup = 4 head blocks of 16, a wavefront each, alone on its SIMD with all its registers (Q 72, O 128); K and V rows in tiles of 32 tokens, staged once for all 64 heads, four
// of them in the LDS.  S and O are computed transposed (tokens x heads, dims x heads), so that a lane owns ONE head: the softmax statistics are
// one value a lane, and S^T leaves the MFMA with a lane's tokens where P^T enters the next one — the probabilities never leave the
// registers (V's rows are read in the order 4 g + (0..3), 16 + 4 g + (0..3) that this gives lane group g), and no wavefront waits for another's scores.
// What bounds it: a tile's 100 MFMAs (1600 cycles) and some 450 other instructions of the same wavefront (96 LDS reads and their waits, the softmax, 9 requests), which one SIMD issues one after
// the other: 1.45 us a tile at 2.1 GHz; without the LDS reads it would be 1.33, without the requests 1.23, without the second bf16 of P 1.21.  So the tile's parts are laid beside each
// other: its probabilities and the requests beside the next one's scores, the next one's largest beside this one's O, one instruction of each kind beside an MFMA.
// Before, two wavefronts a SIMD shared 16 heads in steps of 64 tokens (half of the scores each, exchanged through the LDS, then half of the dims), and two barriers a step kept scores, softmax and O
// apart in both: 3.1 us for 64 tokens, all of O rescaled in nearly every step, and the last step whole where 32 tokens were left.  Decode and merge, before -> here, us: 128 heads, 8
// requests of 2048 .. 8192 tokens 44.5 -> 42.0, 32 of 1000 .. 4000 69.9 -> 60.9, 20 of 2000 .. 8000 76 -> 66, 4 of 8192 .. 32768 66 -> 57, 32 of 250 .. 1000 34.0 -> 32.9; 64 heads, 24 of 1250
// .. 5000 47.4 -> 41.1, 3 of 16384 31.5 -> 29.4, 32 of 500 .. 2000 34.7 -> 32.4.  A call of 8 requests: 1.6 us for the job,
// 3.6 for pages, Q and the first rows, 0.7 the first scores, 17 the tiles, 3 the partial results' stores; over the whole launch the matrix pipe is busy 24 %, the vector ALU 20, the LDS 17, without a
// bank conflict (profiles/expert_prompt_counters.txt).
// The rows are
// packed 1 KiB apart with their 16-byte pieces permuted by mla_swz, which keeps both the fragment reads of 16 rows and the transposed reads of
// 8 rows off each other's banks.
// P enters the product as two bf16, the second what rounding the first left over.  One bf16 is off by its rounding except where P is exactly 1, a
// split's largest entry, and here a split is longer than in mla_decode_kernel: the error against 64-bit sums grew by 1 to 4 % (32 requests
// of 500 tokens, 128 heads 1.77e-3 -> 1.84e-3).  With two it is the outputs' rounding alone, 1.66e-3 at every size, also where P is far below 1: sums are rescaled only when a head's
// largest score has grown by MLA_GROWTH since they last were, for a split's first tile finds most of it and every rescaling is 128 products a lane.  What P is relative to lies that much
// above the largest score then, so that P ends at 1 and sums of it overflow where they did with every maximum followed, not at a 256th of that.
// distinct for 16 rows, also with rows 4 .. 11 flipped by 1 (ds_read_b128 takes lanes 0-3, 12-15, 20-23, 24-27 together); >> 1 distinct for rows
// 0-7 and for 8-15 (ds_read_b64_tr_b16 takes 32 lanes together)
__device__ __forceinline__ uint32_t mla_swz(uint32_t row) { return row & 8 ? ((row & 7) ^ 4) << 1 | 1 : (row & 7) << 1; }
constexpr float MLA_GROWTH = 5.5451774f;   // 8 ln 2
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) void mla_decode_wide_kernel(MlaParams p) {
  constexpr int NWV = 4, NQ = 18, NBUF = 4, REQ = MLA_TILE / NWV + 1;   // REQ: a wavefront's requests of a tile
  constexpr int KA = 6, VA = 2;                                          // fragment reads ahead of their MFMAs: k-steps of the scores, groups of 4 dim tiles of O
  constexpr uint32_t KT_BYTES = MLA_TILE * MLA_DC * 2, KP_BYTES = MLA_TILE * MLA_DR * 2;
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];         // [4][32][1024 B] ckv | [4][32][128 B] k_pe
  const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int hb = blockIdx.y;
  const int head = (hb * 4 + wave) * 16 + (lane & 15);
  MLA_TS(0);

  MlaWork w;
  if (p.jobs) {
    w = mla_pick_job(p, blockIdx.x, lane);
    if (w.req >= 0 && hb == 0 && w.split == 0 && tid == 0) p.njobs[w.qt] = w.nsp;
  } else {
    w.qt = blockIdx.z; w.split = blockIdx.x; w.nsp = p.nsplit;
    mla_find_request(p, w.qt, lane, w.req, w.kv_end, w.page_base, w.app_pos);
  }
  if (w.req < 0) return;
  const int req = __builtin_amdgcn_readfirstlane(w.req), kv_end = __builtin_amdgcn_readfirstlane(w.kv_end);
  const int page_base = __builtin_amdgcn_readfirstlane(w.page_base), app_pos = __builtin_amdgcn_readfirstlane(w.app_pos);
  const int qt = __builtin_amdgcn_readfirstlane(w.qt), split = __builtin_amdgcn_readfirstlane(w.split);
  const int nsp = __builtin_amdgcn_readfirstlane(w.nsp);
  MLA_TS(1);

  // the split's run of 32-token tiles: pairs, but for the context's last one
  const int ntiles = (kv_end + MLA_TILE - 1) / MLA_TILE;
  const int each = 2 * (((kv_end + 2 * MLA_TILE - 1) / (2 * MLA_TILE) + nsp - 1) / nsp);
  const int t_begin = min(split * each, ntiles), t_end = min(t_begin + each, ntiles);

  v4f o[32];     // O^T: dims 16 i + 4 g + (0..3) of the lane's head
#pragma unroll
  for (int i = 0; i < 32; i++) o[i] = v4f{0.f, 0.f, 0.f, 0.f};
  float m_run = -__FLT_MAX__, l_run = 0.f;   // (lowest, not -inf: scores of -inf then weigh 0 also where a split begins with a whole tile of them)

  if (t_begin < t_end) {
    if (app_pos >= 0 && hb == 0 && app_pos / MLA_TILE >= t_begin && app_pos / MLA_TILE < t_end) mla_store_appended(p, req, page_base, app_pos, tid);

    // lane i holds the page of tile pt0 + i (clamped: a tile of this request): one round of the page table for 64 tiles
    auto pages_from = [&](int t0) {
      const int t = min(t0 + lane, ntiles - 1);
      const int pidx_ = page_base + (p.tiles_shift >= 0 ? t >> p.tiles_shift : t * MLA_TILE / p.page_size);
      return p.kv_indices ? p.kv_indices[pidx_] : pidx_;
    };
    int pt0 = t_begin, pages = pages_from(pt0);
    asm volatile("" ::: "memory");   // (in this order: the pages are waited for first)
    v8bf qf[NQ];   // B[k = (lane >> 4) * 8 .. + 7][n = head] of 16 nope and 2 rope k-steps
    {
      const bf16_t* qn = p.q_nope + ((size_t)qt * p.Hq + head) * MLA_DC + g * 8;
      const bf16_t* qr = p.q_pe + ((size_t)qt * p.Hq + head) * MLA_DR + g * 8;
#pragma unroll
      for (int j = 0; j < 16; j++) qf[j] = as_v8bf(*reinterpret_cast<const uint4*>(qn + j * 32));
#pragma unroll
      for (int j = 0; j < 2; j++) qf[16 + j] = as_v8bf(*reinterpret_cast<const uint4*>(qr + j * 32));
    }
    const uint32_t lds0 = (uint32_t)(size_t)(__attribute__((address_space(3))) uint8_t*)smem;
    // Eight ckv rows a wavefront and tile, one 1-KiB row per wave-instruction; k_pe: eight rows in one.  Rows past the context re-read its last one: finite, weighted
    // with exactly 0.  A tile that is all context and does not hold the appended row takes the lanes' offsets from registers: address arithmetic on the scalar
    // unit, 250 instructions for 64 tokens, held a wavefront up for as long as its MFMAs.
    uint32_t ro[MLA_TILE / NWV];
#pragma unroll
    for (int c = 0; c < MLA_TILE / NWV; c++) ro[c] = (uint32_t)((wave + c * NWV) * p.ckv_ts * 2) + ((uint32_t)lane ^ mla_swz(wave + c * NWV)) * 16u;
    const int pr = wave * 8 + (lane >> 3);
    const uint32_t po = (uint32_t)(pr * p.kpe_ts * 2) + ((uint32_t)(lane & 7) ^ ((pr >> 1) & 7)) * 16u;
    uint32_t dK, dP;
    const bf16_t *base_k, *base_p;
    // where tile lies and goes; true: whole rows of the context's cache, which request(0 .. 8) bring
    auto locate = [&](int tile) __attribute__((always_inline)) {
      if (tile - pt0 >= 64) {
        pt0 = tile;
        pages = pages_from(pt0);
        asm volatile("s_waitcnt vmcnt(0)" : "+v"(pages)::"memory");
      }
      const int buf = (tile - t_begin) & (NBUF - 1);
      dK = lds0 + buf * KT_BYTES; dP = lds0 + NBUF * KT_BYTES + buf * KP_BYTES + wave * (8 * MLA_DR * 2);
      const int tok0 = tile * MLA_TILE;
      const int page0 = __builtin_amdgcn_readlane(pages, tile - pt0);
      const size_t row0 = (size_t)page0 * p.page_size + (p.tiles_shift >= 0 ? tok0 & (p.page_size - 1) : tok0 % p.page_size);
      base_k = p.ckv + row0 * p.ckv_ts;
      base_p = p.k_pe + row0 * p.kpe_ts;
      return kv_end - 1 - tok0 >= MLA_TILE - 1 && (unsigned)(app_pos - tok0) >= (unsigned)MLA_TILE;
    };
    auto request = [&](int i) __attribute__((always_inline)) {
      if (i < MLA_TILE / NWV) mla_dma_row_sa(base_k, ro[i], dK + (wave + i * NWV) * (MLA_DC * 2));
      else mla_dma_row_sa(base_p, po, dP);
    };
    auto request_any = [&](int tile) {   // as many requests, of a located tile that ends the context or holds the appended row
      const int tok0 = tile * MLA_TILE, last = kv_end - 1 - tok0;
      for (int c = 0; c < MLA_TILE / NWV; c++) {
        const int r = wave + c * NWV, rr = min(r, last);
        const bf16_t* src = base_k + rr * p.ckv_ts;
        if (tok0 + rr == app_pos) src = p.app_ckv + (size_t)req * MLA_DC;
        mla_dma_row_sa(src, ((uint32_t)lane ^ mla_swz(r)) * 16u, dK + (uint32_t)r * (MLA_DC * 2));
      }
      const int rr = min(pr, last);
      const bf16_t* src = base_p + rr * p.kpe_ts;
      if (tok0 + rr == app_pos) src = p.app_kpe + (size_t)req * MLA_DR;
      mla_dma_row_a(src + ((lane & 7) ^ ((pr >> 1) & 7)) * 8, dP);
    };
#pragma unroll
    for (int c = 0; c < NBUF - 1; c++)
      if (t_begin + c < t_end) {
        if (!locate(t_begin + c)) {
          request_any(t_begin + c);
        } else {
#pragma unroll
          for (int i = 0; i < REQ; i++) request(i);
        }
        if (c == 0) {   // the compiler does not see the requests, so that its wait for these is one for those as well: the first tile comes beside them
#pragma unroll
          for (int j = 0; j < NQ; j++) asm volatile("" : "+a"(qf[j]));
        }
      }
    MLA_TS(2);
    // tile's rows are there for all wavefronts, and all are done with the tile whose buffer the next request takes: what is requested behind it stays in flight
    auto arrived = [&](int tile) __attribute__((always_inline)) {
      if (tile == t_begin && tile + 2 < t_end) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(2 * REQ) : "memory");
      else if (tile + 1 < t_end) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(REQ) : "memory");
      else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
    };

    // fragment addresses within a tile: K rows 16 t + (lane & 15), piece 4 s + g; V rows 4 g + (lane & 15) / 4 (+ 16), piece 2 i + (lane >> 1 & 1)
    const uint32_t kx = (lane & 15) * (MLA_DC * 2) + (((uint32_t)g ^ mla_swz(lane & 15)) * 16);
    const uint32_t px = (lane & 15) * (MLA_DR * 2) + (((uint32_t)g ^ ((lane >> 1) & 7)) * 16);
    const uint32_t vr = 4 * g + ((lane & 15) >> 2);
    const uint32_t vx = vr * (MLA_DC * 2) + ((((lane >> 1) & 1) ^ mla_swz(vr)) * 16) + (lane & 1) * 8;

    // ---- S^T = K Q^T: lane holds tokens 16 t + 4 g + r of its head.  Fragments are read KA k-steps ahead of the MFMAs: fenced, or the compiler reads one
    // fragment ahead and waits for it; between(s): what goes beside k-step s
    v8bf kf[KA + 1][2];
    auto load_k = [&](int tile, int s) __attribute__((always_inline)) {
      const int buf = (tile - t_begin) & (NBUF - 1);
      const uint8_t* a = s < 16 ? smem + buf * KT_BYTES + (kx ^ ((s & 3) * 64)) + (s >> 2) * 256 : smem + NBUF * KT_BYTES + buf * KP_BYTES + (px ^ ((s - 16) * 64));
#pragma unroll
      for (int t = 0; t < 2; t++) kf[s % (KA + 1)][t] = as_v8bf(*reinterpret_cast<const uint4*>(a + t * (s < 16 ? 16 * MLA_DC * 2 : 16 * MLA_DR * 2)));
    };
    auto scores = [&](int tile, v4f (&s2)[2], auto between) __attribute__((always_inline)) {
      s2[0] = s2[1] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < NQ; s++) {
        if (s + KA < NQ) load_k(tile, s + KA);
#pragma unroll
        for (int t = 0; t < 2; t++) s2[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[s % (KA + 1)][t], qf[s], s2[t], 0, 0, 0);
        between(s);
#pragma unroll
        for (int t = 0; t < 2; t++) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x002, 3, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    // in pieces, beside the products of O: 0 the scale, 1 what lies past the context, 2 and 3 the largest
    float mx = 0.f;
    auto prepare = [&](int piece, int tile, v4f (&s2)[2]) __attribute__((always_inline)) {
      if (piece == 0) {
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
          for (int r = 0; r < 4; r++) s2[t][r] *= p.sm_scale;
      } else if (piece == 1) {
        const int ntok = kv_end - tile * MLA_TILE;
        if (ntok < MLA_TILE) {
#pragma unroll
          for (int t = 0; t < 2; t++)
#pragma unroll
            for (int r = 0; r < 4; r++)
              if (16 * t + 4 * g + r >= ntok) s2[t][r] = -__builtin_inff();
        }
      } else if (piece == 2) {
        mx = fmaxf(fmaxf(fmaxf(s2[0][0], s2[0][1]), fmaxf(s2[0][2], s2[0][3])), fmaxf(fmaxf(s2[1][0], s2[1][1]), fmaxf(s2[1][2], s2[1][3])));
      } else {
        mx = pf_max_rows(mx);   // finite: a tile has >= 1 visible token
      }
    };

    typedef __attribute__((address_space(3))) v4s16 lds_v4;
    union VFrag { v4s16 h[2]; v8bf v; };
    VFrag vf[VA + 1][4];
    auto load_v = [&](int tile, int j, int i) __attribute__((always_inline)) {   // the rows' transposed reads, dims 128 i + 16 j
      const uint8_t* a = smem + ((tile - t_begin) & (NBUF - 1)) * KT_BYTES + (vx ^ (j * 32)) + i * 256;
      vf[j % (VA + 1)][i].h[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4*)a);
      vf[j % (VA + 1)][i].h[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4*)(a + 16 * MLA_DC * 2));
    };
    // A tile: its probabilities beside the next one's scores, its share of O beside their largest.
    // MORE: there is a next one.  One instruction of each kind beside an MFMA: a
    // wavefront alone on its SIMD has nobody to fill the matrix pipe while it issues a row of reads.
    auto step = [&](auto more, int tile, v4f (&st)[2], v4f (&sn)[2]) __attribute__((always_inline)) {
      constexpr bool MORE = decltype(more)::value;
      if constexpr (MORE) {
        arrived(tile + 1);
#pragma unroll
        for (int s = 0; s < KA; s++) load_k(tile + 1, s);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int i = 0; i < 32; i++) asm volatile("" : "+a"(o[i]));
      if (__builtin_amdgcn_ballot_w64(mx > m_run) != 0ull) {
        const float m_new = fmaxf(m_run, mx + MLA_GROWTH), alpha = __expf(m_run - m_new);
        m_run = m_new;
        l_run *= alpha;
#pragma unroll
        for (int i = 0; i < 32; i++) {
#pragma unroll
          for (int r = 0; r < 4; r++) o[i][r] *= alpha;
          asm volatile("" : "+a"(o[i]));   // (in the MFMAs' registers on both sides of the branch, or the compiler moves all of them there and back in every tile)
        }
      }
#pragma unroll
      for (int t = 0; t < 2; t++)
#pragma unroll
        for (int r = 0; r < 4; r++) st[t][r] = __expf(st[t][r] - m_run);
      bool bring = false;
      if constexpr (MORE)
        if (tile + NBUF - 1 < t_end) {
          bring = locate(tile + NBUF - 1);
          if (!bring) request_any(tile + NBUF - 1);
        }
      uint32_t hi[4], lo[4];
      float sum = 0.f;
      auto probabilities = [&](int piece) __attribute__((always_inline)) {
        if (piece < 4) {
          const int t = piece >> 1, h = piece & 1;
          hi[piece] = ktx_pk_bf16(st[t][2 * h], st[t][2 * h + 1]);
        } else if (piece < 8) {   // what the rounding left over
          const int t = (piece >> 1) & 1, h = piece & 1;
          lo[piece - 4] = ktx_pk_bf16(st[t][2 * h] - __uint_as_float(hi[piece - 4] << 16), st[t][2 * h + 1] - __uint_as_float(hi[piece - 4] & 0xffff0000u));
        } else if (piece == 8) {
          sum = ((st[0][0] + st[0][1]) + (st[0][2] + st[0][3])) + ((st[1][0] + st[1][1]) + (st[1][2] + st[1][3]));
        } else if (piece == 9) {
          l_run += pf_sum_rows(sum);
        }
      };
      if constexpr (MORE) {
        scores(tile + 1, sn, [&](int s) __attribute__((always_inline)) {
          probabilities(s);
          if (s >= NQ - 4 * VA) load_v(tile, (s - NQ + 4 * VA) / 4, (s - NQ + 4 * VA) % 4);
          if (s >= 1 && s < 1 + REQ && bring) request(s - 1);
        });
      } else {
#pragma unroll
        for (int i = 0; i < 10; i++) probabilities(i);
#pragma unroll
        for (int j = 0; j < 4 * VA; j++) load_v(tile, j / 4, j % 4);
      }
      const v8bf pf = as_v8bf(make_uint4(hi[0], hi[1], hi[2], hi[3])), pl = as_v8bf(make_uint4(lo[0], lo[1], lo[2], lo[3]));
      // ---- O^T += V^T P^T
#pragma unroll
      for (int j = 0; j < 8; j++) {
#pragma unroll
        for (int i = 0; i < 4; i++)
          if (j + VA < 8) load_v(tile, j + VA, i);
#pragma unroll
        for (int i = 0; i < 4; i++) o[i * 8 + j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[j % (VA + 1)][i].v, pf, o[i * 8 + j], 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 4; i++) o[i * 8 + j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[j % (VA + 1)][i].v, pl, o[i * 8 + j], 0, 0, 0);
        if constexpr (MORE)
          if (j >= 1 && j < 5) prepare(j - 1, tile + 1, sn);
#pragma unroll
        for (int i = 0; i < 8; i++) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x002, 3, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    };

    v4f sa[2], sb[2];
    arrived(t_begin);
#pragma unroll
    for (int s = 0; s < KA; s++) load_k(t_begin, s);
    scores(t_begin, sa, [](int) {});
#pragma unroll
    for (int i = 0; i < 4; i++) prepare(i, t_begin, sa);
    MLA_TS(3);
    int tile = t_begin;
    for (; tile + 1 < t_end; tile++) {
      step(std::true_type{}, tile, sa, sb);
      sa[0] = sb[0];
      sa[1] = sb[1];
    }
    step(std::false_type{}, tile, sa, sb);
  }
  MLA_TS(6);

  const int dim0 = 4 * g;   // + 16 i
  if (p.out1) {   // one split holds the whole row: the merge kernel's arithmetic for a single partial (weight 1), in place
    const float inv = t_begin < t_end ? 1.0f / l_run : 0.f;   // (scores of -inf alone: NaN)
    bf16_t* po = p.out1 + ((size_t)qt * p.Hq + head) * MLA_DC + dim0;
#pragma unroll
    for (int i = 0; i < 32; i++)
      *reinterpret_cast<uint2*>(po + i * 16) = make_uint2(ktx_pk_bf16(o[i][0] * inv, o[i][1] * inv), ktx_pk_bf16(o[i][2] * inv, o[i][3] * inv));
    if (p.lse1 && g == 0)
      p.lse1[(size_t)qt * p.Hq + head] = l_run > 0.f ? (m_run + __logf(l_run)) * 1.44269504089f : -__builtin_inff();
    return;
  }
  // ---- partial results: un-normalised O plus (m, l) per head
  const size_t pidx = ((size_t)qt * p.Hq + head) * p.nsplit + split;
  if (g == 0) *reinterpret_cast<float2*>(p.part_ml + pidx * 2) = make_float2(m_run, l_run);
  if (t_begin < t_end) {
    float* po = p.part_o + pidx * MLA_DC + dim0;
#pragma unroll
    for (int i = 0; i < 32; i++) *reinterpret_cast<float4*>(po + i * 16) = make_float4(o[i][0], o[i][1], o[i][2], o[i][3]);
  }
  MLA_TS(7);
}

// merge the KV splits: one 256-thread workgroup per (query token, head, DIMS = 2048 / SL of the 512 output dims), thread (sl, dg) owns splits sl, sl + SL, ... for 8
// dims.  With 16 split lanes that is a quarter of the dims: a workgroup pulls cross-XCD data at only ~65 GB/s, so the many partials of one head are spread over four
// workgroups.  EVERY global load of the kernel — the (m, l) pairs, the partial outputs, the bounds — is issued before the first use: right after the kernel boundary each
// of them is an L2 miss, and a stats -> weights -> addresses -> loads chain would pay that latency three times over.  A dead split's partial may be stale memory, so it is
// selected away (not multiplied by 0).
// SL < 16 (batches that share out the workgroups; ns, twice the mean of a token's splits, to 8: 4 lanes and all of a head's dims, to 32: 8 and half of them): no lane without a split, more
// bytes in flight a thread and fewer workgroups, each of which finds the statistics again.  Us, decode and merge, 16 lanes -> here: 128 heads, 32 of 400 tokens 41.2 -> 31.1, 32 of 1000
// 45.0 -> 35.6, 16 of 2000 36.3 -> 33.8, 8 of 8192 47.5 -> 46.9; 64 heads, 24 of 500 27.3 -> 25.9, 32 of 2000 38.0 -> 35.5; 8 lanes at ns 51 (5 of 8000) lost, 43.6 -> 44.6.  A token that holds
// most of an uneven batch's splits goes round more often, and the batch gains all the same: 128 heads, 31 of 400 and one of 9000 49.2 -> 40.4, 19 of 100 and one of 8000 39.6 -> 36.6, 31 of 200
// and one of 100000 177 -> 169 (profiles/mla_merge_uneven_batches.txt: 26 batches at 64 and 128 heads, none more than 1.5 % slower).
template <int NS, bool JOBS, int SL = 16>   // splits per thread and round; JOBS: a token's number of splits is the decode kernel's (njobs); split lanes
__global__ __launch_bounds__(256) void mla_merge_kernel(MlaParams p, bf16_t* out, float* lse) {
  constexpr int DG = 256 / SL, DIMS = DG * 8;
  __shared__ float s_w[1024];
  __shared__ float s_red[8];
  __shared__ float s_acc[SL][DIMS + 4];
  const int qt = blockIdx.y, h = blockIdx.x, part = blockIdx.z, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int dg = tid % DG, sl = tid / DG;   // dim groups of 8 dims x split lanes
  const size_t base = ((size_t)qt * p.Hq + h) * p.nsplit;
  const int nsp = JOBS ? min(max(p.njobs[qt], 1), p.nsplit) : p.nsplit;   // (no request's token: whatever is there, and nothing is stored)
  // ---- all loads
  int B = p.batch;
  const int bsz_raw = p.d_bsz ? *p.d_bsz : p.batch;
  float2 ml[4];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int s = tid + i * 256;
    ml[i] = s < nsp ? *reinterpret_cast<const float2*>(p.part_ml + (base + s) * 2) : make_float2(0.f, 0.f);
  }
  float4 va[NS], vb[NS];
  const float* po = p.part_o + base * MLA_DC + part * DIMS + dg * 8;
#pragma unroll
  for (int u = 0; u < NS; u++) {
    const int s = min(sl + SL * u, nsp - 1);
    va[u] = *reinterpret_cast<const float4*>(po + (size_t)s * MLA_DC);
    vb[u] = *reinterpret_cast<const float4*>(po + (size_t)s * MLA_DC + 4);
  }
  if (p.d_bsz) B = min(max(bsz_raw, 0), p.batch);
  const int q_total = p.qo_indptr[B];

  // ---- softmax statistics, split-parallel; weights parked in LDS
  float mstar = -__builtin_inff();
#pragma unroll
  for (int i = 0; i < 4; i++)
    if (ml[i].y > 0.f) mstar = fmaxf(mstar, ml[i].x);
  mstar = wave_max(mstar);
  if (lane == 0) s_red[wave] = mstar;
  __syncthreads();
  mstar = fmaxf(fmaxf(s_red[0], s_red[1]), fmaxf(s_red[2], s_red[3]));
  float lsum = 0.f;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int s = tid + i * 256;
    const float w = ml[i].y > 0.f ? __expf(ml[i].x - mstar) : 0.f;
    if (s < nsp) s_w[s] = w;
    lsum += ml[i].y * w;
  }
  lsum = wave_sum(lsum);
  if (lane == 0) s_red[4 + wave] = lsum;
  __syncthreads();
  lsum = (s_red[4] + s_red[5]) + (s_red[6] + s_red[7]);

  float acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  for (int c = 0;; c += SL * NS) {   // (more than one round: a token of the jobs form that holds most of the batch's tiles)
#pragma unroll
  for (int u = 0; u < NS; u++) {
    const int s = c + sl + SL * u;
    const float w = s < nsp ? s_w[s] : 0.f;
    if (w > 0.f) {
      acc[0] += va[u].x * w; acc[1] += va[u].y * w; acc[2] += va[u].z * w; acc[3] += va[u].w * w;
      acc[4] += vb[u].x * w; acc[5] += vb[u].y * w; acc[6] += vb[u].z * w; acc[7] += vb[u].w * w;
    }
  }
  if (!JOBS || c + SL * NS >= nsp) break;
#pragma unroll
  for (int u = 0; u < NS; u++) {
    const int s = min(c + SL * NS + sl + SL * u, nsp - 1);
    va[u] = *reinterpret_cast<const float4*>(po + (size_t)s * MLA_DC);
    vb[u] = *reinterpret_cast<const float4*>(po + (size_t)s * MLA_DC + 4);
  }
  }
#pragma unroll
  for (int q = 0; q < 8; q++) s_acc[sl][dg * 8 + q] = acc[q];
  __syncthreads();
  if (tid < DIMS / 2 && qt < q_total) {   // two dims per thread
    const float inv = lsum > 0.f ? 1.0f / lsum : 0.f;
    float v0 = 0.f, v1 = 0.f;
#pragma unroll
    for (int i = 0; i < SL; i++) { v0 += s_acc[i][2 * tid]; v1 += s_acc[i][2 * tid + 1]; }
    const uint32_t w = (uint32_t)f32_to_bf16(v0 * inv) | ((uint32_t)f32_to_bf16(v1 * inv) << 16);
    *reinterpret_cast<uint32_t*>(out + ((size_t)qt * p.Hq + h) * MLA_DC + part * DIMS + 2 * tid) = w;
    if (lse && tid == 0 && part == 0)
      lse[(size_t)qt * p.Hq + h] = lsum > 0.f ? (mstar + __logf(lsum)) * 1.44269504089f : -__builtin_inff();
  }
}

__global__ void mla_cache_append_kernel(bf16_t* cache, long long ts, int page_size, const bf16_t* ckv, const bf16_t* kpe,
                                        const int32_t* page_idx, const int32_t* page_off, const int32_t* ntok,
                                        int max_tokens, int num_pages) {
  int T = max_tokens;
  if (ntok) T = min(max(*ntok, 0), max_tokens);
  const int t = blockIdx.x;
  if (t >= T) return;
  if (num_pages > 0 && ((unsigned)page_idx[t] >= (unsigned)num_pages || (unsigned)page_off[t] >= (unsigned)page_size)) return;
  bf16_t* dst = cache + ((size_t)page_idx[t] * page_size + page_off[t]) * ts;
  const int i = threadIdx.x;  // 72 threads x 16 B = 576 bf16
  if (i < 64) *reinterpret_cast<uint4*>(dst + i * 8) = *reinterpret_cast<const uint4*>(ckv + (size_t)t * MLA_DC + i * 8);
  else if (i < 72) *reinterpret_cast<uint4*>(dst + i * 8) = *reinterpret_cast<const uint4*>(kpe + (size_t)t * MLA_DR + (i - 64) * 8);
}

static long long* g_mla_dbg = nullptr;
extern "C" int ktx_mla_debug_stamps(long long* d_buf) {   // device buffer of >= 16 * workgroups entries, or NULL to stop
  g_mla_dbg = d_buf;
  return 0;
}

extern "C" size_t ktx_mla_workspace_bytes(const ktx_mla_config* cfg, int max_q_tokens) {
  if (!cfg || max_q_tokens <= 0) return 0;
  // one (O[512], m, l) record per (token, head, split).  The launcher never uses more than ~2048 workgroups, so beyond
  // that the split count shrinks as the token count grows; it also clamps the split count to what the buffer holds.
  const size_t per_split = (size_t)max_q_tokens * cfg->num_heads;
  const size_t cap = (size_t)2048 * 64 + per_split;
  const size_t n = std::max(per_split, std::min(per_split * (size_t)std::max(1, cfg->max_splits), cap));
  return n * (MLA_DC + 2) * sizeof(float);
}

extern "C" int ktx_mla_decode(const ktx_mla_config* cfg, const void* d_q_nope, const void* d_q_pe, const void* d_ckv,
                              const void* d_k_pe, int64_t ckv_token_stride, int64_t kpe_token_stride,
                              const int32_t* d_qo_indptr, const int32_t* d_kv_indptr, const int32_t* d_kv_indices,
                              const int32_t* d_kv_len_arr, const int32_t* d_bsz, int batch, int total_q_tokens,
                              void* d_out, float* d_lse, void* d_workspace, size_t workspace_bytes, void* stream) {
  return ktx_mla_decode_append(cfg, d_q_nope, d_q_pe, const_cast<void*>(d_ckv), const_cast<void*>(d_k_pe), ckv_token_stride,
                               kpe_token_stride, d_qo_indptr, d_kv_indptr, d_kv_indices, d_kv_len_arr, d_bsz, batch,
                               total_q_tokens, nullptr, nullptr, d_out, d_lse, d_workspace, workspace_bytes, stream);
}

static int mla_decode_impl(const ktx_mla_config* cfg, const void* d_q_nope, const void* d_q_pe, void* d_ckv,
                           void* d_k_pe, int64_t ckv_token_stride, int64_t kpe_token_stride,
                           const int32_t* d_qo_indptr, const int32_t* d_kv_indptr, const int32_t* d_kv_indices,
                           const int32_t* d_kv_len_arr, const int32_t* d_bsz, int batch, int total_q_tokens,
                           const void* d_new_ckv, const void* d_new_kpe, void* d_out, float* d_lse,
                           void* d_workspace, size_t workspace_bytes, void* stream, int* partials_nsplit);

extern "C" int ktx_mla_decode_append(const ktx_mla_config* cfg, const void* d_q_nope, const void* d_q_pe, void* d_ckv,
                                     void* d_k_pe, int64_t ckv_token_stride, int64_t kpe_token_stride,
                                     const int32_t* d_qo_indptr, const int32_t* d_kv_indptr, const int32_t* d_kv_indices,
                                     const int32_t* d_kv_len_arr, const int32_t* d_bsz, int batch, int total_q_tokens,
                                     const void* d_new_ckv, const void* d_new_kpe, void* d_out, float* d_lse,
                                     void* d_workspace, size_t workspace_bytes, void* stream) {
  KTX_REQUIRE(d_out, "ktx_mla_decode: null pointer");
  return mla_decode_impl(cfg, d_q_nope, d_q_pe, d_ckv, d_k_pe, ckv_token_stride, kpe_token_stride, d_qo_indptr, d_kv_indptr,
                         d_kv_indices, d_kv_len_arr, d_bsz, batch, total_q_tokens, d_new_ckv, d_new_kpe, d_out, d_lse, d_workspace,
                         workspace_bytes, stream, nullptr);
}

extern "C" int ktx_mla_decode_partials(const ktx_mla_config* cfg, const void* d_q_nope, const void* d_q_pe, void* d_ckv,
                                       void* d_k_pe, int64_t ckv_token_stride, int64_t kpe_token_stride,
                                       const int32_t* d_qo_indptr, const int32_t* d_kv_indptr, const int32_t* d_kv_indices,
                                       const int32_t* d_kv_len_arr, const int32_t* d_bsz, int batch, int total_q_tokens,
                                       const void* d_new_ckv, const void* d_new_kpe, void* d_workspace, size_t workspace_bytes,
                                       int* nsplit_out, void* stream) {
  KTX_REQUIRE(nsplit_out, "ktx_mla_decode_partials: null nsplit_out");
  return mla_decode_impl(cfg, d_q_nope, d_q_pe, d_ckv, d_k_pe, ckv_token_stride, kpe_token_stride, d_qo_indptr, d_kv_indptr,
                         d_kv_indices, d_kv_len_arr, d_bsz, batch, total_q_tokens, d_new_ckv, d_new_kpe, nullptr, nullptr, d_workspace,
                         workspace_bytes, stream, nsplit_out);
}

// mla_decode_wide_kernel or mla_decode_kernel<4, 2> for a call of the 64-head shape?  narrow: the splits that the latter would take.  The wide one
// walks 64 tokens in 2.9 us against 4.2 and shares out what the requests hold, but its first step ends 3 us later, and its shares
// write 256 workgroups' partials.  Measured with the merge (us, <4, 2> | wide, requests of equal length; of unequal ones the wide one gains 5-20 % more):
//   one step of 64 tokens: 24 of 40, 64 heads 19 | 14 (nothing to merge);
//   more workgroups of <4, 2> than CUs, a second round: 16 of 1000, 128 heads 38 | 32; 3 of 8192, 64 heads 34 | 29; 32 of 400, 64 heads (W = 224) 31 | 28;
//     of 200 tokens at most lost: 20 of 200, 128 heads (W = 160) 32 | 32, unequal 27 | 31;
//   one round: as <4, 2>'s splits deepen (in tiles of 32): 128 heads, 8 of 2000 (4) 27 | 29, of 3000 (6) 32 | 32, unequal 30 | 29, of 4500 (9) 38 | 37, unequal 36 | 31, of 7000 (14) 48 | 43; 64
//     heads, 8 of 2000 (4) 25 | 25, 10 24 | 27, 8 of 3000 (6) 27 | 27, 16 32 | 33, unequal 30 | 30, 8 of 4500 (9) 34 | 30, 16 39 | 37, unequal 37 | 32, 20 of 600 (2) 22 | 27.
// Without a hint of the contexts' length: past 16 tokens.
static bool mla_wide_steps(const ktx_mla_config* cfg, int total_q_tokens, int narrow) {
  if (total_q_tokens > 64) return false;
  if (cfg->kv_len_hint <= 0) return total_q_tokens > 16;
  const long hblocks = cfg->num_heads / 64, steps = (cfg->kv_len_hint + 2 * MLA_TILE - 1) / (2 * MLA_TILE);
  if (steps == 1) return true;
  if (narrow * total_q_tokens * hblocks > 256) return steps * total_q_tokens * hblocks >= 192;
  const int tiles = (cfg->kv_len_hint + MLA_TILE - 1) / MLA_TILE;
  return (tiles + narrow - 1) / narrow >= 8;
}

// The jobs form of mla_decode_wide_kernel (see mla_decode_impl): its jobs, and the splits that a token has at most (0: not in this form).
static int mla_jobs(int hblocks, int total_q_tokens) { return std::max(2 * total_q_tokens, 256 / hblocks); }
static int mla_jobs_cap(const ktx_mla_config* cfg, int total_q_tokens, int batch, size_t workspace_bytes) {
  const size_t counts = (size_t)total_q_tokens * 4, rec = (size_t)total_q_tokens * cfg->num_heads * (MLA_DC + 2) * sizeof(float);   // a count, and one split, of every token
  if (cfg->num_heads % 64 != 0 || total_q_tokens < 2 || total_q_tokens > 64 || batch > 64 || workspace_bytes <= counts || ktx_debug_get(7) > 0) return 0;
  return (int)std::min<size_t>(std::min(std::min(256, mla_jobs(cfg->num_heads / 64, total_q_tokens)), std::max(1, cfg->max_splits)), (workspace_bytes - counts) / rec);
}

// Workgroup shape and KV split count of a decode call — one place, because the one-launch decode step (ktx_attn.hip) must
// split the context exactly as the stand-alone kernel does to reproduce its partials bit for bit.
// jobs_cap: mla_jobs_cap's for this call, 0 where it cannot take the jobs form.
static void mla_pick_shape(const ktx_mla_config* cfg, int total_q_tokens, size_t workspace_bytes, int* shape_out, int* nsplit_out,
                           bool* wide_out, int jobs_cap, bool one_launch = false) {
  const int Hq = cfg->num_heads;
  // workgroup shape (head blocks x dim slices): decode-sized calls of many-headed models take 2x4 (32 heads share one staged
  // KV tile, 128 output dims per wave), prompts of those models 4x2, everything else 1x4
  const bool decode_sized = total_q_tokens <= 16;
  // long contexts (many tiles per split): 64 heads per workgroup share each staged tile and twice the splits pay off — measured
  // at 128 heads / 128K tokens (scripts/mla_sweep.py --ctx 131072): 4x2 with 128 splits 103 us, 2x4 with 64 splits 157 us
  // (one_launch: the split rule of csrc/ktx_attn.hip's phase C, which is built on the 2x4 shape — it keeps that shape, with its
  // <= 256 / head-blocks splits, past 8192 tokens: deeper splits instead of the 4x2 shape's wider ones)
  const bool long_hint = decode_sized && cfg->kv_len_hint >= 8192 && Hq % 64 == 0;
  const bool long_ctx = long_hint && !one_launch;
  // a decode BATCH (>= 8 query tokens, each with its own context): every head block of a token re-reads that token's latent rows, so
  // 64 heads per workgroup halve the KV traffic (V3 dims, 8 x 4096 tokens: 150 -> 75 MB per layer; batch-of-8 step 14.47 -> 13.91 ms,
  // profiles/r06_zz_bs8_mla_shape.txt)
  // Fewer (5 and more: what the one-launch step and its companions take stays as it is) of long contexts go to mla_decode_wide_kernel's shares of the batch: the 2x4 shape's workgroups take more
  // than one round of the CUs there, in equal splits that wait for the longest request.  The line is the one of mla_wide_steps, splits (16 of them) of 8 tiles at 128 heads, and lower for more: us,
  // 2x4 | shares, 5 requests of 3600 42 | 29, unequal (a quarter to all, four batches) 26 .. 30 | 25 .. 29, one of 3600 and four of 450 27.4 | 27.4; 7 of 4500 50 | 34, unequal 39 | 30, one and six 31 | 28; 5 of
  // 8000 72 | 36, 56 | 34, 41 | 28; 192 heads, 5 of 3000 40 | 30; 256, 5 of 2600 51 | 32.  Slower from there on: two long requests and three short ones, 1.11 at 3600, 1.05 at 4100, 0.99 at 4500.  Below the
  // line 2x4 stays, also where the 64-head shapes are faster for equal requests (5 of 2000 32 | 26): 6 unequal ones of 3000 take 26.7 | 28.6 (<4, 2>: 29.9), one of 2000 and four of 250 21.4 | 24.4.
  // With a hint far above all contexts the shares are slower, as past 8 requests: hint 6400, 5 of 800 25.2 | 26.8, one of 800 and four of 100 18.3 | 21.7.  (profiles/mla_decode_few_requests.txt)
  const bool few = !one_launch && !long_ctx && total_q_tokens >= 5 && total_q_tokens < 8 && Hq % 64 == 0 && jobs_cap >= 32 && (long)cfg->kv_len_hint * (Hq / 64) > 7168;
  const bool batched = decode_sized && Hq % 64 == 0 && !one_launch && (total_q_tokens >= 8 || few);
  int shape = (Hq % 32 == 0 && Hq >= 64 && decode_sized && !long_ctx && !batched) ? 2 : (Hq % 64 == 0) ? 4 : 1;
  {   // tuning knobs (scripts/mla_sweep.py): 6 = force the workgroup shape, 7 = force the split count
    const int fs = ktx_debug_get(6);
    if ((fs == 1) || (fs == 2 && Hq % 32 == 0) || (fs == 4 && Hq % 64 == 0)) shape = fs;
  }
  const int hbw = shape;
  const int hblocks = Hq / (16 * hbw);
  // KV splits: one 32-token tile per workgroup whenever the grid stays under ~2048 workgroups (measured on 16 heads: extra
  // tiles per workgroup cost more than the extra partials cost the merge kernel), bounded by the workspace — and by the
  // partials themselves: every split writes Hq x 514 floats per token that the merge kernel reads back (at 128 heads and 144
  // splits that was 38 MB per layer, 8x the 4.7 MB of latent rows the attention actually needs), so the split count is
  // capped where the partials reach ~16 MB and at about one workgroup per CU
  int nsplit = std::max(1, 2048 / std::max(1, hblocks * total_q_tokens));
  const size_t per_split_bytes = (size_t)total_q_tokens * Hq * (MLA_DC + 2) * sizeof(float);
  nsplit = std::min<int>(nsplit, std::max<size_t>(16, ((size_t)(long_hint ? 34 : 16) << 20) / per_split_bytes));
  if (long_hint) nsplit = std::min(nsplit, 128);
  if (shape == 2) nsplit = std::min(nsplit, std::max(16, 256 / std::max(1, hblocks * total_q_tokens)));
  if (ktx_debug_get(7) > 0) nsplit = ktx_debug_get(7);
  // no more splits than tiles — and no more than the deepest split needs: with T tiles dealt round-robin the launch takes
  // ceil(T / nsplit) tiles' time, so the smallest split count with that depth writes the fewest partials for the merge to read
  auto splits_of = [&](int unit) {
    if (cfg->kv_len_hint <= 0) return nsplit;
    const int tiles = std::max(1, (cfg->kv_len_hint + unit - 1) / unit), n = std::min(nsplit, tiles), depth = (tiles + n - 1) / n;
    return ktx_debug_get(7) <= 0 ? (tiles + depth - 1) / depth : n;
  };
  const int narrow = splits_of(MLA_TILE);
  const bool wide = shape == 4 && (few || mla_wide_steps(cfg, total_q_tokens, narrow));
  nsplit = wide ? splits_of(2 * MLA_TILE) : narrow;   // (mla_decode_wide_kernel's steps)
  // <= 256 splits: the merge kernel keeps splits/16 partial rows per thread in registers (NS = 16 is its largest, spill-free
  // instantiation); longer contexts simply put more 32-token tiles into each split
  nsplit = std::min(nsplit, std::min(256, std::max(1, cfg->max_splits)));
  nsplit = (int)std::min<size_t>((size_t)nsplit, workspace_bytes / ((size_t)total_q_tokens * Hq * (MLA_DC + 2) * sizeof(float)));
  *shape_out = shape;
  *nsplit_out = nsplit;
  *wide_out = wide;
}
extern "C" int ktx_mla_decode_nsplit(const ktx_mla_config* cfg, int total_q_tokens, size_t workspace_bytes) {   // ktx_internal.h
  int shape = 0, nsplit = 0;
  bool wide = false;
  if (!cfg || total_q_tokens <= 0) return 0;
  // Up to 40 K tokens the one launch wins with deeper 2x4 splits: 61.7 vs 68.4 us per layer at 12 K, 64.1 vs 72.0 at 16 K, 77.9 vs 80.5 at
  // 32 K, 81.7 vs 83.4 at 36 K, even from 40 K on (84.8 / 84.8; 48 K 95.1 vs 89.0 before phase C's staging fast path) — the five launches
  // with the 4x2 shape's 128 splits take over there (profiles/r06_AG_attn_fused_long_ctx.txt, final round-6 kernels; the bound was 12 K
  // before the launch lost 7 us to section 4.1.6).
  const int bound_k = ktx_debug_get(1);   // dev knob 1: the bound in K tokens (scripts/attn_fused_bench.py, ATTN_BOUND_K)
  if (cfg->kv_len_hint >= (bound_k > 0 ? bound_k * 1024 : 40960)) return 0;
  mla_pick_shape(cfg, total_q_tokens, workspace_bytes, &shape, &nsplit, &wide, 0, true);
  return shape == 2 ? nsplit : 0;   // the one-launch step is built on the 2x4 workgroup shape only
}

static int mla_decode_impl(const ktx_mla_config* cfg, const void* d_q_nope, const void* d_q_pe, void* d_ckv,
                           void* d_k_pe, int64_t ckv_token_stride, int64_t kpe_token_stride,
                           const int32_t* d_qo_indptr, const int32_t* d_kv_indptr, const int32_t* d_kv_indices,
                           const int32_t* d_kv_len_arr, const int32_t* d_bsz, int batch, int total_q_tokens,
                           const void* d_new_ckv, const void* d_new_kpe, void* d_out, float* d_lse,
                           void* d_workspace, size_t workspace_bytes, void* stream, int* partials_nsplit) {
  KTX_REQUIRE((d_new_ckv == nullptr) == (d_new_kpe == nullptr), "ktx_mla_decode_append: give both new_ckv and new_kpe or neither");
  KTX_REQUIRE(cfg && d_q_nope && d_q_pe && d_ckv && d_k_pe && d_workspace, "ktx_mla_decode: null pointer");
  KTX_REQUIRE(d_qo_indptr && d_kv_indptr && d_kv_len_arr, "ktx_mla_decode: null index array");
  KTX_REQUIRE(cfg->head_dim_ckv == MLA_DC && cfg->head_dim_kpe == MLA_DR, "ktx_mla_decode: only kv_lora_rank 512 + rope 64");
  KTX_REQUIRE(cfg->num_heads > 0 && cfg->num_heads % 16 == 0, "ktx_mla_decode: num_heads must be a multiple of 16");
  KTX_REQUIRE(batch > 0 && total_q_tokens > 0 && cfg->page_size > 0, "ktx_mla_decode: bad sizes");
  KTX_REQUIRE(cfg->page_size % MLA_TILE == 0, "ktx_mla_decode: page_size must be a multiple of 32 (the reference's caches use 64 and 256)");
  KTX_REQUIRE(ckv_token_stride % 8 == 0 && kpe_token_stride % 8 == 0, "ktx_mla_decode: token strides must be multiples of 8 elements");
  hipStream_t st = (hipStream_t)stream;
  const int Hq = cfg->num_heads;
  int shape = 0, nsplit = 0;
  bool wide = false;
  const int jobs_cap = partials_nsplit ? 0 : mla_jobs_cap(cfg, total_q_tokens, batch, workspace_bytes);
  mla_pick_shape(cfg, total_q_tokens, workspace_bytes, &shape, &nsplit, &wide, jobs_cap);
  const int hbw = shape, nwv = shape == 1 ? 4 : 8;
  const int hblocks = Hq / (16 * hbw);
  KTX_REQUIRE(nsplit >= 1, "ktx_mla_decode: workspace too small");
  const size_t need = (size_t)total_q_tokens * Hq * nsplit * (MLA_DC + 2) * sizeof(float);
  KTX_REQUIRE(workspace_bytes >= need, "ktx_mla_decode: workspace too small");
  MlaParams p;
  p.q_nope = (const bf16_t*)d_q_nope; p.q_pe = (const bf16_t*)d_q_pe; p.ckv = (const bf16_t*)d_ckv; p.k_pe = (const bf16_t*)d_k_pe;
  p.ckv_ts = ckv_token_stride; p.kpe_ts = kpe_token_stride;
  p.qo_indptr = d_qo_indptr; p.kv_indptr = d_kv_indptr; p.kv_indices = d_kv_indices; p.kv_len = d_kv_len_arr; p.d_bsz = d_bsz;
  p.batch = batch; p.total_q = total_q_tokens; p.Hq = Hq; p.page_size = cfg->page_size; p.nsplit = nsplit;
  p.tiles_shift = -1;
  for (int sh = 0; sh < 20; sh++)
    if (cfg->page_size == (MLA_TILE << sh)) p.tiles_shift = sh;
  p.sm_scale = cfg->sm_scale;
  p.part_o = (float*)d_workspace;
  p.part_ml = p.part_o + (size_t)total_q_tokens * Hq * nsplit * MLA_DC;
  p.dbg = g_mla_dbg;
  int only = ktx_debug_get(5);   // measurement knob (include/ktx_moe.h): 1 = split-KV kernel only, 2 = merge only
  if (partials_nsplit) { only = 1; *partials_nsplit = nsplit; }   // the caller merges the partials itself (ktx_linear_forward_batched_merge)
  const bool direct = nsplit == 1 && only == 0;
  // Batches of requests share one workgroup per CU by what they hold: equal splits of unequal contexts wait for the longest, and contexts
  // shorter than the hint leave workgroups idle (8 requests of 2048 .. 8192 tokens, 128 heads, 5121 on average: 51 us with equal splits of
  // the form before, 40 so).
  p.jobs = 0;
  p.njobs = nullptr;
  if (wide && nsplit > 1 && jobs_cap > 1) {
    p.jobs = mla_jobs(hblocks, total_q_tokens); p.nsplit = jobs_cap;
    p.part_ml = p.part_o + (size_t)total_q_tokens * Hq * jobs_cap * MLA_DC;
    p.njobs = reinterpret_cast<int*>(p.part_ml + (size_t)total_q_tokens * Hq * jobs_cap * 2);
  }
  p.out1 = direct ? (bf16_t*)d_out : nullptr;
  p.lse1 = direct ? d_lse : nullptr;
  p.app_ckv = (const bf16_t*)d_new_ckv; p.app_kpe = (const bf16_t*)d_new_kpe; p.ckv_w = (bf16_t*)d_ckv; p.kpe_w = (bf16_t*)d_k_pe;
  const size_t lds = (size_t)(2 * MLA_TILE * MLA_KROW + 2 * MLA_TILE * MLA_DR + nwv * 16 * MLA_TILE) * sizeof(bf16_t) + (size_t)nwv * 512 * sizeof(float) + 16;
  const dim3 grid(nsplit, hblocks, total_q_tokens);
  // algorithmic bytes: the latent rows of the context (hint) + q / out rows; the split partials are an implementation artefact
  const double kv_bytes = (double)std::max(cfg->kv_len_hint, 1) * (MLA_DC + MLA_DR) * 2.0 * batch;
  if (only == 2) {
  } else if (shape == 2) {
    KTX_TIMED(st, kv_bytes + (double)total_q_tokens * Hq * (MLA_DC + MLA_DR + MLA_DC) * 2.0,
              "mla_decode_kernel<2,4> T=%d Hq=%d nsplit=%d", total_q_tokens, Hq, nsplit);
    const hipError_t e2 = ktx_set_max_lds(reinterpret_cast<const void*>(mla_decode_kernel<2, 4>), 128 * 1024);
    KTX_HIP(e2);
    hipLaunchKernelGGL((mla_decode_kernel<2, 4>), grid, dim3(512), lds, st, p);
  } else if (shape == 4 && !wide) {
    KTX_TIMED(st, kv_bytes + (double)total_q_tokens * Hq * (MLA_DC + MLA_DR + MLA_DC) * 2.0,
              "mla_decode_kernel<4,2> T=%d Hq=%d nsplit=%d", total_q_tokens, Hq, nsplit);
    const hipError_t e4 = ktx_set_max_lds(reinterpret_cast<const void*>(mla_decode_kernel<4, 2>), 128 * 1024);
    KTX_HIP(e4);
    hipLaunchKernelGGL((mla_decode_kernel<4, 2>), grid, dim3(512), lds, st, p);
  } else if (wide) {
    KTX_TIMED(st, kv_bytes + (double)total_q_tokens * Hq * (MLA_DC + MLA_DR + MLA_DC) * 2.0,
              "mla_decode_wide_kernel T=%d Hq=%d nsplit=%d", total_q_tokens, Hq, p.nsplit);
    constexpr size_t lds4 = 4 * MLA_TILE * (MLA_DC + MLA_DR) * sizeof(bf16_t);
    KTX_HIP(ktx_set_max_lds(reinterpret_cast<const void*>(mla_decode_wide_kernel), (int)lds4));
    hipLaunchKernelGGL(mla_decode_wide_kernel, p.jobs ? dim3(p.jobs, hblocks) : grid, dim3(256), lds4, st, p);
  } else {
    KTX_TIMED(st, kv_bytes + (double)total_q_tokens * Hq * (MLA_DC + MLA_DR + MLA_DC) * 2.0,
              "mla_decode_kernel<1,4> T=%d Hq=%d nsplit=%d", total_q_tokens, Hq, nsplit);
    const hipError_t e1 = ktx_set_max_lds(reinterpret_cast<const void*>(mla_decode_kernel<1, 4>), 128 * 1024);
    KTX_HIP(e1);
    hipLaunchKernelGGL((mla_decode_kernel<1, 4>), grid, dim3(256), lds, st, p);
  }
  KTX_HIP(hipGetLastError());
  if (only != 1 && !direct) {
    KTX_TIMED(st, (double)total_q_tokens * Hq * MLA_DC * 2.0, "mla_merge_kernel T=%d Hq=%d nsplit=%d", total_q_tokens, Hq, nsplit);
    const int ns = p.jobs ? std::min(p.nsplit, 2 * p.jobs / total_q_tokens) : p.nsplit;   // (jobs: twice the mean; the kernel goes on from there)
    auto merge = [&](auto kern, int parts = 4) { hipLaunchKernelGGL(kern, dim3(Hq, total_q_tokens, parts), dim3(256), 0, st, p, (bf16_t*)d_out, d_lse); };
    if (p.jobs && ns <= 8) merge(mla_merge_kernel<2, true, 4>, 1);
    else if (p.jobs && ns <= 16) merge(mla_merge_kernel<2, true, 8>, 2);
    else if (ns <= 32) p.jobs ? merge(mla_merge_kernel<4, true, 8>, 2) : merge(mla_merge_kernel<2, false>);
    else if (ns <= 64) p.jobs ? merge(mla_merge_kernel<4, true>) : merge(mla_merge_kernel<4, false>);
    else if (ns <= 144) p.jobs ? merge(mla_merge_kernel<9, true>) : merge(mla_merge_kernel<9, false>);
    else p.jobs ? merge(mla_merge_kernel<16, true>) : merge(mla_merge_kernel<16, false>);
  }
  KTX_HIP(hipGetLastError());
  return 0;
}

// =====================================================================================================
// Non-absorbed prompt attention (KDeepseekV2Attention.forward_chunck / forward_linux_flashinfer prefill branch,
// archive/ktransformers/operators/attention.py:349-523: kv_b_proj expands the latents to per-head K_nope / V and a causal
// flash attention runs over qk dim 192 = 128 nope + 64 rope, v dim 128).  The absorbed kernel above spends 2*(576+512) flop
// per (query, key, head) and gives every query token its own workgroup; here it is 2*(192+128) and a workgroup owns 128
// queries of one head.
//   S^T = K Q^T : A = K tile from LDS (rows = keys), B = Q^T from registers; the C layout then leaves a lane with 4
//   consecutive keys of ONE query (lane & 15), so the online softmax is per lane and P never travels through LDS:
//   O^T += V^T P^T : A = V^T tile from LDS (rows = dims; the caller supplies V already transposed, [head][dim][key] — it is
//   the output of a GEMM either way), B = the lane's own P values.  The k-slot -> key map of that product is
//   slot (kc, e) -> key 16*(2*ks + e/4) + 4*kc + e%4, applied to both operands.
// One workgroup: 4 wavefronts x 2 query tiles of 16 = 128 queries, one head; keys in tiles of 64.
// =====================================================================================================
#define PF_BN 64
constexpr int PF_KN = PF_BN * 256, PF_KB = PF_KN + PF_BN * 128, PF_VB = 128 * 128;   // LDS bytes of a key tile: [key][128] | [key][64] | V^T [dim][64 keys]
struct MlaPrefillParams {
  const bf16_t *q_nope, *q_pe;   // [T][H][128] / [T][H][64] with element strides below
  long long qn_ts, qn_hs, qp_ts, qp_hs;
  const bf16_t* k_nope;          // [H][kv_pad][128]
  const bf16_t* k_pe;            // [kv_len][64], token stride kpe_ts
  long long kpe_ts;
  const bf16_t* v_t;             // [H][128][kv_pad]
  bf16_t* out;                   // [T][H][128]
  int T, H, kv_len, kv_pad;
  float sm_scale;
  int nqb;                       // query blocks
  int xcd;                       // 1-D XCD-aware grid of query blocks x splits x H heads (H % 8 == 0); 0: grid (query blocks, heads, splits)
  int nsplit;                    // pieces of a query block's keys, of about as many tiles each
  float* part_o;                 // nsplit > 1: [T][H][nsplit][128] sums, not divided; [T][H][nsplit][2] (largest raw score, sum of the probabilities) behind them
  float* part_ml;
};

// S of the NEXT tile is computed beside the probabilities of this one, and its largest scores are found beside this tile's O: MFMAs and vector instructions that
// do not wait for each other, in one stream (before,
// 1280 cycles of MFMAs and ~1450 of vector ALU a tile ran one after the other, and two workgroups a CU hid a third of that).  That takes a second set of scores, 32
// registers, which the tiles' way through registers left no room for: K, k_pe and V^T come by LDS-DMA, double-buffered, 80 KB a workgroup, two workgroups a CU.
// A lane's 8 probabilities of a half tile are those of 8 keys that follow each other (which K rows a fragment takes is free), so a V^T fragment is one read.
// Rows lie unpadded, their 16-byte pieces permuted so that no read has bank conflicts (ds_read_b128 takes lanes 0-3, 12-15, 20-23 and 24-27 together): with i the lane
// that reads the row, K: piece c in slot c ^ i; k_pe and V^T, 8 pieces a row: c ^ (i >> 1).
// 128 heads, us, one after the other -> here: 1000 tokens behind 3096 367 -> 310 (788 -> 950 TFLOP/s), 2048 of 2048 260 -> 214, 512 of 8192 396 -> 336; 16 heads, 300 of 1500: 50
// -> 38.  Left to its own order the compiler puts the products first, each fragment's read directly before its use, and the softmax behind them: 325 us; with the
// largest scores found beside the products as well, 320.  A running maximum moves somewhere in two fifths of the tiles: one branch for both query tiles costs 8 %.
// DMA false: operands that do not lie on 16 bytes come through registers, into the same places.  Written where they were requested they stood in the step's way; V^T
// waits beside S and K beside O, for which the registers suffice but for 11 of them.  ALONE: workgroups that have a CU each (as many as CUs, or fewer) have twice the registers, and both
// wait for the whole step.  Us, as the tiles' way through registers was before | written at once | now, 8 bytes off: 128 heads, 64 tokens of 4096 125 | 174 | 116 (ALONE; 141 not), 1000 of 4096 370 | 391 |
// 358 (454 ALONE), 1000 of 1000 96 | 97 | 94; 16 heads, 64 of 2000 63.5 | 60.4 | 60.2; 2 bytes off, where the loads themselves are slow: 167 | - | 156, 391 | - | 415, 105 | - | 110, 80 | - | 76.
// (4 bytes a request, by LDS-DMA: 174, 413, 111, 88.)
template <bool DMA, bool ALONE = false, bool SPLIT = false>   // SPLIT: a workgroup has one of p.nsplit pieces of its queries' keys
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(ALONE ? 1 : 2, ALONE ? 1 : 2))) void mla_prefill_kernel(MlaPrefillParams p) {
  constexpr int NU = 2;                              // query tiles of 16 per wavefront: every K fragment read feeds two MFMAs
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];   // [2][PF_KB] | [2][PF_VB]
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // blockIdx -> (head, query block).  XCD-aware (p.nqb > 0: a 1-D grid): workgroup ids are dealt round-robin to the 8 XCDs, so
  // id % 8 picks the XCD; all query blocks of ONE head go to one XCD (head % 8 == XCD) and run there back to back — the head's K / V^T
  // (1 MB at 2048 keys) is fetched into that XCD's L2 once instead of into all eight.  Within a head: heaviest query blocks first
  // (causal: the last block sees the whole context).
  int h, qb, split = 0;
  if (p.xcd) {
    const int id = blockIdx.x, xcd = id & 7, slot = id >> 3, per_head = SPLIT ? p.nqb * p.nsplit : p.nqb;
    h = (slot / per_head) * 8 + xcd;
    qb = slot % per_head;
    if constexpr (SPLIT) { split = qb % p.nsplit; qb /= p.nsplit; }
    qb = p.nqb - 1 - qb;
  } else {
    h = blockIdx.y;
    qb = (int)gridDim.x - 1 - (int)blockIdx.x;
    if constexpr (SPLIT) split = blockIdx.z;
  }
  const int q0 = qb * (64 * NU) + wave * (16 * NU);
  const int qi = lane & 15, g = lane >> 4;
  const int pos_off = p.kv_len - p.T;                // query t sits at position pos_off + t
  const int pos_max = pos_off + min(qb * (64 * NU) + 64 * NU - 1, p.T - 1);
  int ntiles = min(pos_max, p.kv_len - 1) / PF_BN + 1, tile0 = 0;   // the keys' tiles: tile0 .. ntiles - 1
  if constexpr (SPLIT) {
    const int all = ntiles;
    tile0 = all * split / p.nsplit;
    ntiles = all * (split + 1) / p.nsplit;
    if (tile0 == ntiles) {   // (fewer tiles than pieces: a sum of -1 says that no O is there)
      for (int r = tid; r < 64 * NU; r += 256) {
        const int t = qb * (64 * NU) + r;
        if (t < p.T) *reinterpret_cast<float2*>(p.part_ml + (((size_t)t * p.H + h) * p.nsplit + split) * 2) = make_float2(-__builtin_inff(), -1.f);
      }
      return;
    }
  }
  const bf16_t* kn = p.k_nope + (size_t)h * p.kv_pad * 128;
  const bf16_t* vt = p.v_t + (size_t)h * 128 * p.kv_pad;

  // ---- a tile's requests, 10 a wavefront: 4 rows of K, 8 of k_pe or of V^T each.  Rows of k_pe past kv_len read the last one (their scores are masked).  DMA false: a
  // lane's 16 bytes wait in registers until put writes them.
  const uint32_t lds0 = (uint32_t)(uintptr_t)smem;
  const int er = wave * 8 + (lane >> 3), ep = (lane & 7) ^ (wave * 2 + ((lane >> 4) & 1)), vp = (lane & 7) ^ ((wave * 4 + (lane >> 4)) & 7);
  const uint32_t ko_dma = (wave * 4 + (lane >> 4)) * 256 + ((lane & 15) ^ ((wave >> 1) * 4 + (lane >> 4))) * 16, vo_dma = (uint32_t)er * (uint32_t)p.kv_pad * 2u + vp * 16;
  auto bring = [&](const bf16_t* base, uint32_t lane_bytes, uint32_t at, pf_u4& held) __attribute__((always_inline)) {
    if constexpr (DMA) mla_dma_row_sa(base, lane_bytes, lds0 + at);
    else held = *reinterpret_cast<const pf_u4*>(reinterpret_cast<const uint8_t*>(base) + lane_bytes);
  };
  auto put = [&](uint32_t at, const pf_u4& held) __attribute__((always_inline)) {
    if constexpr (!DMA) *reinterpret_cast<pf_u4*>(smem + at + lane * 16) = held;
  };
  auto k_at = [&](int c, int buf) __attribute__((always_inline)) { return (uint32_t)(buf * PF_KB + (c * 4 + wave) * 1024); };   // K: c 0 .. 3, k_pe behind it: 4, 5
  auto v_at = [&](int c, int buf) __attribute__((always_inline)) { return (uint32_t)(2 * PF_KB + buf * PF_VB + (c * 4 + wave) * 1024); };
  auto stage_k = [&](int tile, int buf, pf_u4 (&held)[6]) __attribute__((always_inline)) {
#pragma unroll
    for (int c = 0; c < 4; c++) bring(kn + (size_t)(tile * PF_BN + c * 16) * 128, ko_dma ^ ((c & 1) * 128), k_at(c, buf), held[c]);
#pragma unroll
    for (int c = 4; c < 6; c++) {
      const bf16_t* src = p.k_pe + (size_t)min(tile * PF_BN + (c - 4) * 32 + er, p.kv_len - 1) * p.kpe_ts + ep * 8;
      if constexpr (DMA) mla_dma_row_a(src, lds0 + k_at(c, buf));
      else held[c] = *reinterpret_cast<const pf_u4*>(src);
    }
  };
  auto stage_v = [&](int tile, int buf, pf_u4 (&held)[4]) __attribute__((always_inline)) {
#pragma unroll
    for (int c = 0; c < 4; c++) bring(vt + (size_t)c * 32 * p.kv_pad + tile * PF_BN, vo_dma, v_at(c, buf), held[c]);
  };
  auto put_k = [&](int buf, const pf_u4 (&held)[6]) __attribute__((always_inline)) {
#pragma unroll
    for (int c = 0; c < 6; c++) put(k_at(c, buf), held[c]);
  };
  auto put_v = [&](int buf, const pf_u4 (&held)[4]) __attribute__((always_inline)) {
#pragma unroll
    for (int c = 0; c < 4; c++) put(v_at(c, buf), held[c]);
  };
  {
    pf_u4 hk[6], hv[4];
    stage_k(tile0, 0, hk);
    stage_v(tile0, 0, hv);
    put_k(0, hk);
    put_v(0, hv);
    if (ntiles - tile0 > 1) {
      stage_k(tile0 + 1, 1, hk);
      put_k(1, hk);
    }
  }

  // Q^T fragments: lane (query qi, k-chunk g)
  v8bf qf[NU][6];
  int tq[NU];
#pragma unroll
  for (int u = 0; u < NU; u++) {
    tq[u] = min(q0 + u * 16 + qi, p.T - 1);
    const bf16_t* qn = p.q_nope + (size_t)tq[u] * p.qn_ts + (size_t)h * p.qn_hs + g * 8;
    const bf16_t* qr = p.q_pe + (size_t)tq[u] * p.qp_ts + (size_t)h * p.qp_hs + g * 8;
#pragma unroll
    for (int s = 0; s < 4; s++) qf[u][s] = as_v8bf(*reinterpret_cast<const uint4*>(qn + s * 32));
#pragma unroll
    for (int s = 0; s < 2; s++) qf[u][4 + s] = as_v8bf(*reinterpret_cast<const uint4*>(qr + s * 32));
  }
  v4f o[NU][8];
  float m_run[NU], l_run[NU];
#pragma unroll
  for (int u = 0; u < NU; u++) {
#pragma unroll
    for (int i = 0; i < 8; i++) o[u][i] = v4f{0.f, 0.f, 0.f, 0.f};
    m_run[u] = -__builtin_inff();
    l_run[u] = 0.f;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();

  const int fq = (qi >> 1) & 7;
  const int kq = (qi >> 2) * 8 + (qi & 3);            // row i of a K fragment is key (i >> 2) * 8 + (i & 3), + 4 for odd kt, + 32 for kt >= 2
  const int ko = kq * 256 + ((g ^ qi) << 4), ro = PF_KN + kq * 128 + ((g ^ fq) << 4), vo = 2 * PF_KB + qi * 128 + ((g ^ fq) << 4);
  // ---- S^T = K Q^T: st[u][kt][r] = S[query qi of tile u][key 32*(kt/2) + 8*g + 4*(kt%2) + r].  k-chunk outermost: 4 x NU independent accumulators between two MFMAs of one chain
  auto qk = [&](int buf, v4f (&st)[NU][4]) __attribute__((always_inline)) {
    const uint8_t* kb = smem + buf * PF_KB;
#pragma unroll
    for (int s = 0; s < 6; s++) {
#pragma unroll
      for (int kt = 0; kt < 4; kt++) {
        const v8bf a = as_v8bf(*reinterpret_cast<const uint4*>(s < 4 ? kb + (kt >> 1) * 8192 + (kt & 1) * 1024 + (ko ^ (s * 64)) : kb + (kt >> 1) * 4096 + (kt & 1) * 512 + (ro ^ ((s - 4) * 64))));
#pragma unroll
        for (int u = 0; u < NU; u++) st[u][kt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, qf[u][s], s ? st[u][kt] : v4f{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
      }
    }
  };

  // The causal mask only exists on a query block's last two key tiles: a tile every query of the wavefront sees whole (wave-uniform test) skips it.
  // (the empty asm keeps this a wave-uniform BRANCH: speculated into selects, its compares + selects ran on every tile)
  auto mask = [&](int tile, v4f (&st)[NU][4]) __attribute__((always_inline)) {
    const int j0 = tile * PF_BN;
    if (j0 + PF_BN - 1 <= min(pos_off + min(q0, p.T - 1), p.kv_len - 1)) return;
#pragma unroll
    for (int u = 0; u < NU; u++) {
      const int lim = min(pos_off + tq[u], p.kv_len - 1);       // last visible key of this lane's query
#pragma unroll
      for (int kt = 0; kt < 4; kt++) {
#pragma unroll
        for (int r = 0; r < 4; r++) {
          const int key = j0 + (kt >> 1) * 32 + g * 8 + (kt & 1) * 4 + r;
          st[u][kt][r] = key <= lim ? st[u][kt][r] : -__builtin_inff();
        }
        asm volatile("" : "+v"(st[u][kt]));
      }
    }
  };
  float mx[NU];   // the largest score of a tile, over the query's four key-chunk lanes (qi, qi + 16, + 32, + 48)
  auto largest = [&](const v4f (&st)[NU][4]) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < NU; u++) {
      mx[u] = -__builtin_inff();
#pragma unroll
      for (int kt = 0; kt < 4; kt++)
#pragma unroll
        for (int r = 0; r < 4; r++) mx[u] = fmaxf(mx[u], st[u][kt][r]);
      mx[u] = pf_max_rows(mx[u]);
    }
  };

  // One key tile of parity par: its scores are in st, the largest in mx; MORE: the next tile's go to nx.
  const float cexp = p.sm_scale * 1.44269504088896340736f;
  auto step = [&](auto more, int par, int tile, v4f (&st)[NU][4], v4f (&nx)[NU][4]) __attribute__((always_inline)) {
    constexpr bool MORE = decltype(more)::value;
    pf_u4 hk[6], hv[4];
    if constexpr (MORE) {   // (the buffers' last readers were a step ago)
      if constexpr (DMA) {
        if (tile + 2 < ntiles) stage_k(tile + 2, par, hk);
      } else if constexpr (ALONE) {
        stage_k(min(tile + 2, ntiles - 1), par, hk);
      }
      stage_v(tile + 1, par ^ 1, hv);
    }
    // ---- online softmax, per query (lane & 15): where some lane's running maximum moved, O and the sums are scaled to the new one.  It is kept on the RAW scores;
    // the softmax scale rides in the exponent's multiply: p = exp2(s * c - m * c), c = sm_scale * log2(e).  A lane sums its own keys; the query's four meet at the end.
#pragma unroll
    for (int u = 0; u < NU; u++)
      if (!__all(mx[u] <= m_run[u])) {
        const float m_new = fmaxf(m_run[u], mx[u]);             // finite from tile 0 on: key 0 is visible to every query (SPLIT, tile0 > 0: or the query has seen no key yet)
        const float alpha = SPLIT && m_new == m_run[u] ? 1.f : __builtin_amdgcn_exp2f((m_run[u] - m_new) * cexp);
        m_run[u] = m_new;
        l_run[u] *= alpha;
#pragma unroll
        for (int i = 0; i < 8; i++) o[u][i] *= alpha;
      }
    // ---- the probabilities, beside the next tile's scores
    if constexpr (MORE) qk(par ^ 1, nx);
    uint4 pb[NU][2];
#pragma unroll
    for (int u = 0; u < NU; u++) {
      // (SPLIT: no key seen yet, so that the tile's weigh nothing.  A first tile of scores of -inf gives NaN, shared or not.)
      const float mc = SPLIT && tile0 > 0 && m_run[u] == -__builtin_inff() ? 0.f : -m_run[u] * cexp;
      float sum2[2] = {0.f, 0.f};
      float pv[4][4];
#pragma unroll
      for (int kt = 0; kt < 4; kt++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
          pv[kt][r] = __builtin_amdgcn_exp2f(fmaf(st[u][kt][r], cexp, mc));
          sum2[r & 1] += pv[kt][r];
        }
      l_run[u] += sum2[0] + sum2[1];
#pragma unroll
      for (int ks = 0; ks < 2; ks++)
        pb[u][ks] = make_uint4(ktx_pk_bf16(pv[2 * ks][0], pv[2 * ks][1]), ktx_pk_bf16(pv[2 * ks][2], pv[2 * ks][3]),
                               ktx_pk_bf16(pv[2 * ks + 1][0], pv[2 * ks + 1][1]), ktx_pk_bf16(pv[2 * ks + 1][2], pv[2 * ks + 1][3]));
    }
    if constexpr (MORE) {   // the order of that stream: a fragment's two MFMAs, the read of the fragment four further, the softmax's next instructions
      __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
#pragma unroll
      for (int f = 0; f < 24; f++) {
        __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
        if (f < 20) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x402, 6, 0);
      }
    }
    if constexpr (MORE) {
      // (here, or the compiler moves them behind the mask's branch, away from the products)
#pragma unroll
      for (int u = 0; u < NU; u++) {
        asm volatile("" : "+v"(l_run[u]));
#pragma unroll
        for (int ks = 0; ks < 2; ks++) asm volatile("" : "+v"(pb[u][ks].x), "+v"(pb[u][ks].y), "+v"(pb[u][ks].z), "+v"(pb[u][ks].w));
      }
      mask(tile + 1, nx);
      if constexpr (!DMA && !ALONE) {   // (V^T waited beside S, K does beside O, where the scores before are gone; the last requests repeat)
        put_v(par ^ 1, hv);
        stage_k(min(tile + 2, ntiles - 1), par, hk);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    // ---- O^T += V^T P^T: o[u][i][r] = O[query qi][dim 16*i + 4*g + r], beside the next tile's largest scores
    const uint8_t* vb = smem + par * PF_VB;
#pragma unroll
    for (int ks = 0; ks < 2; ks++) {                  // (key half outermost: 8 x NU independent accumulators)
#pragma unroll
      for (int i = 0; i < 8; i++) {
        const v8bf a = as_v8bf(*reinterpret_cast<const uint4*>(vb + i * 2048 + (vo ^ (ks * 64))));
#pragma unroll
        for (int u = 0; u < NU; u++) o[u][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, as_v8bf(pb[u][ks]), o[u][i], 0, 0, 0);
      }
    }
    if constexpr (MORE) largest(nx);
    __builtin_amdgcn_sched_group_barrier(0x100, 4, 1);
#pragma unroll
    for (int f = 0; f < 16; f++) {
      __builtin_amdgcn_sched_group_barrier(0x008, 2, 1);
      if (f < 12) __builtin_amdgcn_sched_group_barrier(0x100, 1, 1);
    }
    if constexpr (MORE) {
      if constexpr (ALONE) put_v(par ^ 1, hv);
      put_k(par, hk);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // (a step old)
      __syncthreads();
    }
  };
  v4f sa[NU][4], sb[NU][4];
  qk(0, sa);
  __syncthreads();   // (the first step's requests overwrite what this read)
  mask(tile0, sa);
  largest(sa);
  int tile = tile0;
  for (; tile + 2 < ntiles; tile += 2) {
    step(std::true_type{}, 0, tile, sa, sb);
    step(std::true_type{}, 1, tile + 1, sb, sa);
  }
  if (tile + 1 < ntiles) {
    step(std::true_type{}, 0, tile++, sa, sb);
#pragma unroll
    for (int u = 0; u < NU; u++)
#pragma unroll
      for (int kt = 0; kt < 4; kt++) sa[u][kt] = sb[u][kt];
  }
  step(std::false_type{}, (tile - tile0) & 1, tile, sa, sb);
#pragma unroll
  for (int u = 0; u < NU; u++) {
    const int t = q0 + u * 16 + qi;
    const float l = pf_sum_rows(l_run[u]);
    if constexpr (SPLIT) {
      if (t < p.T) {
        const size_t at = ((size_t)t * p.H + h) * p.nsplit + split;
        if (g == 0) *reinterpret_cast<float2*>(p.part_ml + at * 2) = make_float2(m_run[u], l);
        float* po = p.part_o + at * 128 + g * 4;
#pragma unroll
        for (int i = 0; i < 8; i++) *reinterpret_cast<float4*>(po + i * 16) = make_float4(o[u][i][0], o[u][i][1], o[u][i][2], o[u][i][3]);
      }
      continue;
    }
    if (t < p.T) {
      const float inv = l > 0.f ? 1.0f / l : 0.f;
      bf16_t* op = p.out + ((size_t)t * p.H + h) * 128 + g * 4;
#pragma unroll
      for (int i = 0; i < 8; i++)
        *reinterpret_cast<uint2*>(op + i * 16) = make_uint2(ktx_pk_bf16(o[u][i][0] * inv, o[u][i][1] * inv),
                                                            ktx_pk_bf16(o[u][i][2] * inv, o[u][i][3] * inv));
    }
  }
}

// The pieces of a query's keys: out = sum_s w_s O_s / sum_s w_s l_s, w_s = exp2((m_s - max m) c).  Thread = 4 dims of a (token, head), all pieces' loads ahead of the first use.
template <int NS>
__global__ __launch_bounds__(256) void mla_prefill_merge_kernel(MlaPrefillParams p) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x, row = i >> 5;
  if (row >= (long)p.T * p.H) return;
  const int d = (int)(i & 31) * 4;
  const float c = p.sm_scale * 1.44269504088896340736f;
  float2 ml[NS];
  float4 o[NS];
#pragma unroll
  for (int s = 0; s < NS; s++) {
    const size_t at = (size_t)row * p.nsplit + min(s, p.nsplit - 1);
    ml[s] = *reinterpret_cast<const float2*>(p.part_ml + at * 2);
    o[s] = *reinterpret_cast<const float4*>(p.part_o + at * 128 + d);
  }
  float m = -__builtin_inff();
#pragma unroll
  for (int s = 0; s < NS; s++) m = fmaxf(m, ml[s].x);
  float l = 0.f;
  float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
  for (int s = 0; s < NS; s++) {
    if (s >= p.nsplit || ml[s].y < 0.f) continue;   // (a piece without a tile: old memory.  One without a key of the query's weighs 0, which an infinite value makes NaN as in an unshared tile.)
    const float w = __builtin_amdgcn_exp2f((ml[s].x - m) * c);
    l += w * ml[s].y;
    v.x += w * o[s].x; v.y += w * o[s].y; v.z += w * o[s].z; v.w += w * o[s].w;
  }
  const float inv = l > 0.f ? 1.0f / l : 0.f;
  *reinterpret_cast<uint2*>(p.out + (size_t)row * 128 + d) = make_uint2(ktx_pk_bf16(v.x * inv, v.y * inv), ktx_pk_bf16(v.z * inv, v.w * inv));
}

// How many workgroups share a query's keys.  A workgroup of 128 queries and a head alone on its CU takes 1.27 us a key tile, two beside each other 2.0, so that few (query block, head)
// pairs with long contexts leave most of the chip idle: 64 queries of 16 heads behind 6000 tokens are 16 workgroups of 95 tiles, 128 us.  The pieces cost their sums' way to
// memory and back and the merge's launch: this estimate, fitted to 66 calls at 1 to 16 pieces (profiles/mla_prefill_pieces.txt), picks
// a count within 9 % of the best one where it shares, within 6 in all but one, and shares only where it sees a tenth to gain: up to 16 % is left there (16 heads, 1500 queries behind 1000 59.7,
// three pieces 51.5).  Us, whole | here:
// 16 heads, 64 queries behind 1000 29 | 15, 6000 128 | 23, 300 behind 1000 36 | 24, 3000 76 | 32, 800 behind 3000 88 | 56; 64 heads, 64 behind 3000 70 | 31, 150 behind 1000 34 | 28; 128
// heads, 64 behind 3000 72 | 47.  Past 192 pairs, whose workgroups share CUs as it is, 5 to 10 % at most (128 heads, 150 behind 6000 170 | 158) and as often nothing.
// Dev knob 33 (tests): that many.
constexpr int PF_SPLITS = 16;
static int pf_splits(int T, int H, int kv_len) {
  const int tiles = (kv_len + PF_BN - 1) / PF_BN;
  if (ktx_debug_get(33) > 0) return std::min(ktx_debug_get(33), PF_SPLITS);
  const long pairs = (long)((T + 127) / 128) * H;
  if (pairs > 192) return 1;
  auto us = [&](int n) {
    const long each = (pairs * n + 255) / 256;   // workgroups a CU
    return 6.0 + (tiles + n - 1) / n * 1.27 * (each == 1 ? 1.0 : 0.8 * each) + (n > 1 ? 3.0 + (double)T * H * n * 1040e-6 / 6.0 : 0.0);
  };
  int best = 1;
  for (int n = 2; n <= std::min(PF_SPLITS, tiles); n++)
    if (us(n) < us(best)) best = n;
  return us(best) < 0.9 * us(1) ? best : 1;
}
static size_t pf_split_bytes(int T, int H, int nsplit) { return nsplit > 1 ? (size_t)T * H * nsplit * 130 * sizeof(float) : 0; }

extern "C" size_t ktx_mla_prefill_workspace_bytes(int T, int num_heads, int kv_len) {
  return T > 0 && num_heads > 0 && kv_len >= T ? pf_split_bytes(T, num_heads, pf_splits(T, num_heads, kv_len)) : 0;
}

extern "C" int ktx_mla_prefill(int T, int num_heads, int kv_len, int kv_pad, float sm_scale, const void* d_q_nope,
                               int64_t qn_token_stride, int64_t qn_head_stride, const void* d_q_pe, int64_t qp_token_stride,
                               int64_t qp_head_stride, const void* d_k_nope, const void* d_k_pe, int64_t kpe_token_stride,
                               const void* d_v_t, void* d_out, void* stream) {
  return ktx_mla_prefill_ws(T, num_heads, kv_len, kv_pad, sm_scale, d_q_nope, qn_token_stride, qn_head_stride, d_q_pe, qp_token_stride, qp_head_stride, d_k_nope, d_k_pe, kpe_token_stride,
                            d_v_t, d_out, nullptr, 0, stream);
}

extern "C" int ktx_mla_prefill_ws(int T, int num_heads, int kv_len, int kv_pad, float sm_scale, const void* d_q_nope,
                                  int64_t qn_token_stride, int64_t qn_head_stride, const void* d_q_pe, int64_t qp_token_stride,
                                  int64_t qp_head_stride, const void* d_k_nope, const void* d_k_pe, int64_t kpe_token_stride,
                                  const void* d_v_t, void* d_out, void* d_workspace, size_t workspace_bytes, void* stream) {
  KTX_REQUIRE(d_q_nope && d_q_pe && d_k_nope && d_k_pe && d_v_t && d_out, "ktx_mla_prefill: null pointer");
  KTX_REQUIRE(T > 0 && num_heads > 0 && kv_len >= T, "ktx_mla_prefill: need 0 < T <= kv_len (the new tokens are the last T keys)");
  KTX_REQUIRE(kv_pad >= kv_len && kv_pad % PF_BN == 0, "ktx_mla_prefill: kv_pad must be a multiple of 64 covering kv_len");
  KTX_REQUIRE(qn_token_stride % 8 == 0 && qn_head_stride % 8 == 0 && qp_token_stride % 8 == 0 && qp_head_stride % 8 == 0 &&
              kpe_token_stride % 8 == 0, "ktx_mla_prefill: strides must keep 16-byte alignment");
  MlaPrefillParams p;
  p.q_nope = (const bf16_t*)d_q_nope; p.q_pe = (const bf16_t*)d_q_pe;
  p.qn_ts = qn_token_stride; p.qn_hs = qn_head_stride; p.qp_ts = qp_token_stride; p.qp_hs = qp_head_stride;
  p.k_nope = (const bf16_t*)d_k_nope; p.k_pe = (const bf16_t*)d_k_pe; p.kpe_ts = kpe_token_stride;
  p.v_t = (const bf16_t*)d_v_t; p.out = (bf16_t*)d_out;
  p.T = T; p.H = num_heads; p.kv_len = kv_len; p.kv_pad = kv_pad; p.sm_scale = sm_scale;
  constexpr int lds = 2 * (PF_KB + PF_VB);
  const bool aligned = ((reinterpret_cast<uintptr_t>(d_k_nope) | reinterpret_cast<uintptr_t>(d_k_pe) | reinterpret_cast<uintptr_t>(d_v_t)) & 15) == 0;
  p.nqb = (T + 127) / 128;
  p.nsplit = aligned && d_workspace && (reinterpret_cast<uintptr_t>(d_workspace) & 15) == 0 ? pf_splits(T, num_heads, kv_len) : 1;
  if (pf_split_bytes(T, num_heads, p.nsplit) > workspace_bytes) p.nsplit = 1;   // (without scratch: one workgroup for all of a query's keys)
  p.part_o = (float*)d_workspace;
  p.part_ml = p.nsplit > 1 ? p.part_o + (size_t)T * num_heads * p.nsplit * 128 : nullptr;
  void (*kern)(MlaPrefillParams) = p.nsplit > 1 ? mla_prefill_kernel<true, false, true> : aligned ? mla_prefill_kernel<true>
                                   : (long)p.nqb * num_heads <= 256 ? mla_prefill_kernel<false, true> : mla_prefill_kernel<false>;
  KTX_HIP(ktx_set_max_lds(reinterpret_cast<const void*>(kern), lds));
  hipStream_t st = (hipStream_t)stream;
  // per (query, key, head): 2*(192 + 128) flop over the causal half
  KTX_TIMED(st, 0.0, "mla_prefill_kernel T=%d Hq=%d kv=%d splits %d", T, num_heads, kv_len, p.nsplit);
  p.xcd = num_heads % 8 == 0;
  const dim3 grid = p.xcd ? dim3((unsigned)((size_t)p.nqb * num_heads * p.nsplit)) : dim3(p.nqb, num_heads, p.nsplit);
  hipLaunchKernelGGL(kern, grid, dim3(256), lds, st, p);
  KTX_HIP(hipGetLastError());
  if (p.nsplit > 1) {
    const dim3 mgrid((unsigned)(((size_t)T * num_heads + 7) / 8));
    if (p.nsplit <= 2) hipLaunchKernelGGL(mla_prefill_merge_kernel<2>, mgrid, dim3(256), 0, st, p);
    else if (p.nsplit <= 4) hipLaunchKernelGGL(mla_prefill_merge_kernel<4>, mgrid, dim3(256), 0, st, p);
    else if (p.nsplit <= 8) hipLaunchKernelGGL(mla_prefill_merge_kernel<8>, mgrid, dim3(256), 0, st, p);
    else hipLaunchKernelGGL(mla_prefill_merge_kernel<PF_SPLITS>, mgrid, dim3(256), 0, st, p);
    KTX_HIP(hipGetLastError());
  }
  return 0;
}

extern "C" int ktx_mla_cache_append(const ktx_mla_config* cfg, void* d_kv_cache, int64_t token_stride,
                                    const void* d_ckv_new, const void* d_kpe_new, const int32_t* d_page_idx,
                                    const int32_t* d_page_offset, const int32_t* d_ntokens, int max_tokens, int num_pages,
                                    void* stream) {
  KTX_REQUIRE(cfg && d_kv_cache && d_ckv_new && d_kpe_new && d_page_idx && d_page_offset && max_tokens > 0,
              "ktx_mla_cache_append: bad argument");
  KTX_REQUIRE(token_stride >= MLA_DC + MLA_DR && token_stride % 8 == 0, "ktx_mla_cache_append: bad token stride");
  hipLaunchKernelGGL(mla_cache_append_kernel, dim3(max_tokens), dim3(128), 0, (hipStream_t)stream, (bf16_t*)d_kv_cache,
                     (long long)token_stride, cfg->page_size, (const bf16_t*)d_ckv_new, (const bf16_t*)d_kpe_new,
                     d_page_idx, d_page_offset, d_ntokens, max_tokens, num_pages);
  KTX_HIP(hipGetLastError());
  return 0;
}
