// Causal multi-token decode at 16 heads over the fp8 cache (q_seq_len 2 to 4):
// the query rows of one sequence run as one work item.
//
// Planned row by row, each of a sequence's q_seq_len rows gathers the whole
// cache of the sequence again (32 ragged sequences of 512 to 8192 keys, 4 rows:
// 48 us of decode for 64 MB of cache, 5.4 TB/s of gather that is repeated four
// times).  Here an item is {sequence, token range, slot}, and the 16 heads of
// its rows are the 64 columns of one pass: column c is row c / 16, head c % 16
// (columns past q_seq_len rows multiply zeros; a two-row call still reads its
// cache once instead of twice, and the matrix work of 64 columns stays below the
// time of the gather).  Row i sees the sequence's first L - (q_seq_len - 1 - i)
// keys: a per-lane limit in the tiles at the sequence's end.
//
// One work-group of 8 waves per CU, two to a SIMD.  Tiles of 64 tokens in a 4-stage
// LDS ring, in the row layout of mla_tile64.hpp.
// Waves 0-3 score tile t while waves 4-7 run the PV of tile t - 1: as four waves
// doing one after the other, a tile took its whole chain (fragment reads, nine
// MFMAs, softmax, exchange, sixteen MFMAs), about 2.3 us; side by side 1.2, and
// 64 keys more of 256 sequences x 4 rows cost what their gather does (6.1 TB/s).
// The 32 ragged sequences take 24-26 us of decode instead of 48, the call 33.3-35.6
// instead of 58.0; a third of the rest is start-up (Q of 64 columns quantized, 2 us;
// the plan, slots and first rows, 4) and 64 KiB of output per item.
//   Scoring wave w: token half w & 1, column half w >> 1, nine 32x32x64 MFMAs
// (S^T = K . Q^T, Q^T of its 32 columns in 72 registers).  A lane's 16 scores
// are one column's, and the tokens its bytes of the PV operand hold, so P' goes
// through LDS as whole 16-byte fragments.
//   PV wave: latent dims 128 (w - 4) .. +127 of all 64 columns, sixteen 32x32x64
// MFMAs a tile with every K lane in use (two fp8 terms of P', V^T fragments shared
// by both column halves); it also gathers the rows of tile t + 2, nine DMA windows.
// The columns share a tile's V, so at the sequence's end a key that some of them
// must not see is multiplied by their zero P': its NaN codes are read as 0 there (a
// column that sees such a key has a NaN score from the same bytes, and stays NaN).
// Two barriers a tile: (A) tile t landed, P'(t - 1) written, the stage of tile
// t - 2 free; (B) P'(t - 1) in the PV waves' registers, so P'(t) may take its
// place.  Most of the PV runs before B, beside the scores.
// Softmax as in decode_h128.hip: a fixed reference per column (the first tile's
// ceil max, over both token halves), the tile max of a 32-token half in the e8m0 B
// scale of its K block, and a second pass from the maxima of the whole item when a
// tile max lies more than 96 above the reference.
//
// Behavioural reference: competitor_submissions/mi355x_reference/
// reference.py:188-193 (uniform causal rows), mixed-mla/asm_dumps/
// aiter_mla.py:149-470.
#include "mla_internal.hpp"
#include "mla_tile64.hpp"

namespace mla {
namespace {

constexpr float kLog2eR = 1.4426950408889634f;
constexpr float kLn2R = 0.6931471805599453f;
constexpr float kRebaseR = 96.0f;
// The reference of a column whose scores are all -inf so far (or that sees no key):
// below any finite score, which starts the second pass; -inf itself would make the
// differences NaN.
constexpr float kNoScoreR = -3.0e38f;

struct R64 {
  static constexpr int COLS = 64;
  static constexpr int RST = kRowSt, CPR = kRowCh;       // LDS row stride, its chunks
  static constexpr int TSTAGE = 32 * RST;                // 32 rows
  static constexpr int STAGE = 2 * TSTAGE;               // 64 rows
  static constexpr int S = 4, NSL = 4;                   // row stages, slot stages
  static constexpr int NA = STAGE / 1024 / 4;            // 9 one-KiB DMA windows per PV wave
  static constexpr int OFF_SLOT = S * STAGE;             // [NSL][64] int32
  static constexpr int OFF_P = OFF_SLOT + NSL * 256;     // [term][token half][column][lane half] 16 B
  static constexpr int OFF_PS = OFF_P + 2 * 2 * COLS * 2 * 16;  // [token half][column] e8m0
  static constexpr int OFF_X = OFF_PS + 2 * COLS;        // [token half][column] f32 exchange
  static constexpr int OFF_VOTE = OFF_X + 2 * COLS * 4;  // [8] bytes
  static constexpr int LDS = OFF_VOTE + 16;
  static constexpr int OFF_Q = 2 * STAGE;                // Q (prologue): bf16 in stages 2 and 3, fp8 in stage 2
  static constexpr int OST = 2 * 128 + 16;               // output staging: 128 dims of a column
  static_assert(STAGE % 4096 == 0 && COLS * kQKDim <= STAGE, "DMA windows, Q staging");
  static_assert(4 * COLS * OST <= OFF_SLOT && LDS <= 160 * 1024, "LDS");
};

// four e4m3 codes with the NaNs (0x7F, 0xFF) as 0
__device__ __forceinline__ int nan_codes_to_zero(int x) {
  const uint32_t n = (((uint32_t)x & 0x7F7F7F7Fu) + 0x01010101u) & 0x80808080u;  // bit 7 of a NaN's byte
  return (int)((uint32_t)x & ~(n | (n - (n >> 7))));
}

template <bool IDX>
__global__ __launch_bounds__(512, 2) void decode_rows_kernel(const DecodeParams p) {
  using C = R64;
  __shared__ __attribute__((aligned(1024))) uint8_t smem[C::LDS];
  const uint32_t lds0 = (uint32_t)(uintptr_t)smem;
  const int32_t* plan = p.plan;
  // the item count and this item read together (the plan has room for max_items
  // >= gridDim.x items)
  const int nitems = plan[0];
  const int4 it = reinterpret_cast<const int4*>(plan + kPlanHeader)[blockIdx.x];
  if ((int)blockIdx.x >= nitems) return;
  const int b = __builtin_amdgcn_readfirstlane(it.x), t_beg = __builtin_amdgcn_readfirstlane(it.y);
  const int t_end = __builtin_amdgcn_readfirstlane(it.z), slot = __builtin_amdgcn_readfirstlane(it.w);
  const int ntok = t_end - t_beg, ntiles = (ntok + 63) / 64;
  const int qlen = p.plan_qlen, cols = 16 * qlen;

  const int tid = threadIdx.x;
  const int w8 = __builtin_amdgcn_readfirstlane(tid >> 6);
  const bool scorer = w8 < 4;
  const int w = w8 & 3;
  const int lane = tid & 63, l32 = lane & 31, hh = lane >> 5;
  const int th = w & 1, cw = w >> 1;  // a scoring wave's token half and column half
  const int col = 32 * cw + l32;
  float* xch = reinterpret_cast<float*>(smem + C::OFF_X);
  uint8_t* psc = smem + C::OFF_PS;

  // slots of tile t into slot stage t % NSL: scoring wave 0
  auto issue_slots = [&](int t) __attribute__((always_inline)) {
    if constexpr (IDX) {
      if (w8 == 0) dma4_to_lds(p.kv_indices + min(t_beg + 64 * t + lane, t_end - 1), lds0 + C::OFF_SLOT + (t & 3) * 256);
    }
  };
  // rows of tile t: window k of PV wave w puts lane l at chunk position 64 (w +
  // 4k) + l of the stage (row r, position j) and fetches logical chunk j ^ key(r)
  // (wmap[k]: r << 16 | byte offset of the chunk, decoded at use)
  uint32_t wmap[C::NA];
  auto issue_rows = [&](int t) __attribute__((always_inline)) {
    const uint32_t base = __builtin_amdgcn_readfirstlane(lds0 + (t & 3) * C::STAGE + 1024 * w);
    int sl[C::NA];  // every slot read before the first DMA (each an asm barrier)
#pragma unroll
    for (int k = 0; k < C::NA; ++k) {
      asm volatile("" : "+v"(wmap[k]));  // nothing decoded ahead and kept
      if constexpr (IDX) sl[k] = reinterpret_cast<const int*>(smem + C::OFF_SLOT + (t & 3) * 256)[wmap[k] >> 16];
      else sl[k] = min(t_beg + 64 * t + (int)(wmap[k] >> 16), t_end - 1);
    }
    dma16_windows<0, C::NA>(base, [&](auto kt) __attribute__((always_inline)) {
      constexpr int k = decltype(kt)::value;
      return p.k_cache + ((uint64_t)(uint32_t)sl[k] * (uint32_t)p.k_row_stride + (wmap[k] & 0xFFFFu));
    });
  };
  static_assert(C::S == 4 && C::NSL == 4, "stage t & 3");

  if (ntiles > 0) {
#pragma unroll
    for (int j = 0; j < 4; ++j) issue_slots(j);
  }
  // ---- Q: the item's rows as bf16 by LDS-DMA into stages 2 and 3 (nine windows a
  // wave), quantized in place with the per-tensor scale while the rows of the
  // first two tiles fly.  Columns past the rows' re-fetch the last chunk and are
  // zeroed.
  constexpr int QN = C::COLS * kQKDim / 8, QJ = QN / 512;  // 16-byte bf16 chunks, per thread
  static_assert(QJ * 512 == QN && QJ * 8 * 1024 == 2 * C::STAGE, "whole chunks and windows");
  {
    const uint8_t* src = reinterpret_cast<const uint8_t*>(p.q_bf16 + (int64_t)b * cols * kQKDim);
#pragma unroll
    for (int j = 0; j < QJ; ++j) {
      const int off = 1024 * (w8 + 8 * j);
      dma16_to_lds(src + min(off + 16 * lane, cols * kQKDim * 2 - 16), lds0 + C::OFF_Q + off);
    }
  }
  const float kvs = p.kv_scale[0];
  // this lane's column sees keys below vis_end (row col / 16 of the sequence)
  const int vis_end = min(t_end, p.kv_indptr[b + 1] - (qlen - 1 - min(col >> 4, qlen - 1)));

#pragma unroll
  for (int k = 0; k < C::NA; ++k) {
    const int e = 64 * (w + 4 * k) + lane, r = e / C::CPR, j = e - C::CPR * r;
    wmap[k] = ((uint32_t)r << 16) | (uint32_t)(16 * (j ^ row_key(r)));
  }
  if (IDX && w8 == 0) wait_vmcnt<QJ>();  // the slots (Q may be in flight)
  lds_barrier();
  if (!scorer) {  // the first two tiles' rows fly while Q is quantized
    if (ntiles > 0) issue_rows(0);
    if (ntiles > 1) issue_rows(1);
    if (ntiles > 1) wait_vmcnt<2 * C::NA>();  // this wave's share of Q
    else if (ntiles > 0) wait_vmcnt<C::NA>();
    else wait_vmcnt<0>();
  } else {  // the partial maxima (at most 4 x 256)
    uint32_t qm = 0;
#pragma unroll
    for (int j = 0; j < kAmaxMaxBlocks / 256; ++j)
      if (tid + 256 * j < p.q_nparts) qm = max(qm, p.q_partials[tid + 256 * j]);
    const uint32_t m = (uint32_t)wave_max((int)qm);
    if (lane == 0) reinterpret_cast<uint32_t*>(smem + C::OFF_X)[w] = m;
    wait_vmcnt<0>();
  }
  lds_barrier();  // Q and the wave maxima in LDS
  float c;
  {
    const uint4 m = *reinterpret_cast<const uint4*>(smem + C::OFF_X);
    // thread: column tid / 8, its 16-byte bf16 chunks tid % 8 + 8 j; the fp8 row
    // swizzled as the cache rows
    const int qc = tid >> 3, q8 = tid & 7;
    uint4 xq[QJ];
#pragma unroll
    for (int j = 0; j < QJ; ++j) xq[j] = *reinterpret_cast<const uint4*>(smem + C::OFF_Q + qc * 2 * kQKDim + 16 * (q8 + 8 * j));
    const float qs = fp8_scale_from_amax(max(max(m.x, m.y), max(m.z, m.w)));
    const Fp8Quant qq = make_fp8_quant(qs);
    lds_barrier();  // every bf16 chunk read before the fp8 rows overwrite them
#pragma unroll
    for (int j = 0; j < QJ; ++j) {
      const int c16 = (q8 >> 1) + 4 * j;
      *reinterpret_cast<uint2*>(smem + C::OFF_Q + qc * kQKDim + 16 * (c16 ^ row_key(qc)) + 8 * (q8 & 1)) =
          qc < cols ? quant8_fp8(xq[j], qq) : make_uint2(0, 0);
    }
    c = qs * kvs * p.sm_scale * kLog2eR;
  }
  lds_barrier();

  float m_ref = 0.f, m_seen = -__builtin_inff(), l_run = 0.f;
  bool have_ref = false, overflow = false;
  v16f o[2][4];  // PV waves: [column half][dim tile]

  // One pass over the item; both roles run the same barriers: A and B per tile
  // (and one after the last tile's scores), and the reference exchange of a first
  // pass between A and B of tile 0.
  if (scorer) {
    v8i qv[9];
    {
      const uint8_t* qrow = smem + C::OFF_Q + col * kQKDim;
      const int x0 = 16 * ((2 * hh) ^ row_key(col)), x1 = 16 * ((2 * hh + 1) ^ row_key(col));
#pragma unroll
      for (int ks = 0; ks < 9; ++ks) {
        const uint4 a = *reinterpret_cast<const uint4*>(qrow + x0 + 64 * ks);
        const uint4 d = *reinterpret_cast<const uint4*>(qrow + x1 + 64 * ks);
        qv[ks] = v8i{(int)a.x, (int)a.y, (int)a.z, (int)a.w, (int)d.x, (int)d.y, (int)d.z, (int)d.w};
      }
#pragma unroll
      for (int ks = 0; ks < 9; ++ks) asm volatile("" : "+v"(qv[ks]));  // keep resident, no reload
    }
    typedef __attribute__((address_space(3))) v4i lds_v4i;
    // K fragment of step ks: chunks 4 ks + 2 hh + {0, 1} of row l32 of the half
    const uint32_t krow = lds0 + th * C::TSTAGE + l32 * C::RST;
    const uint32_t k0 = krow + 16 * ((2 * hh) ^ row_key(l32)), k1 = krow + 16 * ((2 * hh + 1) ^ row_key(l32));
    for (;;) {
      for (int t = 0; t <= ntiles; ++t) {
        if (IDX && w8 == 0) {  // the slots of tile t + 2 landed (those of t + 3 may be in flight)
          if (t > 0) wait_vmcnt<1>();
        }
        lds_barrier();  // (A)
        if (ntiles > 0) issue_slots(t + 4);  // (past the item: its last token's, never used)
        v16f s = v16f{};
        int4 hi4, lo4;
        int e8 = 0;
        const bool live = t < ntiles;
        if (live) {
          uint32_t a0 = k0 + (t & 3) * C::STAGE, a1 = k1 + (t & 3) * C::STAGE;
          asm volatile("" : "+v"(a0), "+v"(a1));
#pragma unroll
          for (int ks = 0; ks < 9; ++ks) {
            const v4i lo = *(const lds_v4i*)(uintptr_t)(a0 + 64 * ks);
            const v4i hi = *(const lds_v4i*)(uintptr_t)(a1 + 64 * ks);
            s = mfma32_f8(v8i{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]}, qv[ks], s);
          }
          // s[r]: token 8 (r >> 2) + 4 hh + (r & 3) of the half, column `col`
#pragma unroll
          for (int r = 0; r < 16; ++r) s[r] *= c;
          if (t_beg + 64 * (t + 1) > t_end - (qlen - 1)) {
            const int lim = vis_end - (t_beg + 64 * t + 32 * th) - 4 * hh;
#pragma unroll
            for (int r = 0; r < 16; ++r) s[r] = 8 * (r >> 2) + (r & 3) < lim ? s[r] : -__builtin_inff();
          }
          float mx = fmaxf(fmaxf(fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3])), fmaxf(fmaxf(s[4], s[5]), fmaxf(s[6], s[7]))),
                           fmaxf(fmaxf(fmaxf(s[8], s[9]), fmaxf(s[10], s[11])), fmaxf(fmaxf(s[12], s[13]), fmaxf(s[14], s[15]))));
          mx = __builtin_ceilf(xhalf_max(mx));  // -inf where the column sees no token of the half
          if (!have_ref) {
            if (hh == 0) xch[C::COLS * th + col] = mx;
            lds_barrier();
            m_ref = fmaxf(xch[col], xch[C::COLS + col]);
            m_ref = fmaxf(m_ref, kNoScoreR);
            have_ref = true;
          }
          m_seen = fmaxf(m_seen, mx);
          overflow = overflow || mx - m_ref > kRebaseR;  // (m_ref + kRebaseR would round at scores past 2^30)
          // the exponent: clamped (a flagged pass is run again), and finite where
          // the half is masked (its P' is 0 whatever the exponent)
          mx = fminf(fmaxf(mx, m_ref - 160.f), m_ref + kRebaseR);
          // P' = 2^(s - mx + up): up = 8 uses the fp8 range; none where it would
          // round (scores past 2^26 lie 8 apart or more: P' is 1, 2^-8 or next to 0)
          const float up = fabsf(mx) < 67108864.f ? 8.f : 0.f;
          e8 = min(max((int)(mx - m_ref - up) + 127, 0), 254);
          const float sh = up - mx;
          float ps[4] = {0.f, 0.f, 0.f, 0.f};
          int2 q4[4];
#pragma unroll
          for (int q = 0; q < 4; ++q) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              s[4 * q + i] = __builtin_amdgcn_exp2f(s[4 * q + i] + sh);
              ps[i] += s[4 * q + i];
            }
            q4[q] = split4(s[4 * q], s[4 * q + 1], s[4 * q + 2], s[4 * q + 3]);
          }
          l_run = __builtin_fmaf((ps[0] + ps[1]) + (ps[2] + ps[3]), __builtin_amdgcn_exp2f(mx - m_ref - up), l_run);
          hi4 = make_int4(q4[0].x, q4[1].x, q4[2].x, q4[3].x);
          lo4 = make_int4(q4[0].y, q4[1].y, q4[2].y, q4[3].y);
        }
        lds_barrier();  // (B)
        if (live) {
          uint8_t* pw = smem + C::OFF_P + 16 * (2 * (C::COLS * th + col) + hh);
          *reinterpret_cast<int4*>(pw) = hi4;
          *reinterpret_cast<int4*>(pw + 4 * C::COLS * 16) = lo4;
          if (hh == 0) psc[C::COLS * th + col] = (uint8_t)e8;
        }
      }
      // a flagged column on any wave: run the item again from the running maxima
      wait_vmcnt<0>();
      if (lane == 0) smem[C::OFF_VOTE + w] = __any(overflow) ? 1 : 0;
      if (hh == 0) xch[C::COLS * th + col] = m_seen;
      lds_barrier();
      if (__builtin_amdgcn_readfirstlane(*reinterpret_cast<const int*>(smem + C::OFF_VOTE)) == 0) break;
      m_ref = fmaxf(xch[col], xch[C::COLS + col]);
      m_ref = fmaxf(m_ref, kNoScoreR);
      overflow = false;
      l_run = 0.f;
#pragma unroll
      for (int j = 0; j < 4; ++j) issue_slots(j);
      wait_vmcnt<0>();
      lds_barrier();  // slots of tiles 0 .. 3; exchange read
    }
  } else {
    // V^T fragment of dim tile 4w + e: rows T0 + 16 cc of each token half, chunk
    // 2 (4w + e) + (G & 1); the XOR key moves only the chunk's low two bits
    uint32_t va[4];  // [cc][e & 1]; dim tiles e >= 2 are 64 bytes on
    {
      const int G = lane >> 4, m = (lane & 15) >> 1, oo = lane & 1;
      const int T0 = 8 * (m >> 2) + 4 * hh + (m & 3);
#pragma unroll
      for (int cc = 0; cc < 2; ++cc)
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          const int r = T0 + 16 * cc;
          va[2 * cc + e] = lds0 + r * C::RST + 16 * (8 * w + ((2 * e + (G & 1)) ^ row_key(r))) + 8 * oo;
        }
    }
    for (;;) {
#pragma unroll
      for (int i = 0; i < 8; ++i) o[i >> 2][i & 3] = v16f{};
      for (int t = 0; t <= ntiles; ++t) {
        // tile t landed; tile t + 1 (issued after it) may be in flight
        if (t + 1 < ntiles) wait_vmcnt<C::NA>();
        else wait_vmcnt<0>();
        lds_barrier();  // (A)
        v8i pf[2][2];  // [column half][term]: bytes 16 u + i are token half u's
        int bsc[2];
        if (t > 0) {
#pragma unroll
          for (int ch = 0; ch < 2; ++ch) {
            bsc[ch] = psc[C::COLS * hh + 32 * ch + l32];
#pragma unroll
            for (int term = 0; term < 2; ++term) {
              const uint8_t* pr = smem + C::OFF_P + 4 * C::COLS * 16 * term + 16 * (2 * (32 * ch + l32) + hh);
              const int4 u0 = *reinterpret_cast<const int4*>(pr), u1 = *reinterpret_cast<const int4*>(pr + 2 * C::COLS * 16);
              pf[ch][term] = v8i{u0.x, u0.y, u0.z, u0.w, u1.x, u1.y, u1.z, u1.w};
            }
          }
        }
        if (t + 2 < ntiles) issue_rows(t + 2);
        uint32_t a0[2], a1[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          a0[e] = va[e] + ((t - 1) & 3) * C::STAGE;
          a1[e] = va[2 + e] + ((t - 1) & 3) * C::STAGE;
          asm volatile("" : "+v"(a0[e]), "+v"(a1[e]));
        }
        const bool tail = t_beg + 64 * t > t_end - (qlen - 1);  // tile t - 1 holds keys that not every column sees
        auto pv = [&](auto et) __attribute__((always_inline)) {
          constexpr int e = decltype(et)::value;
          const uint32_t x0 = a0[e & 1] + 64 * (e >> 1), x1 = a1[e & 1] + 64 * (e >> 1);
          const v2i r0 = lds_read_tr8(x0), r1 = lds_read_tr8(x1);
          const v2i r2 = lds_read_tr8(x0 + C::TSTAGE), r3 = lds_read_tr8(x1 + C::TSTAGE);
          v8i vf = v8i{r0[0], r0[1], r1[0], r1[1], r2[0], r2[1], r3[0], r3[1]};
          if (tail) {
#pragma unroll
            for (int i = 0; i < 8; ++i) vf[i] = nan_codes_to_zero(vf[i]);
          }
#pragma unroll
          for (int term = 0; term < 2; ++term)
#pragma unroll
            for (int ch = 0; ch < 2; ++ch) o[ch][e] = mfma32_f8_bscale(vf, pf[ch][term], bsc[ch], o[ch][e]);
        };
        if (t > 0) {
          pv(WinK<0>{});
          pv(WinK<1>{});
          pv(WinK<2>{});
        } else if (ntiles > 0 && !have_ref) {
          lds_barrier();  // the scoring waves' reference exchange
          have_ref = true;
        }
        lds_barrier();  // (B)
        if (t > 0) pv(WinK<3>{});
      }
      wait_vmcnt<0>();
      lds_barrier();  // the scoring waves' flags
      if (__builtin_amdgcn_readfirstlane(*reinterpret_cast<const int*>(smem + C::OFF_VOTE)) == 0) break;
      lds_barrier();  // slots of tiles 0 .. 3; every PV wave is done with the ring
      issue_rows(0);
      if (ntiles > 1) issue_rows(1);
    }
  }

  // ---- finish ------------------------------------------------------------------
  // (the flags' barrier above: every wave is past its last read of P', the
  // scales and the ring)
  float* lx = reinterpret_cast<float*>(smem + C::OFF_P);  // [token half][column] row sums
  if (scorer) {
    const float lh = xhalf_sum(l_run);
    if (hh == 0) lx[C::COLS * th + col] = lh;
  }
  lds_barrier();
  if (scorer) {
    if (hh == 0 && th == 0 && col < cols) {
      const float L = lx[col] + lx[C::COLS + col];
      const float lse2 = L > 0.f ? m_ref + __log2f(L) : -__builtin_inff();
      if (slot >= 0) p.part_lse[(int64_t)slot * cols + col] = lse2;
      else if (p.lse_out != nullptr) p.lse_out[(int64_t)b * cols + col] = lse2 * kLn2R;
    }
    return;
  }
  // a PV wave's 128 dims of every column as 16-bit rows in LDS (only it reads
  // them), then 16-byte row segments.  A whole sequence's are the output's bf16.  A
  // piece's are fp16 in 128ths of a code (at most 448 x 128; the combine brings
  // kv_scale in): three bits more than bf16 at the same bytes, as this plan cuts
  // sequences into pieces that row by row stay whole (32 ragged sequences x 4 rows,
  // error against 64 bits: row by row 2.12e-3, here 2.21e-3 with bf16 pieces)
  uint8_t* ob = smem + w * C::COLS * C::OST;
  auto stage = [&](float one, auto pack) __attribute__((always_inline)) {
#pragma unroll
    for (int ch = 0; ch < 2; ++ch) {
      const float L = lx[32 * ch + l32] + lx[C::COLS + 32 * ch + l32];
      const float inv = L > 0.f ? one / L : 0.f;
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const v16f& a = o[ch][e];
          const uint32_t lo = pack(a[4 * q] * inv, a[4 * q + 1] * inv);
          const uint32_t hi = pack(a[4 * q + 2] * inv, a[4 * q + 3] * inv);
          *reinterpret_cast<uint2*>(ob + (32 * ch + l32) * C::OST + 2 * (32 * e + 8 * q + 4 * hh)) = make_uint2(lo, hi);
        }
    }
  };
  if (slot < 0) stage(kvs, [](float a, float b) __attribute__((always_inline)) { return pack_bf16x2(a, b); });
  else stage(128.f, [](float a, float b) __attribute__((always_inline)) { return pack_f16x2(a, b); });
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  uint16_t* dst = (slot < 0 ? p.out + (int64_t)b * cols * kVDim : p.part_o + (int64_t)slot * cols * kVDim) + 128 * w;
#pragma unroll 4
  for (int r = 0; r < C::COLS; r += 4) {
    const int cc = r + (lane >> 4);
    const uint4 v = *reinterpret_cast<const uint4*>(ob + cc * C::OST + 16 * (lane & 15));
    if (cc < cols) *reinterpret_cast<uint4*>(dst + (int64_t)cc * kVDim + 8 * (lane & 15)) = v;
  }
}

}  // namespace

hipError_t launch_decode_rows(const DecodeParams& p, int grid, hipStream_t stream) {
  if (p.kv_indices != nullptr)
    hipLaunchKernelGGL((decode_rows_kernel<true>), dim3(grid), dim3(512), 0, stream, p);
  else
    hipLaunchKernelGGL((decode_rows_kernel<false>), dim3(grid), dim3(512), 0, stream, p);
  return hipGetLastError();
}

}  // namespace mla
