// K3 for few heads (n_heads <= 64: tensor-parallel ranks at TP = 2, 4, 8): sparse MLA forward with
// the operation and the work items of sparse_mla_fwd_kernel (dsa_sparse_fwd.hip).
//
// With 128 heads a gathered KV row feeds 278 KFLOP and the matrix cores bind; with 16 heads it
// feeds 35 KFLOP.  One wave per 32 heads (the 128-head kernel cut down) left three of a CU's four
// SIMDs idle behind a 112 KB ring.  Here four waves share each 32-key tile and the footprint (two
// tiles, no staged index row) lets two workgroups run on a CU:
//   * scores S^T[32 keys x 16 NHT heads] with 16x16x32 MFMAs.  NHT = 1: wave (kt, wh) multiplies
//     16 keys by half of the contraction, and the partial sums meet in LDS (the K tile is read
//     once).  NHT = 2: wave (kt, wh) multiplies 16 keys by one head tile.
//   * O^T += V^T . P^T: wave w owns 128 of the 512 latent dims for every head.  The C layout of
//     S^T (lane group g holds keys 4g .. 4g+3 of each 16-key tile) is the B layout of this product
//     with the k order {4g .. 4g+3, 16 + 4g .. 16 + 4g+3}, which the V^T reads reproduce.
//   * softmax against the per-head reference of the first valid block, redone once with the exact
//     maximum if the headroom is overshot, as in the 128-head kernel.
// What binds is the chain of a block (scores, exchange, softmax, PV) against two waves per SIMD,
// then the LDS port (the gather's writes, K and V^T reads).  So both operands of a block are read
// from LDS at its start, before anything depends on them, no wait or branch sits between those
// reads, and the tile is free at the exchange barrier, behind which block j+2 is gathered into it:
// two blocks in flight with two tiles.  Measured (T = 8192 causal, K = 2048, random rows): 16 heads
// 3.70 -> 1.05-1.1 ms (the gather alone takes 0.62, everything but the gather 0.81), 32 heads 3.72
// -> 1.28, 64 heads (two head groups, each gathering its own rows) 3.11 -> 2.6.  Slower: the gather
// through registers in the MFMA operand layout (1.86; its 64-byte pieces do not coalesce), the
// k-split for two head tiles (1.43 against 1.28: a third barrier), four head tiles in one workgroup
// per CU (2.73), the copies spread between the PV MFMAs (no change; spills at two head tiles).
#include "dsa_fh.h"

namespace dsa {

namespace {

constexpr int kDqk = 576;
constexpr int kDv = 512;
constexpr float kHeadroom = 64.0f;      // log2 headroom above the reference max
template <int NHT>
struct FhSmem {
  union {
    char tile[2][kTileBytes];
    char ostage[16 * NHT][kDv * 2];   // epilogue: bf16 output rows, chunk c of row r at c ^ (r & 7)
  };
  u32x4 xbuf[4][64];                  // NHT = 1: partial S^T of wave w; NHT = 2: P^T fragments of head tile n
  int32_t idx[kFhIdxSlots][64];
  float m[16 * NHT], l[2][16 * NHT], seen[2][16 * NHT], inv_l[16 * NHT];
  int red[kFhWaves];
};

}  // namespace

template <int NHT, bool ROPE>
__global__ __launch_bounds__(256, 2) void sparse_mla_fwd_fh_kernel(SparseFwdParams p) {
  constexpr int QKS = (ROPE ? kDqk : kDv) / 32;      // 32-deep k-steps of the scores
  constexpr int KS = NHT == 1 ? QKS / 2 : QKS;       // k-steps of a wave
  constexpr int KA = QKS / 2;                        // K fragments in registers
  constexpr int DT = 8;                              // 16-dim tiles of a wave's O^T
  static_assert(sizeof(FhSmem<NHT>) <= 80 * 1024, "two workgroups per CU");
  __shared__ __attribute__((aligned(128))) FhSmem<NHT> sm;

  const int item = xcd_remap(blockIdx.x, p.n_xcd);
  if (item >= p.total_q * p.n_split) return;
  const int t = item / p.n_split;
  const int split = item - t * p.n_split;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = lane >> 4, gi = lane & 15;
  const int kt = wave & 1, wh = wave >> 1;           // key tile; k half (NHT = 1) or head tile (NHT = 2)
  const int nt = NHT == 1 ? 0 : wh;                  // head tile of the wave's scores
  const int h0 = blockIdx.y * 16 * NHT;              // first head of the workgroup

  // ---- Q fragments (B operand): lane holds q[head 16 nt + gi][32 ks + 8g .. +7]
  u32x4 qf[KS];
  {
    const bool q_rope = p.q_dim != kDv;
    const int head = h0 + 16 * nt + gi;
    const bool ok = head < p.n_heads;
    const bf16_t* qrow = p.q + (int64_t)t * p.q_stride_t + (int64_t)(ok ? head : 0) * (q_rope ? kDqk : kDv) + 8 * g;
#pragma unroll
    for (int i = 0; i < KS; ++i) {
      const int ks = NHT == 1 ? KS * wh + i : i;
      u32x4 v = u32x4{0, 0, 0, 0};
      if (ks < kDv / 32 || q_rope) v = gload16(qrow + 32 * ks);
      qf[i] = ok ? v : u32x4{0, 0, 0, 0};
    }
  }
  // ---- index row: blocks up to the last valid slot
  const int k_first = split * p.split_keys;
  FhGather<ROPE> gth;
  gth.kv = p.kv;
  gth.idx_row = p.idx + (int64_t)t * p.idx_stride + k_first;
  gth.slots = sm.idx;
  gth.n_slots = max(0, min(p.topk - k_first, p.split_keys));
  gth.lane = lane;
  gth.wave = wave;
  gth.lim = p.causal ? min(p.n_kv, t + 1) : p.n_kv;
  const int nblk = gth.setup(sm.red);

  // score operand (A): key 16 kt + gi, chunk 4 ks + g.  NHT = 1, upper k half: the last two k-steps
  // lie in the rope region.
  const int skey = 16 * kt + gi;
  const uint32_t s_v = fh_row(skey) * kTileVPitch + 16u * g + (NHT == 1 ? 64u * KS * wh : 0u);
  const uint32_t s_r = kTileVBytes + skey * 128u + 16u * ((uint32_t)g ^ ((skey >> 1) & 7u));
  // V^T operand (A): lane feeds keys 4g + gi/4 (+16), dims 128 w + 16 D + 4 (gi % 4)
  const uint32_t pv_lo = fh_row(4 * g + (gi >> 2)) * kTileVPitch + 8u * (gi & 3) + 256u * wave;
  const uint32_t pv_hi = pv_lo + 16u * kTileVPitch;   // fh_row(k + 16) = fh_row(k) + 16
  const uint32_t tile0 = lds_addr(sm.tile[0]);

  auto max4 = [](const f32x4& x) { return fmaxf(fmaxf(x[0], x[1]), fmaxf(x[2], x[3])); };
  auto over_g = [](float v) {   // maximum over the four lane groups of a head
    v = fmaxf(v, __shfl_xor(v, 16, 64));
    return fmaxf(v, __shfl_xor(v, 32, 64));
  };
  auto expo = [&](const f32x4& x, float m, float& sum) {
    float e[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      e[i] = fast_exp2(__builtin_fmaf(x[i], p.scale_log2, -m));
      sum += e[i];
    }
    return u32x2{pack_bf16x2(e[0], e[1]), pack_bf16x2(e[2], e[3])};
  };

  f32x4 o[DT][NHT];
  float m_ref = -INFINITY, m_seen = -INFINITY, l_run = 0.f;
  bool m_set = false;
  for (int pass = 0; pass < 2; ++pass) {
#pragma unroll
    for (int d = 0; d < DT; ++d)
#pragma unroll
      for (int n = 0; n < NHT; ++n) o[d][n] = f32x4{0.f, 0.f, 0.f, 0.f};
    l_run = 0.f;
    if (pass == 1) gth.restart();
    gth.start(tile0, nblk);
    for (int blk = 0; blk < nblk; ++blk) {
      gth.template wait<0>(blk, nblk);
      __syncthreads();
      const uint32_t tb = tile0 + (blk & 1) * kTileBytes;
      uint32_t av = tb + s_v, ar = tb + s_r, lo = tb + pv_lo, hi = tb + pv_hi;
      asm volatile("" : "+v"(av), "+v"(ar), "+v"(lo), "+v"(hi));
      auto k_read = [&](int i) {
        uint32_t a = av + 64u * i;
        if constexpr (ROPE) {
          if (NHT == 1) {
            if (i >= KS - 2) a = wh ? ar ^ (64u * (i - (KS - 2))) : a;
          } else if (i >= kDv / 32) {
            a = ar ^ (64u * (i - kDv / 32));
          }
        }
        return lds_load16(lds_ptr(a));
      };
      const uint32_t xm = gth.entry(blk, lane & 31);
      const uint32_t xv = gth.entry(blk + 2, gth.key_v()), xr = gth.entry(blk + 2, gth.key_r());
      u32x4 ka[KA];
#pragma unroll
      for (int i = 0; i < KA; ++i) ka[i] = k_read(i);
      u32x4 va[DT];
#pragma unroll
      for (int d = 0; d < DT; ++d) {
        const u32x2 a = fh_read_tr16(lo + 32u * d), b = fh_read_tr16(hi + 32u * d);
        va[d] = u32x4{a[0], a[1], b[0], b[1]};
      }
      const uint32_t vmask = (uint32_t)__ballot(gth.ok(xm, blk, lane & 31));
      const bool more = blk + 2 < nblk;
      const TileSrc<kFhWaves> src = gth.sources(blk + 2, xv, xr);

      // ---- S^T = K . Q^T
      f32x4 s = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < KS; ++i) {
        const bf16x8 k = as_bf16x8(ka[i % KA]);
        if (i + KA < KS) ka[i % KA] = k_read(i + KA);
        s = mfma16x16x32(k, as_bf16x8(qf[i]), s);
      }

      // ---- P^T fragments of every head tile: lane holds keys {4g + e, 16 + 4g + e} of head gi
      u32x4 pf[NHT];
      auto mask4 = [&](f32x4& x, int key0) {
        const uint32_t ok = vmask >> key0;
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] = (ok >> e) & 1u ? x[e] : -INFINITY;
      };
      auto gather_next = [&]() {   // the tile is read by nobody any more
        if (more) {
          gth.copy_slice(blk + 4);
          gth.issue(tb, src);
        }
      };
      if constexpr (NHT == 1) {
        lds_store16(&sm.xbuf[wave][lane], __builtin_bit_cast(u32x4, s));
        __syncthreads();
        f32x4 x[2], y[2];
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          x[k] = __builtin_bit_cast(f32x4, lds_load16(&sm.xbuf[k][lane]));
          y[k] = __builtin_bit_cast(f32x4, lds_load16(&sm.xbuf[k + 2][lane]));
        }
        gather_next();
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          x[k] += y[k];
          if (vmask != 0xffffffffu) mask4(x[k], 16 * k + 4 * g);
        }
        const float bm = fmaxf(max4(x[0]), max4(x[1])) * p.scale_log2;
        if (!m_set && vmask != 0u) {
          m_ref = over_g(bm);
          m_set = true;
        }
        m_seen = fmaxf(m_seen, bm);
        const float mu = m_set ? m_ref : 0.f;
        const u32x2 lo2 = expo(x[0], mu, l_run), hi2 = expo(x[1], mu, l_run);
        pf[0] = u32x4{lo2[0], lo2[1], hi2[0], hi2[1]};
      } else {
        if (vmask != 0xffffffffu) mask4(s, 16 * kt + 4 * g);
        if (!m_set && vmask != 0u) {   // the two key tiles' waves agree on the reference (once)
          sm.seen[kt][16 * nt + gi] = over_g(max4(s)) * p.scale_log2;
          __syncthreads();
          m_ref = fmaxf(sm.seen[0][16 * nt + gi], sm.seen[1][16 * nt + gi]);
          m_set = true;
        }
        m_seen = fmaxf(m_seen, max4(s) * p.scale_log2);
        *reinterpret_cast<u32x2*>(reinterpret_cast<char*>(&sm.xbuf[nt][lane]) + 8 * kt) =
            expo(s, m_set ? m_ref : 0.f, l_run);
        __syncthreads();
#pragma unroll
        for (int n = 0; n < NHT; ++n) pf[n] = lds_load16(&sm.xbuf[n][lane]);
        gather_next();
      }

      // ---- O^T += V^T . P^T
#pragma unroll
      for (int d = 0; d < DT; ++d)
#pragma unroll
        for (int n = 0; n < NHT; ++n) o[d][n] = mfma16x16x32(as_bf16x8(va[d]), as_bf16x8(pf[n]), o[d][n]);
    }
    // ---- did any head overshoot its reference?
    __syncthreads();
    if (NHT > 1 || wave == 0) {
      float l = l_run + __shfl_xor(l_run, 16, 64);
      l += __shfl_xor(l, 32, 64);
      const float seen = over_g(m_seen);
      const int h = 16 * nt + gi;
      sm.seen[kt][h] = seen;
      sm.l[kt][h] = l;
      if (NHT == 1) {
        sm.seen[1][h] = seen;
        sm.l[1][h] = 0.f;
      }
      sm.m[h] = m_ref;
    }
    __syncthreads();
    const int h = lane & (16 * NHT - 1);
    const bool over = fmaxf(sm.seen[0][h], sm.seen[1][h]) > sm.m[h] + kHeadroom;
    if (!__any(over)) break;
    m_ref = fmaxf(sm.seen[0][16 * nt + gi], sm.seen[1][16 * nt + gi]);
  }
  // ---- per-head normaliser and LSE, with the attention sink as in sparse_mla_fwd_kernel
  if (threadIdx.x < 16 * NHT) {
    const int h = threadIdx.x, head = h0 + h;
    const bool head_ok = head < p.n_heads;
    const float l = sm.l[0][h] + sm.l[1][h];
    const float ms = m_set ? sm.m[h] : -INFINITY;
    float o_scale = l > 0.f ? 1.f / l : 0.f;
    float lse = -INFINITY;
    if (p.sinks != nullptr) {
      const float s2 = head_ok ? p.sinks[head] * kLog2e : -INFINITY;
      const float mf = fmaxf(ms, s2);
      if (mf != -INFINITY) {
        const float rel = ms == -INFINITY ? 0.f : fast_exp2(ms - mf);
        const float l_tot = l * rel + fast_exp2(s2 - mf);
        o_scale = rel / l_tot;
        lse = (mf + __log2f(l_tot)) * kLn2;
      }
    } else if (l > 0.f) {
      lse = ((ms == -INFINITY ? 0.f : ms) + __log2f(l)) * kLn2;
    }
    sm.inv_l[h] = o_scale;
    if (head_ok) p.lse[(int64_t)item * p.lse_stride_t + head] = lse;
  }
  __syncthreads();
  // ---- output rows through LDS (the tiles are dead), one 1 KB row per store instruction
#pragma unroll
  for (int n = 0; n < NHT; ++n) {
    const float inv = sm.inv_l[16 * n + gi];
    char* row = sm.ostage[16 * n + gi];
#pragma unroll
    for (int d = 0; d < DT; ++d) {
      const int chunk = (16 * wave + 2 * d + (g >> 1)) ^ (gi & 7);
      *reinterpret_cast<u32x2*>(row + 16 * chunk + 8 * (g & 1)) =
          u32x2{pack_bf16x2(o[d][n][0] * inv, o[d][n][1] * inv), pack_bf16x2(o[d][n][2] * inv, o[d][n][3] * inv)};
    }
  }
  __syncthreads();
  bf16_t* obase = p.out + (int64_t)item * p.out_stride_t + (int64_t)h0 * kDv;
  for (int r = wave; r < min(16 * NHT, p.n_heads - h0); r += kFhWaves)
    *reinterpret_cast<u32x4*>(obase + (int64_t)r * kDv + 8 * lane) = lds_load16(sm.ostage[r] + 16 * (lane ^ (r & 7)));
}

// Up to 16 heads: one head tile; up to 64: head groups of two tiles (measured above).
int launch_sparse_mla_fwd_fh(const SparseFwdParams& p, hipStream_t stream) {
  const int nht = p.n_heads <= 16 ? 1 : 2;
  const dim3 grid(xcd_grid(p.total_q * p.n_split, p.n_xcd), (p.n_heads + 16 * nht - 1) / (16 * nht)), block(256);
#define DSA_FH(NHT, ROPE) hipLaunchKernelGGL((sparse_mla_fwd_fh_kernel<NHT, ROPE>), grid, block, 0, stream, p)
  const bool rope = p.q_dim != kDv;   // 512-wide q: no rope part
  if (nht == 1) {
    if (rope) DSA_FH(1, true); else DSA_FH(1, false);
  } else {
    if (rope) DSA_FH(2, true); else DSA_FH(2, false);
  }
#undef DSA_FH
  return hipGetLastError() == hipSuccess ? 0 : -4;
}

}  // namespace dsa
