// B1 and B2 of the sparse MLA backward in one pass over the gathered rows, for few heads (n_heads <=
// 64): S, dP, P, dS and dQ of a query, P and scale * dS staged for the dKV stages as
// bwd_sp_kernel (dsa_sparse_bwd.hip) stages them.
//
// With 128 heads the working set of both does not fit a CU and B2 gathers every row again; with 16 or
// 32 heads per workgroup Q, dO and the fp32 dQ^T accumulator take 180 / 280 registers of a lane, so
// each row is gathered once and dS reaches the dQ product through registers and 4 KB of LDS
// instead of a staged tile read back.  Structure and gather of the few-head forward
// (dsa_sparse_fwd_fh.hip): four waves share each 32-key tile, every LDS operand of a block is read
// at its start, and the tile is refilled behind the exchange barrier.
//   * NHT = 1 (16 heads): wave (kt, r) multiplies the 16 keys of tile kt by Q (r = 0: S, then P) or
//     by dO (r = 1: dP); P and dP are exchanged in fp32, and every wave forms dS of all 32 keys in
//     the B layout of the dQ product.  Two workgroups per CU.
//   * NHT = 2 (32 heads): wave (kt, r) multiplies the 16 keys by Q and dO of head tile r (each K
//     fragment feeds both), forms P and dS, and exchanges dS in bf16.  One workgroup per CU.
//   * dQ^T += K^T . dS^T: wave w owns 128 latent dims and 16 rope dims for every head.
// Measured against the two kernels it replaces: 8192 tokens in 3 documents, K = 2048 (11.3 M pairs),
// 16 heads 3.10 + 3.43 -> 1.21 ms; 777 tokens, 32 heads, K = 512: 120 + 134 -> 98 us; 3.15 M pairs of
// 64 heads 0.98 + 0.83 -> 1.50 ms.
#include "dsa_fh.h"

namespace dsa {

namespace {

constexpr int kDqk = 576;
constexpr int kDv = 512;
constexpr int kBK = kTileKeys;
constexpr int kDqPitch = kDqk * 2 + 16;   // LDS pitch of a staged bf16 dQ row

template <int NHT>
struct BwdFhSmem {
  union {
    char tile[2][kTileBytes];
    char out[16 * NHT][kDqPitch];   // epilogue: bf16 dQ rows
  };
  u32x4 xbuf[4][64];                // NHT = 1: P (slot kt) and dP (slot 2 + kt), fp32; NHT = 2: dS^T fragments
                                    //   of head tile n (slot n)
  int32_t idx[kFhIdxSlots][64];
  float delta[16];
  int red[kFhWaves];
};

// 4 x 4 transpose of 16-bit values inside each quad of lanes: lane j of a quad holds elements
// 0 .. 3 of row j and receives element j of rows 0 .. 3.
struct QuadTranspose {
  uint32_t keep, send, o0, o1;
  bool upper;
  DSA_DEV explicit QuadTranspose(int lane) {
    // v_perm_b32(r, k, sel): bytes 0-3 of k, 4-7 of r
    constexpr uint32_t lo = 0x05040100u, hi = 0x07060302u, lo_x = 0x01000504u, hi_x = 0x03020706u;
    const int j = lane & 3;
    upper = j & 2;
    keep = (j & 1) ? hi : lo;
    send = (j & 1) ? lo : hi;
    o0 = j == 0 ? lo : j == 1 ? lo_x : j == 2 ? hi : hi_x;
    o1 = j == 0 ? hi : j == 1 ? hi_x : j == 2 ? lo : lo_x;
  }
  DSA_DEV u32x2 operator()(const u32x2& x) const {
    // elements {0, 1} or {2, 3} of rows j and j ^ 2, then the lane's element of all four rows
    const uint32_t mine = upper ? x[1] : x[0], theirs = upper ? x[0] : x[1];
    const uint32_t pair = __builtin_amdgcn_update_dpp(0, theirs, 0x4E, 0xf, 0xf, true);   // lane ^ 2
    const uint32_t k = __builtin_amdgcn_perm(pair, mine, keep);      // rows j, j ^ 2
    const uint32_t s = __builtin_amdgcn_perm(pair, mine, send);
    const uint32_t r = __builtin_amdgcn_update_dpp(0, s, 0xB1, 0xf, 0xf, true);           // lane ^ 1: rows j ^ 1, j ^ 3
    return u32x2{__builtin_amdgcn_perm(r, k, o0), __builtin_amdgcn_perm(r, k, o1)};
  }
};

}  // namespace

template <int NHT, bool ROPE>
__global__ __launch_bounds__(256, NHT == 1 ? 2 : 1) void bwd_spdq_fh_kernel(SparseBwdParams p) {
  constexpr int QKS = (ROPE ? kDqk : kDv) / 32;    // 32-deep k-steps of S
  constexpr int VKS = kDv / 32;                    // and of dP
  constexpr int KA = QKS / 2;                      // K fragments in registers
  constexpr int DT = ROPE ? 9 : 8;                 // 16-dim tiles of a wave's dQ^T (the 9th: rope)
  constexpr int kStores = NHT == 1 ? 1 : 2;        // staging stores of a wave per block
  __shared__ __attribute__((aligned(128))) BwdFhSmem<NHT> sm;
  static_assert(NHT > 1 || sizeof(BwdFhSmem<NHT>) <= 80 * 1024, "two workgroups per CU");

  const int t = xcd_remap(blockIdx.x, p.n_xcd);
  if (t >= p.total_q) return;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = lane >> 4, gi = lane & 15;
  const int kt = wave & 1, wr = wave >> 1;         // key tile; product (NHT = 1) or head tile (NHT = 2)
  const int h0 = blockIdx.y * 16 * NHT;            // first head (n_heads is a multiple of 16)
  const int head = h0 + (NHT == 1 ? 0 : 16 * wr) + gi;
  const bool head_ok = NHT == 1 || head < p.n_heads;   // wave-uniform
  const int hs = head_ok ? head : h0 + gi;

  // ---- Q and dO fragments (B operand): lane holds row `hs`, dims 32 ks + 8g .. +7; Delta = dO . O
  const bool q_rope = p.q_dim != kDv;
  const bf16_t* qrow = p.q + (int64_t)t * p.q_stride_t + (int64_t)hs * (q_rope ? kDqk : kDv) + 8 * g;
  const bf16_t* drow = p.dout + (int64_t)t * p.dout_stride_t + (int64_t)hs * kDv + 8 * g;
  const bf16_t* orow = p.out + (int64_t)t * p.out_stride_t + (int64_t)hs * kDv + 8 * g;
  u32x4 qf[QKS], df[NHT == 1 ? 1 : VKS];           // NHT = 1: qf holds Q or dO
  float delta = 0.f;
  auto dot = [&](const u32x4& a, const u32x4& b) {
#pragma unroll
    for (int e = 0; e < 4; ++e) delta += bf16_lo(a[e]) * bf16_lo(b[e]) + bf16_hi(a[e]) * bf16_hi(b[e]);
  };
  u32x4 of[VKS];
  if (NHT > 1 || wr == 0) {
#pragma unroll
    for (int ks = 0; ks < QKS; ++ks) {
      qf[ks] = u32x4{0, 0, 0, 0};
      if (ks < VKS || q_rope) qf[ks] = gload16(qrow + 32 * ks);
    }
  }
  if (NHT > 1 || wr == 1) {
#pragma unroll
    for (int ks = 0; ks < VKS; ++ks) {
      const u32x4 v = gload16(drow + 32 * ks);
      if constexpr (NHT == 1) qf[ks] = v; else df[ks] = v;
      of[ks] = gload16(orow + 32 * ks);
    }
  }
  const float lse = p.lse[(int64_t)t * p.lse_stride_t + hs];
  FhGather<ROPE> gth;
  gth.kv = p.kv;
  gth.idx_row = p.idx + (int64_t)t * p.idx_stride;
  gth.slots = sm.idx;
  gth.n_slots = p.topk;
  gth.lane = lane;
  gth.wave = wave;
  gth.lim = p.causal ? min(p.n_kv, t + p.q_offset + 1) : p.n_kv;
  const int nblk = gth.setup(sm.red);
  const uint32_t tile0 = lds_addr(sm.tile[0]);
  gth.start(tile0, nblk);
  if (NHT > 1 || wr == 1) {
#pragma unroll
    for (int ks = 0; ks < VKS; ++ks) {
      if constexpr (NHT == 1) dot(qf[ks], of[ks]); else dot(df[ks], of[ks]);
    }
    delta += __shfl_xor(delta, 16, 64);
    delta += __shfl_xor(delta, 32, 64);
    if (p.delta_out != nullptr && head_ok && kt == 0 && g == 0) p.delta_out[(int64_t)t * p.n_heads + head] = delta;
  }
  if constexpr (NHT == 1) {
    if (wr == 1 && kt == 0 && g == 0) sm.delta[gi] = delta;
    __syncthreads();
    delta = sm.delta[gi];
  }
  const float delta_s = delta * p.scale, lse2 = lse * kLog2e;
  const bool live = lse != -INFINITY;

  // staged chunks (dsa_common.h): after a 4 x 4 transpose in each lane quad, this lane holds key
  // 16 kt + 4g + lane % 4 of four heads.  NHT = 1: waves 0, 1 store P, waves 2, 3 dS.
  const int64_t st0 = ((int64_t)t * (p.topk_pad / kBK) * (p.n_heads / 16) + (hs >> 4)) * (kStageChunk / 2) +
                      (16 * kt + 4 * g + (lane & 3)) * 16 + (gi & ~3);
  const int64_t st_blk = (int64_t)p.n_heads * kBK;   // elements per block
  const QuadTranspose quad(lane);
  bf16_t* const ps = p.p_stage + st0;
  bf16_t* const ds = p.ds_stage + st0;

  // operand addresses: scores (A): key 16 kt + gi, chunk 4 ks + g; K^T (A): lane feeds keys
  // 4g + gi/4 (+16), dims 128 w + 16 D + 4 (gi % 4) and rope dims 16 w + 4 (gi % 4)
  const int skey = 16 * kt + gi, tkey = 4 * g + (gi >> 2);
  const uint32_t s_v = fh_row(skey) * kTileVPitch + 16u * g;
  const uint32_t s_r = kTileVBytes + skey * 128u + 16u * ((uint32_t)g ^ ((skey >> 1) & 7u));
  const uint32_t kv_lo = fh_row(tkey) * kTileVPitch + 8u * (gi & 3) + 256u * wave;
  const uint32_t kv_hi = kv_lo + 16u * kTileVPitch;
  // (key + 16 leaves (key >> 1) & 7 as it is)
  const uint32_t kr_lo = kTileVBytes + tkey * 128u + 8u * (gi & 1) +
                         16u * ((uint32_t)(2 * wave + ((gi & 3) >> 1)) ^ ((tkey >> 1) & 7u));
  const uint32_t kr_hi = kr_lo + 16u * 128u;

  f32x4 acc[DT][NHT];
#pragma unroll
  for (int d = 0; d < DT; ++d)
#pragma unroll
    for (int n = 0; n < NHT; ++n) acc[d][n] = f32x4{0.f, 0.f, 0.f, 0.f};

  for (int blk = 0; blk < nblk; ++blk) {
    if (head_ok) gth.template wait<kStores>(blk, nblk);
    else gth.template wait<0>(blk, nblk);
    __syncthreads();
    const uint32_t tb = tile0 + (blk & 1) * kTileBytes;
    uint32_t av = tb + s_v, ar = tb + s_r, lo = tb + kv_lo, hi = tb + kv_hi, rlo = tb + kr_lo, rhi = tb + kr_hi;
    asm volatile("" : "+v"(av), "+v"(ar), "+v"(lo), "+v"(hi), "+v"(rlo), "+v"(rhi));
    auto k_read = [&](int ks) { return lds_load16(lds_ptr(ks < VKS ? av + 64u * ks : ar ^ (64u * (ks - VKS)))); };
    const uint32_t xm = gth.entry(blk, lane & 31);
    const uint32_t xv = gth.entry(blk + 2, gth.key_v()), xr = gth.entry(blk + 2, gth.key_r());
    u32x4 ka[KA];
#pragma unroll
    for (int i = 0; i < KA; ++i) ka[i] = k_read(i);
    u32x4 va[DT];
#pragma unroll
    for (int d = 0; d < DT; ++d) {
      const u32x2 a = fh_read_tr16(d < 8 ? lo + 32u * d : rlo), b = fh_read_tr16(d < 8 ? hi + 32u * d : rhi);
      va[d] = u32x4{a[0], a[1], b[0], b[1]};
    }
    const uint32_t vmask = (uint32_t)__ballot(gth.ok(xm, blk, lane & 31));
    const bool more = blk + 2 < nblk;
    const TileSrc<kFhWaves> src = gth.sources(blk + 2, xv, xr);

    // ---- S^T = K . Q^T and dP^T = V . dO^T
    f32x4 s = f32x4{0.f, 0.f, 0.f, 0.f}, dp = f32x4{0.f, 0.f, 0.f, 0.f};
    if constexpr (NHT == 1) {
#pragma unroll
      for (int i = 0; i < QKS; ++i) {
        const bf16x8 k = as_bf16x8(ka[i % KA]);
        if (i + KA < QKS) ka[i % KA] = k_read(i + KA);
        if (i < VKS || wr == 0) s = mfma16x16x32(k, as_bf16x8(qf[i]), s);
      }
    } else {
#pragma unroll
      for (int i = 0; i < QKS; ++i) {
        const bf16x8 k = as_bf16x8(ka[i % KA]);
        if (i + KA < QKS) ka[i % KA] = k_read(i + KA);
        s = mfma16x16x32(k, as_bf16x8(qf[i]), s);
        if (i < VKS) dp = mfma16x16x32(k, as_bf16x8(df[i]), dp);
      }
    }
    // P = 2^(scale_log2 * s - lse2) of keys 16 kt + 4g + e, scale * dS = P * (scale * dP - scale * Delta)
    auto prob = [&](const f32x4& x) {
      const uint32_t ok = live ? vmask >> (16 * kt + 4 * g) : 0u;
      f32x4 r;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float v = fast_exp2(__builtin_fmaf(x[e], p.scale_log2, -lse2));
        r[e] = (ok >> e) & 1u ? v : 0.f;
      }
      return r;
    };
    auto dscore = [&](const f32x4& pr, const f32x4& d) {
      f32x4 r;
#pragma unroll
      for (int e = 0; e < 4; ++e) r[e] = pr[e] * __builtin_fmaf(d[e], p.scale, -delta_s);
      return r;
    };
    auto pack4 = [](const f32x4& x) { return u32x2{pack_bf16x2(x[0], x[1]), pack_bf16x2(x[2], x[3])}; };
    auto refill = [&]() {   // the tile is read by nobody any more
      if (more) {
        gth.copy_slice(blk + 4);
        gth.issue(tb, src);
      }
    };
    u32x4 bf[NHT];   // dS^T fragments: lane holds keys {4g + e, 16 + 4g + e} of head gi
    if constexpr (NHT == 1) {
      if (wr == 0) s = prob(s);
      lds_store16(&sm.xbuf[wave][lane], __builtin_bit_cast(u32x4, s));   // slot kt + 2 wr
      __syncthreads();
      f32x4 pr[2], d[2];
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        pr[k] = __builtin_bit_cast(f32x4, lds_load16(&sm.xbuf[k][lane]));
        d[k] = __builtin_bit_cast(f32x4, lds_load16(&sm.xbuf[2 + k][lane]));
      }
      refill();
      const u32x2 x0 = pack4(dscore(pr[0], d[0])), x1 = pack4(dscore(pr[1], d[1]));
      bf[0] = u32x4{x0[0], x0[1], x1[0], x1[1]};
      bf16_t* const dst = (wr ? ds : ps) + blk * st_blk;
      *reinterpret_cast<u32x2*>(dst) = quad(wr ? (kt ? x1 : x0) : pack4(s));
    } else {
      const f32x4 pr = prob(s);
      const u32x2 x = pack4(dscore(pr, dp));
      *reinterpret_cast<u32x2*>(reinterpret_cast<char*>(&sm.xbuf[wr][lane]) + 8 * kt) = x;
      __syncthreads();
#pragma unroll
      for (int n = 0; n < NHT; ++n) bf[n] = lds_load16(&sm.xbuf[n][lane]);
      refill();
      if (head_ok) {
        *reinterpret_cast<u32x2*>(ps + blk * st_blk) = quad(pack4(pr));
        *reinterpret_cast<u32x2*>(ds + blk * st_blk) = quad(x);
      }
    }
    // ---- dQ^T += K^T . dS^T
#pragma unroll
    for (int d = 0; d < DT; ++d)
#pragma unroll
      for (int n = 0; n < NHT; ++n) acc[d][n] = mfma16x16x32(as_bf16x8(va[d]), as_bf16x8(bf[n]), acc[d][n]);
  }

  // ---- dQ rows through LDS (the tiles are dead), then coalesced 16-byte stores.  Lane holds head
  // 16 n + gi, dims 128 w + 16 d + 4g .. +3 (d = 8: 512 + 16 w + 4g ..)
  __syncthreads();
#pragma unroll
  for (int n = 0; n < NHT; ++n) {
    char* row = sm.out[16 * n + gi];
#pragma unroll
    for (int d = 0; d < DT; ++d) {
      const int dim = d < 8 ? 128 * wave + 16 * d + 4 * g : kDv + 16 * wave + 4 * g;
      *reinterpret_cast<u32x2*>(row + 2 * dim) =
          u32x2{pack_bf16x2(acc[d][n][0], acc[d][n][1]), pack_bf16x2(acc[d][n][2], acc[d][n][3])};
    }
  }
  __syncthreads();
  const int rows = min(16 * NHT, p.n_heads - h0);
  const int qc = (q_rope ? kDqk : kDv) / 8;   // 16-byte chunks of a dq row
  bf16_t* dq_t = p.dq + (int64_t)t * p.dq_stride_t + (int64_t)h0 * (8 * qc);
  for (int c = threadIdx.x; c < rows * qc; c += 256) {
    const int r = c / qc, q = c - r * qc;
    *reinterpret_cast<u32x4*>(dq_t + (int64_t)r * (8 * qc) + 8 * q) = lds_load16(sm.out[r] + 16 * q);
  }
}

// Up to 16 heads: one head tile; up to 64: head groups of two tiles.
void launch_bwd_spdq_fh(const SparseBwdParams& p, hipStream_t stream) {
  const int nht = p.n_heads <= 16 ? 1 : 2;
  const dim3 grid(xcd_grid(p.total_q, p.n_xcd), (p.n_heads + 16 * nht - 1) / (16 * nht)), block(256);
#define DSA_FH(NHT, ROPE) hipLaunchKernelGGL((bwd_spdq_fh_kernel<NHT, ROPE>), grid, block, 0, stream, p)
  const bool rope = p.q_dim != kDv;   // 512-wide q: no rope part
  if (nht == 1) {
    if (rope) DSA_FH(1, true); else DSA_FH(1, false);
  } else {
    if (rope) DSA_FH(2, true); else DSA_FH(2, false);
  }
#undef DSA_FH
}

}  // namespace dsa
