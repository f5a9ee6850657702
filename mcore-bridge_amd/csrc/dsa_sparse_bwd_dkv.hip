// dKV of the sparse MLA backward by key tiles, without per-pair rows (the alternative to B3 + B4 + B5 of
// dsa_sparse_bwd.hip where a query selects a good part of the keys it sees).
//
// B3 writes a 1152-byte row per selected (query, key) pair and B5 reads it back: at few heads that is
// nearly all of the backward (16 heads: 35 KFLOP per row of 1152 bytes out and in).  Here a workgroup
// keeps dKV of 128 keys in registers (128 x 576 fp32, 288 registers of a lane) and walks the queries
// that select any of them; per query and group of 16 heads
//   dKV[128 x 576] += dS^T[128 x 16] . Q[16 x 576],  dKV[128 x 512] += P^T[128 x 16] . dO[16 x 512]
// with the staged P / dS chunks gathered by key through an inverse index (a key that the query did not
// select reads zeros).  The matrix work is that of every (query, key tile) pair that meets, 128 keys
// wide, so it pays by the share of visible keys that are selected; no pair rows, no pair order, and
// the sums stay in fp32 (B3 rounds every pair's row to bf16).
//   dkv_inverse_kernel   per query: slot of every key of the tiles it selects from
//   dkv_tile_kernel      work item (key tile, split of the queries): partial dKV of the tile
//   dkv_sum_kernel       per key: the splits' partials in split order (deterministic)
// A step (query, 16 heads) of one CU takes 1.45 us for 1152 cycles of MFMAs per wave; what bounds it is
// the chain of a wave alone on its SIMD: barrier, transposed reads, MFMAs (without the copies 7 % less
// time, without the MFMAs 18 %; copies ordered further ahead, or code without branches: the same).
// Whole backward, T = 8192, K = 2048, 16 heads: 8840 us by rows, 2839 by tiles; 64 heads 12900, 10820.
// A split is every S-th chunk of 16 queries, all splits of an XCD walking theirs from the last query
// down: the workgroups of an XCD then stream the same Q / dO rows through its L2, and under the causal
// mask the tiles with most queries start first.
#include "dsa_bwd_g.h"
#include "dsa_common.h"
#include "dsa_kernels.h"

namespace dsa {

namespace {

constexpr int kKeys = kDkvKeys;                    // 128 keys per tile
constexpr int kWaves = 4;
constexpr int kInvPass = 16384;                    // keys per LDS pass of the inverse
constexpr uint32_t kNone = 0xffffffffu;
constexpr int kQPart = 16 * kDqk * 2;              // Q rows of 16 heads
constexpr int kOPart = 16 * kDv * 2;               // dO rows
constexpr int kSPart = 4 * kStageChunk;            // dS (or P) of 128 keys x 16 heads
constexpr int kStepBytes = kQPart + kOPart + 2 * kSPart;
constexpr int kRing = 3;
constexpr int kInvSlots = 8;
constexpr int kListLen = 2048;                     // queries of a segment
constexpr int kSumThreads = 192;

struct DkvSmem {
  char ring[kRing][kStepBytes];   // Q | dO (16-byte chunk c of row r at c ^ 2 (r & 3)) | dS | P (stage_unit)
  uint16_t inv[kInvSlots][kKeys]; // inverse rows of the queries in flight
  uint32_t list[kListLen];        // query | key-subtile mask << 28, last query first
  int scan[kWaves];
};
static_assert(sizeof(DkvSmem) <= 160 * 1024, "LDS budget");

}  // namespace

// One workgroup per query: scatter the row's slots into an LDS table of the keys, then write the
// inverse rows of the tiles that hold any (tile-major, 128 slots each, 0xffff = not selected) and
// every tile's flag byte: bits 0-3 the 32-key subtiles that hold a key, bit 7 a key that the row
// repeats (the table keeps one of its slots; dkv_sum_kernel adds the others).
__global__ __launch_bounds__(256) void dkv_inverse_kernel(SparseBwdParams p, DkvParams d) {
  extern __shared__ uint32_t tab[];
  __shared__ int dup[kInvPass / kKeys];
  const int t = blockIdx.x;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int32_t* row = p.idx + (int64_t)t * p.idx_stride;
  const int lim = p.causal ? min(p.n_kv, t + p.q_offset + 1) : p.n_kv;
  for (int k0 = 0; k0 < d.n_tiles * kKeys; k0 += kInvPass) {
    const int nt = min(kInvPass / kKeys, d.n_tiles - k0 / kKeys);             // tiles of this pass
    const int live = max(0, min(nt, (lim - k0 + kKeys - 1) / kKeys));         // tiles a key can lie in
    for (int k = threadIdx.x; k < live * kKeys; k += 256) tab[k] = kNone;
    for (int k = threadIdx.x; k < live; k += 256) dup[k] = 0;
    __syncthreads();
    if (live > 0)
      for (int j = threadIdx.x; j < p.topk; j += 256) {
        const int v = row[j];
        if (v >= k0 && v < lim && v - k0 < live * kKeys)
          if (atomicExch(&tab[v - k0], (uint32_t)j) != kNone) dup[(v - k0) / kKeys] = 1;
      }
    __syncthreads();
    for (int i = wave; i < live; i += kWaves) {
      const uint32_t a = tab[i * kKeys + 2 * lane], b = tab[i * kKeys + 2 * lane + 1];
      const uint64_t m = __ballot(a != kNone || b != kNone);
      const int64_t at = (int64_t)(k0 / kKeys + i) * p.total_q + t;
      if (m) reinterpret_cast<uint32_t*>(d.inv)[at * (kKeys / 2) + lane] = (a & 0xffffu) | b << 16;
      if (lane == 0) {
        int f = dup[i] ? 128 : 0;
#pragma unroll
        for (int s = 0; s < 4; ++s) f |= ((m >> (16 * s)) & 0xffffu) ? 1 << s : 0;
        d.flags[at] = (uint8_t)f;
      }
    }
    for (int i = live + threadIdx.x; i < nt; i += 256) d.flags[(int64_t)(k0 / kKeys + i) * p.total_q + t] = 0;
    __syncthreads();   // the next pass clears the table
  }
}

// Wave w owns dims 128 w .. +127 (and rope dims 32 w .. +31 for w < 2) of all 128 keys: the latent
// accumulators (16 tiles) pinned in AccVGPRs, the rope ones in VGPRs.  Per step (query, head group)
// it reads 9 transposed fragments of Q / dO and the 8 fragments of dS and P, for 36 (32) MFMAs.
// Copies of step s + 2 are issued under step s's MFMAs.
template <bool ROPE>
__global__ __launch_bounds__(256, 1) void dkv_tile_kernel(SparseBwdParams p, DkvParams d) {
  __shared__ __attribute__((aligned(128))) DkvSmem sm;
  const int tile = blockIdx.x / d.n_split, split = blockIdx.x - tile * d.n_split;
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int hb = lane >> 5, g = lane >> 4, gi = lane & 15;
  const int nhg = p.n_heads / 16;
  const bool rope_wave = ROPE && w < 2;

  f32x16 acc[4][4], racc[4];   // [dim tile 4w + i][key subtile]; rope dim tile 16 + w
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int k = 0; k < 4; ++k) acc[i][k] = f32x16{};
#pragma unroll
  for (int k = 0; k < 4; ++k) racc[k] = f32x16{};
  mfma_acc_drain();

  // copies of a step by this wave: 1 KB pieces j = 4 i + w of Q (j < QJ) then dO, at these offsets
  // from the head group's rows; then dS and P of key subtile w
  constexpr int QJ = ROPE ? kQPart / 1024 : 16, NJ = QJ + kOPart / 1024;
  constexpr int NI = (NJ + kWaves - 1) / kWaves;
  constexpr int QROW = ROPE ? kDqk * 2 : kDv * 2;   // bytes of a q row
  uint32_t off[NI];
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int j = kWaves * i + w;
    if (j < QJ) {
      const int c = j * 64 + lane, r = c / (QROW / 16), slot = c - r * (QROW / 16);
      off[i] = r * QROW + 16 * (slot ^ (2 * (r & 3)));
    } else {
      const int r = j - QJ;
      off[i] = r * (kDv * 2) + 16 * (lane ^ (2 * (r & 3)));
    }
  }
  const uint32_t sk = 32 * w + stage_unit_key(lane), sc = 16 * stage_unit_half(lane);
  const uint32_t ring0 = lds_addr(sm.ring[0]);
  const int64_t st_row = (int64_t)(p.topk_pad / kBK) * nhg * kStageChunk;   // staged bytes per query
  struct Step {   // step = (list entry e, head group hg)
    int e, hg;
  };
  auto next = [&](Step x) { return x.hg + 1 < nhg ? Step{x.e, x.hg + 1} : Step{x.e + 1, 0}; };
  auto entry = [&](int e) { return __builtin_amdgcn_readfirstlane(sm.list[e]); };
  auto copy_inv = [&](int e) {   // inverse row of list entry e (waves 2 and 3, the same bytes)
    const int t = (int)(entry(e) & 0x0fffffffu);
    async_copy4_unordered(d.inv + ((int64_t)tile * p.total_q + t) * kKeys + 2 * lane,
                          __builtin_amdgcn_readfirstlane(lds_addr(sm.inv[e % kInvSlots])));
  };
  struct Src {
    const char *q, *o, *ds, *ps;
    uint32_t dst;
  };
  auto step_src = [&](Step x, int ring) {
    const int e = x.e, hg = x.hg, t = (int)(entry(e) & 0x0fffffffu);
    Src r;
    r.q = reinterpret_cast<const char*>(p.q + (int64_t)t * p.q_stride_t) + (int64_t)hg * 16 * QROW;
    r.o = reinterpret_cast<const char*>(p.dout + (int64_t)t * p.dout_stride_t) + (int64_t)hg * kOPart;
    const uint32_t slot = sm.inv[e % kInvSlots][sk];
    const int64_t at = (int64_t)t * st_row + ((int64_t)(slot >> 5) * nhg + hg) * kStageChunk + (slot & 31u) * 32u + sc;
    const char* zero = reinterpret_cast<const char*>(kZero16);
    r.ds = slot == 0xffffu ? zero : reinterpret_cast<const char*>(p.ds_stage) + at;
    r.ps = slot == 0xffffu ? zero : reinterpret_cast<const char*>(p.p_stage) + at;
    r.dst = ring0 + (uint32_t)ring * kStepBytes;
    return r;
  };
  auto copy_part = [&](const Src& r, int i) {   // i < NI: Q / dO pieces; NI, NI + 1: dS, P
    if (i < NI) {
      const int j = kWaves * i + w;
      if (j < NJ) copy_row16(r.dst + (j < QJ ? 0 : kQPart - QJ * 1024) + 1024u * j, j < QJ ? r.q : r.o, off[i]);
    } else {
      async_copy16_unordered(i == NI ? r.ds : r.ps, r.dst + kQPart + kOPart + (i - NI) * kSPart + w * kStageChunk);
    }
  };
  // operand addresses inside a step (transposing reads as in bwd_g_kernel: head row tr_h, column tr_c)
  const int tr_h = 8 * (g >> 1) + (gi >> 2), tr_c = 16 * (g & 1) + 4 * (gi & 3), tr_sw = 2 * (gi >> 2);
  auto tr_off = [&](int rp, int mt) {
    const int cb = 64 * mt + 2 * tr_c;
    return (uint32_t)(tr_h * rp + 16 * ((cb >> 4) ^ tr_sw) + (cb & 15));
  };
  uint32_t qo[5], oo[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    qo[i] = tr_off(QROW, 4 * w + i);
    oo[i] = kQPart + tr_off(kDv * 2, 4 * w + i);
  }
  qo[4] = tr_off(QROW, 16 + (w & 1));
  const uint32_t so = kQPart + kOPart + 16 * stage_unit(lane & 31, hb);

  const int n_chunks = (p.total_q + kDkvQChunk - 1) / kDkvQChunk;
  const int my_chunks = split < n_chunks ? (n_chunks - split + d.n_split - 1) / d.n_split : 0;
  const int n_pos = my_chunks * kDkvQChunk;
  bool any = false;
  int dups = 0;
  for (int seg = 0; seg < n_pos; seg += kListLen) {
    // ---- the segment's queries that select from the tile, last query first
    int t8[8], f8[8], cnt = 0;
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int pos = seg + (int)threadIdx.x * 8 + u;
      const int c = split + (my_chunks - 1 - pos / kDkvQChunk) * d.n_split;
      t8[u] = c * kDkvQChunk + kDkvQChunk - 1 - pos % kDkvQChunk;
      f8[u] = pos < n_pos && t8[u] < p.total_q ? d.flags[(int64_t)tile * p.total_q + t8[u]] : 0;
      cnt += (f8[u] & 15) != 0;
      dups |= f8[u] & 128;
    }
    int before = cnt;   // inclusive scan over the wave, then the waves
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int v = __shfl_up(before, o, 64);
      if (lane >= o) before += v;
    }
    if (lane == 63) sm.scan[w] = before;
    wait_vmcnt0();
    __syncthreads();
    int at = before - cnt, total = 0;
#pragma unroll
    for (int i = 0; i < kWaves; ++i) {
      if (i < w) at += sm.scan[i];
      total += sm.scan[i];
    }
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (f8[u] & 15) sm.list[at++] = (uint32_t)t8[u] | (uint32_t)(f8[u] & 15) << 28;
    __syncthreads();
    const int n_list = __builtin_amdgcn_readfirstlane(total), n_steps = n_list * nhg;
    if (n_steps == 0) continue;
    any = true;
    Step cur{0, 0}, ahead{0, 0}, far{0, 0};   // steps s, s + 2, and the query of step s + 4
    for (int i = 0; i < 4; ++i) {
      if (w >= 2) copy_inv(min(far.e, n_list - 1));
      far = next(far);
    }
    wait_vmcnt0();
    __syncthreads();
    for (int s = 0; s < min(2, n_steps); ++s) {
      const Src r = step_src(ahead, s);
      ahead = next(ahead);
#pragma unroll
      for (int i = 0; i < NI + 2; ++i) copy_part(r, i);
    }
    int ring = 0;   // ring slot of step s
    for (int s = 0; s < n_steps; ++s) {
      // step s's copies done; at least 10 of step s + 1's are younger (8 or 9 pieces, dS, P, and an
      // inverse row from waves 2 and 3 after the first)
      if (s + 1 < n_steps) wait_vmcnt<10>();
      else wait_vmcnt0();
      __syncthreads();
      const bool more = s + 2 < n_steps;
      Src nx{};
      if (more) {
        nx = step_src(ahead, ring == 0 ? 2 : ring - 1);   // (s + 2) % 3
        ahead = next(ahead);
        if (w >= 2) copy_inv(min(far.e, n_list - 1));
        far = next(far);
      }
      const uint32_t mask = entry(cur.e) >> 28;
      cur = next(cur);
      const uint32_t base = ring0 + (uint32_t)ring * kStepBytes;
      ring = ring == 2 ? 0 : ring + 1;
      auto tr = [&](uint32_t o, uint32_t rows4) {
        const u32x2 lo = lds_read_tr16(lds_ptr(base + o)), hi = lds_read_tr16(lds_ptr(base + o + rows4));
        return u32x4{lo[0], lo[1], hi[0], hi[1]};
      };
      u32x4 qb[5], ob[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) qb[i] = tr(qo[i], 4 * QROW);
      if (rope_wave) qb[4] = tr(qo[4], 4 * QROW);
#pragma unroll
      for (int i = 0; i < 4; ++i) ob[i] = tr(oo[i], 4 * kDv * 2);
      auto keys = [&](auto kc) {
        constexpr int k = decltype(kc)::value;
        if (more) {   // copies of step s + 2: three or so per key subtile
#pragma unroll
          for (int i = k * (NI + 2) / 4; i < (k + 1) * (NI + 2) / 4; ++i) copy_part(nx, i);
        }
        if (!((mask >> k) & 1u)) return;
        const u32x4 a = lds_load16(lds_ptr(base + so + k * kStageChunk));
        const u32x4 b = lds_load16(lds_ptr(base + so + kSPart + k * kStageChunk));
#pragma unroll
        for (int i = 0; i < 4; ++i) mfma32x32x16_cA(acc[i][k], a, qb[i]);
        if (rope_wave) mfma32x32x16_cV(racc[k], a, qb[4]);
#pragma unroll
        for (int i = 0; i < 4; ++i) mfma32x32x16_cA(acc[i][k], b, ob[i]);
      };
      static_for<0, 4>(keys);
    }
    __syncthreads();   // list and ring free
  }
  mfma_acc_drain();
  // ---- partial tile: rows of 576 floats; lane holds dim lane % 32 of a dim tile, keys (i/4)*8 +
  // 4 hb + i%4 of a key subtile
  dups = __any(dups) ? 2 : 0;
  if (lane == 0) sm.scan[w] = dups;
  __syncthreads();
  if (threadIdx.x == 0)
    d.used[tile * d.n_split + split] = (any ? 1 : 0) | sm.scan[0] | sm.scan[1] | sm.scan[2] | sm.scan[3];
  if (!any) return;
  float* part = d.part + ((int64_t)tile * d.n_split + split) * (kKeys * kDqk);
#pragma unroll
  for (int k = 0; k < 4; ++k)
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      float* row = part + (32 * k + (j >> 2) * 8 + 4 * hb + (j & 3)) * kDqk + (lane & 31);
#pragma unroll
      for (int i = 0; i < 4; ++i) row[32 * (4 * w + i)] = acc[i][k][j];
      if (rope_wave) row[32 * (16 + w)] = racc[k][j];
    }
}

// One workgroup per key: the splits' partials in split order.  Two things the tiles leave to a walk
// over the queries, in query order (neither occurs with indices of a top-k over finite inputs):
//   a row that repeats the key: its slots hold the same P and dS, the table keeps one of them;
//   a sum that is not finite: a key that a query does not select met it as 0 * (its Q or dO), NaN if
//   those are not finite, so the key is summed again over the queries that select it.
__global__ __launch_bounds__(kSumThreads) void dkv_sum_kernel(SparseBwdParams p, DkvParams d) {
  __shared__ int slot_of[kSumThreads];   // slot | 1 << 16 where the row repeats a key of the tile, or -1
  __shared__ int count;
  const int key = blockIdx.x, tile = key / kKeys, kk = key - tile * kKeys;
  const int c = threadIdx.x;   // 4 dims
  const uint8_t* used = d.used + tile * d.n_split;
  const float* part = d.part + (int64_t)tile * d.n_split * (kKeys * kDqk) + (int64_t)kk * kDqk + 4 * c;
  const bool has = c < (p.q_dim == kDv ? kDv : kDqk) / 4;
  f32x4 sum = f32x4{0.f, 0.f, 0.f, 0.f};
  int seen = 0;
#pragma unroll 4
  for (int x = 0; x < d.n_split; ++x) {
    const int u = used[x];
    seen |= u;
    if ((u & 1) && has) sum += __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(part + (int64_t)x * (kKeys * kDqk)));
  }
  bool nonfinite = false;
#pragma unroll
  for (int i = 0; i < 4; ++i) nonfinite |= (__float_as_uint(sum[i]) & 0x7f800000u) == 0x7f800000u;
  const bool again = __syncthreads_or(nonfinite);
  if (again) sum = f32x4{0.f, 0.f, 0.f, 0.f};
  if (again || (seen & 2)) {
    const int nhg = p.n_heads / 16;
    for (int t0 = 0; t0 < p.total_q; t0 += kSumThreads) {
      const int tc = t0 + c;
      int mine = -1;
      if (tc < p.total_q) {
        const int64_t at = (int64_t)tile * p.total_q + tc;
        const int f = d.flags[at];
        if ((f & 128) || (again && (f & 15))) {
          const int held = d.inv[at * kKeys + kk];
          if (held != 0xffff) mine = held | (f & 128 ? 1 << 16 : 0);
        }
      }
      slot_of[c] = mine;
      __syncthreads();
      for (int i = 0; i < min(kSumThreads, p.total_q - t0); ++i) {
        const int so = slot_of[i];
        if (so < 0) continue;
        const int t = t0 + i, j = so & 0xffff;
        int n = again ? 1 : 0;   // times the pair enters
        if (so >> 16) {
          if (c == 0) count = 0;
          __syncthreads();
          const int32_t* row = p.idx + (int64_t)t * p.idx_stride;
          int same = 0;
          for (int x = c; x < p.topk; x += kSumThreads) same += row[x] == key;
          if (same) atomicAdd(&count, same);
          __syncthreads();
          n += count - 1;
          __syncthreads();   // read before the next reset
        }
        if (n == 0 || !has) continue;
        const int64_t st = ((int64_t)t * (p.topk_pad / kBK) + (j >> 5)) * nhg * (kStageChunk / 2) + (j & 31) * 16;
        f32x4 one = f32x4{0.f, 0.f, 0.f, 0.f};
        for (int hg = 0; hg < nhg; ++hg) {
          const bf16_t* ds = p.ds_stage + st + hg * (kStageChunk / 2);
          const bf16_t* ps = p.p_stage + st + hg * (kStageChunk / 2);
          const bf16_t* q = p.q + (int64_t)t * p.q_stride_t + (int64_t)hg * 16 * p.q_dim + 4 * c;
          const bf16_t* o = p.dout + (int64_t)t * p.dout_stride_t + (int64_t)hg * 16 * kDv + 4 * c;
          const bool latent = 4 * c < kDv;
          u32x2 qv[16], ov[16];
#pragma unroll
          for (int h = 0; h < 16; ++h) {
            qv[h] = *reinterpret_cast<const u32x2*>(q + h * p.q_dim);
            ov[h] = latent ? *reinterpret_cast<const u32x2*>(o + h * kDv) : u32x2{0, 0};
          }
#pragma unroll
          for (int h = 0; h < 16; ++h)
#pragma unroll
            for (int x = 0; x < 4; ++x) {
              const uint32_t qx = qv[h][x >> 1], ox = ov[h][x >> 1];
              one[x] += (float)ds[h] * __uint_as_float(x & 1 ? qx & 0xffff0000u : qx << 16);
              if (latent) one[x] += (float)ps[h] * __uint_as_float(x & 1 ? ox & 0xffff0000u : ox << 16);
            }
        }
        sum += (float)n * one;
      }
      __syncthreads();   // slot_of free
    }
  }
  if (c < kDqk / 4) {
    f32x4* out = reinterpret_cast<f32x4*>(p.dkv + (int64_t)key * p.dkv_stride + 4 * c);
    *out = p.dkv_accumulate ? *out + sum : sum;
  }
}

int dkv_tiles(int n_kv) { return (n_kv + kKeys - 1) / kKeys; }

// Splits of the queries, in multiples of the 8 XCDs, of 8 chunks of queries or more: work items (one per
// CU at a time) for about two rounds of the chip.  Their lengths differ under a causal mask, and every
// item costs a partial tile of 295 KB out and in.  Whole backward, 1024 / 512 / 256 items: T = 4096,
// 16 heads, K = 512: 756 / 673 / 934 us; T = 2048, 64 heads, K = 1024: 1258 / 1205 / 1406; equal at
// T = 8192 and above.
int dkv_splits(int total_q, int n_kv) {
  const int tiles = dkv_tiles(n_kv), chunks = (total_q + kDkvQChunk - 1) / kDkvQChunk;
  const int want = (512 + 8 * tiles - 1) / (8 * tiles), most = chunks / 8 > 1 ? chunks / 8 : 1;
  return 8 * (want < most ? want : most);
}

void launch_dkv_inverse(const SparseBwdParams& p, const DkvParams& d, hipStream_t stream) {
  const size_t lds = sizeof(uint32_t) * (size_t)(d.n_tiles * kKeys < kInvPass ? d.n_tiles * kKeys : kInvPass);
  hipLaunchKernelGGL(dkv_inverse_kernel, dim3(p.total_q), dim3(256), lds, stream, p, d);
}

void launch_dkv_tiles(const SparseBwdParams& p, const DkvParams& d, hipStream_t stream) {
  const dim3 grid(d.n_tiles * d.n_split);
  if (p.q_dim == kDv) hipLaunchKernelGGL(dkv_tile_kernel<false>, grid, dim3(256), 0, stream, p, d);
  else hipLaunchKernelGGL(dkv_tile_kernel<true>, grid, dim3(256), 0, stream, p, d);
}

void launch_dkv_sum(const SparseBwdParams& p, const DkvParams& d, hipStream_t stream) {
  hipLaunchKernelGGL(dkv_sum_kernel, dim3(p.n_kv), dim3(kSumThreads), 0, stream, p, d);
}

}  // namespace dsa
