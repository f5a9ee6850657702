// The gather of the few-head kernels (dsa_sparse_fwd_fh.hip, dsa_sparse_bwd_fh.hip): four waves fill
// 32-key tiles of the layout of dsa_kvtile.h with another row order, from a ring of index slices
// instead of a whole index row in LDS, so that two tiles are all that a workgroup needs.
#pragma once
#include "dsa_common.h"
#include "dsa_kernels.h"
#include "dsa_kvtile.h"

namespace dsa {

constexpr int kFhWaves = 4;
constexpr int kFhIdxSlots = 4;   // ring of index slices (block b's 32 entries at b % 4; a copy writes 64)

// V row of block key k: keys 8j .. 8j+7 sit two rows apart, so that a transposing read of 32 lanes
// (8 keys, 32 bytes each) covers all banks; 16 consecutive keys still cover 16 consecutive rows.
constexpr uint32_t fh_row(uint32_t k) { return (k & 16u) | ((k & 7u) << 1) | ((k >> 3) & 1u); }

typedef short fh_s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) fh_s16x4 fh_lds_s16x4;
DSA_DEV u32x2 fh_read_tr16(uint32_t a) {
  fh_s16x4 r = __builtin_amdgcn_ds_read_tr16_b64_v4i16((fh_lds_s16x4*)(lds_ptr(a)));
  return __builtin_bit_cast(u32x2, r);
}

template <bool ROPE>
struct FhGather {
  static constexpr int kCopies = tile_copies_per_wave<kFhWaves, ROPE>();   // per wave and block
  const bf16_t* kv;
  const int32_t* idx_row;
  int32_t (*slots)[64];
  int n_slots, lane, wave;
  uint32_t lim;   // valid ids: 0 .. lim - 1

  // Last valid slot + 1 in blocks; leaves the first slices in the ring.  `red`: one int per wave.
  // Retires every load in flight (nothing compiler-visible is left).
  DSA_DEV int setup(int* red) {
    int last = -1;
    constexpr int kBatch = 8;   // loads in flight per thread
    for (int j0 = threadIdx.x; j0 < n_slots; j0 += kBatch * 256) {
      int v[kBatch];
#pragma unroll
      for (int i = 0; i < kBatch; ++i) v[i] = j0 + i * 256 < n_slots ? idx_row[j0 + i * 256] : -1;
#pragma unroll
      for (int i = 0; i < kBatch; ++i)
        if ((uint32_t)v[i] < lim) last = j0 + i * 256;
      if (j0 < kFhIdxSlots * kTileKeys) slots[j0 / kTileKeys][j0 % kTileKeys] = v[0];
    }
    last = wave_max_i(last);
    if (lane == 0) red[wave] = last;
    wait_vmcnt0();
    __syncthreads();
#pragma unroll
    for (int w = 0; w < kFhWaves; ++w) last = max(last, red[w]);
    return __builtin_amdgcn_readfirstlane((last + kTileKeys) / kTileKeys);
  }

  // Raw entry of key `key` of block blk, and whether it names a key.  No branch between the reads of
  // the entries and their use: a wait for one would be a wait for every LDS read in flight.
  DSA_DEV uint32_t entry(int blk, int key) const { return (uint32_t)slots[blk % kFhIdxSlots][key]; }
  DSA_DEV bool ok(uint32_t x, int blk, int key) const { return (x < lim) & (blk * kTileKeys + key < n_slots); }

  DSA_DEV int key_v() const { return wave + kFhWaves * (lane & 7); }   // this lane's key of the row copies
  DSA_DEV int key_r() const { return 8 * wave + (lane >> 3); }         // and of the rope copy
  // Gather sources of block blk from its raw entries rv (key_v) and rr (key_r); no key: row 0.
  DSA_DEV TileSrc<kFhWaves> sources(int blk, uint32_t rv, uint32_t rr) const {
    TileSrc<kFhWaves> src;
    const char* base = reinterpret_cast<const char*>(kv);
    src.v = base + (uint64_t)(ok(rv, blk, key_v()) ? rv : 0u) * (kLatent * 2);
    if constexpr (ROPE)
      src.rope[0] = base + (uint64_t)(ok(rr, blk, key_r()) ? rr : 0u) * (kLatent * 2) +
                    (64 + ((lane & 7) ^ ((key_r() >> 1) & 7))) * 16;
    return src;
  }
  // Copies of one block into the tile at LDS address `tile`: keys wave + 4k, then a rope group.
  DSA_DEV void issue(uint32_t tile, const TileSrc<kFhWaves>& src) const {
    const TileDst d = tile_dst<kFhWaves>(tile, wave);   // row fh_row(wave) = 2 wave
    const char* row[2] = {gather_row<kFhWaves>(src, 0), gather_row<kFhWaves>(src, 1)};
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_nop 4");
    static_for<0, kCopies>([&](auto kc) {
      constexpr int k = decltype(kc)::value;
      if constexpr (k < 8) copy_row16_at<fh_row(kFhWaves * k) * kTileVPitch>(d.v, row[k & 1], (uint32_t)lane * 16u);
      else copy16_at<0>(src.rope[0], d.rope);
      row[k & 1] = gather_row<kFhWaves>(src, k + 2);
      __builtin_amdgcn_sched_barrier(0);
    });
  }
  // Index slice of block blk (past the row: its last entry again), by wave 0.
  DSA_DEV void copy_slice(int blk) const {
    if (wave == 0)
      async_copy4_unordered(idx_row + min(blk * kTileKeys + lane, n_slots - 1),
                            __builtin_amdgcn_readfirstlane(lds_addr(slots[blk % kFhIdxSlots])));
  }
  // First slices again (a second pass over the row).
  DSA_DEV void restart() const {
    for (int b = 0; b < kFhIdxSlots; ++b) copy_slice(b);
    wait_vmcnt0();
    __syncthreads();
  }
  // Blocks 0 and 1 into the two tiles.
  DSA_DEV void start(uint32_t tile0, int nblk) const {
    for (int b = 0; b < min(nblk, 2); ++b)
      issue(tile0 + b * kTileBytes, sources(b, entry(b, key_v()), entry(b, key_r())));
  }
  // Block blk's copies done, those of block blk + 1 (issued after them, behind a slice by wave 0 from
  // the loop on, and followed by at least `extra` more vector-memory instructions) left in flight.
  template <int EXTRA>
  DSA_DEV void wait(int blk, int nblk) const {
    if (blk + 1 >= nblk) wait_vmcnt0();
    else if (blk == 0) wait_vmcnt<kCopies>();
    else if (wave == 0) wait_vmcnt<kCopies + EXTRA + 1>();
    else wait_vmcnt<kCopies + EXTRA>();
  }
};

}  // namespace dsa
