// Prompt chunks over the packed q4/q8 cache at head_dim 128 (more than
// kQSlabMaxHeads virtual heads per KV head; fp16 or bf16 q, scales, biases
// and outputs): the shared-tile kernel of the fp16 cache with its 32-row
// K/V1/V2 tiles dequantised into LDS by the workgroup that attends them.
//
// The decode kernels hold 8 (head, row) pairs per workgroup at group size 64,
// so a 512-row chunk at GQA 4 unpacked every cache row 256 times; here a
// workgroup of NW waves x NCB x 16 virtual heads unpacks it once.  What
// bounds it is what bounds sdpa_prefill_kernel -- the SIMD's MFMA plus VALU
// issue -- and unpacking adds ~14 VALU instructions per thread, tensor and
// tile to it (~50 on ~130).
//   - every thread holds one 8-code chunk per tensor (two at 4 waves) and its
//     scale and bias, loaded one tile ahead of their use: a 16-byte fp16
//     chunk each, written at the swizzled place the tile math reads;
//   - two LDS stages: while tile i is attended, tile i + 1 is dequantised
//     into the other stage and tile i + 2 is in flight; one barrier per tile;
//   - values are s * u + b with one rounding to fp16 (the operand of the
//     matrix cores; scores, sums and partials stay fp32).  They are scaled by
//     a power of two per workgroup and tensor, found from the scales and
//     biases of the rows it reads, so that every finite cache fits fp16:
//     2^-e_K goes into the softmax scale, 2^-e_V into the result.  bf16 rows
//     of q are scaled the same way, per row.
#pragma once

#include "sdpa_qslab.hpp"

namespace motif {

// 8 codes as fp16 s * u + b (one rounding each): two codes become 1024 + u in
// the halves of one word, a packed subtract leaves u exactly, a packed fma
// gives the value.
template <int BITS>
__device__ inline uint4 dequant8_f16(const uint32_t (&w)[BITS / 4], half2_t s2, half2_t b2) {
  const half2_t k1024 = half2_t{(_Float16)1024.f, (_Float16)1024.f};
  uint32_t h[4];
  const uint32_t lo = w[0] & 0x0F0F0F0Fu, hi = (w[0] >> 4) & 0x0F0F0F0Fu;  // q4 nibble planes
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    uint32_t x;
    if constexpr (BITS == 8)
      x = __builtin_amdgcn_perm(0x64646464u, w[i / 2], (i & 1) ? 0x04030402u : 0x04010400u);
    else
      x = __builtin_amdgcn_perm(hi, lo, 0x0C000C00u | ((4u + i) << 16) | (uint32_t)i) | 0x64006400u;
    h[i] = h2_bits(__builtin_elementwise_fma(as_h2(x) - k1024, s2, b2));
  }
  return make_uint4(h[0], h[1], h[2], h[3]);
}

template <int BITS, typename E, int NW, int NCB>
__global__ void __launch_bounds__(NW * 64) __attribute__((amdgpu_waves_per_eu(2, 2)))
sdpa_qprefill_kernel(SdpaArgs a) {
  using Acc = SwizzledTileAcc<half_t>;
  using V8 = Acc::V8;
  constexpr bool kBf16 = std::is_same<E, bf16_t>::value;
  constexpr int D = 128;
  constexpr int TR = kPrefillTileRows;  // 32
  constexpr int RB = D * BITS / 8;      // packed bytes per row
  constexpr int CB = BITS;              // packed bytes per 8-code chunk
  constexpr int CPT = 8 / NW;           // chunks per thread and tensor
  static_assert(NW == 4 || NW == 8, "4 or 8 waves");
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 15;
  const int blk = lane >> 4;

  int qblk, unit, split;
  if (!prefill_block_coords(a, blockIdx.x, qblk, unit, split)) return;  // grid padding
  const int wg_vh0 = qblk * NW * 16 * NCB;
  int vh[NCB], lim[NCB], lim_lo[NCB];
  bool col_ok[NCB];
#pragma unroll
  for (int cb = 0; cb < NCB; ++cb) {
    const int v0 = wg_vh0 + (wave * NCB + cb) * 16;
    vh[cb] = v0 + col;
    col_ok[cb] = vh[cb] < a.GV;
    lim[cb] = col_ok[cb] ? vhead_limit(a, vh[cb]) : 0;
    lim_lo[cb] = qslab_block_limit_lo(a, v0);
  }
  const int r_end = max(vhead_limit_max(a, wg_vh0, min(NW * 16 * NCB, a.GV - wg_vh0)), 0);
  // The visible rows [0, r_end) in 32-row tiles, dealt to the splits round
  // robin (every split of a block gets the same count, +-1).
  const int ns = a.nsplit;
  const int n_vis = (r_end + TR - 1) / TR;
  const int ntiles = n_vis > split ? (n_vis - split + ns - 1) / ns : 0;
  const long qrow0 = (long)unit * a.GV;

  // Rows [0, r_end) through range-checked resources (past the end: zeros).
  const int lg = a.group_size == 128 ? 0 : a.group_size == 64 ? 1 : 2;  // log2(groups per row)
  const long hrow0 = (long)unit * a.kv_cap;
  const unsigned dbytes = (unsigned)r_end * RB;
  const unsigned sbytes = (unsigned)r_end << (lg + 1);
  auto head_scales = [&](const void* p) { return (const uint16_t*)p + (hrow0 << lg); };
  const __amdgpu_buffer_rsrc_t rd[3] = {
      uniform_stream_rsrc((const uint8_t*)a.kd + hrow0 * RB, dbytes),
      uniform_stream_rsrc((const uint8_t*)a.v1d + hrow0 * RB, dbytes),
      uniform_stream_rsrc((const uint8_t*)a.v2d + hrow0 * RB, dbytes)};
  const __amdgpu_buffer_rsrc_t rsc[3] = {uniform_stream_rsrc(head_scales(a.ks), sbytes),
                                         uniform_stream_rsrc(head_scales(a.v1s), sbytes),
                                         uniform_stream_rsrc(head_scales(a.v2s), sbytes)};
  const __amdgpu_buffer_rsrc_t rbi[3] = {uniform_stream_rsrc(head_scales(a.kb), sbytes),
                                         uniform_stream_rsrc(head_scales(a.v1b), sbytes),
                                         uniform_stream_rsrc(head_scales(a.v2b), sbytes)};

  // Chunk k of a thread: row tid / 16 + (TR / CPT) k of the tile, codes 8 c ..
  // 8 c + 7 with c = tid % 16; 16 lanes cover a row.
  const int crow = tid >> 4;
  const int cchunk = tid & 15;
  const int cgroup = (8 * cchunk) >> (7 - lg);
  struct Packed {
    uint32_t w[3][CPT][CB / 4];
    uint32_t s[3][CPT], b[3][CPT];
  };
  auto load = [&](Packed& P, int i) {  // tile i of this split (past the last: zeros)
    const unsigned row0 = (unsigned)((i * ns + split) * TR + crow);
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      const unsigned row = row0 + (unsigned)(TR / CPT * k);
      const unsigned off = row * RB + (unsigned)(cchunk * CB);
      const unsigned soff = ((row << lg) + (unsigned)cgroup) * 2u;
#pragma unroll
      for (int t = 0; t < 3; ++t) {
        if constexpr (CB == 8) {
          const uint2 x = bload2(rd[t], off);
          P.w[t][k][0] = x.x;
          P.w[t][k][1] = x.y;
        } else {
          P.w[t][k][0] = bload1(rd[t], off);
        }
        P.s[t][k] = __builtin_amdgcn_raw_buffer_load_b16(rsc[t], soff, 0, 0);
        P.b[t][k] = __builtin_amdgcn_raw_buffer_load_b16(rbi[t], soff, 0, 0);
      }
    }
  };
  Packed P;
  load(P, 0);

  // Powers of two of K, V1 and V2 from the scales and biases of this split's
  // rows.
  // Stage st, tensor t: 32 rows x 256 bytes, 16-byte chunk c of row r at byte
  // r * 256 + (c ^ (r % 16)) * 16; the split partials are staged there at the end.
  constexpr int TB = TR * D * 2;
  constexpr int LDS_BYTES = 6 * TB > NW * kStageWaveBytes ? 6 * TB : NW * kStageWaveBytes;
  __shared__ __attribute__((aligned(16))) uint8_t ring[LDS_BYTES];
  __shared__ float wmax[3][NW];
  int ex[3];
  {
    float m[3];
    scan_scales<E>(a, hrow0, lg, split * TR, ns * TR, ntiles, r_end, tid, NW * 64, m);
#pragma unroll
    for (int t = 0; t < 3; ++t) {
      const float x = group_max<64>(m[t]);
      if (lane == 0) wmax[t][wave] = x;
    }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < 3; ++t) {
      float x = wmax[t][0];
#pragma unroll
      for (int w = 1; w < NW; ++w) x = fmaxf(x, wmax[t][w]);
      ex[t] = __builtin_amdgcn_readfirstlane(value_exp<E>(x));
    }
  }

  // Q^T, B operand: lane (col, blk) holds its column's channels 32*s + 8*blk
  // .. +7 for k-step s; bf16 rows times 2^-e, e per row, as fp16.
  V8 qb[NCB][4];
  float qsc[NCB];
#pragma unroll
  for (int cb = 0; cb < NCB; ++cb) {
    const uint16_t* qp =
        (const uint16_t*)a.q + (qrow0 + (col_ok[cb] ? vh[cb] : 0)) * D + 8 * blk;
    uint4 w[4];
#pragma unroll
    for (int s = 0; s < 4; ++s)
      w[s] = col_ok[cb] ? *reinterpret_cast<const uint4*>(qp + 32 * s) : make_uint4(0, 0, 0, 0);
    int qe = 0;
    if constexpr (kBf16) qe = q_row_f16(w);
#pragma unroll
    for (int s = 0; s < 4; ++s) qb[cb][s] = __builtin_bit_cast(V8, w[s]);
    qsc[cb] = scaled_qscale(a.qscale, ex[0] + qe);
  }

  half2_t h2[3];
#pragma unroll
  for (int t = 0; t < 3; ++t) {
    const _Float16 v = (_Float16)ldexpf(1.f, -max(ex[t], 0));  // fp16 rows only: e <= 11
    h2[t] = half2_t{v, v};
  }
  auto dequant_store = [&](const Packed& X, int st) {
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      const int row = crow + TR / CPT * k;
#pragma unroll
      for (int t = 0; t < 3; ++t)
        *reinterpret_cast<uint4*>(&ring[(3 * st + t) * TB + row * 256 + (cchunk ^ (row % 16)) * 16]) =
            dequant8_f16<BITS>(X.w[t][k], scale_pair<E>(X.s[t][k], ex[t], h2[t]),
                               scale_pair<E>(X.b[t][k], ex[t], h2[t]));
    }
  };

  Acc acc[NCB];
#pragma unroll
  for (int cb = 0; cb < NCB; ++cb) acc[cb].init();
  dequant_store(P, 0);
  load(P, 1);
  qslab_barrier();
  // The tile count is uniform over the workgroup, so every barrier is reached
  // by all of its threads.  Barrier i ends tile i: every wave is done with
  // stage i % 2 (its LDS accesses completed) and tile i + 1 is in the other.
  for (int i = 0; i < ntiles; ++i) {
    const uint8_t* tl = ring + (i & 1) * 3 * TB;
    floatx4 sacc[NCB][2];
    tile_scores_n<half_t, NCB>(tl, qb, sacc, col, blk);
    dequant_store(P, (i + 1) & 1);
    load(P, i + 2);
    V8 pb[NCB];
    const int t0 = (i * ns + split) * TR;
#pragma unroll
    for (int cb = 0; cb < NCB; ++cb)
      pb[cb] = acc[cb].softmax(sacc[cb], t0, r_end, lim[cb], qsc[cb], blk,
                               t0 + TR <= min(r_end, lim_lo[cb]));
    tile_pv_n<half_t, NCB>(acc, pb, tl + TB, tl + 2 * TB, col, blk);
    qslab_barrier();
  }

  // The values' powers of two; a value past the fp16 range (an fp16 cache's
  // s * u + b can be, by the rounding of s) stays finite in an fp16 partial.
  if (ex[1] != 0 || ex[2] != 0) {
#pragma unroll
    for (int cb = 0; cb < NCB; ++cb) {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          acc[cb].acc1[j][r] = ldexpf(acc[cb].acc1[j][r], ex[1]);
          acc[cb].acc2[j][r] = ldexpf(acc[cb].acc2[j][r], ex[2]);
          if (ns > 1 && a.part_f16) {
            const float hi = 65504.f * acc[cb].accl[0];
            acc[cb].acc1[j][r] = fminf(fmaxf(acc[cb].acc1[j][r], -hi), hi);
            acc[cb].acc2[j][r] = fminf(fmaxf(acc[cb].acc2[j][r], -hi), hi);
          }
        }
      }
    }
  }
  if (ns > 1) {
    // Partials through the ring, free after the last barrier.
    float* lds = reinterpret_cast<float*>(ring) + wave * (kStageWaveBytes / 4);
#pragma unroll
    for (int cb = 0; cb < NCB; ++cb) {
      const int c0 = vh[cb] - col;
      store_partials_staged<half_t>(acc[cb], lds, a.part_o, a.part_ml, qrow0 + c0,
                                    min(16, a.GV - c0), ns, split, col, blk, a.part_f16);
    }
    return;
  }
#pragma unroll
  for (int cb = 0; cb < NCB; ++cb)
    if (col_ok[cb]) acc[cb].template store_y<E>(a.y, qrow0 + vh[cb], blk);
}

}  // namespace motif
