// dK and dV of the first backward with two waves per 32 keys (kernel 2 of
// fhog_bwd.hip, same math and bit-identical results):
//   wave A of a pair holds K and accumulates dV:  P = exp(scale Q K^T - L),
//                                                 dV = P^T dO;
//   wave B holds V and accumulates dK:            dP = dO V^T, dS = P (dP - D),
//                                                 dK = scale dS^T Q.
// P crosses from A to B through LDS, in fp32 and in the accumulator layout
// (lane l of B reads the 16 values lane l of A wrote, four conflict-free
// 16-byte accesses each way), so dS is formed from the same fp32 values as in
// one wave, and every sum runs in the same order.
//
// Why. One wave that does both halves holds K, V and both accumulators: at
// D = 128 (2-byte) 401 registers, which ran as two passes over halves of the
// output columns, forming the scores twice (12 d instead of 8 d matrix flops
// per pair); at D = 256 and for fp32 one wave per SIMD. Half of that state is
// about 120 (D = 64), 185 (128) and 256 registers (256; fp32: 135 and 214), so two
// or three waves share each SIMD and the scores are formed once. A pair also
// takes half the time per tile, and a workgroup is 64 keys instead of 128, so
// small and grouped-head grids spread over twice as many CUs. The price is the
// exchange: 8 KiB of LDS traffic beside 32 KiB of operand reads per 32 x 32
// tile at D = 128 (at D = 64 beside 16 KiB). What bounds it is latency: at B2
// N8192 H16 D = 128 the matrix pipes are busy 47 % of the cycles and the LDS 63 %, 24
// points of it bank conflicts, while a wave waits half of its time for operands, the
// exchange and the barriers.
//
// First backward (dQ kernel included), us, before -> with this kernel, causal
// bf16 unless named: B2 N2048 H32 over 8 key heads D128 642 -> 364; B4 N2048
// H16 D128 359 -> 285; B2 N8192 H16 D128 2380 -> 1890; B2 N2048 H8 D256
// 463 -> 271; fp32 B2 N2048 H8 D64 513 -> 377, B1 N2048 H8 D128 non-causal
// 943 -> 678; D64 B1 N4096 H12 184 -> 166, B1 N512 H12 31.1 -> 27.6.
//
// Both waves work on the same tile; a barrier before it orders the ring and
// one in its middle the exchange, which needs one buffer per pair and a ring of
// two stages, so that two or three workgroups share a CU (a wave B one tile
// behind A needs one barrier, but a ring stage and a buffer more: 0-3 % slower).
// The two roles run separate copies of the sweep and must reach the same barriers:
// every one of them stands outside the role's and the mask's branches, and the number
// of tiles is the workgroup's.
#pragma once

#include "fhog_device.h"
#include "fhog_params.h"

namespace fhog {

namespace {

constexpr int kPairs = 2;  // four pairs (128 keys) per workgroup: 4-10 % slower
constexpr int kWaves = 2 * kPairs;
constexpr int kThreads = 64 * kWaves;

template <typename T, int D, bool CAUSAL, int OCC>
__global__ void __launch_bounds__(kThreads)
__attribute__((amdgpu_waves_per_eu(OCC, OCC)))
bwd_pair_kernel(BwdParams<T> p, int chunk, int fold) {
  typedef SwzTile<T, D> G;
  constexpr int KS = D / 16;
  constexpr int DT = D / 32;
  constexpr int BKB = 32 * kPairs;
  constexpr int BQ = 32;
  constexpr int NST = 2;
  constexpr int kTile = G::kElems * (int)sizeof(T);
  // Statistics area as in bwd_k_kernel: two 256-byte rows (L, D of the tile's
  // 32 queries, then a copy that nothing reads).
  constexpr int kStatRow = 64 * (int)sizeof(float);
  constexpr int kSR = kStatRow / (int)sizeof(float);
  constexpr int kStage = 2 * kTile + 2 * kStatRow;  // Q, dO, statistics
  constexpr int kPer = G::kLoads / kPairs;
  constexpr int kExch = 32 * 32 * (int)sizeof(float);
  constexpr int kStatWave = kWaves - 1;
  __shared__ __attribute__((aligned(1024))) char s_q[NST * kStage];
  __shared__ __attribute__((aligned(1024))) char s_p[kPairs * kExch];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int pair = wave % kPairs;
  const int wave_role = wave / kPairs;  // 0 = A (S, P, dV), 1 = B (dP, dS, dK)
  const int n = lane & 31, g = lane >> 5;
  const int nbh = p.batch * p.kv_heads;
  const int nkb = (p.nk + BKB - 1) / BKB;
  const GridSlot gs = grid_slot(blockIdx.x, nbh, nkb, chunk);
  // causal: the longest key columns come first, up to rank `fold`; the ranks
  // from there on run backwards (fold_rank)
  const int kb = folded(gs.rank, nkb, fold);
  const int bh = gs.pair;
  const int b = bh / p.kv_heads, hk = bh % p.kv_heads;
  const int grp = p.heads / p.kv_heads;  // query heads per key/value head
  const long rs = (long)p.heads * D;      // query-side row stride
  const long rsk = (long)p.kv_heads * D;  // key-side row stride
  // query head hk * grp + gi: tensors at qbase + gi * D, statistics at sbase + gi * nq
  const long qbase = ((long)b * p.nq * p.heads + (long)hk * grp) * D;
  const long kbase = ((long)b * p.nk * p.kv_heads + hk) * D;
  const long sbase = ((long)b * p.heads + (long)hk * grp) * p.nq;
  const int k0 = kb * BKB + pair * 32;
  const int kj = k0 + n;
  const bool kvalid = kj < p.nk;
  const float scale = p.scale;

  // Iteration i visits query tile qt_begin + i / grp of query head
  // hk * grp + i % grp: the heads of a group share each tile's causal bounds.
  const int nqt = (p.nq + BQ - 1) / BQ;
  const int qt_begin = CAUSAL ? max(0, kb * BKB - p.coff) / BQ : 0;
  const int total = nqt > qt_begin ? (nqt - qt_begin) * grp : 0;

  f32x16 acc[DT];  // A: dV, B: dK
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) acc[dt] = zero16();

  if (total > 0) {
    const float c2 = scale * kLog2e;
    const float inv_scale = 1.0f / scale;

    // Wave w streams part w % kPairs of tensor w / kPairs (0 = Q, 1 = dO); the
    // last wave also the tile's L and D, which it rewrites in LDS, once they
    // have landed, as the initial values of the S and dP accumulators.
    SwzFrags<T, D> fr;
    fr.init(lane);
    const int tensor = wave / kPairs;
    const T* src = (tensor == 0 ? p.q : p.dout) + qbase;
    const uint32_t row_bytes = (uint32_t)(rs * (long)sizeof(T));
    TileDma<T, D, kPer> dma;
    dma.init(row_bytes, BQ, lane, kPer * pair);
    const uint32_t lds0 = lds_base_u32(s_q);
    // Sources of the next tile to issue, advanced with the cursor (bwd_k_kernel).
    const T* gnext = src + (long)qt_begin * BQ * rs;
    const long row_step = (long)BQ * rs - (long)(grp - 1) * D;
    const long soff0 = sbase + (long)qt_begin * BQ;
    const float* lnext = p.lse + soff0;
    const float* dnext = p.delta + soff0;
    const long stat_step = (long)BQ - (long)(grp - 1) * p.nq;
    auto issue = [&](int i, GroupCursor c) {
      const int q0t = (qt_begin + c.qt) * BQ;
      const uint32_t stage = lds0 + (uint32_t)(((uint32_t)i % NST) * kStage);
      const int nvalid = p.nq - q0t;
      if (nvalid >= BQ) {
        dma.issue(stage + tensor * kTile, gnext);
      } else {
        TileDma<T, D, kPer> part;
        part.init(row_bytes, nvalid, lane, kPer * pair);
        part.issue(stage + tensor * kTile, gnext);
      }
      if (wave == kStatWave) {
        // lane l reads query q0t + (l % 32); rows past nq repeat row nq - 1
        const uint32_t voff = 4u * (uint32_t)min(n, nvalid - 1);
        dma4s(lnext, voff, stage + 2 * kTile);
        dma4s(dnext, voff, stage + 2 * kTile + kStatRow);
      }
    };
    auto advance = [&](GroupCursor& c) {
      const bool last = c.gi + 1 == grp;
      gnext += last ? row_step : (long)D;
      lnext += last ? stat_step : (long)p.nq;
      dnext += last ? stat_step : (long)p.nq;
      c.next(grp);
    };
    auto finish_stats = [&](int i) {
      if (wave == kStatWave && g == 0) {
        float* st = reinterpret_cast<float*>(s_q + ((uint32_t)i % NST) * kStage + 2 * kTile);
        st[n] = -st[n] * inv_scale;
        st[kSR + n] = -st[kSR + n];
      }
    };

    auto sweep = [&](auto role) {
      V8<T> res[KS];  // A: K, B: V
      const T* rsrc = role ? p.v : p.k;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const long off = kbase + (long)kj * rsk + 16 * ks + 8 * g;
        res[ks] = kvalid ? *reinterpret_cast<const V8<T>*>(rsrc + off) : zero8<T>();
      }
      // Retire the key-side loads before the ring starts (see fwd_kernel).
      wait_vmem();
      GroupCursor nxt;  // iteration of the next tile to issue
      issue(0, nxt);
      advance(nxt);

      // After its first barrier of iteration i every wave is done with tile
      // i - 1, whose stage tile i + 1 takes, and with the exchange buffer.
      GroupCursor cur;  // iteration i
      for (int i = 0; i < total; ++i, cur.next(grp)) {
        wait_vmem();
        finish_stats(i);
        __syncthreads();
        if (i + 1 < total) {
          issue(i + 1, nxt);
          advance(nxt);
        }
        const int q0 = (qt_begin + cur.qt) * BQ;
        const bool active = k0 < p.nk && (!CAUSAL || q0 + BQ - 1 >= k0 - p.coff);
        const uint32_t slot = ((uint32_t)i % NST) * kStage;
        const uint32_t sa = lds0 + slot;  // Q at 0, dO at kTile
        float* xp = reinterpret_cast<float*>(s_p + pair * kExch) + 4 * lane;
        // Register r holds query 8 (r / 4) + 4 g + r % 4 of the tile. A starts at
        // -L / scale and ends as P, B starts at -D and ends as dS / scale.
        f32x16 C;
        if (active) {
          const float* sc = reinterpret_cast<const float*>(s_q + slot + 2 * kTile) + role * kSR;
#pragma unroll
          for (int a = 0; a < 4; ++a) {
            const f32x4 v = *reinterpret_cast<const f32x4*>(sc + 8 * a + 4 * g);
#pragma unroll
            for (int j = 0; j < 4; ++j) C[4 * a + j] = v[j];
          }
          const uint32_t srow = sa + role * kTile;
#pragma unroll
          for (int ks = 0; ks < KS; ++ks) C = mma<T>(fr.rowf(srow, 0, ks), res[ks], C);
          if (role == 0) {
#pragma unroll
            for (int r = 0; r < 16; ++r) C[r] = exp2_fast(C[r] * c2);
            if ((q0 + BQ > p.nq) || (CAUSAL && q0 < k0 + 31 - p.coff)) {
              // visible iff query >= key - coff (causal) and query < nq
              const int qlo = (CAUSAL ? kj - p.coff : 0) - q0, qhi = p.nq - q0;
#pragma unroll
              for (int r = 0; r < 16; ++r) {
                const int m = crow(r, g);
                if (m < qlo || m >= qhi) C[r] = 0.f;
              }
            }
#pragma unroll
            for (int a = 0; a < 4; ++a)
              *reinterpret_cast<f32x4*>(xp + 256 * a) = f32x4{C[4 * a], C[4 * a + 1], C[4 * a + 2], C[4 * a + 3]};
          }
        }
        __syncthreads();
        if (active) {
          if (role == 1) {
#pragma unroll
            for (int a = 0; a < 4; ++a) {
              const f32x4 P = *reinterpret_cast<const f32x4*>(xp + 256 * a);
#pragma unroll
              for (int j = 0; j < 4; ++j) C[4 * a + j] = P[j] * C[4 * a + j];
            }
          }
          const uint32_t scol = sa + (1 - role) * kTile;
#pragma unroll
          for (int s = 0; s < 2; ++s) {
            const V8<T> o = cvt8<T>(s ? hi8(C) : lo8(C));
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) acc[dt] = mma<T>(fr.trf(scol, 0, dt, s), o, acc[dt]);
          }
        }
      }
    };
    // Up to 256-byte rows the sweep is compiled once per role (D = 64 B1 N4096
    // H12 169 -> 163 us for the first backward, D = 128 with 8 key heads 371 ->
    // 355); at 512-byte rows two copies spill in the loop (D = 256 B2 N2048 H8
    // 271 us with one, 338 with two).
    if constexpr (D * sizeof(T) >= 512) {
      sweep(wave_role);
    } else {
      if (wave_role == 0)
        sweep(std::integral_constant<int, 0>{});
      else
        sweep(std::integral_constant<int, 1>{});
    }
  }

  if (kvalid) {
    T* dst = (wave_role ? p.dk : p.dv) + kbase + (long)kj * rsk;
    const float f = wave_role ? scale : 1.0f;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
#pragma unroll
      for (int a = 0; a < 4; ++a) {
        f32x4 x;
#pragma unroll
        for (int j = 0; j < 4; ++j) x[j] = acc[dt][4 * a + j] * f;
        *reinterpret_cast<V4<T>*>(dst + 32 * dt + 8 * a + 4 * g) = cvt4<T>(x);
      }
    }
  }
}

template <typename T, int D, bool CAUSAL, int OCC>
hipError_t launch_occ(const BwdParams<T>& p, int nkb, int npairs, int cus, hipStream_t stream) {
  hipLaunchKernelGGL((bwd_pair_kernel<T, D, CAUSAL, OCC>), dim3(nkb * npairs), dim3(kThreads), 0, stream, p,
                     grid_chunk(npairs, nkb, OCC * cus), fold_rank(CAUSAL, nkb, npairs, cus));
  return hipGetLastError();
}

}  // namespace

template <typename T, int D, bool CAUSAL>
hipError_t launch_bwd_pair(const BwdParams<T>& p, hipStream_t stream) {
  const int nkb = (p.nk + 32 * kPairs - 1) / (32 * kPairs);
  const int npairs = p.batch * p.kv_heads;
  const int cus = resident_workgroups(1);
  [[maybe_unused]] const int waves = bwd_pair_waves(mask_of(CAUSAL, p), npairs, D, (int)sizeof(T), cus);
  if constexpr (sizeof(T) == 4 && D == 64) {
    return launch_occ<T, D, CAUSAL, 3>(p, nkb, npairs, cus, stream);
  } else {
    if constexpr (sizeof(T) == 2 && D == 128) {
      if (waves == 3) return launch_occ<T, D, CAUSAL, 3>(p, nkb, npairs, cus, stream);
    }
    if constexpr (sizeof(T) == 2 && D == 64) {
      if (waves == 4) return launch_occ<T, D, CAUSAL, 4>(p, nkb, npairs, cus, stream);
    }
    return launch_occ<T, D, CAUSAL, 2>(p, nkb, npairs, cus, stream);
  }
}

}  // namespace fhog
