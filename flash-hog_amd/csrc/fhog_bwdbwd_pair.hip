// Stage 2 of the Flash-HOG double backward (pass 4: dK2, dV2) with two waves
// per 32 keys. The math is that of fhog_bwdbwd.hip's stage 2
// (flash_hog/_jax_refs/jax_impl.py:273-336, the pass split of
// flash_hog/jax/_pallas_gpu_kernel.py:309-391), split so that each wave of a
// pair does four of the eight products:
//   wave A holds K, ddK:  S, ddS -> P = exp(S'), t = ddS - dD,
//                         dV2 = sum_i (P t) dO;
//   wave B holds V, ddV:  u = dP - D, dPa' = dPa - (D dD + B),
//                         dK2 = scale sum_i (P u) ddQ + P (dPa' + u t) Q.
// P and t cross from A to B through LDS in fp32, in the accumulator layout
// (lane l of B reads what lane l of A wrote). Products, sums and roundings are
// bwdbwd_k_kernel's, in the same order, so at D = 64 the two kernels give the
// same bits and the launch may choose between them by grid shape.
//
// Why. One wave with K, ddK, V, ddV, both accumulators and four score tiles
// takes 256 registers at D = 64, more than a SIMD can share at D = 128 (which
// ran 16 keys per wave on the 16x16x32 instruction, reading each query-side
// tile from LDS twice as often), and 256 + 130 (D = 64) or 512 with 600 bytes
// of spill (D = 128) for fp32. Half of that state fits two waves per SIMD at
// D = 128 and for fp32 at D = 64, and one wave without spill at D = 256 and
// for fp32 at D = 128. Per 32 x 32 tile at D = 128 a pair reads 48 KiB and
// exchanges 16 KiB, against 96 KiB with 16 keys per wave. What
// bounds it is latency: at B2 N8192 H16 the matrix pipes are busy 47 % of the cycles
// and the LDS 51 %, 18 points of it bank conflicts; a wave waits 44 % of its time.
//
// Stage 2, us, before -> with this kernel: causal bf16 B2 N8192 H16 D128
// 2525 -> 2189, B2 N2048 H32 over 8 key heads D128 574 -> 396, B2 N2048 H8
// D256 278 -> 213; fp32 B2 N2048 H8 D64 565 -> 366, B1 N2048 H8 D128
// non-causal 1285 -> 665; D = 64 small grids: B1 N1024 H12 42.4 -> 35.7, B1
// N4096 H12 161 -> 144. At D = 64 the exchange is two thirds of the operand
// reads, and grids that fill the chip keep bwdbwd_k_kernel (B4 N2048 H16 147
// against 184).
//
// The two roles run separate copies of the sweep and must reach the same barriers:
// every one of them stands outside the role's and the mask's branches, and the number
// of tiles is the workgroup's.
#include <cmath>
#include <type_traits>

#include "fhog_device.h"
#include "fhog_params.h"

namespace fhog {

namespace {

constexpr int kPairs = 2;
constexpr int kWaves = 2 * kPairs;
constexpr int kThreads = 64 * kWaves;

// Waves per SIMD: two up to 256-byte rows, one (512 registers) above. A third
// at 256-byte rows spills (B2 N8192 H16 D128 3213 us).
template <typename T, int D> struct Occupancy {
  static constexpr int value = D * sizeof(T) >= 512 ? 1 : 2;
};

template <typename T, int D, bool CAUSAL, bool PRE>
__global__ void __launch_bounds__(kThreads)
__attribute__((amdgpu_waves_per_eu(Occupancy<T, D>::value, Occupancy<T, D>::value)))
bwdbwd_pair_kernel(BwdBwdParams<T> p, int chunk, int fold) {
  typedef SwzTile<T, D> G;
  constexpr int KS = D / 16;
  constexpr int DT = D / 32;
  constexpr int BKB = 32 * kPairs;
  constexpr int BQ = 32;
  constexpr int NST = 2;
  constexpr int kTile = G::kElems * (int)sizeof(T);
  constexpr int kStat = 4 * BQ * (int)sizeof(float);
  constexpr int kStage = 3 * kTile + kStat;  // Q, dO, ddQ, constants
  constexpr int kPart = G::kLoads / kWaves;   // loads of each tensor per wave
  constexpr int kStatWave = kWaves - 1;
  constexpr int kExch = 32 * 32 * (int)sizeof(float);  // one of P and t
  __shared__ __attribute__((aligned(1024))) char s_q[NST * kStage];
  __shared__ __attribute__((aligned(1024))) char s_x[kPairs * 2 * kExch];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int pair = wave % kPairs;
  const int wave_role = wave / kPairs;  // 0 = A (S, ddS, dV2), 1 = B (dP, dPa, dK2)
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
  const int qfirst = first_contributing_query(p, kj, CAUSAL);

  // Iteration i visits query tile qt_begin + i / grp of query head
  // hk * grp + i % grp (the group reduction of _pallas_gpu_kernel.py:333-370).
  const int nqt = (p.nq + BQ - 1) / BQ;
  const int qt_begin = CAUSAL ? max(0, kb * BKB - p.coff) / BQ : 0;
  const int total = __builtin_amdgcn_readfirstlane(nqt > qt_begin ? (nqt - qt_begin) * grp : 0);

  f32x16 acc[DT];  // A: dV2, B: dK2
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) acc[dt] = zero16();

  if (total > 0) {
    const float scale = p.scale;
    const float inv_scale = 1.0f / scale;
    SwzFrags<T, D> fr;
    fr.init(lane);
    // Wave w streams quarter w of each of the three tiles, the last wave also
    // the row statistics.
    const uint32_t row_bytes = (uint32_t)(rs * (long)sizeof(T));
    TileDma<T, D, kPart> dma;
    dma.init(row_bytes, BQ, lane, kPart * wave);
    const uint32_t lds0 = lds_base_u32(s_q);
    long gnext = qbase + (long)qt_begin * BQ * rs;
    const long row_step = (long)BQ * rs - (long)(grp - 1) * D;
    auto issue = [&](int i, GroupCursor c) {
      const int q0t = (qt_begin + c.qt) * BQ;
      const uint32_t stage = lds0 + (uint32_t)(((uint32_t)i % NST) * kStage);
      if (q0t + BQ <= p.nq) {
        dma.issue(stage, p.q + gnext);
        dma.issue(stage + kTile, p.dout + gnext);
        dma.issue(stage + 2 * kTile, p.ddq + gnext);
      } else {
        TileDma<T, D, kPart> part;
        part.init(row_bytes, p.nq - q0t, lane, kPart * wave);
        part.issue(stage, p.q + gnext);
        part.issue(stage + kTile, p.dout + gnext);
        part.issue(stage + 2 * kTile, p.ddq + gnext);
      }
      if (wave == kStatWave) {
        const uint32_t off = 4u * (uint32_t)min(q0t + n, p.nq - 1);
        const long sb = sbase + (long)c.gi * p.nq;
        const uint32_t dst = stage + 3 * kTile;
        if (g == 0) {
          dma4s(p.lse + sb, off, dst);
          dma4s(p.ddelta + sb, off, dst + 256);
        } else {
          dma4s(p.delta + sb, off, dst);
          dma4s(p.bstat + sb, off, dst + 256);
        }
      }
    };
    auto advance = [&](GroupCursor& c) {
      gnext += c.gi + 1 == grp ? row_step : (long)D;
      c.next(grp);
    };
    auto finish_stats = [&](int i) {
      if (g == 0) {
        float* st = reinterpret_cast<float*>(s_q + ((uint32_t)i % NST) * kStage + 3 * kTile);
        const float L = st[n], Dq = st[BQ + n], dDq = st[2 * BQ + n], Bq = st[3 * BQ + n];
        st[n] = PRE ? -L : -L * inv_scale;
        st[BQ + n] = PRE ? -dDq : -dDq * inv_scale;
        st[2 * BQ + n] = -Dq;
        st[3 * BQ + n] = -fmaf(Dq, dDq, Bq);
      }
    };

    GroupCursor nxt;  // iteration of the next tile to issue
    issue(0, nxt);
    advance(nxt);

    // Compiled once per role: one loop for both took 256 registers and spilled
    // 37 in it at D = 128 (7678 against 2189 us at B2 N8192 H16).
    auto sweep = [&](auto role_tag) {
      constexpr int role = decltype(role_tag)::value;
      V8<T> r0[KS], r1[KS];  // A: K, ddK; B: V, ddV
      const T* src0 = role ? p.v : p.k;
      const T* src1 = role ? p.ddv : p.ddk;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const long off = kbase + (long)kj * rsk + 16 * ks + 8 * g;
        r0[ks] = kvalid ? *reinterpret_cast<const V8<T>*>(src0 + off) : zero8<T>();
        r1[ks] = kvalid ? *reinterpret_cast<const V8<T>*>(src1 + off) : zero8<T>();
      }
      if constexpr (PRE && role == 0) {
        // scale is a power of two: K and ddK carry it exactly (bwdbwd_k_kernel)
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            r0[ks][e] = (T)((float)r0[ks][e] * scale);
            r1[ks][e] = (T)((float)r1[ks][e] * scale);
          }
      }
      const float c2 = PRE ? kLog2e : scale * kLog2e;
      // Retire the key-side loads, and with them the first tile, before the loop.
      wait_vmem();
      if (wave == kStatWave) finish_stats(0);

      // After its first barrier of iteration i every wave is done with tile
      // i - 1, whose stage tile i + 1 takes, and with the exchange buffer.
      GroupCursor cur;  // iteration i
      for (int i = 0; i < total; ++i, cur.next(grp)) {
        wait_vmem();
        __syncthreads();
        if (i + 1 < total) {
          issue(i + 1, nxt);
          advance(nxt);
        }
        const int q0 = (qt_begin + cur.qt) * BQ;
        const bool active = k0 < p.nk && (!CAUSAL || q0 + BQ - 1 >= k0 - p.coff);
        const uint32_t slot = ((uint32_t)i % NST) * kStage;
        const uint32_t sa = lds0 + slot;  // Q, dO, ddQ
        float* xp = reinterpret_cast<float*>(s_x + pair * 2 * kExch) + 4 * lane;  // P, then t
        // The accumulators start at the per-query constants (register r holds
        // query 8 (r / 4) + 4 g + r % 4 of the tile): A's end as S' and ddS - dD
        // (both over scale unless PRE), B's as u and dPa'.
        f32x16 C0, C1;
        if (active) {
          const float* sc = reinterpret_cast<const float*>(s_q + slot + 3 * kTile) + 2 * BQ * role;
#pragma unroll
          for (int a = 0; a < 4; ++a) {
            const f32x4 v0 = *reinterpret_cast<const f32x4*>(sc + 8 * a + 4 * g);
            const f32x4 v1 = *reinterpret_cast<const f32x4*>(sc + BQ + 8 * a + 4 * g);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              C0[4 * a + j] = v0[j];
              C1[4 * a + j] = v1[j];
            }
          }
          if constexpr (role == 0) {
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) {
              const V8<T> qa = fr.rowf(sa, 0, ks);
              const V8<T> dqa = fr.rowf(sa, 2 * kTile, ks);
              C0 = mma<T>(qa, r0[ks], C0);
              C1 = mma<T>(dqa, r0[ks], C1);
              C1 = mma<T>(qa, r1[ks], C1);
            }
#pragma unroll
            for (int r = 0; r < 16; ++r) {
              C0[r] = exp2_fast(C0[r] * c2);
              if (!PRE) C1[r] *= scale;
            }
            if ((q0 + BQ > p.nq) || (CAUSAL && q0 < k0 + 31 - p.coff) || p.nk == 1) {
              // a pair enters iff qfirst <= query < nq
              const int qlo = qfirst - q0, qhi = p.nq - q0;
#pragma unroll
              for (int r = 0; r < 16; ++r) {
                const int m = crow(r, g);
                if (m < qlo || m >= qhi) C0[r] = 0.f;
              }
            }
#pragma unroll
            for (int a = 0; a < 4; ++a) {
              *reinterpret_cast<f32x4*>(xp + 256 * a) = f32x4{C0[4 * a], C0[4 * a + 1], C0[4 * a + 2], C0[4 * a + 3]};
              *reinterpret_cast<f32x4*>(xp + 1024 + 256 * a) =
                  f32x4{C1[4 * a], C1[4 * a + 1], C1[4 * a + 2], C1[4 * a + 3]};
            }
          } else {
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) {
              const V8<T> doa = fr.rowf(sa, kTile, ks);
              C0 = mma<T>(doa, r0[ks], C0);
              C1 = mma<T>(doa, r1[ks], C1);
            }
          }
        }
        __syncthreads();
        if (active) {
#pragma unroll
          for (int s = 0; s < 2; ++s) {
            if constexpr (role == 0) {
              f32x8 vddP;
#pragma unroll
              for (int e = 0; e < 8; ++e) vddP[e] = C0[8 * s + e] * C1[8 * s + e];
              const V8<T> odP = cvt8<T>(vddP);
#pragma unroll
              for (int dt = 0; dt < DT; ++dt) acc[dt] = mma<T>(fr.trf(sa, kTile, dt, s), odP, acc[dt]);
            } else {
              f32x8 vdS, vdS2;
#pragma unroll
              for (int a = 0; a < 2; ++a) {
                const f32x4 P = *reinterpret_cast<const f32x4*>(xp + 256 * (2 * s + a));
                const f32x4 t = *reinterpret_cast<const f32x4*>(xp + 1024 + 256 * (2 * s + a));
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                  const int r = 8 * s + 4 * a + j;
                  const float x = fmaf(C0[r], t[j], C1[r]);  // dP2 - B
                  vdS[4 * a + j] = P[j] * C0[r];
                  vdS2[4 * a + j] = P[j] * x;
                }
              }
              const V8<T> oS = cvt8<T>(vdS);
              const V8<T> oS2 = cvt8<T>(vdS2);
#pragma unroll
              for (int dt = 0; dt < DT; ++dt) {
                acc[dt] = mma<T>(fr.trf(sa, 2 * kTile, dt, s), oS, acc[dt]);
                acc[dt] = mma<T>(fr.trf(sa, 0, dt, s), oS2, acc[dt]);
              }
            }
          }
        }
        // The next tile's statistics, whose DMA went out with this iteration's issue.
        if (wave == kStatWave && i + 1 < total) {
          wait_vmem();
          finish_stats(i + 1);
        }
      }
    };
    if (wave_role == 0)
      sweep(std::integral_constant<int, 0>{});
    else
      sweep(std::integral_constant<int, 1>{});
  }

  if (kvalid) {
    T* dst = (wave_role ? p.dk2 : p.dv2) + kbase + (long)kj * rsk;
    const float f = wave_role ? p.scale : 1.0f;
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

}  // namespace

template <typename T, int D, bool CAUSAL>
hipError_t launch_bwdbwd_stage2_pair(const BwdBwdParams<T>& p, hipStream_t stream) {
  const int nkb = (p.nk + 32 * kPairs - 1) / (32 * kPairs);
  const int npairs = p.batch * p.kv_heads;
  const int cus = resident_workgroups(1);
  const int fold = fold_rank(CAUSAL && Occupancy<T, D>::value == 2, nkb, npairs, cus);
  const int chunk = grid_chunk(npairs, nkb, Occupancy<T, D>::value * cus);
  const dim3 grid(nkb * npairs);
  int e2;
  constexpr bool kPre = std::is_same_v<T, __bf16>;
  if (kPre && std::frexp(p.scale, &e2) == 0.5f)  // scale = 2^(e2 - 1)
    hipLaunchKernelGGL((bwdbwd_pair_kernel<T, D, CAUSAL, kPre>), grid, dim3(kThreads), 0, stream, p, chunk, fold);
  else
    hipLaunchKernelGGL((bwdbwd_pair_kernel<T, D, CAUSAL, false>), grid, dim3(kThreads), 0, stream, p, chunk, fold);
  return hipGetLastError();
}

#define FHOG_INST(T, D, C) template hipError_t launch_bwdbwd_stage2_pair<T, D, C>(const BwdBwdParams<T>&, hipStream_t);
FHOG_INST(__bf16, 64, true)
FHOG_INST(__bf16, 64, false)
FHOG_INST(__bf16, 128, true)
FHOG_INST(__bf16, 128, false)
FHOG_INST(__bf16, 256, true)
FHOG_INST(__bf16, 256, false)
FHOG_INST(_Float16, 64, true)
FHOG_INST(_Float16, 64, false)
FHOG_INST(_Float16, 128, true)
FHOG_INST(_Float16, 128, false)
FHOG_INST(_Float16, 256, true)
FHOG_INST(_Float16, 256, false)
FHOG_INST(float, 64, true)
FHOG_INST(float, 64, false)
FHOG_INST(float, 128, true)
FHOG_INST(float, 128, false)
#undef FHOG_INST

}  // namespace fhog
