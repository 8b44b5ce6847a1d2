// Stage 1 of the Flash-HOG double backward (passes 1-3) in one sweep over the keys
// with two waves per 32 queries, for 2-byte types at D = 128. The algebra, its
// rounding and the special rows are those of fhog_bwdbwd_fused.hip; its eleven
// products are split between the waves of a pair:
//   wave A holds Q, ddQ:  S, ddS -> P, x = P ddS, dD; sum P ddV + x V and sum P K;
//   wave B holds dO:      u = dP - D, dPa -> P u, X; sum P u ddK + X K and sum P u K.
// P and x cross from A to B through LDS in fp32, in the accumulator layout (lane l
// of B reads what lane l of A wrote); at the end A hands dD and sum P K to B, which
// forms dQ2 and the statistics, and forms ddO itself.
//
// Why. The four accumulators of 32 queries do not fit one wave, so the fused
// kernel gives a wave 16 queries on the 16x16x32 instruction and reads each
// key-side tile from LDS once per 16 queries: 128 KiB per 32 x 32 tile. Two waves
// share the accumulators of 32 queries (two each, 256 registers) on the 32x32x16
// instruction and read 72 KiB, with 16 KiB of exchange. What bounds it is
// latency: at B2 N8192 H16 the matrix pipes are busy 51 % of the cycles and the LDS
// 49 %, 21 points of it bank conflicts; two waves per SIMD each wait 43 % of their time,
// and 20-88 bytes per lane are spilled, part of them in the loop.
//
// Two workgroup shapes give the same bits (stage1_pairs_rule): two pairs (two
// workgroups per CU) for grids that do not fill the chip and where 128-query blocks would
// waste rows, four (waves w and w + 4, the two of a pair, share a SIMD; the key-side
// tiles are streamed half as often) for the others.
// Stage 1, us, before -> with this kernel: B2 N8192 H16 causal bf16 2924 -> 2743, B4
// N2048 H16 non-causal 759 -> 679, B2 N2048 H32 over 8 key heads 397 -> 372, B1
// N1024 H8 73 -> 66.
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

constexpr int kOcc = 2;  // waves per SIMD

template <typename T, int D, bool CAUSAL, bool PRE, int PAIRS>
__global__ void __launch_bounds__(128 * PAIRS)
__attribute__((amdgpu_waves_per_eu(kOcc, kOcc)))
bwdbwd_fused_pair_kernel(BwdBwdParams<T> p, int chunk, int fold) {
  typedef SwzTile<T, D> G;
  constexpr int KS = D / 16;
  constexpr int DT = D / 32;
  constexpr int kWaves = 2 * PAIRS;
  constexpr int BQ = 32 * PAIRS;  // queries per workgroup
  constexpr int BK = 32;
  constexpr int NST = 2;  // a third stage with four pairs: within 1 %
  constexpr int kTile = G::kElems * (int)sizeof(T);
  constexpr int kStage = 4 * kTile;           // K, V, ddK, ddV
  constexpr int kPart = G::kLoads / kWaves;   // loads of each tensor per wave
  constexpr int kExch = 32 * 32 * (int)sizeof(float);  // one of P and x
  constexpr int kAcc = DT * 16 * 64 * (int)sizeof(float);  // one accumulator of a wave
  static_assert(PAIRS * kAcc <= NST * kStage, "the accumulator exchange reuses the ring");
  __shared__ __attribute__((aligned(1024))) char s_kv[NST * kStage];
  __shared__ __attribute__((aligned(1024))) char s_x[PAIRS * 2 * kExch];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int pair = wave % PAIRS;
  const int wave_role = wave / PAIRS;  // 0 = A, 1 = B
  const int n = lane & 31, g = lane >> 5;
  const int nqb = (p.nq + BQ - 1) / BQ;
  const int nbh = p.batch * p.heads;
  const GridSlot gs = grid_slot(blockIdx.x, nbh, nqb, chunk);
  // causal: the longest query rows first, up to rank `fold`; the ranks from
  // there on run backwards (fold_rank)
  const int rank = folded(gs.rank, nqb, fold);
  const int qb = CAUSAL ? nqb - 1 - rank : rank;
  const int bh = gs.pair;
  const int b = bh / p.heads, h = bh % p.heads;
  const int hk = h / (p.heads / p.kv_heads);
  const long rs = (long)p.heads * D;      // query-side row stride
  const long rsk = (long)p.kv_heads * D;  // key-side row stride
  const long qbase = ((long)b * p.nq * p.heads + h) * D;
  const long kbase = ((long)b * p.nk * p.kv_heads + hk) * D;
  const long sbase = (long)bh * p.nq;
  const int q0 = qb * BQ + pair * 32;
  const int qi = q0 + n;
  const bool qvalid = qi < p.nq;

  int kend = p.nk;
  if (CAUSAL) kend = min(kend, qb * BQ + BQ + p.coff);
  const int nkt = __builtin_amdgcn_readfirstlane(kend > 0 ? (kend + BK - 1) / BK : 0);
  int wend = p.nk;
  if (CAUSAL) wend = max(0, min(wend, q0 + 32 + p.coff));
  const int wkt = q0 < p.nq ? (wend + BK - 1) / BK : 0;  // tiles with work for this pair

  SwzFrags<T, D> fr;
  fr.init(lane);
  const uint32_t row_bytes = (uint32_t)(rsk * (long)sizeof(T));
  TileDma<T, D, kPart> dma;
  dma.init(row_bytes, BK, lane, kPart * wave);
  const uint32_t lds0 = lds_base_u32(s_kv);
  long gnext = kbase;
  auto issue = [&](int kt) {
    const uint32_t stage = lds0 + (uint32_t)(((uint32_t)kt % NST) * kStage);
    const int nvalid = p.nk - kt * BK;
    if (nvalid >= BK) {
      dma.issue(stage, p.k + gnext);
      dma.issue(stage + kTile, p.v + gnext);
      dma.issue(stage + 2 * kTile, p.ddk + gnext);
      dma.issue(stage + 3 * kTile, p.ddv + gnext);
    } else {
      TileDma<T, D, kPart> part;
      part.init(row_bytes, nvalid, lane, kPart * wave);
      part.issue(stage, p.k + gnext);
      part.issue(stage + kTile, p.v + gnext);
      part.issue(stage + 2 * kTile, p.ddk + gnext);
      part.issue(stage + 3 * kTile, p.ddv + gnext);
    }
    gnext += BK * rsk;
  };

  const float scale = p.scale;
  // A lane past the last query loads the last query's row (its results are
  // never stored, and no product mixes queries).
  const long roff = qbase + (long)min(qi, p.nq - 1) * rs;
  if (nkt > 0) issue(0);

  // Compiled once per role, so that neither keeps the other's operands.
  auto sweep = [&](auto role_tag) {
    constexpr int role = decltype(role_tag)::value;
    V8<T> r0[KS], r1[role == 0 ? KS : 1];  // A: Q, ddQ; B: dO
    float dpart = 0.f;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const long off = roff + 16 * ks + 8 * g;
      if constexpr (role == 0) {
        r0[ks] = *reinterpret_cast<const V8<T>*>(p.q + off);
        r1[ks] = *reinterpret_cast<const V8<T>*>(p.ddq + off);
      } else {
        r0[ks] = *reinterpret_cast<const V8<T>*>(p.dout + off);
        dpart = dot8<T>(*reinterpret_cast<const V8<T>*>(p.o + off), r0[ks], dpart);
      }
    }
    if constexpr (PRE && role == 0) {
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          r0[ks][e] = (T)((float)r0[ks][e] * scale);
          r1[ks][e] = (T)((float)r1[ks][e] * scale);
        }
    }
    const float c2 = PRE ? kLog2e : scale * kLog2e;
    const float Di = role ? xgroup_sum(dpart) : 0.f;
    const float nL2 = role ? 0.f : -p.lse[sbase + min(qi, p.nq - 1)] * kLog2e;

    f32x16 acc0[DT], acc1[DT];  // A: ddO part, sum P K; B: dQ2 part, sum P u K
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) acc0[dt] = acc1[dt] = zero16();
    float s0 = 0.f, s1 = 0.f;  // A: sum x, sum T(x); B: sum X, sum P u
    wait_vmem();

    // After its first barrier of iteration t every wave is done with tile t - 1,
    // whose stage tile t + 1 takes, and with the exchange buffer.
    for (int t = 0; t < nkt; ++t) {
      wait_vmem();
      __syncthreads();
      if (t + 1 < nkt) issue(t + 1);
      const bool active = t < wkt;
      const uint32_t sa = lds0 + (uint32_t)(((uint32_t)t % NST) * kStage);
      float* xp = reinterpret_cast<float*>(s_x + pair * 2 * kExch) + 4 * lane;  // P, then x
      f32x16 C0, C1;
      if (active) {
        if constexpr (role == 0) {
          C0 = zero16();
          C1 = zero16();
#pragma unroll
          for (int ks = 0; ks < KS; ++ks) {
            const V8<T> kf = fr.rowf(sa, 0, ks);
            const V8<T> dkf = fr.rowf(sa, 2 * kTile, ks);
            C0 = mma<T>(kf, r0[ks], C0);
            C1 = mma<T>(kf, r1[ks], C1);
            C1 = mma<T>(dkf, r0[ks], C1);
          }
#pragma unroll
          for (int r = 0; r < 16; ++r) C0[r] = exp2_fast(fmaf(C0[r], c2, nL2));
          const int k0 = t * BK;
          if ((k0 + BK > p.nk) || (CAUSAL && k0 + BK - 1 > q0 + p.coff)) {
            const int klim = min(p.nk - 1, CAUSAL ? qi + p.coff : p.nk - 1) - k0;  // last visible key, tile-relative
#pragma unroll
            for (int r = 0; r < 16; ++r)
              if (crow(r, g) > klim) C0[r] = 0.f;
          }
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            C1[r] = PRE ? C0[r] * C1[r] : C0[r] * (C1[r] * scale);
            s0 += C1[r];
          }
#pragma unroll
          for (int a = 0; a < 4; ++a) {
            *reinterpret_cast<f32x4*>(xp + 256 * a) = f32x4{C0[4 * a], C0[4 * a + 1], C0[4 * a + 2], C0[4 * a + 3]};
            *reinterpret_cast<f32x4*>(xp + 1024 + 256 * a) =
                f32x4{C1[4 * a], C1[4 * a + 1], C1[4 * a + 2], C1[4 * a + 3]};
          }
        } else {
#pragma unroll
          for (int r = 0; r < 16; ++r) C0[r] = -Di;
          C1 = zero16();
#pragma unroll
          for (int ks = 0; ks < KS; ++ks) {
            C0 = mma<T>(fr.rowf(sa, kTile, ks), r0[ks], C0);
            C1 = mma<T>(fr.rowf(sa, 3 * kTile, ks), r0[ks], C1);
          }
        }
      }
      __syncthreads();
      if (active) {
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          if constexpr (role == 0) {
            const V8<T> oP = cvt8<T>(s ? hi8(C0) : lo8(C0));
            const V8<T> ox = cvt8<T>(s ? hi8(C1) : lo8(C1));
            s1 = add_sum8<T>(ox, s1);
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) {
              acc0[dt] = mma<T>(fr.trf(sa, 3 * kTile, dt, s), oP, acc0[dt]);
              acc0[dt] = mma<T>(fr.trf(sa, kTile, dt, s), ox, acc0[dt]);
              acc1[dt] = mma<T>(fr.trf(sa, 0, dt, s), oP, acc1[dt]);
            }
          } else {
            f32x8 vu, vX;
#pragma unroll
            for (int a = 0; a < 2; ++a) {
              const f32x4 P = *reinterpret_cast<const f32x4*>(xp + 256 * (2 * s + a));
              const f32x4 x = *reinterpret_cast<const f32x4*>(xp + 1024 + 256 * (2 * s + a));
#pragma unroll
              for (int j = 0; j < 4; ++j) {
                const int r = 8 * s + 4 * a + j;
                vu[4 * a + j] = P[j] * C0[r];
                vX[4 * a + j] = fmaf(x[j], C0[r], P[j] * C1[r]);
                s0 += vX[4 * a + j];
                s1 += vu[4 * a + j];
              }
            }
            const V8<T> ou = cvt8<T>(vu);
            const V8<T> oX = cvt8<T>(vX);
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) {
              const V8<T> tK = fr.trf(sa, 0, dt, s);
              acc0[dt] = mma<T>(fr.trf(sa, 2 * kTile, dt, s), ou, acc0[dt]);
              acc0[dt] = mma<T>(tK, oX, acc0[dt]);
              acc1[dt] = mma<T>(tK, ou, acc1[dt]);
            }
          }
        }
      }
    }

    // A hands sum P K and dD to B through the ring, which no wave reads any more.
    __syncthreads();
    s0 = xgroup_sum(s0);
    s1 = xgroup_sum(s1);
    float* xa = reinterpret_cast<float*>(s_kv + pair * kAcc) + 4 * lane;
    float* xd = reinterpret_cast<float*>(s_x + pair * 2 * kExch) + lane;
    if constexpr (role == 0) {
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int a = 0; a < 4; ++a)
          *reinterpret_cast<f32x4*>(xa + 256 * (4 * dt + a)) =
              f32x4{acc1[dt][4 * a], acc1[dt][4 * a + 1], acc1[dt][4 * a + 2], acc1[dt][4 * a + 3]};
      *xd = s0;
    }
    __syncthreads();
    if constexpr (role == 0) {
      if (qvalid) {
        T* ddo = p.ddo + roff;
        const T* o = p.o + roff;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
          for (int a = 0; a < 4; ++a) {
            const int d = 32 * dt + 8 * a + 4 * g;
            const V4<T> o4 = *reinterpret_cast<const V4<T>*>(o + d);
            f32x4 y;
#pragma unroll
            for (int j = 0; j < 4; ++j) y[j] = acc0[dt][4 * a + j] - s1 * (float)o4[j];
            *reinterpret_cast<V4<T>*>(ddo + d) = cvt4<T>(y);
          }
      }
    } else {
      const float dD = *xd;
      const float c = s0 - dD * s1;
      const bool one_key = (CAUSAL ? min(p.nk, qi + p.coff + 1) : p.nk) == 1;
      if (qvalid) {
        if (g == 0) {
          p.delta[sbase + qi] = Di;
          p.ddelta[sbase + qi] = dD;
          p.bstat[sbase + qi] = c - Di * dD;
        }
        T* dq2 = p.dq2 + roff;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
          for (int a = 0; a < 4; ++a) {
            const f32x4 pk = *reinterpret_cast<const f32x4*>(xa + 256 * (4 * dt + a));
            f32x4 x;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              const int r = 4 * a + j;
              x[j] = one_key ? 0.f : scale * (acc0[dt][r] - dD * acc1[dt][r] - c * pk[j]);
            }
            *reinterpret_cast<V4<T>*>(dq2 + 32 * dt + 8 * a + 4 * g) = cvt4<T>(x);
          }
      }
    }
  };
  if (wave_role == 0)
    sweep(std::integral_constant<int, 0>{});
  else
    sweep(std::integral_constant<int, 1>{});
}

template <typename T, int D, bool CAUSAL, int PAIRS>
hipError_t launch_pairs(const BwdBwdParams<T>& p, int cus, hipStream_t stream) {
  const int nqb = (p.nq + 32 * PAIRS - 1) / (32 * PAIRS);
  const int npairs = p.batch * p.heads;
  const int fold = fold_rank(CAUSAL && PAIRS == 2, nqb, npairs, cus);
  const int chunk = grid_chunk(npairs, nqb, PAIRS == 2 ? 2 * cus : cus);
  const dim3 grid(nqb * npairs), block(128 * PAIRS);
  int e2;
  constexpr bool kPre = std::is_same_v<T, __bf16>;
  if (kPre && std::frexp(p.scale, &e2) == 0.5f)  // scale = 2^(e2 - 1)
    hipLaunchKernelGGL((bwdbwd_fused_pair_kernel<T, D, CAUSAL, kPre, PAIRS>), grid, block, 0, stream, p, chunk, fold);
  else
    hipLaunchKernelGGL((bwdbwd_fused_pair_kernel<T, D, CAUSAL, false, PAIRS>), grid, block, 0, stream, p, chunk, fold);
  return hipGetLastError();
}

}  // namespace

template <typename T, bool CAUSAL>
hipError_t launch_bwdbwd_stage1_fused_pair(const BwdBwdParams<T>& p, hipStream_t stream) {
  const int cus = resident_workgroups(1);
  if (stage1_pairs_rule(mask_of(CAUSAL, p), p.batch * p.heads, cus) == 2)
    return launch_pairs<T, 128, CAUSAL, 2>(p, cus, stream);
  return launch_pairs<T, 128, CAUSAL, 4>(p, cus, stream);
}

#define FHOG_INST(T, C) \
  template hipError_t launch_bwdbwd_stage1_fused_pair<T, C>(const BwdBwdParams<T>&, hipStream_t);
FHOG_INST(__bf16, true)
FHOG_INST(__bf16, false)
FHOG_INST(_Float16, true)
FHOG_INST(_Float16, false)
#undef FHOG_INST

}  // namespace fhog
