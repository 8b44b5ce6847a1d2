// Stage 1 of the Flash-HOG double backward (passes 1-3) for fp32, in two sweeps
// over the keys with two waves per 32 queries, for grids that do not fill the chip. The math follows
// flash_hog/_jax_refs/jax_impl.py:273-336 and the pass split of
// flash_hog/jax/_pallas_gpu_kernel.py:149-278.
//
// Sweep 1 (passes 1+2) forms S, ddS, dP and, per row, dD = sum ddS P,
// r2 = sum dP P, r3 = sum dP ddS P and P ddV; then
// r1 = sum_j P dPa = <dO_i, (P ddV)_i> and B = r1 - dD r2 - D dD + r3, which is
// rowsum(dP2 P) expanded. Sweep 2 (pass 3) forms S, ddS, dP, dPa again and adds
// dS ddK + dS2 K to dQ2 and ddP V to ddO, whose P ddV part came from sweep 1.
// (The one-sweep form of fhog_bwdbwd_fused.hip does two products fewer, but its
// sums cancel: the 2-byte types' roundings hide that, fp32's would not.)
//
// Of the 13 products wave A of a pair does seven, wave B six:
//   A holds Q, ddQ.  Sweep 1: S, ddS -> P, x = P ddS, dD.
//                    Sweep 2: S, ddS -> P, t = ddS - dD; ddO += (P t) V.
//   B holds dO.      Sweep 1: dP -> r2, r3; P ddV.
//                    Sweep 2: dP, dPa -> u, dP2 - B; dQ2 += (P u) ddK + ... K.
// P and x (sweep 1), P and t (sweep 2) cross from A to B through LDS in the
// accumulator layout (lane l of B reads what lane l of A wrote); between the
// sweeps dD goes to B and P ddV to A. Products, sums and roundings are those of
// one wave per 32 queries, in the same order.
//
// Why. One wave per 32 queries holds Q, ddQ, dO and two accumulators: one wave
// per SIMD and 128 queries per workgroup, so a causal grid of one workgroup per
// CU takes as long as its longest block. Half of that state (D = 64, 186
// registers) lets two waves share a SIMD, and a block is 64 queries at half the
// time per tile. Two waves wait for each other in every tile, though, and wave A
// has more to do in sweep 1: on grids that fill the chip bwdbwd_q_kernel
// (fhog_bwdbwd.hip) is faster, and the launch chooses by grid size
// (stage1_qpair_rule). Bound by the fp32 matrix rate and, small grids, by the chain of a
// block: stage 1 at B2 N2048 H8 D64 causal 887 -> 631 us, at B1 N2048 H8 D128
// non-causal 1647 -> 1255.
//
// The two roles run separate copies of the sweep and must reach the same barriers:
// every one of them stands outside the role's and the mask's branches, and the number
// of tiles is the workgroup's.
#include "fhog_device.h"
#include "fhog_params.h"

#include <type_traits>

namespace fhog {

namespace {

constexpr int kPairs = 2;
constexpr int kWaves = 2 * kPairs;
constexpr int kThreads = 64 * kWaves;

template <int D> struct Occupancy {
  static constexpr int value = D == 64 ? 2 : 1;
};

template <int D, bool CAUSAL>
__global__ void __launch_bounds__(kThreads)
__attribute__((amdgpu_waves_per_eu(Occupancy<D>::value, Occupancy<D>::value)))
bwdbwd_qpair_kernel(BwdBwdParams<float> p, int chunk, int fold) {
  typedef float T;
  typedef SwzTile<T, D> G;
  constexpr int KS = D / 16;       // 16-deep steps over the head dim
  constexpr int DT = D / 32;       // 32-wide output column blocks
  constexpr int BQ = 32 * kPairs;  // queries per workgroup
  constexpr int BK = 32;           // keys per streamed tile
  constexpr int NST = 2;
  constexpr int kTile = G::kElems * (int)sizeof(T);
  constexpr int kStage = 4 * kTile;                    // K, V, ddK, ddV
  constexpr int kPart = G::kLoads / kWaves;            // loads of each tensor per wave
  constexpr int kExch = 32 * 32 * (int)sizeof(float);  // one tile of the exchange
  __shared__ __attribute__((aligned(1024))) char s_kv[NST * kStage];
  __shared__ __attribute__((aligned(1024))) char s_x[kPairs * 2 * kExch];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int pair = wave % kPairs;
  const int wave_role = wave / kPairs;  // 0 = A, 1 = B
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
  const int nkt = __builtin_amdgcn_readfirstlane(kend > 0 ? (kend + BK - 1) / BK : 0);  // tiles the workgroup streams
  int wend = p.nk;
  if (CAUSAL) wend = max(0, min(wend, q0 + 32 + p.coff));
  const int wkt = q0 < p.nq ? (wend + BK - 1) / BK : 0;  // tiles with work for this pair

  SwzFrags<T, D> fr;
  fr.init(lane);

  // Wave w streams quarter w of each tile; the key sequence is streamed twice
  // (iterations 0 .. nkt-1 and nkt .. 2 nkt - 1).
  const uint32_t row_bytes = (uint32_t)(rsk * (long)sizeof(T));
  TileDma<T, D, kPart> dma;
  dma.init(row_bytes, BK, lane, kPart * wave);
  const uint32_t lds0 = lds_base_u32(s_kv);
  const int total = 2 * nkt;
  auto issue = [&](int it) {
    const int kt = it < nkt ? it : it - nkt;
    const int nvalid = p.nk - kt * BK;
    const uint32_t stage = lds0 + (uint32_t)(((uint32_t)it % NST) * kStage);
    const long off = kbase + (long)kt * BK * rsk;
    if (nvalid >= BK) {
      dma.issue(stage, p.k + off);
      dma.issue(stage + kTile, p.v + off);
      dma.issue(stage + 2 * kTile, p.ddk + off);
      dma.issue(stage + 3 * kTile, p.ddv + off);
    } else {
      TileDma<T, D, kPart> part;
      part.init(row_bytes, nvalid, lane, kPart * wave);
      part.issue(stage, p.k + off);
      part.issue(stage + kTile, p.v + off);
      part.issue(stage + 2 * kTile, p.ddk + off);
      part.issue(stage + 3 * kTile, p.ddv + off);
    }
  };
  // Waits for tile `it`, then starts streaming the next one into the stage
  // every wave finished reading in the previous iteration (as it did the
  // exchange buffer).
  auto advance = [&](int it) {
    wait_vmem();
    __syncthreads();
    if (it + 1 < total) issue(it + 1);
  };
  const float scale = p.scale;
  const float c2 = scale * kLog2e;
  float* const xp = reinterpret_cast<float*>(s_x + pair * 2 * kExch) + 4 * lane;
  auto put = [&](int which, const f32x16& v) {
#pragma unroll
    for (int a = 0; a < 4; ++a)
      *reinterpret_cast<f32x4*>(xp + 1024 * which + 256 * a) = f32x4{v[4 * a], v[4 * a + 1], v[4 * a + 2], v[4 * a + 3]};
  };
  auto get = [&](int which, int a) { return *reinterpret_cast<const f32x4*>(xp + 1024 * which + 256 * a); };

  // Compiled once per role, so that neither keeps the other's operands.
  auto sweeps = [&](auto role_tag) {
    constexpr int role = decltype(role_tag)::value;
    V8<T> r0[KS], r1[role == 0 ? KS : 1];  // A: Q, ddQ; B: dO
    float dpart = 0.f;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const long off = qbase + (long)qi * rs + 16 * ks + 8 * g;
      if constexpr (role == 0) {
        r0[ks] = qvalid ? *reinterpret_cast<const V8<T>*>(p.q + off) : zero8<T>();
        r1[ks] = qvalid ? *reinterpret_cast<const V8<T>*>(p.ddq + off) : zero8<T>();
      } else {
        r0[ks] = qvalid ? *reinterpret_cast<const V8<T>*>(p.dout + off) : zero8<T>();
        const V8<T> of = qvalid ? *reinterpret_cast<const V8<T>*>(p.o + off) : zero8<T>();
#pragma unroll
        for (int e = 0; e < 8; ++e) dpart += of[e] * r0[ks][e];
      }
    }
    const float nL2 = role == 0 && qvalid ? -p.lse[sbase + qi] * kLog2e : 0.f;
    // Retire the query-side loads before the ring starts (see fwd_kernel).
    wait_vmem();
    if (total > 0) issue(0);

    // A: S and ddS (over scale) of the tile at sa, S turned into P and masked.
    f32x16 C0, C1;
    auto scores_a = [&](uint32_t sa, int kt) {
      C0 = zero16();
      C1 = zero16();
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const V8<T> kf = fr.rowf(sa, 0, ks);
        C0 = mma<T>(kf, r0[ks], C0);
        C1 = mma<T>(kf, r1[role == 0 ? ks : 0], C1);
        C1 = mma<T>(fr.rowf(sa, 2 * kTile, ks), r0[ks], C1);
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) C0[r] = exp2_fast(fmaf(C0[r], c2, nL2));
      const int k0 = kt * BK;
      if ((k0 + BK > p.nk) || (CAUSAL && k0 + BK - 1 > q0 + p.coff)) {
        const int klim = min(p.nk - 1, CAUSAL ? qi + p.coff : p.nk - 1) - k0;  // last visible key, tile-relative
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (crow(r, g) > klim) C0[r] = 0.f;
      }
    };

    // ---- sweep 1: A: dD; B: r2, r3 and P ddV ----
    f32x16 acc[DT];  // B: P ddV, then dQ2; A: ddO
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) acc[dt] = zero16();
    float dd_acc = 0.f, r2 = 0.f, r3 = 0.f;
    for (int it = 0; it < nkt; ++it) {
      advance(it);
      const uint32_t sa = lds0 + (uint32_t)(((uint32_t)it % NST) * kStage);  // K, V, ddK, ddV
      const bool active = it < wkt;
      if (active) {
        if constexpr (role == 0) {
          scores_a(sa, it);
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            C1[r] = C1[r] * C0[r];
            dd_acc += C1[r];
          }
          put(0, C0);
          put(1, C1);
        } else {
          C0 = zero16();
#pragma unroll
          for (int ks = 0; ks < KS; ++ks) C0 = mma<T>(fr.rowf(sa, kTile, ks), r0[ks], C0);
        }
      }
      __syncthreads();
      if constexpr (role == 1) {
        if (active) {
#pragma unroll
          for (int s = 0; s < 2; ++s) {
            f32x8 P;
#pragma unroll
            for (int a = 0; a < 2; ++a) {
              const f32x4 Pa = get(0, 2 * s + a), xa = get(1, 2 * s + a);
#pragma unroll
              for (int j = 0; j < 4; ++j) {
                const float dP = C0[8 * s + 4 * a + j];
                r3 = fmaf(dP, xa[j], r3);
                r2 = fmaf(dP, Pa[j], r2);
                P[4 * a + j] = Pa[j];
              }
            }
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) acc[dt] = mma<T>(fr.trf(sa, 3 * kTile, dt, s), P, acc[dt]);
          }
        }
      }
    }

    // ---- between the sweeps: dD to B, P ddV to A, the statistics to memory ----
    const float Di = xgroup_sum(dpart);
    float dD = xgroup_sum(dd_acc) * scale;
    float Bi = 0.f;
    __syncthreads();  // the exchange buffer is free
    if constexpr (role == 0) *(xp - 3 * lane) = dD;
    __syncthreads();
    if constexpr (role == 1) {
      dD = *(xp - 3 * lane);
      // r1 = <dO_i, (P ddV)_i>: the accumulator holds lane = query, registers = columns.
      float r1s = 0.f;
      if (qvalid) {
        const T* dorow = p.dout + qbase + (long)qi * rs;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
#pragma unroll
          for (int a = 0; a < 4; ++a) {
            const V4<T> x = *reinterpret_cast<const V4<T>*>(dorow + 32 * dt + 8 * a + 4 * g);
#pragma unroll
            for (int j = 0; j < 4; ++j) r1s = fmaf(x[j], acc[dt][4 * a + j], r1s);
          }
        }
      }
      Bi = xgroup_sum(r1s) - dD * xgroup_sum(r2) - Di * dD + xgroup_sum(r3) * scale;
      if (qvalid && g == 0) {
        p.delta[sbase + qi] = Di;
        p.ddelta[sbase + qi] = dD;
        p.bstat[sbase + qi] = Bi;
      }
    }
    // two column blocks at a time, the size of the buffer
#pragma unroll
    for (int d0 = 0; d0 < DT; d0 += 2) {
      __syncthreads();
      if constexpr (role == 1) {
        put(0, acc[d0]);
        put(1, acc[d0 + 1]);
        acc[d0] = acc[d0 + 1] = zero16();
      }
      __syncthreads();
      if constexpr (role == 0) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int a = 0; a < 4; ++a) {
            const f32x4 v = get(i, a);
#pragma unroll
            for (int j = 0; j < 4; ++j) acc[d0 + i][4 * a + j] = v[j];
          }
      }
    }

    // ---- sweep 2: A: ddO += P t V; B: dQ2 += P u ddK + P (dPa + u t - c) K ----
    const float nD = -Di, ndD = -dD, nc = -(Di * dD + Bi);
    for (int it = nkt; it < total; ++it) {
      advance(it);
      const uint32_t sa = lds0 + (uint32_t)(((uint32_t)it % NST) * kStage);  // K, V, ddK, ddV
      const bool active = it - nkt < wkt;
      if (active) {
        if constexpr (role == 0) {
          scores_a(sa, it - nkt);
#pragma unroll
          for (int r = 0; r < 16; ++r) C1[r] = fmaf(C1[r], scale, ndD);  // ddS - dD
          put(0, C0);
          put(1, C1);
        } else {
          C0 = zero16();
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
        // one 16-key half at a time
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          if constexpr (role == 0) {
            f32x8 ddP;
#pragma unroll
            for (int e = 0; e < 8; ++e) ddP[e] = C0[8 * s + e] * C1[8 * s + e];
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) acc[dt] = mma<T>(fr.trf(sa, kTile, dt, s), ddP, acc[dt]);
          } else {
            f32x8 dS, dS2;
#pragma unroll
            for (int a = 0; a < 2; ++a) {
              const f32x4 P = get(0, 2 * s + a), t = get(1, 2 * s + a);
#pragma unroll
              for (int j = 0; j < 4; ++j) {
                const int r = 8 * s + 4 * a + j;
                const float u = C0[r] + nD;                    // dP - D
                const float x = fmaf(u, t[j], C1[r]) + nc;     // dP2 - B
                dS[4 * a + j] = P[j] * u;
                dS2[4 * a + j] = P[j] * x;
              }
            }
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) {
              acc[dt] = mma<T>(fr.trf(sa, 2 * kTile, dt, s), dS, acc[dt]);
              acc[dt] = mma<T>(fr.trf(sa, 0, dt, s), dS2, acc[dt]);
            }
          }
        }
      }
    }

    if (qvalid) {
      T* dst = (role ? p.dq2 : p.ddo) + qbase + (long)qi * rs;
      // A row that sees exactly one key has a constant softmax: its dQ2 is
      // exactly 0, while the sums above cancel only to rounding of c.
      const bool one_key = (CAUSAL ? min(p.nk, qi + p.coff + 1) : p.nk) == 1;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
#pragma unroll
        for (int a = 0; a < 4; ++a) {
          f32x4 x;
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            x[j] = acc[dt][4 * a + j];
            if constexpr (role == 1) x[j] = one_key ? 0.f : x[j] * scale;
          }
          *reinterpret_cast<V4<T>*>(dst + 32 * dt + 8 * a + 4 * g) = x;
        }
      }
    }
  };
  if (wave_role == 0)
    sweeps(std::integral_constant<int, 0>{});
  else
    sweeps(std::integral_constant<int, 1>{});
}

}  // namespace

template <int D, bool CAUSAL>
hipError_t launch_bwdbwd_stage1_qpair(const BwdBwdParams<float>& p, hipStream_t stream) {
  const int nqb = (p.nq + 32 * kPairs - 1) / (32 * kPairs);
  const int npairs = p.batch * p.heads;
  const int cus = resident_workgroups(1);
  hipLaunchKernelGGL((bwdbwd_qpair_kernel<D, CAUSAL>), dim3(nqb * npairs), dim3(kThreads), 0, stream, p,
                     grid_chunk(npairs, nqb, Occupancy<D>::value * cus),
                     fold_rank(CAUSAL && Occupancy<D>::value == 2, nqb, npairs, cus));
  return hipGetLastError();
}

#define FHOG_INST(D, C) template hipError_t launch_bwdbwd_stage1_qpair<D, C>(const BwdBwdParams<float>&, hipStream_t);
FHOG_INST(64, true)
FHOG_INST(64, false)
FHOG_INST(128, true)
FHOG_INST(128, false)
#undef FHOG_INST

}  // namespace fhog
