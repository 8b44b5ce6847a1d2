// dQ and D of the first backward with two waves per 32 queries (kernel 1 of
// fhog_bwd.hip, same math and bit-identical results): wave A of a pair holds Q
// and forms P = exp(scale Q K^T - L), wave B holds dO and forms D and
// u = dO V^T - D. Each writes its 32 x 32 tile to LDS in fp32, in the accumulator
// layout, and reads the other's, so both have dS = P u and each accumulates
// half of dQ's columns.
//
// Why. One wave per 32 queries holds Q, dO and all of dQ: at 2-byte D = 256 and
// for fp32 that ran one wave per SIMD (D = 256: 450 registers), 128 queries per
// workgroup, so a causal grid of one workgroup per CU was as long as its longest
// block. Half of that state lets two waves share a SIMD (230 registers at
// D = 256, 124 and 197 for fp32), and a 64-query block takes half the time per
// tile. The price is 16 KiB of exchange per tile beside 48 KiB of operand reads
// at D = 256 (24 at 2-byte D = 128, where the split loses on grids that fill the
// chip: B2 N2048 H32 362 -> 388 us).
//
// First backward (dK/dV kernel included), us, before -> with this kernel: B2
// N2048 H8 D256 causal bf16 247 -> 199, B4 N2048 H16 D256 642 -> 600, fp32 B2
// N2048 H8 D64 causal 378 -> 289, B4 N2048 H16 D64 1015 -> 976, B1 N2048 H8 D128
// non-causal 680 -> 494; 2-byte small grids: B1 N2048 H8 D128 118 -> 109.
//
// The two roles run separate copies of the sweep and must reach the same barriers:
// every one of them stands outside the role's and the mask's branches, and the number
// of tiles is the workgroup's.
#include "fhog_device.h"
#include "fhog_params.h"

namespace fhog {

namespace {

constexpr int kPairs = 2;
constexpr int kWaves = 2 * kPairs;
constexpr int kThreads = 64 * kWaves;
// At least this many waves per SIMD; the narrower instances' registers allow
// three or four (a bound of two: 430 -> 481 us for the first backward at B128 N512
// H12 D64 causal).
constexpr int kOcc = 2;
template <typename T, int D, bool CAUSAL>
__global__ void __launch_bounds__(kThreads)
__attribute__((amdgpu_waves_per_eu(kOcc, 8)))
bwd_qpair_kernel(BwdParams<T> p, int chunk, int fold) {
  typedef SwzTile<T, D> G;
  constexpr int KS = D / 16;
  constexpr int DT = D / 64;  // 32-column blocks of dQ per wave
  constexpr int BQ = 32 * kPairs;
  constexpr int BK = 32;
  constexpr int NST = 2;  // a third stage leaves room for one workgroup per CU at 512-byte rows, and gains nothing below
  constexpr int kTile = G::kElems * (int)sizeof(T);
  constexpr int kStage = 2 * kTile;  // K, V
  constexpr int kPer = G::kLoads / kPairs;
  constexpr int kExch = 32 * 32 * (int)sizeof(float);  // one of P and u
  __shared__ __attribute__((aligned(1024))) char s_kv[NST * kStage];
  __shared__ __attribute__((aligned(1024))) char s_x[kPairs * 2 * kExch];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int pair = wave % kPairs;
  const int wave_role = wave / kPairs;  // 0 = A (S, P), 1 = B (D, dP, u)
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

  // Keys [0, kend) are visible to some query of the workgroup, [0, wend) to
  // some query of this pair.
  int kend = p.nk;
  if (CAUSAL) kend = min(kend, qb * BQ + BQ + p.coff);
  const int nkt = __builtin_amdgcn_readfirstlane(kend > 0 ? (kend + BK - 1) / BK : 0);
  int wend = p.nk;
  if (CAUSAL) wend = max(0, min(wend, q0 + 32 + p.coff));
  const int wkt = q0 < p.nq ? (wend + BK - 1) / BK : 0;

  SwzFrags<T, D> fr;
  fr.init(lane);
  const int tensor = wave / kPairs;  // 0 = K, 1 = V
  const T* src = (tensor == 0 ? p.k : p.v) + kbase;
  const uint32_t row_bytes = (uint32_t)(rsk * (long)sizeof(T));
  TileDma<T, D, kPer> dma;
  dma.init(row_bytes, BK, lane, kPer * pair);
  const uint32_t lds0 = lds_base_u32(s_kv);
  auto issue = [&](int kt) {
    const int nvalid = p.nk - kt * BK;
    const uint32_t dst = lds0 + tensor * kTile + (uint32_t)(((uint32_t)kt % NST) * kStage);
    const T* gsrc = src + (long)kt * BK * rsk;
    if (nvalid >= BK) {
      dma.issue(dst, gsrc);
    } else {
      TileDma<T, D, kPer> part;
      part.init(row_bytes, nvalid, lane, kPer * pair);
      part.issue(dst, gsrc);
    }
  };

  const float scale = p.scale;
  // Compiled once per role, so that neither keeps the other's temporaries.
  auto sweep = [&](auto role_tag) {
    constexpr int role = decltype(role_tag)::value;
    V8<T> res[KS];  // A: Q, B: dO
    const T* rsrc = role ? p.dout : p.q;
    float dpart = 0.f;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const long off = qbase + (long)qi * rs + 16 * ks + 8 * g;
      res[ks] = qvalid ? *reinterpret_cast<const V8<T>*>(rsrc + off) : zero8<T>();
      if constexpr (role == 1) {
        const V8<T> of = qvalid ? *reinterpret_cast<const V8<T>*>(p.o + off) : zero8<T>();
        if constexpr (sizeof(T) == 2) {
          dpart = dot8<T>(of, res[ks], dpart);
        } else {
#pragma unroll
          for (int e = 0; e < 8; ++e) dpart += (float)of[e] * (float)res[ks][e];
        }
      }
    }
    const float Di = xgroup_sum(dpart);
    const float nL2 = qvalid && role == 0 ? -p.lse[sbase + qi] * kLog2e : 0.f;
    const float c2 = scale * kLog2e;
    constexpr bool kU0 = D == 64;  // as in bwd_q_kernel: the dP accumulator starts at -D
    f32x16 acc[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) acc[dt] = zero16();

    // Retire the query-side loads before the ring starts (see fwd_kernel).
    wait_vmem();
#pragma unroll
    for (int i = 0; i < NST - 1; ++i)
      if (i < nkt) issue(i);

    // After its first barrier of iteration kt every wave is done with tile
    // kt - 1, whose stage tile kt + 1 takes, and with the exchange buffer.
    for (int kt = 0; kt < nkt; ++kt) {
      wait_tile<NST, kPer>(kt, nkt);
      __syncthreads();
      if (kt + NST - 1 < nkt) issue(kt + NST - 1);
      const bool active = kt < wkt;
      const uint32_t sa = lds0 + (uint32_t)(((uint32_t)kt % NST) * kStage);  // K at 0, V at kTile
      float* xp = reinterpret_cast<float*>(s_x + pair * 2 * kExch) + 4 * lane;  // P, then u
      f32x16 C;
      if (active) {
#pragma unroll
        for (int r = 0; r < 16; ++r) C[r] = kU0 && role ? -Di : 0.f;
        const uint32_t srow = sa + role * kTile;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) C = mma<T>(fr.rowf(srow, 0, ks), res[ks], C);
        if constexpr (role == 0) {
#pragma unroll
          for (int r = 0; r < 16; ++r) C[r] = exp2_fast(fmaf(C[r], c2, nL2));
          const int k0 = kt * BK;
          if ((k0 + BK > p.nk) || (CAUSAL && k0 + BK - 1 > q0 + p.coff)) {
            const int klim = min(p.nk - 1, CAUSAL ? qi + p.coff : p.nk - 1) - k0;  // last visible key, tile-relative
#pragma unroll
            for (int r = 0; r < 16; ++r)
              if (crow(r, g) > klim) C[r] = 0.f;
          }
        } else if constexpr (!kU0) {
#pragma unroll
          for (int r = 0; r < 16; ++r) C[r] -= Di;
        }
#pragma unroll
        for (int a = 0; a < 4; ++a)
          *reinterpret_cast<f32x4*>(xp + 1024 * role + 256 * a) =
              f32x4{C[4 * a], C[4 * a + 1], C[4 * a + 2], C[4 * a + 3]};
      }
      __syncthreads();
      if (active) {
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          f32x8 vdS;
#pragma unroll
          for (int a = 0; a < 2; ++a) {
            const f32x4 y = *reinterpret_cast<const f32x4*>(xp + 1024 * (1 - role) + 256 * (2 * s + a));
#pragma unroll
            for (int j = 0; j < 4; ++j) vdS[4 * a + j] = C[8 * s + 4 * a + j] * y[j];  // dS / scale
          }
          const V8<T> oS = cvt8<T>(vdS);
#pragma unroll
          for (int dt = 0; dt < DT; ++dt) acc[dt] = mma<T>(fr.trf(sa, 0, role * DT + dt, s), oS, acc[dt]);
        }
      }
    }

    if (qvalid) {
      T* dq = p.dq + qbase + (long)qi * rs + role * (D / 2);
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
#pragma unroll
        for (int a = 0; a < 4; ++a) {
          f32x4 x;
#pragma unroll
          for (int j = 0; j < 4; ++j) x[j] = acc[dt][4 * a + j] * scale;
          *reinterpret_cast<V4<T>*>(dq + 32 * dt + 8 * a + 4 * g) = cvt4<T>(x);
        }
      }
      if (role == 1 && g == 0) p.delta[sbase + qi] = Di;
    }
  };
  if (wave_role == 0)
    sweep(std::integral_constant<int, 0>{});
  else
    sweep(std::integral_constant<int, 1>{});
}

}  // namespace

template <typename T, int D, bool CAUSAL>
hipError_t launch_bwd_qpair(const BwdParams<T>& p, hipStream_t stream) {
  const int nqb = (p.nq + 32 * kPairs - 1) / (32 * kPairs);
  const int npairs = p.batch * p.heads;
  const int cus = resident_workgroups(1);
  hipLaunchKernelGGL((bwd_qpair_kernel<T, D, CAUSAL>), dim3(nqb * npairs), dim3(kThreads), 0, stream, p,
                     grid_chunk(npairs, nqb, kOcc * cus), fold_rank(CAUSAL, nqb, npairs, cus));
  return hipGetLastError();
}

#define FHOG_INST(T, D, C) template hipError_t launch_bwd_qpair<T, D, C>(const BwdParams<T>&, hipStream_t);
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
