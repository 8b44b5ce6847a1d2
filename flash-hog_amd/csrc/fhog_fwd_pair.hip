// Flash attention forward with two waves per 32 queries, for 2-byte types at
// D = 256 and for fp32 on small grids (fhog_fwd.hip holds the other kernel and
// the definitions of O and L, fhog_grid.h the rule between them). Each wave of a pair holds half of Q's and
// half of O's columns: it forms its half of the contraction of S^T = K Q^T, adds
// its partner's half through LDS (fp32, accumulator layout: lane l reads what
// lane l of the partner wrote), takes the softmax of the whole tile and
// accumulates its columns of O^T = V^T P^T. Both add the same two numbers, so
// both hold the same P, running maximum and row sum.
//
// Why. One wave with all of Q and O ran one wave per SIMD at D = 256 (422
// registers) and fp32 D = 128, and 128-query workgroups made causal grids of one
// workgroup per CU as long as their longest block. Half of that state lets two
// waves share each SIMD, and a 64-query block takes half the matrix time per
// tile; the price is the softmax done twice and 16 KiB of exchange per tile
// beside 32 KiB of operand reads at D = 256. us, before -> with this kernel: B2
// N2048 H8 D256 causal bf16 107 -> 77, B4 N2048 H16 D256 248 -> 212, fp32 B2 N2048
// H8 D64 causal 140 -> 99, fp32 B1 N2048 H8 D128 non-causal 271 -> 166.
//
// The two halves run separate copies of the sweep and must reach the same barriers:
// every one of them stands outside the half's and the mask's branches, and the number
// of tiles is the workgroup's.
#include "fhog_device.h"
#include "fhog_params.h"

namespace fhog {

namespace {

constexpr int kPairs = 2;
constexpr int kWaves = 2 * kPairs;
constexpr int kThreads = 64 * kWaves;
// At least this many waves per SIMD; the fp32 D = 64 instance's 118 registers
// allow more (a bound of two: 312 -> 329 us at B4 N2048 H16 causal).
constexpr int kOcc = 2;

template <typename T, int D, bool CAUSAL>
__global__ void __launch_bounds__(kThreads)
__attribute__((amdgpu_waves_per_eu(kOcc, 8)))
fwd_pair_kernel(FwdParams<T> p, int chunk, int fold) {
  typedef SwzTile<T, D> G;
  constexpr int KS = D / 32;  // 16-deep steps of half the head dim
  constexpr int DT = D / 64;  // 32-wide column blocks of half of O
  constexpr int BQ = 32 * kPairs;
  constexpr int BK = 32;
  constexpr int NST = 2;
  constexpr int kTile = G::kElems * (int)sizeof(T);
  constexpr int kStage = 2 * kTile;  // K, V
  constexpr int kPer = G::kLoads / kPairs;
  constexpr int kExch = 32 * 32 * (int)sizeof(float);
  __shared__ __attribute__((aligned(1024))) char s_kv[NST * kStage];
  __shared__ __attribute__((aligned(1024))) char s_x[kWaves * kExch];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int pair = wave % kPairs;
  const int half = wave / kPairs;
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
  const int tensor = wave / kPairs;  // this wave streams half of each tile of K (0) or V (1)
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
  float* const xp = reinterpret_cast<float*>(s_x + wave * kExch) + 4 * lane;
  const float* const yp = reinterpret_cast<const float*>(s_x + (wave ^ kPairs) * kExch) + 4 * lane;

  auto sweep = [&](auto half_tag) {
    constexpr int HALF = decltype(half_tag)::value;
    // A negative scale is applied as |scale| to -Q (fwd_kernel).
    const bool negate = p.scale < 0.f;
    V8<T> qf[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const long off = qbase + (long)qi * rs + 16 * (HALF * KS + ks) + 8 * g;
      qf[ks] = qvalid ? *reinterpret_cast<const V8<T>*>(p.q + off) : zero8<T>();
      if (negate) qf[ks] = -qf[ks];
    }
    const float c2 = fabsf(p.scale) * kLog2e;  // > 0
    constexpr float kBound = 256.f;            // bound on P
    float m = -1e30f;                          // running row max of the log2-domain logits (possibly stale)
    float lpart = 0.f;                         // this lane's share of the running row sum
    f32x16 acc[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) acc[dt] = zero16();

    // Retire the query loads before the ring starts (fwd_kernel).
    wait_vmem();
    if (nkt > 0) issue(0);

    // After its first barrier of iteration kt every wave is done with tile
    // kt - 1, whose stage tile kt + 1 takes, and with the exchange buffer.
    for (int kt = 0; kt < nkt; ++kt) {
      wait_vmem();
      __syncthreads();
      if (kt + 1 < nkt) issue(kt + 1);
      const bool active = kt < wkt;
      const uint32_t sa = lds0 + (uint32_t)(((uint32_t)kt % NST) * kStage);  // K at 0, V at kTile
      f32x16 S;
      if (active) {
        S = zero16();
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) S = mma<T>(fr.rowf(sa, 0, HALF * KS + ks), qf[ks], S);
#pragma unroll
        for (int a = 0; a < 4; ++a)
          *reinterpret_cast<f32x4*>(xp + 256 * a) = f32x4{S[4 * a], S[4 * a + 1], S[4 * a + 2], S[4 * a + 3]};
      }
      __syncthreads();
      if (active) {
#pragma unroll
        for (int a = 0; a < 4; ++a) {
          const f32x4 y = *reinterpret_cast<const f32x4*>(yp + 256 * a);
#pragma unroll
          for (int j = 0; j < 4; ++j) S[4 * a + j] += y[j];
        }
        const int k0 = kt * BK;
        if ((k0 + BK > p.nk) || (CAUSAL && k0 + BK - 1 > q0 + p.coff)) {
          const int klim = min(p.nk - 1, CAUSAL ? qi + p.coff : p.nk - 1) - k0;  // last visible key, tile-relative
#pragma unroll
          for (int r = 0; r < 16; ++r)
            if (crow(r, g) > klim) S[r] = -INFINITY;
        }
        // The lazy rescale of fwd_kernel.
        f32x16 P;
        float psum = 0.f;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          P[r] = exp2_fast(fmaf(S[r], c2, -m));  // masked: exp2(-inf) = 0
          psum += P[r];
        }
        if (__any(!(psum <= kBound))) {
          float mloc = S[0];
#pragma unroll
          for (int r = 1; r < 16; ++r) mloc = fmaxf(mloc, S[r]);
          const float mnew = fmaxf(m, xgroup_max(mloc * c2));
          const float alpha = exp2_fast(m - mnew);
          lpart *= alpha;
#pragma unroll
          for (int dt = 0; dt < DT; ++dt) acc[dt] *= alpha;
          m = mnew;
          psum = 0.f;
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            P[r] = exp2_fast(fmaf(S[r], c2, -m));
            psum += P[r];
          }
        }
        lpart += psum;
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          const V8<T> oP = cvt8<T>(s ? hi8(P) : lo8(P));
#pragma unroll
          for (int dt = 0; dt < DT; ++dt) acc[dt] = mma<T>(fr.trf(sa, kTile, HALF * DT + dt, s), oP, acc[dt]);
        }
      }
    }

    // A query that sees no key gets O = 0 and L = +inf (fwd_kernel).
    const float l = xgroup_sum(lpart);
    if (qvalid) {
      const float inv = l > 0.f ? 1.f / l : 0.f;
      T* o = p.o + qbase + (long)qi * rs + HALF * (D / 2);
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
#pragma unroll
        for (int a = 0; a < 4; ++a) {
          f32x4 x;
#pragma unroll
          for (int j = 0; j < 4; ++j) x[j] = acc[dt][4 * a + j] * inv;
          *reinterpret_cast<V4<T>*>(o + 32 * dt + 8 * a + 4 * g) = cvt4<T>(x);
        }
      }
      if (HALF == 0 && g == 0) p.lse[sbase + qi] = l > 0.f ? (m + __log2f(l)) * kLn2 : INFINITY;
    }
  };
  if (half == 0)
    sweep(std::integral_constant<int, 0>{});
  else
    sweep(std::integral_constant<int, 1>{});
}

}  // namespace

template <typename T, int D, bool CAUSAL>
hipError_t launch_fwd_pair(const FwdParams<T>& p, hipStream_t stream) {
  const int nqb = (p.nq + 32 * kPairs - 1) / (32 * kPairs);
  const int npairs = p.batch * p.heads;
  const int cus = resident_workgroups(1);
  hipLaunchKernelGGL((fwd_pair_kernel<T, D, CAUSAL>), dim3(nqb * npairs), dim3(kThreads), 0, stream, p,
                     grid_chunk(npairs, nqb, kOcc * cus), fold_rank(CAUSAL, nqb, npairs, cus));
  return hipGetLastError();
}

#define FHOG_INST(T, D, C) template hipError_t launch_fwd_pair<T, D, C>(const FwdParams<T>&, hipStream_t);
FHOG_INST(__bf16, 256, true)
FHOG_INST(__bf16, 256, false)
FHOG_INST(_Float16, 256, true)
FHOG_INST(_Float16, 256, false)
FHOG_INST(float, 64, true)
FHOG_INST(float, 64, false)
FHOG_INST(float, 128, true)
FHOG_INST(float, 128, false)
#undef FHOG_INST

}  // namespace fhog
