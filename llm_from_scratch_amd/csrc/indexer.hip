// FP8 lightning-indexer scores for gfx950 (the DSA indexer's fp8_index,
// model/attention/utils.py:175-250 of the reference):
//
//   o[b, m, n] = k_s[b, n] * sum_h relu(q[b, m, h, :] . k[b, n, :]) * q_s[b, m, h]
//
// q, k e4m3fn; the dot products on v_mfma_f32_16x16x128_f8f6f4 (head dim
// d <= 128, zero-padded to 128), fp32 everywhere after.  A 16-head block of
// q[b, m] is the first operand and a 16-key block of k[b] the second, so
// lane l ends with key (l % 16) and heads 4(l / 16) .. +3 of the block: the
// ReLU, the head weights and three of the head sums stay in the lane; the
// sums of four key blocks then meet by halving (lane distance 16, 32), which
// leaves lane l with key l of the 64, a whole line per store.
//
// Bound: the VALU beside the MFMAs.  A score costs a multiply that clamps to
// [0, 1] (ReLU: |q . k| < 2^25, so the scores are taken times 2^-25, exactly)
// and an fma; the scale comes back as 2^12 in the weights and 2^13 at the end,
// powers of two.  fmaxf costs two v_max_f32 (the first quiets a signaling
// NaN), which run at half the rate of a multiply: 1 x 4096 x 4096, 64 heads,
// D 128: 190 -> 173 us.  The same bits as fmaxf while no weight makes a
// product lose bits below 2^-149 or a sum pass 2^128 on one scale and not on
// the other: every weight 0 or in [2^-95, 2^95) (scores are multiples of
// 2^-18, at most 128 of them meet).  A query with any other weight -- larger,
// smaller, infinite, NaN -- sits the walk out and is computed after it, with
// fmaxf and its weights unscaled (a second form inside the walk cost it 1 %
// and, at few heads, registers past an occupancy step: 8.6 -> 10.7 us).
//
// One workgroup per (b, 8 queries, chunk of nchunk keys), one wave per
// query; the wave keeps its query's H/16 operand fragments in registers.
// The chunk's keys pass through LDS in tiles of 128, loaded once for the
// eight waves (double-buffered, the next tile's global loads in flight
// during the current tile's MFMAs).  Operand K bytes: lane l supplies
// 16-byte chunks g and g + 4 (g = l / 16) of the 128-byte row for both q
// and k -- the same permutation of the head dim on both sides -- so the
// sixteen rows of one LDS read hit every bank once with the swizzle below.
#include "common.h"

namespace lfs {
namespace {

typedef int v8i __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));

constexpr int IDX_QPW = 8;  // queries (waves) per workgroup
// Keys per LDS tile: a barrier each, and the next tile's loads have one tile
// of MFMAs to land (4096 x 4096, 64 heads: 64 keys 151 us, 128 144, 256 143).
constexpr int IDX_KT = 128;
// Keys per workgroup, a multiple of the tile: every workgroup loads its
// queries first (64 KB at 64 heads of 128), so as many as still leave four
// workgroups per CU, two rounds (4096 x 4096: 512 keys 173 us, 1024 158, 2048
// 151, 4096 the same); below that short chunks, to spread a few queries'
// keys over the CUs.
constexpr int IDX_CHUNKS[] = {2048, 1024, 512, 256};
constexpr int64_t IDX_MIN_WG = 1024;

// head weights whose scores may be summed on the scale of 2^-13 (see above)
__device__ __forceinline__ bool weight_scales(float w) {
  const unsigned e = (__float_as_uint(w) >> 23) & 0xFF;
  return (e >= 127 - 95 && e < 127 + 95) || w == 0.f;
}

// byte offset of 16-byte chunk c of key row r in an LDS tile of D-byte rows
template <int D>
__device__ __forceinline__ int kswz(int r, int c) {
  if constexpr (D == 128) return r * 128 + ((c ^ (((r >> 1) & 7) ^ ((r & 1) << 2))) << 4);
  else if constexpr (D == 64) return r * 64 + ((c ^ ((r >> 2) & 3)) << 4);
  else return r * D + (c << 4);
}

// One wave's query against its workgroup's keys with fmaxf and the weights as
// they are, 16 keys and 16 heads at a time out of memory: the same products and
// sums.  Every index is formed again from an opaque thread id, so that the walk
// before it holds no register for it.
template <int HB, int D>
__device__ __attribute__((noinline)) void index_apart(const uint8_t* __restrict__ q, const float* __restrict__ q_s,
                                            const uint8_t* __restrict__ k, const float* __restrict__ k_s,
                                            float* __restrict__ o, int M, int N, int H, int64_t k_stride_b,
                                            int64_t ks_stride_b, int nchunk) {
  unsigned tid = threadIdx.x;
  asm volatile("" : "+v"(tid));
  const int lane = tid & 63, c16 = lane & 15, g = lane >> 4;
  const int b = blockIdx.z, m = blockIdx.y * IDX_QPW + __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n_begin = blockIdx.x * nchunk, n_end = min(N - n_begin, nchunk) + n_begin;
  const bool lo_ok = 16 * g < D, hi_ok = 16 * (g + 4) < D;
  const int64_t qrow = ((int64_t)b * M + m) * H;
  auto row = [&](const uint8_t* p, bool ok) -> v8i {
    uint4 lo = make_uint4(0, 0, 0, 0), hi = make_uint4(0, 0, 0, 0);
    if (ok && lo_ok) lo = *reinterpret_cast<const uint4*>(p + 16 * g);
    if (ok && hi_ok) hi = *reinterpret_cast<const uint4*>(p + 16 * (g + 4));
    return v8i{(int)lo.x, (int)lo.y, (int)lo.z, (int)lo.w, (int)hi.x, (int)hi.y, (int)hi.z, (int)hi.w};
  };
#pragma unroll 1
  for (int n0 = n_begin; n0 < n_end; n0 += 16) {
    const int n = n0 + c16;
    const v8i kf = row(k + (int64_t)b * k_stride_b + (int64_t)min(n, N - 1) * D, true);
    float acc = 0.f;
#pragma unroll 1
    for (int h0 = 0; h0 < 16 * HB; h0 += 16) {
      const v4f z = {0.f, 0.f, 0.f, 0.f};
      const v8i qf = row(q + (qrow + h0 + c16) * D, h0 + c16 < H);
      const v4f s = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(qf, kf, z, 0, 0, 0, 0, 0, 0);
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        const int hr = h0 + 4 * g + x;
        acc = fmaf(fmaxf(s[x], 0.f), hr < H ? q_s[qrow + hr] : 0.f, acc);
      }
    }
    acc = xor_sum<32>(xor_sum<16>(acc));
    if (g == 0 && n < n_end) o[((int64_t)b * M + m) * N + n] = acc * k_s[(int64_t)b * ks_stride_b + n];
  }
}

// HB: 16-head blocks.  The bound keeps 128 heads of 64 at 128 registers (130
// without: a workgroup per CU fewer, 110 -> 120 us at 2048 x 4096).
template <int HB, int D>
__global__ __launch_bounds__(64 * IDX_QPW, HB == 8 && D == 64 ? 4 : 1) void fp8_index_kernel(
    const uint8_t* __restrict__ q, const float* __restrict__ q_s, const uint8_t* __restrict__ k,
    const float* __restrict__ k_s, float* __restrict__ o, int M, int N, int H, int64_t k_stride_b,
    int64_t ks_stride_b, int nchunk) {
  constexpr int CPR = D / 16;                 // 16-byte chunks per key row
  constexpr int TCH = IDX_KT * CPR;           // chunks per LDS tile
  constexpr int NT = 64 * IDX_QPW;
  constexpr int CPT = (TCH + NT - 1) / NT;    // chunks per thread per tile
  __shared__ __attribute__((aligned(16))) uint8_t kt[2][IDX_KT * D];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int b = blockIdx.z, m = blockIdx.y * IDX_QPW + wave;
  bool active = m < M;  // inactive waves still take part in the barriers
  const int n_begin = blockIdx.x * nchunk;
  const int n_end = min(N - n_begin, nchunk) + n_begin;
  const int c16 = lane & 15, g = lane >> 4;
  const bool lo_ok = 16 * g < D, hi_ok = 16 * (g + 4) < D;  // this lane's chunks g, g + 4 exist

  // q fragments (head hb*16 + c16, chunks g and g + 4) and the weights of
  // the heads this lane's results belong to
  v8i qf[HB];
  float qw[HB][4];
  bool scaled = true;
  const int64_t qrow = ((int64_t)b * M + min(m, M - 1)) * H;
#pragma unroll
  for (int hb = 0; hb < HB; ++hb) {
    const int h = hb * 16 + c16;
    uint4 lo = make_uint4(0, 0, 0, 0), hi = make_uint4(0, 0, 0, 0);
    if (h < H) {
      const uint8_t* p = q + (qrow + h) * D;
      if (lo_ok) lo = *reinterpret_cast<const uint4*>(p + 16 * g);
      if (hi_ok) hi = *reinterpret_cast<const uint4*>(p + 16 * (g + 4));
    }
    qf[hb] = v8i{(int)lo.x, (int)lo.y, (int)lo.z, (int)lo.w, (int)hi.x, (int)hi.y, (int)hi.z, (int)hi.w};
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int hr = hb * 16 + 4 * g + r;
      const float w = hr < H ? q_s[qrow + hr] : 0.f;
      scaled = scaled && weight_scales(w);
      qw[hb][r] = w * 0x1p12f;
    }
  }
  const bool apart = active && __any(!scaled);  // the wave's lanes hold all heads of its query
  active = active && !apart;

  const uint8_t* kb = k + (int64_t)b * k_stride_b;
  const float* ksb = k_s + (int64_t)b * ks_stride_b;
  float* orow = o + ((int64_t)b * M + m) * N;
  // chunk u of tile starting at key t0: key t0 + u / CPR (clamped to the
  // last key; those rows are never stored), chunk u % CPR
  auto load_tile = [&](uint4 (&kr)[CPT], int t0) {
#pragma unroll
    for (int e = 0; e < CPT; ++e) {
      const int u = threadIdx.x + NT * e;
      kr[e] = make_uint4(0, 0, 0, 0);
      if (u < TCH) kr[e] = *reinterpret_cast<const uint4*>(kb + (int64_t)min(t0 + u / CPR, N - 1) * D + (u % CPR) * 16);
    }
  };
  auto store_tile = [&](const uint4 (&kr)[CPT], int buf) {
#pragma unroll
    for (int e = 0; e < CPT; ++e) {
      const int u = threadIdx.x + NT * e;
      if (u < TCH) *reinterpret_cast<uint4*>(&kt[buf][kswz<D>(u / CPR, u % CPR)]) = kr[e];
    }
  };

  const int ntiles = (n_end - n_begin + IDX_KT - 1) / IDX_KT;
  uint4 kr[CPT];
  load_tile(kr, n_begin);
  store_tile(kr, 0);
  __syncthreads();
  for (int ti = 0; ti < ntiles; ++ti) {
    const int t0 = n_begin + ti * IDX_KT;
    const int buf = ti & 1;
    if (ti + 1 < ntiles) load_tile(kr, t0 + IDX_KT);
    if (active) {
      const uint8_t* tile = kt[buf];
#pragma unroll
      for (int k64 = 0; k64 < IDX_KT; k64 += 64) {
        float sum[4];
#pragma unroll
        for (int st = 0; st < 4; ++st) {
          const int r = k64 + 16 * st + c16;
          uint4 lo = make_uint4(0, 0, 0, 0), hi = make_uint4(0, 0, 0, 0);
          if (lo_ok) lo = *reinterpret_cast<const uint4*>(tile + kswz<D>(r, g));
          if (hi_ok) hi = *reinterpret_cast<const uint4*>(tile + kswz<D>(r, g + 4));
          const v8i kf = v8i{(int)lo.x, (int)lo.y, (int)lo.z, (int)lo.w, (int)hi.x, (int)hi.y, (int)hi.z, (int)hi.w};
          float acc = 0.f;
#pragma unroll
          for (int hb = 0; hb < HB; ++hb) {
            const v4f z = {0.f, 0.f, 0.f, 0.f};
            // D[head][key]: lane holds key c16, heads hb*16 + 4g .. +3
            const v4f s = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(qf[hb], kf, z, 0, 0, 0, 0, 0, 0);
#pragma unroll
            for (int x = 0; x < 4; ++x)
              acc = fmaf(__builtin_amdgcn_fmed3f(s[x] * 0x1p-25f, 0.f, 1.f), qw[hb][x], acc);
          }
          sum[st] = acc;
        }
        const float tot = halve<32>(halve<16>(sum[0], sum[1]), halve<16>(sum[2], sum[3]));
        const int n = t0 + k64 + lane;
        if (n < n_end) orow[n] = (tot * 0x1p13f) * ksb[n];
      }
    }
    if (ti + 1 < ntiles) store_tile(kr, buf ^ 1);  // buffer buf ^ 1 was last read in tile ti - 1
    __syncthreads();
  }
  if (apart) index_apart<HB, D>(q, q_s, k, k_s, o, M, N, H, k_stride_b, ks_stride_b, nchunk);
}

}  // namespace
}  // namespace lfs

using namespace lfs;

extern "C" int lfs_fp8_index(const void* q, const float* q_s, const void* k, const float* k_s, float* o,
                             int64_t B, int32_t M, int32_t N, int32_t H, int32_t D, int64_t k_stride_b,
                             int64_t ks_stride_b, void* stream) {
  LFS_REQUIRE(B >= 0 && M >= 0 && N >= 0 && H > 0, "fp8_index: bad shape");
  LFS_REQUIRE(D == 32 || D == 64 || D == 128, "fp8_index: head_dim must be 32, 64 or 128 (got %d)", D);
  LFS_REQUIRE(H <= 128, "fp8_index: at most 128 heads (got %d)", H);
  if (B == 0 || M == 0 || N == 0) return 0;
  LFS_REQUIRE(q && q_s && k && k_s && o, "fp8_index: null pointer");
  LFS_REQUIRE(k_stride_b >= (int64_t)N * D && ks_stride_b >= N, "fp8_index: k batch stride too small");
  LFS_REQUIRE(((((uintptr_t)q) | ((uintptr_t)k)) & 15u) == 0 && (k_stride_b % 16) == 0,
              "fp8_index: q and k rows must be 16-byte aligned");
  LFS_REQUIRE(B < 65536 && (M + IDX_QPW - 1) / IDX_QPW < 65536, "fp8_index: grid too large");
  const int64_t rows = B * ((M + IDX_QPW - 1) / IDX_QPW);
  int nchunk = IDX_KT;
  for (const int c : IDX_CHUNKS)
    if (rows * (((int64_t)N + c - 1) / c) >= IDX_MIN_WG) {
      nchunk = c;
      break;
    }
  const dim3 grid((unsigned)(((int64_t)N + nchunk - 1) / nchunk), (unsigned)((M + IDX_QPW - 1) / IDX_QPW), (unsigned)B);
  hipStream_t st = (hipStream_t)stream;
  const int hb = (H + 15) / 16;
  const uint8_t *qq = (const uint8_t*)q, *kk = (const uint8_t*)k;
#define LFS_IX(HB, DD)                                                                                       \
  hipLaunchKernelGGL((fp8_index_kernel<HB, DD>), grid, dim3(64 * IDX_QPW), 0, st, qq, q_s, kk, k_s, o, M, N, H, \
                     k_stride_b, ks_stride_b, nchunk)
#define LFS_IXD(HB)                    \
  case HB:                             \
    if (D == 128) LFS_IX(HB, 128);     \
    else if (D == 64) LFS_IX(HB, 64);  \
    else LFS_IX(HB, 32);               \
    break;
  switch (hb) {
    LFS_IXD(1) LFS_IXD(2) LFS_IXD(3) LFS_IXD(4) LFS_IXD(5) LFS_IXD(6) LFS_IXD(7) LFS_IXD(8)
    default: LFS_REQUIRE(false, "fp8_index: unsupported head count %d", H);
  }
#undef LFS_IXD
#undef LFS_IX
  return check_launch("fp8_index");
}
