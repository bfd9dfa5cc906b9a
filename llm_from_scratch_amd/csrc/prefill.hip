// Varlen causal prefill attention for gfx950 (the prefill half of the
// engine step).
//
// Sequence i of the batch has lq = cu_q[i+1] - cu_q[i] new query tokens
// (rows cu_q[i] .. of q) at positions lk - lq .. lk - 1 of its context of
// lk = cu_k[i+1] - cu_k[i] keys; query token p attends to keys 0 .. p
// (causal, aligned to the end of the context, as with a cached prefix).
// Key t of sequence i is row cu_k[i] + t of k / v (contiguous mode) or slot
// block_table[i][t / BS] * BS + t % BS of the KV pool (paged mode, a
// prefix-cache hit: the cached blocks and the just-stored new tokens).
//
// A kv head's work in one sequence is a list of lq * G rows (row r: query
// token r / G, query head r % G of the group), so a wave's 32 rows are full
// whatever G is.  One workgroup takes 32 * NW consecutive rows, one wave 32
// of them; the waves share 64-key K / V tiles in LDS, copied there directly
// (global_load_lds, no registers), the next tile's copies in flight while
// the current one is computed, one barrier per tile.  Per tile and wave:
//   S^T = K Q^T   v_mfma_f32_32x32x16_bf16: K rows from LDS as the A operand,
//                 Q^T preloaded as the B operand; lane l ends with the scores
//                 of row l % 32 for keys 8i + 4(l / 32) .. +3 of each 32-key
//                 block, so that max and sum need an exchange with lane
//                 l ^ 32 only;
//   softmax       online, log2 domain; O and the sum are rescaled only in
//                 the tiles where a row's maximum grows (not a looser bound:
//                 the weight of the largest key is then 1 and rounds to bf16
//                 exactly, which a lag of up to 2^8 gives up for 3 % of time
//                 and 3-4 % more error).  A tile's sum runs over the keys of
//                 each (key % 16) / 4 in turn, then (0 + 1) + (2 + 3): with
//                 the MFMAs' own order (eight k-indexes at a time) that makes
//                 the results those of 16x16x32 MFMAs over the same tiles,
//                 bit for bit;
//   O^T += V^T P^T  P^T is the B operand straight from the softmax registers:
//                 MFMA k-index 8h + j (h = l / 32) of key step x of a 32-key
//                 block stands for key 8x + 4h + j (j < 4) or 16 + 8x + 4h +
//                 j - 4 -- the same permutation of the keys on both operands
//                 leaves the sum unchanged; V^T is
//                 read transposed from the row-major V tile
//                 (ds_read_b64_tr_b16: 16 lanes read 4 keys x 16 dims and
//                 each gets one dim's four keys).
//
// Why this shape: 32x32 MFMAs do 32 rows per K and V^T fragment read (the
// 16x16 form read twice the LDS bytes per product and needed two exchanges
// for max and two for the sum), rows of all heads of the group keep the waves
// full for any G, and copying straight to LDS took the V transpose, its
// registers and its 32-bit LDS writes out.  Bound: at D = 128 the MFMAs are
// busy 45 % of the cycles and the VALU 55 % (the clock falls to 1.9 GHz under
// the load), at D = 64 the VALU 75 %: exp2 takes 8 cycles a wave, and
// max, fma, sum and rounding 2.5-5 each, per score.  Measured in turn on one
// card against a 16-row tile form (a wave per head, V transposed through
// registers): six prompts of 700-6000 tokens, half of each cached (GQA 32 / 8,
// D 128, paged): 1870 -> 568 us, 278 -> 914 TFLOP/s; 16 x 2048 tokens (12 / 4,
// D 64): 259 -> 149 us.  Short prompts keep that form (below).
// Not faster: 8 waves, 32-key tiles at three waves per SIMD, the next tile's
// scores computed beside this tile's weights, deeper operand reads, the sum
// on the MFMAs or v_dot2 (which does not overlap the MFMAs).
#include "common.h"

namespace lfs {
namespace {

typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef short v4s __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(3))) uint8_t lds_u8;

constexpr int KT = 64;               // keys per tile
constexpr int NW = 4;                // waves per workgroup
constexpr int RW = 32;               // rows (query token, head) per wave
// Workgroups per grid row: a launch takes less than 2^32 threads in x (a few
// prompts padded to a long max_seqlen_q pass that: 2^24 workgroups).  A
// multiple of 8, so the id in x fixes the XCD.  Ids past the last work item
// fall past the last tile.
constexpr int64_t kGridX = 1 << 20;

// N copies of 16 bytes per lane, from base + off[c] (per lane) to LDS address
// lds + 1024 c + 16 * lane.  The kernel waits for them before its barrier
// (the compiler does not see that they write LDS).  m0 is kept for the
// compiler; an LDS copy may not be the instruction after a write of m0.
template <int N>
__device__ __forceinline__ void copy_rows(const uint8_t* base, const unsigned (&off)[N], unsigned lds) {
  const uint64_t b = (uint64_t)(uintptr_t)base;
  i32x4 rsrc;
  rsrc[0] = __builtin_amdgcn_readfirstlane((int)(uint32_t)b);
  rsrc[1] = __builtin_amdgcn_readfirstlane((int)(uint32_t)(b >> 32)) & 0xFFFF;
  rsrc[2] = -1;
  rsrc[3] = 0x00020000;
  const unsigned dst = __builtin_amdgcn_readfirstlane(lds);
  unsigned keep;
  if constexpr (N == 2) {
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\tbuffer_load_dwordx4 %2, %4, 0 offen lds\n\t"
                 "s_add_u32 m0, m0, 0x400\n\ts_nop 0\n\tbuffer_load_dwordx4 %3, %4, 0 offen lds\n\ts_mov_b32 m0, %0"
                 : "=&s"(keep) : "s"(dst), "v"(off[0]), "v"(off[1]), "s"(rsrc) : "memory", "scc");
  } else {
    static_assert(N == 4, "2 or 4 copies per wave");
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\tbuffer_load_dwordx4 %2, %6, 0 offen lds\n\t"
                 "s_add_u32 m0, m0, 0x400\n\ts_nop 0\n\tbuffer_load_dwordx4 %3, %6, 0 offen lds\n\t"
                 "s_add_u32 m0, m0, 0x400\n\ts_nop 0\n\tbuffer_load_dwordx4 %4, %6, 0 offen lds\n\t"
                 "s_add_u32 m0, m0, 0x400\n\ts_nop 0\n\tbuffer_load_dwordx4 %5, %6, 0 offen lds\n\ts_mov_b32 m0, %0"
                 : "=&s"(keep) : "s"(dst), "v"(off[0]), "v"(off[1]), "v"(off[2]), "v"(off[3]), "s"(rsrc)
                 : "memory", "scc");
  }
}
__device__ __forceinline__ u32x4 lds_read16(unsigned a) {
  return *(const __attribute__((address_space(3))) u32x4*)(uintptr_t)a;
}
__device__ __forceinline__ void lds_write8(unsigned a, uint2 v) {
  typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
  *(__attribute__((address_space(3))) u32x2*)(uintptr_t)a = u32x2{v.x, v.y};
}
__device__ __forceinline__ uint2 lds_read_tr(unsigned a) {
  return __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                                       (__attribute__((address_space(3))) v4s*)(uintptr_t)a));
}

// 16-byte chunk c of key row r of a tile sits in chunk slot c ^ f(r).  K: the
// sixteen rows of an operand read (one chunk index) touch every bank once.
// V: the four rows of a transposed read (64 bytes each for 32 lanes) do.
template <int D>
__device__ __forceinline__ int kswz(int r) {
  return D == 64 ? (((r >> 1) & 7) ^ ((r & 1) << 2)) : (r & 15);
}
template <int D>
__device__ __forceinline__ int vswz(int r) {
  return D == 64 ? ((r >> 1) & 1) << 2 : (r & 3) << 2;
}

// x / v.d for x < 2^31, by the reciprocal that div_by() rounded up: the product's
// high word is the quotient or one more.
struct Div {
  unsigned d, inv;
};
inline Div div_by(unsigned d) { return Div{d, d == 1 ? 0u : (unsigned)((0xFFFFFFFFull + d) / d)}; }
__device__ __forceinline__ unsigned operator/(unsigned x, Div v) {
  const unsigned q = v.inv != 0 ? __umulhi(x, v.inv) : x;
  return q * v.d > x ? q - 1 : q;
}

// Inclusive sum over the wave's lanes.
__device__ __forceinline__ int scan_sum(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xF, 0xF, false);  // row_shr 1, 2, 4, 8
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xF, 0xF, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xF, 0xF, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xF, 0xF, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xA, 0xF, false);  // row_bcast 15: rows 1 and 3
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xC, 0xF, false);  // row_bcast 31: rows 2 and 3
  return v;
}

// A sequence's first query row and token, and their numbers.
struct Seq {
  int q0, lq, k0, lk;
};

// Row tile `tile` of sequence `seq` (the i-th) that comes at place `rank` when
// all tiles of R rows are ordered by the number of KT-key tiles they walk,
// longest first.  A launch fills the chip in id order and deals ids to the
// shader engines in turn, so ids in any other order leave engines or the tail
// idle (six cached prompts of 700-6000 tokens: 700 us with the sequences
// interleaved tile by tile, 551 us ranked).  With B <= 64 sequences lane s
// holds sequence s; N(c), the tiles that walk at least c key tiles, is one sum
// over the wave, and a binary search finds the largest c with N(c) > rank: the
// same few hundred cycles for any B (testing 64 thresholds a pass, each a loop
// over B, took 0.2 us per sequence from every workgroup, also from the empty
// ones of a ragged batch, which now leave after the first sum).  False (nothing
// set) for larger batches, whose many sequences even out, and for contexts
// whose arithmetic would not fit; tile is -1 past the last.
template <int R>
__device__ __forceinline__ bool ranked_item(const int32_t* cu_q, const int32_t* cu_k, int B, Div G, int rtiles,
                                            int rank, int& i, int& tile, Seq& seq) {
  if (B > 64) return false;
  const int lane = threadIdx.x & 63;
  int q0 = 0, lq = 0, k0 = 0, lk = 0, nt = 0, off = 0, most = 0;
  if (lane < B) {
    q0 = cu_q[lane], lq = cu_q[lane + 1] - q0;
    k0 = cu_k[lane], lk = cu_k[lane + 1] - k0;
    off = lk - lq;
    if (lq > 0) {
      if (off < 0 || lk > 1 << 26) {
        most = 1 << 30;
      } else {
        const unsigned tiles = ((unsigned)lq * G.d + R - 1) / R;
        nt = min((int)tiles, rtiles);
        most = (off + (int)((tiles * R - 1) / G) + KT) / KT;  // key tiles of the last tile (its full rows)
      }
    }
  }
  if (__any(most >= 1 << 30)) return false;
  // tiles of the lane's sequence that walk at least c >= 1 key tiles, and of all
  auto count = [&](int c) { return max(0, nt - max(0, (int)G.d * (KT * (c - 1) - off)) / R); };
  auto total = [&](int c) { return __builtin_amdgcn_readlane(scan_sum(count(c)), 63); };
  tile = -1;
  i = 0;
  int tlo = total(1), thi = 0;
  if (tlo <= rank) return true;
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) most = max(most, __shfl_xor(most, d, 64));
  int lo = 1, hi = __builtin_amdgcn_readfirstlane(most) + 1;  // N(lo) > rank >= N(hi) = thi
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1, n = total(mid);
    if (n > rank) lo = mid;
    else hi = mid, thi = n;
  }
  rank -= thi;
  const int n = count(lo), m = n - count(hi), incl = scan_sum(m);
  i = __builtin_ctzll(__ballot(incl > rank));
  tile = __builtin_amdgcn_readlane(nt - n - incl + m, i) + rank;
  seq.q0 = __builtin_amdgcn_readlane(q0, i), seq.lq = __builtin_amdgcn_readlane(lq, i);
  seq.k0 = __builtin_amdgcn_readlane(k0, i), seq.lk = __builtin_amdgcn_readlane(lk, i);
  return true;
}

template <int D, bool PAGED>
__global__ __launch_bounds__(64 * NW, 2) void prefill_attention_kernel(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ k, const uint16_t* __restrict__ v,
    const int32_t* __restrict__ cu_q, const int32_t* __restrict__ cu_k, const int32_t* __restrict__ bt,
    int64_t bt_stride, int64_t num_slots, uint16_t* __restrict__ out, Div dB, Div dHkv, Div G, Div dBS,
    int rtiles, int xshift, float scale_log2) {
  constexpr int NDC = D / 16;            // 16-dim MFMA k steps of S
  constexpr int NDB = D / 32;            // 32-dim blocks of O^T
  constexpr int RB = 2 * D;              // bytes of a tile row
  constexpr int TB = KT * RB;            // bytes of a tile
  constexpr int RPC = 1024 / RB;         // rows per copy instruction
  constexpr int NC = TB / 1024 / NW;     // copies per wave, tile and operand
  constexpr int RPW = KT / NW;           // tile rows a wave copies
  constexpr int NB = KT / 32;            // 32-key blocks of S^T
  static_assert(RPW <= 16 && RPW == NC * RPC, "a wave copies rows of one 16-key half");
  __shared__ __attribute__((aligned(1024))) uint8_t smem[4 * TB];  // K0, K1, V0, V1

  const int B = (int)dB.d, Hkv = (int)dHkv.d, BS = (int)dBS.d;
  // Work item of this workgroup.  Workgroup ids are dealt round-robin to the
  // 8 XCDs: XCD x takes kv head x >> xshift (2^xshift = 8 / Hkv where Hkv
  // divides 8: every 2^xshift-th row tile of it), so that a pair's K and V are
  // read through one or few L2s and ragged sequences still load the XCDs
  // evenly.
  int rank = blockIdx.y * gridDim.x + blockIdx.x, kh;
  if (xshift >= 0) {
    kh = (rank & 7) >> xshift;
    rank = ((rank >> 3) << xshift) + ((rank & 7) - (kh << xshift));
  } else {
    const int r = (int)((unsigned)rank / dHkv);
    kh = rank - r * Hkv;
    rank = r;
  }
  int i, tile;
  Seq seq;
  if (!ranked_item<RW * NW>(cu_q, cu_k, B, G, rtiles, rank, i, tile, seq)) {
    const int r = (int)((unsigned)rank / dB);
    i = rank - r * B;
    tile = rtiles - 1 - r;
    seq.q0 = cu_q[i], seq.lq = cu_q[i + 1] - seq.q0;
    seq.k0 = cu_k[i], seq.lk = cu_k[i + 1] - seq.k0;
  }
  const int q0 = seq.q0, lq = seq.lq, k0 = seq.k0, lk = seq.lk;
  if (tile < 0 || (int64_t)tile * (RW * NW) >= (int64_t)lq * G.d) return;  // the whole workgroup
  const unsigned r0 = (unsigned)tile * (RW * NW);  // its first row
  const int off = lk - lq;                 // position of query token 0
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int c32 = lane & 31, h = lane >> 5;
  const int Hq = Hkv * (int)G.d;
  const unsigned rows = (unsigned)lq * G.d;
  // this lane's row; rows past the sequence are computed as its last row and not stored
  const unsigned row = r0 + RW * wave + c32;
  const int tq = min(row, rows - 1) / G, hq = min(row, rows - 1) - tq * G.d;
  const int qp = off + tq;                 // its position
  // positions of the wave's first and last row, and of the workgroup's last
  const int pfirst = __builtin_amdgcn_readfirstlane(off + (int)(min(r0 + RW * wave, rows - 1) / G));
  const int plast = r0 + RW * wave >= rows  // (-1: none, the wave only copies)
                        ? -1 : __builtin_amdgcn_readfirstlane(off + (int)(min(r0 + RW * wave + RW - 1, rows - 1) / G));
  const int wlast = off + (int)(min(r0 + RW * NW - 1, rows - 1) / G);
  const int nkt = min(lk, wlast + 1) <= 0 ? 0 : (min(lk, wlast + 1) + KT - 1) / KT;
  const int64_t rowb = (int64_t)Hkv * RB;  // bytes per token of k / v
  const uint8_t* kb = reinterpret_cast<const uint8_t*>(k) + (int64_t)kh * RB;
  const uint8_t* vb = reinterpret_cast<const uint8_t*>(v) + (int64_t)kh * RB;
  const unsigned lbase = (unsigned)(uintptr_t)(const lds_u8*)smem;

  // Copies: instruction c of a wave fills rows RPW * wave + RPC * c .. of a
  // tile; lane l writes chunk slot l % (D / 8) of row l / (D / 8) and so
  // fetches the chunk that belongs there.
  const int crow = RPW * wave + lane / (D / 8);  // row of instruction 0
  unsigned krow[NC], vrow[NC];  // byte offsets from local row 0
  const int crow0 = PAGED ? crow & 15 : crow;
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const int r = crow + RPC * c;
    krow[c] = (unsigned)(crow0 + RPC * c) * (unsigned)rowb + (((lane % (D / 8)) ^ kswz<D>(r)) << 4);
    vrow[c] = (unsigned)(crow0 + RPC * c) * (unsigned)rowb + (((lane % (D / 8)) ^ vswz<D>(r)) << 4);
  }
  // Keys past the context read the row of key lk - 1: their weights are 0,
  // but their V rows still enter the product, so they must hold finite data
  // (pool slots past a sequence's keys may hold anything).  Paged: BS % 16
  // == 0, so the 16-key half that a wave copies rows of lies in one block;
  // an invalid table entry reads slot 0.  The entry is loaded one tile ahead.
  const int hoff = (RPW * wave) & ~15;  // the wave's half within a tile
  int blk = 0, boff = 0, lblk = 0, loff = 0;  // block and offset of the half's first key, and of key lk - 1
  if constexpr (PAGED) {
    boff = hoff;
    while (boff >= BS) boff -= BS, ++blk;
    lblk = (int)((unsigned)max(lk - 1, 0) / dBS), loff = max(lk - 1, 0) - lblk * BS;
  }
  auto entry = [&](int t) -> int {  // table entry of the half that starts at key t
    int64_t e = (int64_t)i * bt_stride + min((int64_t)(t < lk ? blk : lblk), bt_stride - 1);
    asm volatile("" : "+v"(e));  // a vector load: it returns before the barrier, with the copies
    return bt[e];
  };
  int next = 0;
  if constexpr (PAGED) next = entry(hoff);
  // copies of the K or V rows of the tile at key t0 into buffer buf (0 / 1;
  // V tiles are buffers 2 / 3); first: token or slot of its local row 0
  auto fetch = [&](const uint8_t* base, int64_t first, int t0, int buf, const unsigned (&rows16)[NC]) {
    const int valid = PAGED ? max(0, lk - 1 - (t0 + hoff)) : lk - 1 - t0;  // last local row that may be read
    const uint8_t* p = base + first * rowb;
    const unsigned dst = lbase + buf * TB + RPW * wave * RB;
    if (valid >= (PAGED ? 15 : KT - 1)) {
      copy_rows<NC>(p, rows16, dst);
    } else {
      unsigned at[NC];
#pragma unroll
      for (int c = 0; c < NC; ++c)  // rows past the last one read it
        at[c] = rows16[c] - (unsigned)max(0, crow0 + RPC * c - valid) * (unsigned)rowb;
      copy_rows<NC>(p, at, dst);
    }
  };
  int64_t kfirst = 0;  // local row 0 of the K tile last fetched
  auto fetch_k = [&](int t0, int buf) {
    if constexpr (PAGED) {
      const int b = __builtin_amdgcn_readfirstlane(next);
      kfirst = b < 0 || (int64_t)b * BS >= num_slots ? 0 : (int64_t)b * BS + (t0 + hoff < lk ? boff : loff);
      boff += KT;
      while (boff >= BS) boff -= BS, ++blk;
    } else {
      kfirst = (int64_t)k0 + t0;
    }
    fetch(kb, kfirst, t0, buf, krow);
    if constexpr (PAGED) next = entry(t0 + KT + hoff);
  };

  // Q^T (B operand): lane l supplies row l % 32, dims 16c + 8h .. +7
  v8bf qb[NDC];
  {
    const uint16_t* qr = q + ((int64_t)(q0 + tq) * Hq + (int64_t)kh * G.d + hq) * D + 8 * h;
#pragma unroll
    for (int c = 0; c < NDC; ++c) {
      qb[c] = __builtin_bit_cast(v8bf, *reinterpret_cast<const uint4*>(qr + 16 * c));
    }
  }
  v16f o[NDB];
#pragma unroll
  for (int db = 0; db < NDB; ++db)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[db][r] = 0.f;
  float m_run = -INFINITY, l_run = 0.f;

  // LDS addresses of the operand reads (tile 0, key 0); further chunks and
  // dim blocks are an xor, further keys an immediate offset
  const unsigned ka = lbase + c32 * RB + ((h ^ kswz<D>(c32)) << 4);
  const int il = lane & 15, gq = (lane >> 4) & 1;
  const unsigned va = lbase + 2 * TB + (4 * h + (il >> 2)) * RB +
                      (((2 * gq + ((il & 3) >> 1)) ^ vswz<D>(4 * h + (il >> 2))) << 4) + 8 * (il & 1);

  // The maximum the weights are taken against: 0 for a row that sees no key (a
  // position below 0), so that it ends as 0; else the running maximum, also
  // where that stays -infinity (every score overflowed), which makes the row
  // NaN, as a softmax over it is.
  const float m_none = qp < 0 ? 0.f : -INFINITY;
  float m_exp = m_none;
  float alpha = 1.f;   // the tile's rescaling of O and of the sum
  // the causal mask, only where the tile reaches past the wave's first row;
  // then the running maximum, and O and the sum on its scale
  auto mask_max = [&](v16f (&s)[NB], int t0) {
#pragma unroll
    for (int b = 0; b < NB; ++b) s[b] *= scale_log2;
    if (t0 + KT - 1 > pfirst) {
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (t0 + 32 * b + 8 * (r / 4) + 4 * h + r % 4 > qp) s[b][r] = -INFINITY;
    }
    float mx = s[0][0];
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[b][r]);
    mx = xor_max<32>(mx);
    alpha = 1.f;
    if (__any(mx > m_run)) {
      const float m_new = fmaxf(m_run, mx);
      alpha = m_new == m_run ? 1.f : __builtin_amdgcn_exp2f(m_run - m_new);
#pragma unroll
      for (int db = 0; db < NDB; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[db][r] *= alpha;
      m_run = m_new;
      m_exp = m_new == -INFINITY ? m_none : m_new;
    }
  };
  // weights of a tile on the hardware exp2 (results below 2^-126 flush to
  // 0), rounded to bf16, and their sum
  auto weights = [&](const v16f (&s)[NB], uint32_t (&pw)[NB][8]) {
    float ps[2] = {0.f, 0.f};
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int r = 0; r < 16; r += 2) {
        const float x = __builtin_amdgcn_exp2f(s[b][r] - m_exp);
        const float y = __builtin_amdgcn_exp2f(s[b][r + 1] - m_exp);
        pw[b][r / 2] = pack_bf16x2(x, y);
        ps[r / 4 & 1] += x;
        ps[r / 4 & 1] += y;
      }
    l_run = fmaf(l_run, alpha, xor_sum<32>(ps[0]) + xor_sum<32>(ps[1]));
  };
  auto k_frag = [&](int n, int buf) -> u32x4 {  // of MFMA n of S^T: 32-key block n % NB, 16 dims n / NB
    return lds_read16((ka ^ (32 * (n / NB))) + buf * TB + n % NB * 32 * RB);
  };
  auto v_frag = [&](int n, int buf) -> uint4 {  // of MFMA n of O^T: dim block n % NDB, key step n / NDB
    const unsigned a = (va ^ (64 * (n % NDB))) + buf * TB + (32 * (n / NDB / 2) + 8 * (n / NDB % 2)) * RB;
    const uint2 lo = lds_read_tr(a), hi = lds_read_tr(a + 16 * RB);
    return make_uint4(lo.x, lo.y, hi.x, hi.y);
  };
  constexpr int NS = NB * NDC, NP = KT / 16 * NDB;  // MFMAs of S^T and of O^T per tile
  constexpr int AH = 4;                             // operand reads ahead of them
  if (nkt > 0) {
    fetch_k(0, 0);
    fetch(vb, kfirst, 0, 2, vrow);
  }
  for (int j = 0; j < nkt; ++j) {
    const int t0 = j * KT, buf = j & 1;
    // tile j is in LDS for every wave; every wave is done with tile j - 1,
    // whose buffers the next copies fill
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    u32x4 kf[AH];
#pragma unroll
    for (int n = 0; n < AH; ++n) kf[n] = k_frag(n, buf);
    __builtin_amdgcn_sched_barrier(0);
    if (j + 1 < nkt) {
      fetch_k(t0 + KT, buf ^ 1);
      fetch(vb, kfirst, t0 + KT, 2 + (buf ^ 1), vrow);
    }
    if (t0 > plast) continue;  // the wave's rows end before this tile (it still copies)
    v16f s[NB];
    uint32_t pw[NB][8];
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int r = 0; r < 16; ++r) s[b][r] = 0.f;
#pragma unroll
    for (int n = 0; n < NS; ++n) {
      s[n % NB] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, kf[n % AH]), qb[n / NB], s[n % NB],
                                                          0, 0, 0);
      if (n + AH < NS) kf[n % AH] = k_frag(n + AH, buf);
      __builtin_amdgcn_sched_barrier(0);
    }
    uint4 vf[AH];
#pragma unroll
    for (int n = 0; n < AH; ++n) vf[n] = v_frag(n, buf);
    __builtin_amdgcn_sched_barrier(0);
    mask_max(s, t0);
    weights(s, pw);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int n = 0; n < NP; ++n) {
      const uint32_t* p = &pw[n / NDB / 2][n / NDB % 2 * 2];
      o[n % NDB] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, vf[n % AH]),
                                                           __builtin_bit_cast(v8bf, make_uint4(p[0], p[1], p[4], p[5])),
                                                           o[n % NDB], 0, 0, 0);
      if (n + AH < NP) vf[n % AH] = v_frag(n + AH, buf);
      __builtin_amdgcn_sched_barrier(0);
    }
  }

  // ---- normalise and store: lane l holds row l % 32, dims 32db + 8i + 4h .. +3,
  // 16 bytes of a line per row and instruction: the rows go through LDS
  // (swizzled as K's) and leave it with D / 8 lanes on each.  Stored from the
  // registers, a workgroup's lines were written in pieces for 1 us at D = 128
  // (32 / 8 heads, 64 prompts of 64: 25.6 -> 21.1 us, 65 of 128 64 -> 38, 64
  // of 512 300 -> 255).
  __syncthreads();  // every wave is done with the K and V tiles
  const unsigned ob = lbase + wave * (RW * RB);
  {
    const float inv = l_run > 0.f ? 1.f / l_run : 0.f;
#pragma unroll
    for (int db = 0; db < NDB; ++db)
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        uint2 w;
        w.x = pack_bf16x2(o[db][4 * x] * inv, o[db][4 * x + 1] * inv);
        w.y = pack_bf16x2(o[db][4 * x + 2] * inv, o[db][4 * x + 3] * inv);
        lds_write8(ob + c32 * RB + (((4 * db + x) ^ kswz<D>(c32)) << 4) + 8 * h, w);
      }
  }
  wave_lds_fence();
#pragma unroll
  for (int it = 0; it < RW / RPC; ++it) {
    const int r = RPC * it + lane / (D / 8), c = lane % (D / 8);
    const unsigned orow = r0 + RW * wave + r;
    const u32x4 v = lds_read16(ob + r * RB + ((c ^ kswz<D>(r)) << 4));
    if (orow < rows) {
      const int t = orow / G;
      *reinterpret_cast<u32x4*>(out + ((int64_t)(q0 + t) * Hq + (int64_t)kh * G.d + (orow - t * G.d)) * D + 8 * c) = v;
    }
  }
}

// ---- short prompts ----
//
// One workgroup per (sequence, 16 query tokens, kv head), one wave per query
// head of the group; 64-key K and V tiles go through registers into LDS, V
// transposed, and 16x16x32 MFMAs make the same sums.  Twice the waves of the
// kernel above at half the work each: where a call is one or few tiles long it
// ends sooner (the softmax of 16 rows a wave against 32), and never when tiles
// follow each other.  The rule is at prefill_short().
constexpr int QT = 16;                // query tokens per wave (one MFMA column block)
constexpr int NH = KT / 16;           // 16-key halves (S MFMA row blocks) per tile
constexpr int NKS = KT / 32;          // 32-key MFMA k steps of P.V per tile
constexpr int VT_PITCH = 2 * KT + 8;  // bytes per dim row of the transposed V tile (+ pad)

template <int D, int G, bool PAGED>
__global__ __launch_bounds__(64 * G) void prefill_short_kernel(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ k, const uint16_t* __restrict__ v,
    const int32_t* __restrict__ cu_q, const int32_t* __restrict__ cu_k, const int32_t* __restrict__ bt,
    int64_t bt_stride, Div dBS, int64_t num_slots, uint16_t* __restrict__ out, int Hkv, int qtiles, float scale_log2) {
  constexpr int NDC = D / 32;                        // 32-dim chunks (MFMA k steps of S)
  constexpr int NDB = D / 16;                        // 16-dim blocks of O^T
  constexpr int CPK = D / 8;                         // 16-byte chunks of a key row
  constexpr int VUN = KT / 2 * CPK;                  // (key pair, chunk) units of a V tile
  constexpr int NT = 64 * G;                         // threads
  constexpr int VPT = (VUN + NT - 1) / NT;           // units per thread
  constexpr int KUN = KT * CPK;                      // 16-byte chunks of a K tile
  constexpr int KPT = (KUN + NT - 1) / NT;           // chunks per thread
  __shared__ __attribute__((aligned(16))) uint8_t vt[2][D * VT_PITCH];
  __shared__ __attribute__((aligned(16))) uint8_t kt[2][KT * 2 * D];

  // each XCD takes a contiguous range of (sequence, kv head) pairs, whose
  // query tiles, last to first, share its L2
  const int nwg = gridDim.x * gridDim.y;
  int wid = blockIdx.y * gridDim.x + blockIdx.x;
  if ((nwg & 7) == 0) wid = (wid & 7) * (nwg >> 3) + (wid >> 3);
  const int pair = wid / qtiles;
  const int i = pair / Hkv, kh = pair - i * Hkv;
  const int tq0 = (qtiles - 1 - (wid - pair * qtiles)) * QT;  // the first query
  const int q0 = cu_q[i], lq = cu_q[i + 1] - q0;
  if (tq0 >= lq) return;  // the whole workgroup
  const int k0 = cu_k[i], lk = cu_k[i + 1] - k0;
  const int off = lk - lq;  // position of query token 0
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int h = kh * G + wave, Hq = Hkv * G;
  const int c16 = lane & 15, g = lane >> 4;
  const int64_t row = (int64_t)Hkv * D;  // elements per token row of k / v
  const int64_t hoff = (int64_t)kh * D;

  // Keys past the context read the row of key lk - 1: their weights are 0, but
  // their V rows still enter the product.  Paged: one table entry per 16-key
  // half (BS % 16 == 0); an invalid one reads slot 0.
  auto half_slot = [&](int tstart) -> int64_t {
    const int tc = min(tstart, lk - 1), c = (int)((unsigned)tc / dBS), BS = (int)dBS.d;
    const int32_t blk = bt[(int64_t)i * bt_stride + min((int64_t)c, bt_stride - 1)];
    return blk < 0 || (int64_t)blk * BS >= num_slots ? 0 : (int64_t)blk * BS + (tc - c * BS);
  };
  auto key_elem = [&](const int64_t (&hs)[NH], int t0, int kx) -> int64_t {  // key t0 + kx, kx < KT
    if constexpr (PAGED) return (hs[kx >> 4] + max(0, min(kx & 15, lk - 1 - (t0 + (kx & ~15))))) * row + hoff;
    else return ((int64_t)k0 + min(t0 + kx, lk - 1)) * row + hoff;
  };
  auto halves = [&](int64_t (&hs)[NH], int t0) {
#pragma unroll
    for (int hf = 0; hf < NH; ++hf) hs[hf] = PAGED ? half_slot(t0 + 16 * hf) : 0;
  };

  // Q^T (B operand): lane l supplies query tq0 + l % 16, dims 32c + 8g .. +7
  v8bf qb[NDC];
  {
    const int tq = tq0 + c16;
#pragma unroll
    for (int c = 0; c < NDC; ++c) {
      uint4 w = make_uint4(0, 0, 0, 0);
      if (tq < lq) w = *reinterpret_cast<const uint4*>(q + ((int64_t)(q0 + tq) * Hq + h) * D + c * 32 + g * 8);
      qb[c] = __builtin_bit_cast(v8bf, w);
    }
  }
  // this lane's query position; rows past lq are computed (finite) and not stored
  const int qp = min(off + tq0 + c16, lk - 1);
  // keys up to the last query of the tile
  const int nkt = (max(min(lk, off + tq0 + QT), 0) + KT - 1) / KT;

  // K tile in LDS: key rows of 2D bytes, 16-byte chunk c of row r at kswz
  auto kat = [](int r, int c) -> int { return r * 2 * D + ((c ^ kswz<D>(r)) << 4); };
  // chunk u of the tile: key u / CPK, chunk u % CPK (a row per CPK lanes)
  auto load_k = [&](uint4 (&kr)[KPT], const int64_t (&hs)[NH], int t0) {
#pragma unroll
    for (int e = 0; e < KPT; ++e) {
      const int u = threadIdx.x + NT * e;
      kr[e] = make_uint4(0, 0, 0, 0);
      if (u < KUN) kr[e] = *reinterpret_cast<const uint4*>(k + key_elem(hs, t0, u / CPK) + (u % CPK) * 8);
    }
  };
  auto store_kt = [&](const uint4 (&kr)[KPT], int buf) {
#pragma unroll
    for (int e = 0; e < KPT; ++e) {
      const int u = threadIdx.x + NT * e;
      if (u < KUN) *reinterpret_cast<uint4*>(&kt[buf][kat(u / CPK, u % CPK)]) = kr[e];
    }
  };
  // V unit u of a tile: key pair kp (keys 2kp, 2kp + 1), 16-byte chunk cc of
  // both rows; eight consecutive units cover the chunks of one pair (whole
  // rows per eight lanes), the pair index is swizzled by the chunk's high
  // half so that a wave's 32-bit LDS writes below hit distinct banks
  auto vunit = [&](int u, int& kp, int& cc) {
    cc = (u & 7) + 8 * ((u >> 3) / (KT / 2) % (CPK / 8));
    const int kpl = (u >> 3) % (KT / 2);
    kp = (kpl + 8 * ((u & 7) >> 2)) % (KT / 2);
  };
  auto load_v = [&](uint4 (&vr)[VPT][2], const int64_t (&hs)[NH], int t0) {
#pragma unroll
    for (int e = 0; e < VPT; ++e) {
      const int u = threadIdx.x + NT * e;
      vr[e][0] = vr[e][1] = make_uint4(0, 0, 0, 0);
      if (u < VUN) {
        int kp, cc;
        vunit(u, kp, cc);
        vr[e][0] = *reinterpret_cast<const uint4*>(v + key_elem(hs, t0, 2 * kp) + cc * 8);
        vr[e][1] = *reinterpret_cast<const uint4*>(v + key_elem(hs, t0, 2 * kp + 1) + cc * 8);
      }
    }
  };
  // transposed store: dim d of keys (2kp, 2kp + 1) as one 32-bit word at
  // vt[d][2kp]
  auto store_vt = [&](const uint4 (&vr)[VPT][2], int buf) {
#pragma unroll
    for (int e = 0; e < VPT; ++e) {
      const int u = threadIdx.x + NT * e;
      if (u < VUN) {
        int kp, cc;
        vunit(u, kp, cc);
        const uint32_t* a = reinterpret_cast<const uint32_t*>(&vr[e][0]);
        const uint32_t* b = reinterpret_cast<const uint32_t*>(&vr[e][1]);
#pragma unroll
        for (int x = 0; x < 4; ++x) {
          // dims 8cc + 2x (low halves) and 8cc + 2x + 1 (high halves)
          const uint32_t lo = (a[x] & 0xFFFFu) | (b[x] << 16);
          const uint32_t hi = (a[x] >> 16) | (b[x] & 0xFFFF0000u);
          *reinterpret_cast<uint32_t*>(&vt[buf][(8 * cc + 2 * x) * VT_PITCH + kp * 4]) = lo;
          *reinterpret_cast<uint32_t*>(&vt[buf][(8 * cc + 2 * x + 1) * VT_PITCH + kp * 4]) = hi;
        }
      }
    }
  };

  v4f o[NDB];
#pragma unroll
  for (int db = 0; db < NDB; ++db) o[db] = v4f{0.f, 0.f, 0.f, 0.f};
  float m_run = -INFINITY, l_run = 0.f;

  uint4 kr[KPT], vr[VPT][2];
  int64_t hs[NH];
  if (nkt > 0) {
    halves(hs, 0);
    load_k(kr, hs, 0);
    load_v(vr, hs, 0);
  }
  for (int j = 0; j < nkt; ++j) {
    const int t0 = j * KT;
    const int buf = j & 1;
    store_kt(kr, buf);
    store_vt(vr, buf);
    // K and V^T of tile j visible to every wave.  The buffers written next
    // (tile j+1) were last read in tile j-1, which every wave finished
    // before this barrier.
    __syncthreads();
    if (j + 1 < nkt) {
      halves(hs, t0 + KT);
      load_k(kr, hs, t0 + KT);
      load_v(vr, hs, t0 + KT);
    }
    const uint8_t* kb8 = kt[buf];

    // ---- S^T for the 16-key halves; the causal mask only where the tile
    // reaches past the tile's first query position
    const bool need_mask = t0 + KT - 1 > off + tq0;
    float s[NH][4];
    float tmax = -INFINITY;
#pragma unroll
    for (int kb = 0; kb < NH; ++kb) {
      v4f sc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int c = 0; c < NDC; ++c) {
        const uint4 kf = *reinterpret_cast<const uint4*>(kb8 + kat(16 * kb + c16, 4 * c + g));
        sc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, kf), qb[c], sc, 0, 0, 0);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        s[kb][r] = sc[r] * scale_log2;
        if (need_mask && t0 + 16 * kb + 4 * g + r > qp) s[kb][r] = -INFINITY;
        tmax = fmaxf(tmax, s[kb][r]);
      }
    }
    tmax = fmaxf(tmax, __shfl_xor(tmax, 16, 64));
    tmax = fmaxf(tmax, __shfl_xor(tmax, 32, 64));
    const float m_new = fmaxf(m_run, tmax), m_exp = m_new == -INFINITY && qp < 0 ? 0.f : m_new;
    const float alpha = m_new == m_run ? 1.f : __builtin_amdgcn_exp2f(m_run - m_new);
    float psum = 0.f;
    float p[NH][4];
#pragma unroll
    for (int kb = 0; kb < NH; ++kb)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        p[kb][r] = __builtin_amdgcn_exp2f(s[kb][r] - m_exp);
        psum += p[kb][r];
      }
    psum += __shfl_xor(psum, 16, 64);
    psum += __shfl_xor(psum, 32, 64);
    l_run = l_run * alpha + psum;
    m_run = m_new;

    // ---- O^T = O^T * alpha + V^T P^T, one MFMA k step per 32 keys
    v8bf pb[NKS];
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        pb[ks][r] = (__bf16)p[2 * ks][r];
        pb[ks][4 + r] = (__bf16)p[2 * ks + 1][r];
      }
    const uint8_t* vb = vt[buf];
#pragma unroll
    for (int db = 0; db < NDB; ++db) {
      const int dim = db * 16 + c16;
#pragma unroll
      for (int r = 0; r < 4; ++r) o[db][r] *= alpha;
#pragma unroll
      for (int ks = 0; ks < NKS; ++ks) {
        const uint2 lo = *reinterpret_cast<const uint2*>(vb + dim * VT_PITCH + (32 * ks + 4 * g) * 2);
        const uint2 hi = *reinterpret_cast<const uint2*>(vb + dim * VT_PITCH + (32 * ks + 16 + 4 * g) * 2);
        const uint4 w = make_uint4(lo.x, lo.y, hi.x, hi.y);
        o[db] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, w), pb[ks], o[db], 0, 0, 0);
      }
    }
  }

  // ---- normalise and store: lane l holds query tq0 + l % 16, dims 16db + 4g .. +3
  const int tq = tq0 + c16;
  if (tq < lq) {
    const float inv = l_run > 0.f ? 1.f / l_run : 0.f;
    uint16_t* dst = out + ((int64_t)(q0 + tq) * Hq + h) * D;
#pragma unroll
    for (int db = 0; db < NDB; ++db) {
      uint2 w;
      w.x = pack_bf16x2(o[db][0] * inv, o[db][1] * inv);
      w.y = pack_bf16x2(o[db][2] * inv, o[db][3] * inv);
      *reinterpret_cast<uint2*>(dst + db * 16 + 4 * g) = w;
    }
  }
}

// Whether a call goes to prefill_short_kernel: few and short tiles.  With w = B *
// q heads * 16-token tiles (its waves) and t = 64-key tiles of the longest
// context, to 256 keys: at D = 64 w * t <= 4096 (3072 from t = 3; one head a
// group, whose workgroup is a single wave, one tile and w <= 1024); at D = 128,
// where half as many workgroups fit a CU, w * t <= 2304 and groups of 2-6 (a
// single wave copies too slowly, eight hold a CU's LDS).  Through a block table
// one tile only, as its look-ups come before every tile's loads (16 of 64 keys
// 0.94 of the long form's time, 64 of 128 1.02, 64 of 256 1.06).
// us, short / long.  12 / 4 heads of 64: 1 prompt of 64 4.5 / 5.7, of 128 5.7 /
// 6.5, of 256 8.3 / 8.5, of 384 10.8 / 10.3; 64 prompts of 64 7.1 / 7.6, 32 of
// 128 8.9 / 8.0.  8 / 8 of 64: 1 of 64 4.9 / 5.5, 64 of 64 9.3 / 6.8.  32 / 8 of
// 128: 1 of 64 5.4 / 6.8, 8 of 64 6.0 / 7.3, 4 of 128 7.6 / 8.7, 8 of 128 9.8 /
// 9.6, 4 of 192 11.4 / 10.6.  8 / 8 of 128: 1 of 64 7.0 / 6.6.
inline bool prefill_short(bool paged, int64_t B, int Hq, int G, int D, int64_t max_q, int64_t max_k) {
  if (max_k > (paged ? KT : 256) || max_q > max_k) return false;
  const int64_t w = B * Hq * ((max_q + QT - 1) / QT), t = (max_k + KT - 1) / KT;
  if (D == 64) return G == 1 ? w * t <= 1024 && t == 1 : w * t <= (t <= 2 ? 4096 : 3072) && (G < 8 || t <= 3);
  return G >= 2 && G <= 6 && w * t <= 2304;
}

}  // namespace
}  // namespace lfs

using namespace lfs;

extern "C" int lfs_prefill_attention(const void* q, const void* k, const void* v, const int32_t* cu_seqlens_q,
                                     const int32_t* cu_seqlens_k, const int32_t* block_tables,
                                     int64_t bt_stride, int32_t block_size, int64_t num_slots, void* out,
                                     int64_t B, int32_t num_q_heads, int32_t num_kv_heads, int32_t head_dim,
                                     int32_t max_seqlen_q, float scale, void* stream) {
  return lfs_prefill_attention_max_k(q, k, v, cu_seqlens_q, cu_seqlens_k, block_tables, bt_stride, block_size, num_slots,
                                     out, B, num_q_heads, num_kv_heads, head_dim, max_seqlen_q, INT32_MAX, scale, stream);
}

extern "C" int lfs_prefill_attention_max_k(const void* q, const void* k, const void* v, const int32_t* cu_seqlens_q,
                                           const int32_t* cu_seqlens_k, const int32_t* block_tables,
                                           int64_t bt_stride, int32_t block_size, int64_t num_slots, void* out,
                                           int64_t B, int32_t num_q_heads, int32_t num_kv_heads, int32_t head_dim,
                                           int32_t max_seqlen_q, int32_t max_seqlen_k, float scale, void* stream) {
  const int Hq = num_q_heads, Hkv = num_kv_heads, D = head_dim;
  LFS_REQUIRE(B >= 0 && Hq > 0 && Hkv > 0 && max_seqlen_q >= 0, "prefill_attention: bad shape");
  LFS_REQUIRE(D == 64 || D == 128, "prefill_attention: head_dim must be 64 or 128 (got %d)", D);
  LFS_REQUIRE(Hq % Hkv == 0 && Hq / Hkv <= 8,
              "prefill_attention: num_q_heads (%d) must be a multiple of num_kv_heads (%d), ratio <= 8", Hq, Hkv);
  if (B == 0 || max_seqlen_q == 0) return 0;
  LFS_REQUIRE(q && k && v && cu_seqlens_q && cu_seqlens_k && out, "prefill_attention: null pointer");
  LFS_REQUIRE(((((uintptr_t)q) | ((uintptr_t)k) | ((uintptr_t)v) | ((uintptr_t)out)) & 15u) == 0,
              "prefill_attention: q, k, v and out must be 16-byte aligned");
  if (block_tables != nullptr) {
    LFS_REQUIRE(block_size > 0 && block_size % 16 == 0 && num_slots >= block_size && bt_stride > 0,
                "prefill_attention: bad paged KV geometry (block_size must be a multiple of 16)");
  }
  const int G = Hq / Hkv;
  const int64_t rtiles = ((int64_t)max_seqlen_q * G + RW * NW - 1) / (RW * NW);
  const int xshift = Hkv <= 8 && 8 % Hkv == 0 ? __builtin_ctz(8 / Hkv) : -1;
  const int64_t nt = xshift > 0 ? (rtiles + (1 << xshift) - 1) >> xshift << xshift : rtiles;
  LFS_REQUIRE(B * nt < ((1ll << 31) - kGridX) / Hkv && Hkv < 65536, "prefill_attention: grid too large");
  const int64_t wgs = B * nt * Hkv;
  const dim3 grid((unsigned)(wgs < kGridX ? wgs : kGridX), (unsigned)((wgs + kGridX - 1) / kGridX));
  const float sl2 = scale * 1.4426950408889634f;
  hipStream_t st = (hipStream_t)stream;
  if (prefill_short(block_tables != nullptr, B, Hq, G, D, max_seqlen_q, max_seqlen_k)) {
    const int qtiles = (max_seqlen_q + QT - 1) / QT;
    const dim3 sgrid((unsigned)(B * qtiles), (unsigned)Hkv);
#define LFS_PSP(DD, GG, PG)                                                                                        \
  hipLaunchKernelGGL((prefill_short_kernel<DD, GG, PG>), sgrid, dim3(64 * GG), 0, st, (const uint16_t*)q,         \
                     (const uint16_t*)k, (const uint16_t*)v, cu_seqlens_q, cu_seqlens_k, block_tables, bt_stride, \
                     div_by(PG ? block_size : 1), num_slots, (uint16_t*)out, Hkv, qtiles, sl2)
#define LFS_PS(DD, GG)                                                                                             \
  case GG:                                                                                                         \
    if (block_tables != nullptr) LFS_PSP(DD, GG, true);                                                            \
    else LFS_PSP(DD, GG, false);                                                                                   \
    break;
    if (D == 64) {
      switch (G) {
        LFS_PS(64, 1) LFS_PS(64, 2) LFS_PS(64, 3) LFS_PS(64, 4) LFS_PS(64, 5) LFS_PS(64, 6) LFS_PS(64, 7) LFS_PS(64, 8)
      }
    } else {
      switch (G) { LFS_PS(128, 2) LFS_PS(128, 3) LFS_PS(128, 4) LFS_PS(128, 5) LFS_PS(128, 6) }
    }
#undef LFS_PS
#undef LFS_PSP
    return check_launch("prefill_attention");
  }
  const Div dBS = div_by(block_tables != nullptr ? block_size : 1);
#define LFS_PF(DD, PG)                                                                                             \
  hipLaunchKernelGGL((prefill_attention_kernel<DD, PG>), grid, dim3(64 * NW), 0, st, (const uint16_t*)q,        \
                     (const uint16_t*)k, (const uint16_t*)v, cu_seqlens_q, cu_seqlens_k, block_tables,             \
                     PG ? bt_stride : 0, num_slots, (uint16_t*)out, div_by((unsigned)B), div_by(Hkv), div_by(G),   \
                     dBS, (int)rtiles, xshift, sl2)
  if (block_tables != nullptr) {
    if (D == 64) LFS_PF(64, true);
    else LFS_PF(128, true);
  } else {
    if (D == 64) LFS_PF(64, false);
    else LFS_PF(128, false);
  }
#undef LFS_PF
  return check_launch("prefill_attention");
}
