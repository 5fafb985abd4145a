// nibble_mfma.hip — attention over sealed int4 nibble pages on the matrix cores (head_dim 128).
//
// Same contract as nib_attn_kernel (nibble_kv.hip) for the sealed pages of an item: key position p counts for query
// position P when p <= P and, with a window w > 0, p + w > P; softmax with a running maximum in log2 units; the
// split partials (m, l, unnormalised acc) go to the same workspace rows, and the same merge kernel finishes them.
// The item's active fp32 page is taken along by the workgroups of its last split.
//
// Layout. A workgroup = 4 wavefronts serves one (item, query token, KV head, group of 4 query heads, context
// split); each wavefront walks 64-slot tiles = four 16-token chunks of pages (chunk G of a tile on lanes
// 16G..16G+15, a page of N tokens giving ceil(N/16) chunks).
//   staging:  global_load_lds copies a chunk's 16 K rows and 16 V rows of this KV head (64 B each) into LDS, the
//             four 16-byte pieces of row r stored in the order piece ^ (r & 3) so that the lanes' row reads below
//             hit different banks; the next tile's copies start as soon as this tile's words are in registers.
//   K phase:  lane = token. Half a word of nibbles becomes the f16 B operand (n - 8, exact) of v_mfma_f32_4x4x4f16
//             with its four dims in the order the masks take them (0 4 1 5 or 2 6 3 7 of the word); the 4 query heads
//             (split into f16 hi + lo for fp32-grade scores, dims in the same order) are broadcast as the A operand,
//             accumulating one score per head in the lane. One accumulator pair per scale block of the row (the
//             page's block size is 32, 64 or a multiple of 128): score = sum over blocks of k_scale * acc.
//   softmax:  one running maximum per head for each chunk group (a 16-lane DPP row, so the maximum is four DPP
//             steps), merged across the groups once after the loop; p goes to LDS with the tokens' V scales.
//   V phase:  lane (G, t) owns dims 8t..8t+7 of chunk G's tokens: it reads word t of four rows, transposes the
//             4 x 8 nibbles with v_perm into eight f16 B operands (4 tokens x 1 dim), and the A operand is p times
//             the V scale of its 32-dim block for those 4 tokens, as f16 hi + lo.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <utility>

#include "cf_device.hpp"
#include "nibble_kv.hpp"
#include "nibble_page.hpp"
#include "nibble_query.hpp"
#include "nibble_work.hpp"

namespace cfnib {
namespace {

typedef _Float16 half4_t __attribute__((ext_vector_type(4)));
typedef float float4_t __attribute__((ext_vector_type(4)));
typedef _Float16 half2_t __attribute__((ext_vector_type(2)));

constexpr int kD = 128;
constexpr int kWaves = 4;
constexpr uint32_t kRowBytes = kD / 2;                    // nibbles of one token's row of one KV head
constexpr uint32_t kChunkStride = 16 * kRowBytes + 64;   // staged 16-row chunk + a bank offset between chunks
constexpr uint32_t kTileBytes = 4 * kChunkStride;
constexpr float kNegInf = -__builtin_huge_valf();
constexpr float kLowest = -__FLT_MAX__;  // running maximum before the first token: below or equal to every finite score
constexpr float kWeightTop = 32768.0f;                    // of a weight in the accumulators' unit
constexpr int kUnitMax = 100;  // units 2^-100 to 2^100: V scales from 2^-85 (smaller ones lose bits) to 2^115

__device__ inline half4_t as_half4(uint32_t lo, uint32_t hi) {
  half4_t h;
  uint32_t *w = reinterpret_cast<uint32_t *>(&h);
  w[0] = lo;
  w[1] = hi;
  return h;
}

// Nibbles -> f16 values n - 8, exact: a nibble in bits 0-3 of a half under the exponent of 1024 (ulp 1) is 1024 + n,
// one in bits 4-7 under the exponent of 64 (ulp 1/16) is 64 + n, so that two masks of a word serve four nibbles, and
// one packed f16 add per two values takes the rest off. (The nibbles alone, as f16 denormals n * 2^-24 with the offset
// folded out of the sums, cost a third less, but the matrix cores align a denormal's product by its nominal exponent:
// the error against float64 grew from 3e-7 to 2e-5 - 2e-4.)
__device__ inline uint32_t and_or(uint32_t x, uint32_t mask, uint32_t bits) {  // one VALU (hipcc makes two with literals)
  uint32_t r;
  asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(r) : "v"(x), "s"(mask), "v"(bits));
  return r;
}
__device__ inline uint32_t low_nibbles(uint32_t x) {
  return __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2_t, and_or(x, 0x000F000Fu, 0x64006400u)) -
                                          half2_t{static_cast<_Float16>(1032.0f), static_cast<_Float16>(1032.0f)});
}
__device__ inline uint32_t high_nibbles(uint32_t x) {
  return __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2_t, and_or(x, 0x00F000F0u, 0x54005400u)) -
                                          half2_t{static_cast<_Float16>(72.0f), static_cast<_Float16>(72.0f)});
}

// K operand of half a word of nibbles n0..n7: values of {n0, n4, n1, n5} (U = 0) or {n2, n6, n3, n7} (U = 1), the order
// the masks take them in; the query operand holds its dims in the same order.
template <int U>
__device__ inline half4_t k_quad(uint32_t w) {
  const uint32_t x = U ? w >> 8 : w;
  return as_half4(low_nibbles(x), high_nibbles(x));
}
// dim inside the word of element e of half u
__device__ constexpr int k_dim(int u, int e) { return 2 * u + 4 * (e & 1) + (e >> 1); }

// Pointers read from the item table are generic; these casts make their loads global (vector) or constant
// (scalar) accesses, which the compiler does not have to order against the LDS DMA the way it orders FLAT loads.
#define CF_GLOBAL __attribute__((address_space(1)))
#define CF_CONST __attribute__((address_space(4)))
template <typename T>
__device__ inline const CF_GLOBAL T *gptr(const T *p) {
  return (const CF_GLOBAL T *)p;  // an address-space conversion (C-style cast)
}
template <typename T>
__device__ inline const CF_CONST T *cptr(const T *p) {
  return (const CF_CONST T *)p;
}

// Elements at byte offsets o0 and o1 of a query row (both loads in flight before either is converted).
__device__ inline float2 load_q2(const void *base, uint32_t type, uint64_t o0, uint64_t o1) {
  const CF_GLOBAL char *p = gptr(static_cast<const char *>(base));
  if (type == CF_DEVICE_F32)
    return make_float2(*reinterpret_cast<const CF_GLOBAL float *>(p + o0), *reinterpret_cast<const CF_GLOBAL float *>(p + o1));
  const uint16_t a = *reinterpret_cast<const CF_GLOBAL uint16_t *>(p + o0);
  const uint16_t b = *reinterpret_cast<const CF_GLOBAL uint16_t *>(p + o1);
  if (type == CF_DEVICE_F16)
    return make_float2(static_cast<float>(__builtin_bit_cast(_Float16, a)), static_cast<float>(__builtin_bit_cast(_Float16, b)));
  return make_float2(__uint_as_float(uint32_t(a) << 16), __uint_as_float(uint32_t(b) << 16));
}

// Maximum over the 16 lanes of a DPP row for four values at once; every lane of the row receives them. One asm
// statement with the four chains interleaved, so that each DPP source was written three VALU instructions earlier (a
// DPP read needs two wait states after the write of its source), behind one s_nop for the values' own writes.
__device__ inline void row_max4(float (&x)[4]) {
#define CF_DPP4(CTL)                                                                                               \
  "v_max_f32_dpp %0, %0, %0 " CTL "\n\tv_max_f32_dpp %1, %1, %1 " CTL "\n\tv_max_f32_dpp %2, %2, %2 " CTL       \
  "\n\tv_max_f32_dpp %3, %3, %3 " CTL "\n\t"
  asm volatile("s_nop 1\n\t"
               CF_DPP4("quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf")
               CF_DPP4("quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf")
               CF_DPP4("row_half_mirror row_mask:0xf bank_mask:0xf")
               CF_DPP4("row_mirror row_mask:0xf bank_mask:0xf")
               : "+v"(x[0]), "+v"(x[1]), "+v"(x[2]), "+v"(x[3]));
#undef CF_DPP4
}

// Two products a0 * b0 and a1 * b1 as f16 hi + lo (cfd::split2_mul_f16 with a factor each).
__device__ inline void split2p_f16(float a0, float b0, float a1, float b1, _Float16 &h0, _Float16 &l0, _Float16 &h1,
                                   _Float16 &l1) {
  const auto h = __builtin_amdgcn_cvt_pkrtz(a0 * b0, a1 * b1);
  h0 = static_cast<_Float16>(h[0]);
  h1 = static_cast<_Float16>(h[1]);
  l0 = static_cast<_Float16>(__builtin_fmaf(a0, b0, -static_cast<float>(h[0])));
  l1 = static_cast<_Float16>(__builtin_fmaf(a1, b1, -static_cast<float>(h[1])));
}

// LDS reads of the tile loop, in inline asm with their wait: the compiler cannot tell the tile being read from the one
// the next tile's global_load_lds copies are filling, and puts s_waitcnt vmcnt(0), the whole memory latency of the
// prefetch, before a plain read (at four tiles a wave the MFMA kernel took 67 us with plain reads).
typedef uint32_t uint4_t __attribute__((ext_vector_type(4)));
typedef uint32_t uint2_t __attribute__((ext_vector_type(2)));
__device__ inline uint32_t lds_addr(const void *p) { return static_cast<uint32_t>(reinterpret_cast<uintptr_t>(p)); }
__device__ inline void lds_read4_b128(uint4_t (&v)[4], uint32_t a0, uint32_t a1, uint32_t a2, uint32_t a3) {
  asm volatile(
      "ds_read_b128 %0, %4\n\tds_read_b128 %1, %5\n\tds_read_b128 %2, %6\n\tds_read_b128 %3, %7\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3])
      : "v"(a0), "v"(a1), "v"(a2), "v"(a3)
      : "memory");
}
// V phase: p and V scales of the lane's 16 slots (16 floats each from `p` and `s`), and one word of each of the 16
// rows: rows 4 tq + k at ak + 256 tq bytes (kRowBytes = 64).
__device__ inline void lds_read_v(float4_t (&pv)[4], float4_t (&sv)[4], uint2_t (&w)[4][2], uint32_t p, uint32_t s,
                                  uint32_t a0, uint32_t a1, uint32_t a2, uint32_t a3) {
  static_assert(kRowBytes == 64, "row offsets of the reads below");
  asm volatile(
      "ds_read2_b32 %8, %18 offset0:0 offset1:64\n\tds_read2_b32 %9, %18 offset0:128 offset1:192\n\t"
      "ds_read2_b32 %10, %19 offset0:0 offset1:64\n\tds_read2_b32 %11, %19 offset0:128 offset1:192\n\t"
      "ds_read2_b32 %12, %20 offset0:0 offset1:64\n\tds_read2_b32 %13, %20 offset0:128 offset1:192\n\t"
      "ds_read2_b32 %14, %21 offset0:0 offset1:64\n\tds_read2_b32 %15, %21 offset0:128 offset1:192\n\t"
      "ds_read_b128 %0, %16\n\tds_read_b128 %1, %16 offset:16\n\tds_read_b128 %2, %16 offset:32\n\t"
      "ds_read_b128 %3, %16 offset:48\n\tds_read_b128 %4, %17\n\tds_read_b128 %5, %17 offset:16\n\t"
      "ds_read_b128 %6, %17 offset:32\n\tds_read_b128 %7, %17 offset:48\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(pv[0]), "=&v"(pv[1]), "=&v"(pv[2]), "=&v"(pv[3]), "=&v"(sv[0]), "=&v"(sv[1]), "=&v"(sv[2]), "=&v"(sv[3]),
        "=&v"(w[0][0]), "=&v"(w[0][1]), "=&v"(w[1][0]), "=&v"(w[1][1]), "=&v"(w[2][0]), "=&v"(w[2][1]), "=&v"(w[3][0]),
        "=&v"(w[3][1])
      : "v"(p), "v"(s), "v"(a0), "v"(a1), "v"(a2), "v"(a3)
      : "memory");
}

__device__ inline void wave_sync_lds() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Attention of 4 query heads over the item's fp32 active page by one workgroup, on the VALU in fp32: a 16-lane row per
// token (see the call), two tokens' loads in flight. m, l and acc as in nib_mfma_kernel (m per row of lanes, l summed
// over lanes at the end: the row's first lane holds it).
__device__ void active_page(const AttnItem &it, const AttnShape &sh, uint32_t h, uint32_t qt, uint32_t qc, bool open,
                            int wave, int G, int t, float (&m)[4], float (&l)[4], float4_t (&acc)[8]) {
  const uint32_t gqa = sh.gqa, n = it.active_count;
  float q[4][8];
  {
    uint64_t off[4];
    bool ok[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      ok[j] = qc * 4 + j < gqa;
      off[j] = uint64_t(qt) * it.q_token_stride + uint64_t(h * gqa + (ok[j] ? qc * 4 + j : 0u)) * it.q_head_stride +
               uint64_t(8 * t) * it.q_elem_stride;
    }
    const bool packed = ((reinterpret_cast<uintptr_t>(it.q) | it.q_token_stride | it.q_head_stride) & 15u) == 0u;
    load_rows8<4>(q, it.q, it.q_type, off, it.q_elem_stride, packed);
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int e = 0; e < 8; ++e) q[j][e] = ok[j] ? q[j][e] : 0.0f;
  }
  const Visible seen = visible_range(it.q_begin + qt, it.window, open ? kOpenWindow : 0u);
  constexpr int kIn = 2;
  for (uint32_t t0 = 4u * wave + G; t0 < n; t0 += 16u * kIn) {  // (the rows of a wave may leave at different times)
    float4_t k[kIn][2], v[kIn][2];
#pragma unroll
    for (int u = 0; u < kIn; ++u) {
      const uint64_t base = (uint64_t(min(t0 + 16u * u, n - 1u)) * sh.kv_heads + h) * kD + 8u * t;
      const CF_GLOBAL float4_t *kp = reinterpret_cast<const CF_GLOBAL float4_t *>(gptr(it.active_k) + base);
      const CF_GLOBAL float4_t *vp = reinterpret_cast<const CF_GLOBAL float4_t *>(gptr(it.active_v) + base);
      k[u][0] = kp[0];
      k[u][1] = kp[1];
      v[u][0] = vp[0];
      v[u][1] = vp[1];
    }
#pragma unroll
    for (int u = 0; u < kIn; ++u) {
      const uint32_t tok = t0 + 16u * u, pos = it.active_begin + tok;
      const bool valid = tok < n && seen(pos);
      const float kf[8] = {k[u][0].x, k[u][0].y, k[u][0].z, k[u][0].w, k[u][1].x, k[u][1].y, k[u][1].z, k[u][1].w};
      const float vf[8] = {v[u][0].x, v[u][0].y, v[u][0].z, v[u][0].w, v[u][1].x, v[u][1].y, v[u][1].z, v[u][1].w};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        float d = 0.0f;
#pragma unroll
        for (int e = 0; e < 8; ++e) d = fmaf(q[j][e], kf[e], d);
        const float s = cfd::row16_sum(d) * it.scale_log2;
        if (!valid) continue;  // the whole row of lanes
        const float mn = fmaxf(m[j], s);
        // the maximum is never -inf (kLowest): a score of -inf (the tail's values are not checked) has no weight, and
        // one that is no number makes the row NaN, in a row of lanes that counts when states are merged
        const float a = __builtin_amdgcn_exp2f(m[j] - mn), p = __builtin_amdgcn_exp2f(s - mn);
        m[j] = mn;
        l[j] = l[j] * a + (t == 0 ? p : 0.0f);
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[e][j] = fmaf(p, vf[e], acc[e][j] * a);
      }
    }
  }
}

// MODE 1 / 2 / 4: sealed pages with that many scale blocks per row (block size known for the request).
// MODE kMfmaContract: a batched-items request (two's-complement nibbles, per-row scale blocks, no causal bound and
// an inclusive window): each page's own block size (a multiple of 32) gives one scale per 32-dim quarter of a row,
// and pages that mfma_page_ok refuses are left to the VALU kernel.
template <int MODE>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3, 3))) void nib_mfma_kernel(const AttnItem *__restrict__ items, WorkList work, AttnShape sh,
                                                       uint32_t qchunks, float *__restrict__ ws) {
  constexpr bool PG = MODE == static_cast<int>(kMfmaContract);
  constexpr int NB = PG ? 4 : MODE;
  constexpr uint32_t sx = PG ? 0x88888888u : 0u;  // two's-complement nibbles -> offset-8 (n ^ 8 = n + 8 mod 16)
  __shared__ __attribute__((aligned(16))) uint8_t s_kv[kWaves][2][kTileBytes];  // [wave][K, V]
  __shared__ __attribute__((aligned(16))) float s_p[kWaves][4][64];                // p per [head][slot]
  __shared__ __attribute__((aligned(16))) float s_vs[kWaves][NB][64];              // V scales per slot
  // A unit of `work` is one (item, query token, chunk of query heads, split) over all KV heads. Consecutive workgroups
  // go to consecutive XCDs, and a unit's KV heads read interleaved pieces of the same lines (a token's rows of all
  // heads lie side by side, 64 bytes each, its scales 16 bytes each), so the heads of a unit are 8 workgroups apart:
  // one XCD's L2, close in time. (Heads across XCDs fetched 1.5x the bytes at 32 sequences of 32768 tokens.)
  const uint32_t kvh = sh.kv_heads, gqa = sh.gqa;
  const uint32_t block = work_block(), oct = block / (8u * kvh), in_oct = block - oct * (8u * kvh);
  const uint32_t unit = 8u * oct + (in_oct & 7u), h = in_oct >> 3;
  if (unit >= work.total) return;
  const uint32_t ii = work_item(work.first, work.items, unit);
  const AttnItem &it = items[ii];
  // the item's units: split fastest, then the chunk of query heads, the query token
  const uint32_t local = unit - work.first[ii];
  const uint32_t y = local / it.page_splits, split = local - y * it.page_splits;
  const uint32_t qt = y / qchunks, qc = y - qt * qchunks;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int G = lane >> 4, t = lane & 15;
  const uint32_t qpos = it.q_begin + qt;
  const uint32_t window = it.window;

  const uint32_t cpp = (sh.page_size + 15u) / 16u;
  const uint32_t nchunks = it.page_count * cpp;
  const uint32_t ntiles = (nchunks + 3u) / 4u;
  const uint32_t tb = split * it.units_per_split;
  const uint32_t te = min(ntiles, tb + it.units_per_split);
  const cf_device_page_descriptor *pages = it.pages;

  float m_run[4], l_run[4];
  float4_t acc[8];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    m_run[j] = kLowest;
    l_run[j] = 0.0f;
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) acc[e] = float4_t{0, 0, 0, 0};
  // acc is kept in units of 2^-vunit (one per 16-lane row), which the largest V scale met so far sets: f16 hi + lo holds
  // a weight p * v_scale to 2^-25 of the unit, and in units of 1, with V scales around 0.3, that quantised small weights
  // (relative error of an output row against float64, 26 items of 500-12000 tokens: 3.2e-7, in this unit 2.4e-7)
  int vunit = kUnitMax;
  float vfac = ldexpf(1.0f, vunit);

  // per-lane metadata of the tile in flight: this lane's token (row of chunk G), its visibility and scales
  bool n_ok = false;
  float n_ks[NB], n_vs[NB];
#pragma unroll
  for (int s = 0; s < NB; ++s) n_ks[s] = n_vs[s] = 0.0f;

  // Chunks are counted over the item's pages, cpp to a page; a wave's next tile is 16 chunks on, so the position of
  // its tiles' chunk 0 (page, chunk of the page; wave-uniform) advances without a division.
  struct Pos {
    uint32_t page, sub;
  };
  const uint32_t step_p = 4u * kWaves / cpp, step_s = 4u * kWaves % cpp;
  auto next_chunk = [&](Pos p) { return p.sub + 1u < cpp ? Pos{p.page, p.sub + 1u} : Pos{p.page + 1u, 0u}; };
  auto next_tile = [&](Pos p) {
    p.page += step_p;
    p.sub += step_s;
    if (p.sub >= cpp) {
      p.sub -= cpp;
      ++p.page;
    }
    return p;
  };
  // Descriptor fields of this lane's chunk (G) of a tile, fetched one tile ahead of its copies with vector loads
  // (they land under the same vmcnt wait as the copies, and unlike scalar loads they do not hold up the LDS reads).
  // A chunk past the item's pages reads the last page's descriptor and counts no tokens.
  struct TileDesc {
    const uint8_t *kp, *vp;
    const float *ks, *vs;
    uint32_t tb, tc, bs, sub;
    bool in;
  };
  auto fetch = [&](Pos p0, TileDesc &d) {
    const Pos p1 = next_chunk(p0), p2 = next_chunk(p1), p3 = next_chunk(p2);
    const uint32_t pg = G == 0 ? p0.page : G == 1 ? p1.page : G == 2 ? p2.page : p3.page;
    d.sub = G == 0 ? p0.sub : G == 1 ? p1.sub : G == 2 ? p2.sub : p3.sub;
    d.in = pg < it.page_count;
    const CF_GLOBAL cf_device_page_descriptor *gp = gptr(pages) + min(pg, it.page_count - 1u);
    d.kp = gp->key_payload;
    d.vp = gp->value_payload;
    d.ks = gp->key_scales;
    d.vs = gp->value_scales;
    d.tb = gp->token_begin;
    d.tc = gp->token_count;
    d.bs = gp->block_size;
    if constexpr (PG) {  // a refused page: no tokens here (the VALU kernel reads it)
      d.in = d.in && mfma_page_ok(d.kp, d.vp, d.ks, d.vs, d.bs, gp->head_dim, d.tc, it.mfma_cap);
    }
  };
  // lane part of a copy's source offset: lane -> row r of the chunk, 16-byte piece (swizzled), this KV head
  const uint32_t copy_r = static_cast<uint32_t>(lane) >> 2;
  const uint32_t copy_off = h * kRowBytes + 16u * ((static_cast<uint32_t>(lane) & 3u) ^ (copy_r & 3u));
  // Copies of a tile's K (which = 0) or V rows into the wave's buffer (the descriptors have landed).
  auto stage = [&](const TileDesc &d, int which) {
    const uint32_t mtc = d.in ? d.tc : 0u;
    const uint64_t mp = reinterpret_cast<uintptr_t>(which ? d.vp : d.kp);
    auto uni = [](uint32_t v, int src) { return static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(v), src)); };
#pragma unroll
    for (int C = 0; C < 4; ++C) {
      const uint32_t tc = uni(mtc, 16 * C), off = uni(d.sub, 16 * C) * 16u;
      if (off >= tc) continue;  // past the pages, a refused page, a partial page's empty chunk: masked slots
      const uint8_t *src = reinterpret_cast<const uint8_t *>(
          uint64_t(uni(static_cast<uint32_t>(mp), 16 * C)) | (uint64_t(uni(static_cast<uint32_t>(mp >> 32), 16 * C)) << 32));
      // slots past the page's tokens re-read its last row; a page's payload is below 4 GiB (checked by the launch)
      const uint32_t goff = min(off + copy_r, tc - 1u) * (kvh * kRowBytes) + copy_off;
      __builtin_amdgcn_global_load_lds(reinterpret_cast<const CF_GLOBAL uint32_t *>(gptr(src) + goff),
                                       (__attribute__((address_space(3))) void *)(&s_kv[wave][which][C * kChunkStride]),
                                       16, 0, 0);
    }
  };
  // this lane's visibility and scales for a tile
  auto load_scales = [&](const TileDesc &d) {
    const uint32_t mtc = d.in ? d.tc : 0u;
    n_ok = false;
    const uint32_t tok = d.sub * 16u + static_cast<uint32_t>(t);
    if (d.sub * 16u < mtc) {
      const uint32_t pos = d.tb + tok;
      const uint32_t row = min(tok, mtc - 1u) * kvh + h;  // token-head row of the page
      if constexpr (PG) {
        n_ok = tok < mtc && (window == 0u || uint64_t(pos) + window >= qpos);
        // ceil(128 / block_size) blocks per row; quarter s (dims 32 s .. 32 s + 31) lies in block 32 s / block_size
        const uint32_t bs = d.bs, rb = row * ((128u + bs - 1u) / bs);
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          const uint32_t bi = rb + (32u * s) / bs;
          n_ks[s] = gptr(d.ks)[bi];
          n_vs[s] = gptr(d.vs)[bi];
        }
      } else {
        n_ok = tok < mtc && pos <= qpos && (window == 0u || uint64_t(pos) + window > qpos);
        // first scale of the row: block = row * 128 / block_size (block_size 32 / 64 / a multiple of 128)
        const uint32_t bi = NB == 4 ? row * 4u : NB == 2 ? row * 2u : row / (d.bs / 128u);
#pragma unroll
        for (int s = 0; s < NB; ++s) {
          n_ks[s] = gptr(d.ks)[bi + s];
          n_vs[s] = gptr(d.vs)[bi + s];
        }
      }
    }
  };

  uint32_t tile = tb + wave;
  TileDesc dnext;
  Pos pos{4u * tile / cpp, 4u * tile % cpp};  // of the tile that `dnext` describes
  if (tile < te) fetch(pos, dnext);  // in flight while the queries are loaded and split

  // ---- queries (scaled to log2 units) as f16 hi + lo in LDS, in the K operand's dim order, then in registers
  _Float16(*s_q)[4][kD] = reinterpret_cast<_Float16(*)[4][kD]>(&s_p[0][0][0]);
  static_assert(sizeof(s_p) >= 2 * 4 * kD * sizeof(_Float16), "query staging fits the probability tiles");
  {
    const int i = 2 * threadIdx.x, j = i / kD, dd = i % kD;  // elements dd and dd + 1 of operand order
    const bool ok = qc * 4 + j < gqa;
    const uint64_t row = uint64_t(qt) * it.q_token_stride + uint64_t(h * gqa + (ok ? qc * 4 + j : 0u)) * it.q_head_stride;
    auto dim = [](int x) { return (x & ~7) + k_dim((x >> 2) & 1, x & 3); };
    const float2 q = load_q2(it.q, it.q_type, row + uint64_t(dim(dd)) * it.q_elem_stride,
                             row + uint64_t(dim(dd + 1)) * it.q_elem_stride);
    cfd::split_mul_f16(ok ? q.x : 0.0f, it.scale_log2, s_q[0][j][dd], s_q[1][j][dd]);
    cfd::split_mul_f16(ok ? q.y : 0.0f, it.scale_log2, s_q[0][j][dd + 1], s_q[1][j][dd + 1]);
  }
  if (tile < te) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    stage(dnext, 0);
    stage(dnext, 1);
    load_scales(dnext);
    pos = next_tile(pos);
    if (tile + kWaves < te) fetch(pos, dnext);
  }
  __syncthreads();
  half4_t qhi[2], qlo[2];
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    const int qd = 16 * c + (lane >> 2);
    qhi[c] = *reinterpret_cast<const half4_t *>(&s_q[0][lane & 3][4 * qd]);
    qlo[c] = *reinterpret_cast<const half4_t *>(&s_q[1][lane & 3][4 * qd]);
  }
  __syncthreads();  // the query staging aliases the probability tiles
  // ---- the item's fp32 active page, with its last split: lane group G of wave w takes tokens 4 w + G, 4 w + G + 16,
  // ...; lane t owns dims 8t..8t+7 as in the V phase, so the page joins the wavefront's own state. Here, before the
  // tiles, its loads share the wait for the first tile's copies. (A launch of its own for the tails took 14 us of a
  // batch and added partials to merge.)
  if (it.active_count != 0u && split + 1u == it.page_splits)
  {
    active_page(it, sh, h, qt, qc, PG, wave, G, t, m_run, l_run, acc);
    // into the unit of its own magnitude
    float top = 0.0f;
#pragma unroll
    for (int e = 0; e < 8; ++e)
#pragma unroll
      for (int j = 0; j < 4; ++j) top = fmaxf(top, __builtin_fabsf(acc[e][j]));
    top = cfd::row16_max(top);
    if (top > 0.0f) vunit = min(max(15 - __builtin_amdgcn_frexp_expf(top), -kUnitMax), kUnitMax);
    vfac = ldexpf(1.0f, vunit);
#pragma unroll
    for (int e = 0; e < 8; ++e)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[e][j] *= vfac;
  }

  for (; tile < te; tile += kWaves) {
    // this tile's rows and scales and the next tile's descriptors have landed. K and V have one buffer each: the next
    // tile's K copies start when this tile's K words are in registers, its V copies, scales and the descriptors after
    // it when the V words are, so that each is in flight for about half a tile (with two buffers of each, two instead
    // of three workgroups fit a CU).
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    wave_sync_lds();
    const bool more = tile + kWaves < te;
    const bool tok_ok = n_ok;

    // ---- K: one score per head for this lane's token
    // four independent accumulator chains (x hi / lo): chain c holds quads of scale block c / CPS, and the quad
    // order below makes consecutive MFMAs hit different chains
    constexpr int CPS = 4 / NB;  // chains per scale block
    float4_t sa[4], sb[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) sa[c] = sb[c] = float4_t{0, 0, 0, 0};
    {
      const uint32_t kb = lds_addr(&s_kv[wave][0][G * kChunkStride + t * kRowBytes]);
      uint4_t pc[4];
      lds_read4_b128(pc, kb + 16 * (t & 3), kb + 16 * (1 ^ (t & 3)), kb + 16 * (2 ^ (t & 3)), kb + 16 * (3 ^ (t & 3)));
      if (more) stage(dnext, 0);
      uint32_t w16[16];
#pragma unroll
      for (int k = 0; k < 16; ++k) w16[k] = pc[k / 4][k % 4] ^ sx;
      [&]<int... I>(std::integer_sequence<int, I...>) {
        (
            [&] {
              constexpr int c = I % 4;                         // chain
              constexpr int blk = c / CPS, sub = c % CPS;      // scale block, position among its chains
              constexpr int q = blk * (32 / NB) + CPS * (I / 4) + sub;  // operand quad (half a word)
              const half4_t b = k_quad<q & 1>(w16[q / 2]);
              sa[c] = __builtin_amdgcn_mfma_f32_4x4x4f16(qhi[q / 16], b, sa[c], 4, q % 16, 0);
              sb[c] = __builtin_amdgcn_mfma_f32_4x4x4f16(qlo[q / 16], b, sb[c], 4, q % 16, 0);
            }(),
            ...);
      }(std::make_integer_sequence<int, 32>{});
    }
    // softmax: one running maximum per head for each 16-lane chunk group (a DPP row), merged after the loop
    float sc[4], mx[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      float v = 0.0f;
#pragma unroll
      for (int c = 0; c < 4; ++c) v = fmaf(n_ks[c / CPS], sa[c][j] + sb[c][j], v);
      sc[j] = tok_ok ? v : kNegInf;
      mx[j] = sc[j];
    }
    row_max4(mx);
    // V scales in the accumulators' unit: a weight p * v_scale * 2^vunit stays below 2^15 (by magnitude: the scales of
    // pages that a caller publishes may be negative)
    float vs[NB], vmax = 0.0f;
#pragma unroll
    for (int s = 0; s < NB; ++s) {
      vs[s] = n_vs[s] * vfac;
      vmax = fmaxf(vmax, __builtin_fabsf(vs[s]));
    }
    // raise the running maxima and the unit (and rescale the accumulators) only when some lane's grew
    bool grow = vmax >= kWeightTop;
#pragma unroll
    for (int j = 0; j < 4; ++j) grow |= mx[j] > m_run[j];
    if (__ballot(grow) != 0) {
      float top = 0.0f;
#pragma unroll
      for (int s = 0; s < NB; ++s) top = fmaxf(top, __builtin_fabsf(n_vs[s]));
      const int un = min(vunit, max(15 - __builtin_amdgcn_frexp_expf(cfd::row16_max(top)), -kUnitMax)), du = un - vunit;
      vunit = un;
      vfac = ldexpf(1.0f, un);
#pragma unroll
      for (int s = 0; s < NB; ++s) vs[s] = n_vs[s] * vfac;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float mn = fmaxf(m_run[j], mx[j]);
        const float alpha = __builtin_amdgcn_exp2f(m_run[j] - mn);
        l_run[j] *= alpha;
        const float beta = ldexpf(alpha, du);
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[e][j] *= beta;
        m_run[j] = mn;
      }
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float p = __builtin_amdgcn_exp2f(sc[j] - m_run[j]);  // 0 for a score of -inf
      l_run[j] += p;
      s_p[wave][j][lane] = p;
    }
#pragma unroll
    for (int s = 0; s < NB; ++s) s_vs[wave][s][lane] = vs[s];
    wave_sync_lds();

    // ---- V: out[head][8t + e] += sum over 4 tokens of p * v_scale * (nibble - 8)
    {
      const uint32_t vb = lds_addr(&s_kv[wave][1][G * kChunkStride]) + 4u * (t & 3);
      const int vset = NB == 4 ? (t >> 2) : NB == 2 ? (t >> 3) : 0;
      float4_t pv[4], sv[4];
      uint2_t wv[4][2];  // [row of a quad k][tq pair]: word t of rows 4 tq + k
      lds_read_v(pv, sv, wv, lds_addr(&s_p[wave][lane & 3][16 * G]), lds_addr(&s_vs[wave][vset][16 * G]),
                 vb + 16 * (t >> 2), vb + kRowBytes + 16 * ((t >> 2) ^ 1), vb + 2 * kRowBytes + 16 * ((t >> 2) ^ 2),
                 vb + 3 * kRowBytes + 16 * ((t >> 2) ^ 3));
      if (more) {
        stage(dnext, 1);
        load_scales(dnext);
        pos = next_tile(pos);
        if (tile + 2 * kWaves < te) fetch(pos, dnext);
      }
#pragma unroll
      for (int tq = 0; tq < 4; ++tq) {
        const float4_t pp = pv[tq], vv = sv[tq];
        half4_t a, al;  // p * v_scale as f16 hi + lo (fp32-grade weights, like the query operand)
        _Float16 h[4], l[4];
        split2p_f16(pp.x, vv.x, pp.y, vv.y, h[0], l[0], h[1], l[1]);
        split2p_f16(pp.z, vv.z, pp.w, vv.w, h[2], l[2], h[3], l[3]);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          a[k] = h[k];
          al[k] = l[k];
        }
        uint32_t wk[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) wk[k] = wv[k][tq / 2][tq % 2] ^ sx;
        half4_t bv[8];
#pragma unroll
        for (int j = 0; j < 4; ++j) {  // byte j of the four words: dims 8t + 2j (low nibbles), 8t + 2j + 1 (high)
          const uint32_t sel = uint32_t(j) | 0x0c00u | (uint32_t(4 + j) << 16) | 0x0c000000u;
          const uint32_t x01 = __builtin_amdgcn_perm(wk[1], wk[0], sel);  // [w0.bj, 0, w1.bj, 0]
          const uint32_t x23 = __builtin_amdgcn_perm(wk[3], wk[2], sel);
          bv[2 * j] = as_half4(low_nibbles(x01), low_nibbles(x23));
          bv[2 * j + 1] = as_half4(high_nibbles(x01), high_nibbles(x23));
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[e] = __builtin_amdgcn_mfma_f32_4x4x4f16(a, bv[e], acc[e], 0, 0, 0);
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[e] = __builtin_amdgcn_mfma_f32_4x4x4f16(al, bv[e], acc[e], 0, 0, 0);
      }
    }
    wave_sync_lds();
  }

  // ---- wavefront partial: bring the four chunk groups to a common maximum, then sum them (l over all lanes)
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const float mw = cfd::rows4_max(m_run[j]);
    const float f = __builtin_amdgcn_exp2f(m_run[j] - mw);
    const float g = ldexpf(f, -vunit);
    l_run[j] = cfd::rows4_sum(cfd::row16_sum(l_run[j] * f));
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e][j] = cfd::rows4_sum(acc[e][j] * g);
    m_run[j] = l_run[j] == 0.0f ? kNegInf : mw;  // nothing seen
  }
  __syncthreads();  // every wave is done with its tile buffers: reuse them for the partials
  float(*red)[4][kD + 2] = reinterpret_cast<float(*)[4][kD + 2]>(&s_kv[0][0][0]);
  if (lane < 16) {
#pragma unroll
    for (int e = 0; e < 8; ++e)
#pragma unroll
      for (int j = 0; j < 4; ++j) red[wave][j][8 * t + e] = acc[e][j];
  }
  if (lane < 4) {
    red[wave][lane][kD] = m_run[lane];
    red[wave][lane][kD + 1] = l_run[lane];
  }
  __syncthreads();
  const uint32_t stride = kD + 4u;
  float *base = ws + it.ws_offset + (uint64_t(split) * it.q_tokens + qt) * sh.q_heads * stride;
  for (int i = threadIdx.x; i < 4 * kD; i += 256) {
    const int j = i / kD, dd = i % kD;
    if (qc * 4 + j >= gqa) continue;
    float m = kNegInf;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) m = fmaxf(m, red[w][j][kD]);
    float l = 0.0f, o = 0.0f;
    if (m != kNegInf)
#pragma unroll
      for (int w = 0; w < kWaves; ++w) {
        const float mw = red[w][j][kD];
        if (mw == kNegInf) continue;
        const float f = __builtin_amdgcn_exp2f(mw - m);
        l = fmaf(red[w][j][kD + 1], f, l);
        o = fmaf(red[w][j][dd], f, o);
      }
    float *row = base + uint64_t(h * gqa + qc * 4 + j) * stride;
    row[dd] = o;
    if (dd == 0) {
      row[kD] = m;
      row[kD + 1] = l;
    }
  }
}

}  // namespace

uint64_t nib_mfma_units(const AttnItem &it, const AttnShape &sh) {
  return uint64_t(it.page_splits) * it.q_tokens * ((sh.gqa + 3u) / 4u);
}

hipError_t launch_nib_mfma(uint32_t nb, const AttnItem *items, const WorkList &work, const AttnShape &sh, float *ws,
                           hipStream_t stream) {
  if (sh.head_dim != kD || work.total == 0) return hipSuccess;
  const uint32_t qchunks = (sh.gqa + 3u) / 4u;
  const uint64_t blocks = (uint64_t(work.total) + 7u) / 8u * 8u * sh.kv_heads;
  if (blocks > 0x7fffffffu) return hipErrorInvalidValue;
  const dim3 grid = work_grid(blocks);
  switch (nb) {
    case 1: nib_mfma_kernel<1><<<grid, 256, 0, stream>>>(items, work, sh, qchunks, ws); break;
    case 2: nib_mfma_kernel<2><<<grid, 256, 0, stream>>>(items, work, sh, qchunks, ws); break;
    case kMfmaContract: nib_mfma_kernel<kMfmaContract><<<grid, 256, 0, stream>>>(items, work, sh, qchunks, ws); break;
    default: nib_mfma_kernel<4><<<grid, 256, 0, stream>>>(items, work, sh, qchunks, ws); break;
  }
  return hipPeekAtLastError();
}

}  // namespace cfnib
