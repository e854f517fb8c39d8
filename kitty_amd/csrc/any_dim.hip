// The quantized-KV path for head dimensions other than 128 (64 and 256).
//
// The reference takes the head dimension from the model's config and promotes a quarter of the key
// channels (kitty.py:39-44); its kernels take D as a parameter (kitty_quant_pack.py:42-45, 180-181;
// kitty_attention.py:59-62, 253-254).  The other kernels of this library are written for D = 128, the
// size of every model the reference names.  The kernels here cover the other sizes with the same
// arithmetic and the same storage format, one template parameter for D:
//
//   attn_any_kernel<D, false, 1>              decode attention over few tokens, split pass (the reference's order of
//                                             operations: fp16 dequantization with both roundings; matrix cores)
//   attn_any_kernel<D, true, NT>              chunked-prefill attention, in one pass or in shares
// Decode attention otherwise: any_decode.hip.
//
// Wire format for general D (PAGE = 128 tokens): a K page-head is 32 D bytes of low plane (channel d at
// 32 d), 32 d_boost bytes of high plane (slot s at 32 (D + s)) and D bytes of slot map; a V page-head is
// 128 rows of D / 4 bytes; metadata as for D = 128 with D resp. 128 (scale, zero) pairs per head.
#include <cmath>
#include <type_traits>

#include "any_dim.h"

namespace kitty {
// merge pass over independent rows (rows_merge.hip)
void launch_rows_merge(int D, const float* ws_ml, const float* ws_acc, void* out, int64_t rows, int num_splits,
                       bool keep_nan, hipStream_t stream);
namespace {

// Column tiles of 16 query rows per workgroup in chunked prefill: what 256 registers, that is two workgroups on a compute unit,
// leave room for.  (200 tokens over 8000 at D = 64, one share's worth of rounds each: 124 us with four, whose loop spills, 99
// with three; with 512 registers and the accumulators copied between the paths' registers, 141.)
// At D = 64 three, or two where blocks of 32 rows leave less of the chunk's edge empty; each block also costs what unpacking
// a tile does, about 0.6 of a column tile.  (1000 rows of seven heads: 650 us with three, 730 with two; 16 of four: 19 and 16.)
int prefill_tiles(int D, int G, int Tq) {
  if (D != 64) return 1;
  auto blocks = [&](int nt) { const int pb = 16 * nt / G > 0 ? 16 * nt / G : 1; return (Tq + pb - 1) / pb; };
  return blocks(2) * 2.6f < blocks(3) * 3.6f ? 2 : 3;
}

// ---------------------------------------------------------------------------------------------
// attention
// ---------------------------------------------------------------------------------------------
// LDS of one workgroup: the packed bytes of a tile as they lie in memory, or (at the end) one round of the
// sum over the wavefronts.
struct AnyLds {
  int zero_row, k_meta, v_raw, v_meta, bytes;
  __host__ __device__ AnyLds(int D, int DB) {
    zero_row = k_head_bytes_d(D, DB);          // 32 zero bytes: the high-plane row of a channel that has none
    k_meta = zero_row + kRowBytes;
    v_raw = k_meta + 4 * D;
    v_meta = v_raw + v_head_bytes_d(D);
    bytes = v_meta + 4 * kPage;
    if (bytes < 16384) bytes = 16384;
  }
  // with the operands of NT column tiles of query rows
  int with_q(int D, int NT) const { return bytes + D / 32 * NT * 1024; }
};

// 16 NT query rows of one (batch row, kv head) against a range of 128-token tiles, on the matrix cores.
// Decode (PREFILL false): grid (splits, H_KV, B); the rows are the G heads of the group; the partial
// (running max in log2 units, running sum, un-normalised output) goes to the split-K workspace.
// Prefill: grid (blocks of 16 NT / G chunk positions x splits, H_KV, B); row r is head r / PB at chunk position
// p0 + r % PB; after the layer's own tiles come the chunk's rows, causally; the normalised output goes to
// out [B, T_q, H_Q, D], or with ws_ml set a partial per row to the workspace.
//
// What bounds it is turning codes into fp16 numbers with the reference's two roundings: 6 vector instructions
// per two key codes, 4 per two value codes, once per code.  So every code is unpacked in the register in which the
// matrix instruction takes it, by one lane of one wavefront: the packed bytes of a tile go to LDS as they
// are (loaded into registers while the tile before is worked on), a transposing read hands lane n the 8 codes
// 8n .. 8n+7 of several plane rows, and `(X >> 2u) & mask` is then one register of the operand of
//   S^T[token 8n + u][row] = sum_ch  K[token][ch] * Q[row][ch]           (A = K, B = Q in registers)
//   O^T[ch 8n + u][row]    = sum_tok V[tok][ch]   * P^T[tok][row]        (A = V, B = P)
// Wavefront w owns tokens 8i + 2w and 8i + 2w + 1 of every tile, with a running maximum, a sum and an output of its
// own: its accumulator of the first product holds, lane for lane, the B operand of the second (lane group kg:
// tokens 32kg + 8j + 2w, + 1), and the wavefronts meet only where a tile is staged and once at the end.
// fp16 rows (sink, windows, the chunk) are loaded from memory in operand order.
// Probabilities stay fp32 numbers: 32768 p is split into three fp16 numbers, each a matrix operand of its own.
// Together they are the fp32 number itself from 2^-16 of the row's largest probability on; below that they miss it by
// at most 2^-40 of the largest.
// For decode, sharing a tile among four wavefronts pays where there are few tiles (few_tiles in any_decode.hip).
template <int D, bool PREFILL, int NT>
__global__ __launch_bounds__(256, 2) void attn_any_kernel(
    kitty_kv_layer L, const uint8_t* __restrict__ q, int64_t q_stride_b, int64_t q_stride_h, int64_t q_stride_t,
    const uint8_t* __restrict__ k_new, const uint8_t* __restrict__ v_new, int64_t new_stride_b,
    int64_t new_stride_h, int64_t new_stride_t, int H_Q, int Tq, float scaling, float* __restrict__ ws_ml,
    float* __restrict__ ws_acc, int num_splits, __half* __restrict__ out) {
  static_assert(D == 64 || D == 256, "128 has kernels of its own");
  constexpr int kHalves = D == 256 ? 2 : 1;      // V rows in pieces of 128 channels
  constexpr int kU = D == 256 ? 8 : 4;           // channels of a lane within a piece
  constexpr int kOT = kHalves * kU;              // 16-channel tiles of the output
  constexpr int kRows = 16 * NT;
  constexpr int kKIter = (kRowBytes * 2 * D + D) / 16 / 256 + 1;
  constexpr int kVIter = (D + 127) / 128;
  const int h = blockIdx.y, b = blockIdx.z;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, kg = lane >> 4, n = lane & 15;
  const int G = H_Q / L.H_KV;
  const int DB = L.D_BOOSTED;
  const SeqCounts c = load_counts(L, b);
  const int PB = PREFILL ? max(1, kRows / G) : 1;
  const int split = PREFILL ? (int)blockIdx.x % num_splits : (int)blockIdx.x;
  const int p0 = PREFILL ? ((int)blockIdx.x / num_splits) * PB : 0;
  const int kv_chunk = PREFILL ? min(Tq, p0 + PB) : 0;           // chunk tokens this workgroup can see
  const int n_tiles = c.ntiles + (kv_chunk + kPage - 1) / kPage;
  int tile_begin, tile_end;
  if (D == 64) {   // shares that differ by at most one tile
    const int least = n_tiles / num_splits, longer = n_tiles - least * num_splits;
    tile_begin = split * least + min(split, longer), tile_end = tile_begin + least + (split < longer ? 1 : 0);
  } else {         // equal ones (the last shorter): at D = 256 the compiler's code for the above costs 5 %
    const int share = (n_tiles + num_splits - 1) / num_splits;
    tile_begin = min(split * share, n_tiles), tile_end = min(n_tiles, tile_begin + share);
  }
  int bad_page = 0;

  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  __shared__ float s_m[4][kRows], s_l[4][kRows];
  const AnyLds at(D, DB);
  if (tid < 2) ((uint4*)(lds + at.zero_row))[tid] = uint4{0u, 0u, 0u, 0u};

  // the query rows as operands, one copy in LDS for the four wavefronts (16 bytes a lane): k-slots 0..3 of chunk kc
  // are channels 32 kc + 4 kg .., 4..7 those 16 further
  uint4* const s_q = (uint4*)(lds + at.bytes);   // [D / 32][NT][64 lanes]
  int qpos[NT], qhead[NT];   // chunk position (decode: 0), -1 = no such row; head within the group
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    const int r = 16 * nt + n, g = r / PB, pos = p0 + r % PB;
    const bool ok = g < G && pos < (PREFILL ? Tq : 1);
    qpos[nt] = ok ? pos : -1;
    qhead[nt] = g;
    const uint8_t* row = q + (int64_t)b * q_stride_b + (int64_t)(h * G + (ok ? g : 0)) * q_stride_h +
                         (int64_t)(ok ? pos : 0) * q_stride_t;
#pragma unroll
    for (int kc = w; kc < D / 32; kc += 4) {
      const uint2 x0 = *(const uint2*)(row + (32 * kc + 4 * kg) * 2);
      const uint2 x1 = *(const uint2*)(row + (32 * kc + 16 + 4 * kg) * 2);
      s_q[(kc * NT + nt) * 64 + lane] = ok ? uint4{x0.x, x0.y, x1.x, x1.y} : uint4{0u, 0u, 0u, 0u};
    }
  }

  float4v O[kOT][NT];
  float m_run[NT], l_run[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    m_run[nt] = -INFINITY, l_run[nt] = 0.f;
#pragma unroll
    for (int t = 0; t < kOT; ++t) O[t][nt] = float4v{0.f, 0.f, 0.f, 0.f};
  }
  const float sc2 = scaling * kLog2e;
  const int64_t sink_base = (int64_t)b * L.sink_stride_b + (int64_t)h * L.sink_stride_h;
  const int64_t win_base = (int64_t)b * L.win_stride_b + (int64_t)h * L.win_stride_h;
  const int k_words = k_head_bytes_d(D, DB) / 16;

  // the packed bytes of a tile on their way to LDS
  uint4v pk[kKIter] = {}, pv[kVIter] = {}, pm = {};
  auto k_is_packed = [&](int tile) { return tile > 0 && tile < c.ntiles && tile - 1 < c.pk; };
  auto v_is_packed = [&](int tile) { return tile > 0 && tile < c.ntiles && tile - 1 < c.pv; };
  // Whole packed tiles first, in a loop of their own: as branches of one loop the packed and the other paths have the
  // accumulators copied from one set of registers to another at every tile (150 of 1270 instructions a tile at D = 64).
  // (Decode has few tiles a workgroup: one loop, 9 KB of code less; 12000 tokens of one kv head at D = 256 20.7 us so, 22.0.)
  const int full_begin = max(tile_begin, 1);
  const int full_end = PREFILL ? max(full_begin, min(tile_end, 1 + min(min(c.pk, c.pv), c.nbody / kPage))) : full_begin;
  auto next_of = [&](int tile) {   // full_begin .. full_end - 1, then the others
    const bool full = tile >= full_begin && tile < full_end;
    const int t = full && tile + 1 == full_end && tile_begin < full_begin ? tile_begin : tile + 1;
    return !full && t >= full_begin && t < full_end ? full_end : t;
  };
  int64_t id_k = 0, id_v = 0;   // of the tile fetched next, asked for one tile ahead: the load behind them waits for nothing
  auto ask = [&](int tile) {
    if (tile < tile_end && k_is_packed(tile)) id_k = page_id(L.page_table_k, (int64_t)b * L.page_table_k_stride_b + tile - 1);
    if (tile < tile_end && v_is_packed(tile)) id_v = page_id(L.page_table_v, (int64_t)b * L.page_table_v_stride_b + tile - 1);
  };
  auto fetch = [&](int tile) {
    if (k_is_packed(tile)) {
      const int64_t pg = checked_page(id_k, L.cache_pages_k, bad_page);
      const uint4v* src = (const uint4v*)(L.key_cache + pg * L.key_cache_stride_page + (int64_t)h * k_head_bytes_d(D, DB));
#pragma unroll
      for (int i = 0; i < kKIter; ++i)
        if (i * 256 + tid < k_words) pk[i] = src[i * 256 + tid];
      if (tid < D / 4)
        pm = ((const uint4v*)((const uint8_t*)L.key_meta + pg * L.key_meta_stride_page + (int64_t)h * D * 4))[tid];
    }
    if (v_is_packed(tile)) {
      const int64_t pg = checked_page(id_v, L.cache_pages_v, bad_page);
      const uint4v* src = (const uint4v*)(L.value_cache + pg * L.value_cache_stride_page + (int64_t)h * v_head_bytes_d(D));
#pragma unroll
      for (int i = 0; i < kVIter; ++i)
        if (i * 256 + tid < 2 * D) pv[i] = src[i * 256 + tid];
      if (tid >= 64 && tid < 96)
        pm = ((const uint4v*)((const uint8_t*)L.value_meta + pg * L.value_meta_stride_page + (int64_t)h * kPage * 4))[tid - 64];
    }
    ask(next_of(tile));
  };
  auto stage = [&](int tile) {
    if (k_is_packed(tile)) {
#pragma unroll
      for (int i = 0; i < kKIter; ++i)
        if (i * 256 + tid < k_words) ((uint4v*)lds)[i * 256 + tid] = pk[i];
      if (tid < D / 4) ((uint4v*)(lds + at.k_meta))[tid] = pm;
    }
    if (v_is_packed(tile)) {
#pragma unroll
      for (int i = 0; i < kVIter; ++i)
        if (i * 256 + tid < 2 * D) ((uint4v*)(lds + at.v_raw))[i * 256 + tid] = pv[i];
      if (tid >= 64 && tid < 96) ((uint4v*)(lds + at.v_meta))[tid - 64] = pm;
    }
  };

  auto step = [&](auto full_, int tile) {
    constexpr bool FULL = decltype(full_)::value;
    const bool chunk = !FULL && tile >= c.ntiles;              // a tile of the new chunk (prefill only)
    const int chunk_t0 = chunk ? (tile - c.ntiles) * kPage : 0;
    const int body = tile - 1;                                  // -1 = sink
    const int ntok = FULL ? kPage : chunk ? min(kPage, kv_chunk - chunk_t0) : tile == 0 ? c.sink : min(kPage, c.nbody - body * kPage);
    const bool k_packed = FULL || k_is_packed(tile), v_packed = FULL || v_is_packed(tile);
    __syncthreads();   // everyone is done with the tile before
    stage(tile);
    __syncthreads();
    const int after = next_of(tile);
    if (after < tile_end) fetch(after);
    if (ntok <= 0) return;   // an empty sink

    // ---- logits of tokens 8i + 2w + e: S[e][nt][j] is token 32 kg + 8 j + 2 w + e, row 16 nt + n -------------------
    float4v S[2][NT];
#pragma unroll
    for (int e = 0; e < 2; ++e)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) S[e][nt] = float4v{0.f, 0.f, 0.f, 0.f};
    if (k_packed) {
      const uint8_t* idx = lds + kRowBytes * (D + DB);
      const int quarter = (n & 3) * 8;
#pragma unroll 2
      for (int kc = 0; kc < D / 32; ++kc) {
        const int r0 = 32 * kc + 4 * kg, mine = r0 + (n >> 2);
        uint32_t X[4], H[4], sc[4], zr[4];
        lds_tr(lds + mine * kRowBytes + quarter, X[0], X[1]);
        lds_tr(lds + (mine + 16) * kRowBytes + quarter, X[2], X[3]);
        const int s0 = idx[mine], s1 = idx[mine + 16];
        lds_tr(lds + (s0 < DB ? (D + s0) * kRowBytes : at.zero_row) + quarter, H[0], H[1]);
        lds_tr(lds + (s1 < DB ? (D + s1) * kRowBytes : at.zero_row) + quarter, H[2], H[3]);
        const uint4 m0 = *(const uint4*)(lds + at.k_meta + r0 * 4), m1 = *(const uint4*)(lds + at.k_meta + (r0 + 16) * 4);
        sc[0] = low_halves(m0.x, m0.y), zr[0] = high_halves(m0.x, m0.y);
        sc[1] = low_halves(m0.z, m0.w), zr[1] = high_halves(m0.z, m0.w);
        sc[2] = low_halves(m1.x, m1.y), zr[2] = high_halves(m1.x, m1.y);
        sc[3] = low_halves(m1.z, m1.w), zr[3] = high_halves(m1.z, m1.w);
        uint4 qq[NT];
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) qq[nt] = s_q[(kc * NT + nt) * 64 + lane];
        uint32_t a0[4], a1[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const uint32_t lo = X[i] >> (4 * w), hi = (H[i] >> (4 * w)) << 2;   // code e: bits 2e, 2e + 1 of lo, two further up in hi
          const uint32_t c0 = (lo & 0x00030003u) | (hi & ~0x00030003u), c1 = (lo & 0x000c000cu) | (hi & ~0x000c000cu);
          a0[i] = dequant_word<0>((c0 & 0x000f000fu) | kCodeMagic, sc[i], zr[i]);
          a1[i] = dequant_word<2>((c1 & 0x003c003cu) | kCodeMagic, sc[i], zr[i]);
        }
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
          S[0][nt] = mfma16(a0, qq[nt], S[0][nt]);
          S[1][nt] = mfma16(a1, qq[nt], S[1][nt]);
        }
      }
    } else {
      const uint8_t* base = chunk ? k_new + (int64_t)b * new_stride_b + (int64_t)h * new_stride_h + (int64_t)chunk_t0 * new_stride_t
                          : tile == 0 ? (const uint8_t*)L.sink_k + sink_base : (const uint8_t*)L.qbuf_k + win_base;
      const int64_t stride = chunk ? new_stride_t : (int64_t)(2 * D);
      int first = 8 * n + 2 * w;
      asm volatile("" : "+v"(first));   // these addresses are formed here, not kept in registers over the packed tiles
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        // a token past the end repeats the last one: its logits are masked below
        const uint8_t* row = base + (int64_t)min(first + e, ntok - 1) * stride;
#pragma unroll 4
        for (int kc = 0; kc < D / 32; ++kc) {
          const uint2 x0 = *(const uint2*)(row + (32 * kc + 4 * kg) * 2);
          const uint2 x1 = *(const uint2*)(row + (32 * kc + 16 + 4 * kg) * 2);
          const uint32_t a[4] = {x0.x, x0.y, x1.x, x1.y};
#pragma unroll
          for (int nt = 0; nt < NT; ++nt) S[e][nt] = mfma16(a, s_q[(kc * NT + nt) * 64 + lane], S[e][nt]);
        }
      }
    }

    // ---- online softmax of this wavefront's tokens ----------------------------------------------
    uint32_t pr[kProbParts][NT][4];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
#pragma unroll
      for (int e = 0; e < 2; ++e) S[e][nt] *= sc2;
      if (chunk || ntok < kPage) {
        // tokens of the tile this row sees: all of them, or (the chunk's own tiles) those up to its position
        const int lim = chunk ? min(ntok, qpos[nt] - chunk_t0 + 1) : ntok;
#pragma unroll
        for (int e = 0; e < 2; ++e)
#pragma unroll
          for (int j = 0; j < 4; ++j)
            if (32 * kg + 8 * j + 2 * w + e >= lim) S[e][nt][j] = -INFINITY;
      }
      float mx = fmaxf(fmaxf(fmaxf(S[0][nt][0], S[0][nt][1]), fmaxf(S[0][nt][2], S[0][nt][3])),
                       fmaxf(fmaxf(S[1][nt][0], S[1][nt][1]), fmaxf(S[1][nt][2], S[1][nt][3])));
      mx = max_over_lane_groups(mx);
      const float m_old = m_run[nt], m_new = fmaxf(m_old, mx);
      if (__any(m_new > m_old)) {
        const float alpha = m_old == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m_old - m_new);
        l_run[nt] *= alpha;
#pragma unroll
        for (int t = 0; t < kOT; ++t) O[t][nt] *= alpha;
        m_run[nt] = m_new;
      }
      const float ref = m_run[nt] == -INFINITY ? 0.f : m_run[nt];
      float sum = 0.f;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float p0v = __builtin_amdgcn_exp2f(S[0][nt][j] - ref), p1v = __builtin_amdgcn_exp2f(S[1][nt][j] - ref);
        sum += p0v + p1v;
        float x0 = p0v * kProbScale, x1 = p1v * kProbScale;
#pragma unroll
        for (int i = 0; i < kProbParts; ++i) {
          const half2v part = {(_Float16)x0, (_Float16)x1};
          pr[i][nt][j] = __builtin_bit_cast(uint32_t, part);
          x0 -= (float)part[0], x1 -= (float)part[1];   // exact
        }
      }
      l_run[nt] += sum;
    }

    // ---- O += P V over the same tokens ------------------------------------------------------------
    const int t0 = 32 * kg + 2 * w;   // register j of an operand: tokens t0 + 8 j, t0 + 8 j + 1
    auto weigh = [&](uint32_t (&a)[4], int t, bool infinities) {
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) O[t][nt] = mfma16(a, pr[0][nt], O[t][nt]);
      if (infinities) {
#pragma unroll
        for (int j = 0; j < 4; ++j) a[j] = finite_word(a[j]);
      }
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int i = 1; i < kProbParts; ++i) O[t][nt] = mfma16(a, pr[i][nt], O[t][nt]);
    };
    if (v_packed) {
      uint32_t sc[4], zr[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        uint2 mm = *(const uint2*)(lds + at.v_meta + (t0 + 8 * j) * 4);
        if (ntok < kPage) {           // a token that does not count is 0, whatever its bytes say
          if (t0 + 8 * j >= ntok) mm.x = 0u;
          if (t0 + 8 * j + 1 >= ntok) mm.y = 0u;
        }
        sc[j] = low_halves(mm.x, mm.y), zr[j] = high_halves(mm.x, mm.y);
      }
      // 3 scale + zero stays finite where both are below 2^13; elsewhere a value may be infinite
      uint32_t big = 0u;
#pragma unroll
      for (int j = 0; j < 4; ++j) big |= ((sc[j] & 0x7fff7fffu) + 0x10001000u) | ((zr[j] & 0x7fff7fffu) + 0x10001000u);
      const bool wild = __any((big & 0x80008000u) != 0u);
      const int rr = n >> 2, tok = t0 + (rr & 1) + 8 * (rr >> 1);
#pragma unroll
      for (int hf = 0; hf < kHalves; ++hf) {
        // D = 64: a row has 8 pieces; lanes n and n + 8 both receive piece n % 8 and take its lower and upper four codes
        const uint8_t* p = lds + at.v_raw + tok * (D / 4) + hf * kRowBytes + (D == 64 ? n & 1 : n & 3) * 8;
        uint32_t X[4];
        lds_tr(p, X[0], X[1]);
        lds_tr(p + 16 * (D / 4), X[2], X[3]);
        if (D == 64) {
#pragma unroll
          for (int j = 0; j < 4; ++j) X[j] >>= n & 8;
        }
        uint32_t X10[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) X10[j] = X[j] >> 10;
        auto piece = [&](auto u_, bool infinities) {
          constexpr int u = decltype(u_)::value;
          uint32_t a[4];
#pragma unroll
          for (int j = 0; j < 4; ++j) a[j] = dequant_v<u>(X[j], X10[j], kCodeMagic, sc[j], zr[j]);
          weigh(a, hf * kU + u, infinities);
        };
        auto pieces = [&](bool infinities) {
          piece(std::integral_constant<int, 0>{}, infinities), piece(std::integral_constant<int, 1>{}, infinities);
          piece(std::integral_constant<int, 2>{}, infinities), piece(std::integral_constant<int, 3>{}, infinities);
          if constexpr (kU == 8) {
            piece(std::integral_constant<int, 4>{}, infinities), piece(std::integral_constant<int, 5>{}, infinities);
            piece(std::integral_constant<int, 6>{}, infinities), piece(std::integral_constant<int, 7>{}, infinities);
          }
        };
        if (wild) pieces(true);
        else pieces(false);
      }
    } else {
      int first = t0;
      asm volatile("" : "+v"(first));   // as above
      // rows u < lows of one tensor, then the ring's (a tail tile only)
      const int u0 = chunk || tile == 0 ? 0 : (body - c.pv) * kPage, lows = chunk || tile == 0 ? kPage : c.rv;
      const uint8_t* low = chunk ? v_new + (int64_t)b * new_stride_b + (int64_t)h * new_stride_h + (int64_t)chunk_t0 * new_stride_t
                         : tile == 0 ? (const uint8_t*)L.sink_v + sink_base : (const uint8_t*)L.qbuf_v + win_base;
      const int64_t stride = chunk ? new_stride_t : (int64_t)(2 * D);
      const uint8_t* ring = (const uint8_t*)L.local_v + win_base;
      const uint8_t* rows[8];   // the rows of tokens t0 + 8 j + e
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int u = u0 + min(first + 8 * (i >> 1) + (i & 1), ntok - 1);
        const int64_t in_low = (int64_t)u * stride, in_ring = (int64_t)((c.off + u - lows) & (kPage - 1)) * (2 * D);
        rows[i] = (u < lows ? low : ring) + (u < lows ? in_low : in_ring);
      }
#pragma unroll
      for (int hf = 0; hf < kHalves; ++hf) {
        const int ch = D == 256 ? 128 * hf + 8 * n : 8 * (n & 7) + 4 * (n >> 3);
        asm volatile("" ::: "memory");   // one piece's rows in flight at a time: both would cost 32 registers more
        typedef uint32_t words __attribute__((ext_vector_type(kU / 2)));
        words x[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          x[i] = *(const words*)(rows[i] + ch * 2);
          if (first + 8 * (i >> 1) + (i & 1) >= ntok) x[i] = words{};   // probability 0 times what a dead row may hold must be 0
        }
#pragma unroll
        for (int u = 0; u < kU; ++u) {
          uint32_t a[4];
#pragma unroll
          for (int j = 0; j < 4; ++j)
            a[j] = u & 1 ? high_halves(x[2 * j][u >> 1], x[2 * j + 1][u >> 1]) : low_halves(x[2 * j][u >> 1], x[2 * j + 1][u >> 1]);
          weigh(a, hf * kU + u, true);
        }
      }
    }
  };
  const int first = full_begin < full_end ? full_begin : tile_begin;
  if (first < tile_end) ask(first), fetch(first);
  if constexpr (PREFILL) {
#pragma unroll 1
    for (int tile = full_begin; tile < full_end; ++tile) step(std::true_type{}, tile);
  }
#pragma unroll 1
  for (int tile = full_begin < full_end && tile_begin >= full_begin ? full_end : tile_begin; tile < tile_end; tile = next_of(tile))
    step(std::false_type{}, tile);

  if (tid == 0) report_bad_page(L, b, bad_page);
  // ---- the wavefronts' partials meet: a common maximum, then sums of four output tiles at a time ---------------
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    float l = l_run[nt];
    l += __shfl_xor(l, 16);
    l += __shfl_xor(l, 32);
    if (kg == 0) s_m[w][16 * nt + n] = m_run[nt], s_l[w][16 * nt + n] = l;
  }
  __syncthreads();
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    const int r = 16 * nt + n;
    const float mm = fmaxf(fmaxf(s_m[0][r], s_m[1][r]), fmaxf(s_m[2][r], s_m[3][r]));
    const float own = m_run[nt] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m_run[nt] - mm) * (1.f / kProbScale);
#pragma unroll
    for (int t = 0; t < kOT; ++t) O[t][nt] *= own;
  }
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    // (this thread's part of the result: 4 channels of row n of column tile nt)
    const int r = 16 * nt + n;
    float mm = -INFINITY, l = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) mm = fmaxf(mm, s_m[i][r]);
#pragma unroll
    for (int i = 0; i < 4; ++i)   // (a wavefront whose logits are all NaN has -inf for a maximum and NaN for a sum, which must stay)
      l += s_l[i][r] * (s_m[i][r] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(s_m[i][r] - mm));
    const bool partial = !PREFILL || ws_ml != nullptr;
    int64_t row = 0;   // of the workspace, or of out
    if (PREFILL) row = ((int64_t)b * Tq + qpos[nt]) * H_Q + h * G + qhead[nt];
    else row = (int64_t)b * H_Q + h * G + qhead[nt];
    if (partial) row = row * num_splits + split;
    if (partial && qpos[nt] >= 0 && w == 0 && kg == 0) {
      if (l != l) mm = 0.f;   // a share of nothing but NaN counts, whatever the number of shares (the merge passes over -inf)
      *(float2*)(ws_ml + row * 2) = float2{mm, l};
    }
#pragma unroll
    for (int t4 = 0; t4 < kOT; t4 += 4) {
      __syncthreads();
#pragma unroll
      for (int t = 0; t < 4; ++t) ((float4v*)lds)[(w * 4 + t) * 64 + lane] = O[t4 + t][nt];
      __syncthreads();
      float4v o = float4v{0.f, 0.f, 0.f, 0.f};   // tile t4 + w, summed over the wavefronts
#pragma unroll
      for (int i = 0; i < 4; ++i) o += ((const float4v*)lds)[(i * 4 + w) * 64 + lane];
      if (qpos[nt] >= 0) {
        const int t = t4 + w;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int x = 4 * kg + j;
          const int ch = D == 256 ? 128 * (t >> 3) + 8 * x + (t & 7) : 8 * (x & 7) + 4 * (x >> 3) + t;
          if (partial) ws_acc[row * D + ch] = o[j];
          else out[row * D + ch] = __float2half_rn(l > 0.f ? o[j] / l : 0.f);
        }
      }
    }
  }
}

}  // namespace

// decode over few tiles
void launch_decode_by_tile(const kitty_kv_layer& L, const void* q, int B, int H_Q, float scaling, float* ws_ml, float* ws_acc,
                           int num_splits, hipStream_t stream) {
  const dim3 grid(num_splits, L.H_KV, B), block(256);
  const int64_t row = (int64_t)L.D * 2;
  const auto kernel = L.D == 64 ? attn_any_kernel<64, false, 1> : attn_any_kernel<256, false, 1>;
  hipLaunchKernelGGL(kernel, grid, block, AnyLds(L.D, L.D_BOOSTED).with_q(L.D, 1), stream, L, (const uint8_t*)q, H_Q * row, row, (int64_t)0,
                     nullptr, nullptr, (int64_t)0, (int64_t)0, (int64_t)0, H_Q, 1, scaling, ws_ml, ws_acc, num_splits, nullptr);
}

namespace {
// chunk positions per workgroup
int any_positions(int D, int G, int Tq) {
  const int rows = 16 * prefill_tiles(D, G, Tq);
  return rows / G > 0 ? rows / G : 1;
}
// Shares of ceil(tiles / s) tiles, as the kernel cuts them at D = 256, may leave the last of them empty: 65 tiles in 64 shares are
// 33 of two.  Those workgroups would load the queries and write partials for the merge to read.
int without_empty_shares(int D, int tiles, int s) {
  if (D == 64) return s;   // shares that differ by at most one tile
  const int share = (tiles + s - 1) / s;
  return (tiles + share - 1) / share;
}
}  // namespace

// Shares of a chunk's walk.  The device holds two workgroups per compute unit at a time (their registers); a share takes as
// long as its tiles and one more (its start and its end), and rounds that are not full overlap with the next by about a half.
// A share more also costs the merge its partials: a tile's time is some 4 us, in which it reads 12 MB.  At least two tiles
// each.  200 tokens over 8000 at D = 64, 136 workgroups: 99 us with 7 shares (two rounds of 93 %), 105 with 3, 125 with 4;
// 1000 over 30000 (334): 650 with 3, 968 with 1.  200 over 4000 at D = 256 (200): 121 with 5, 131 with 2, 140 with 3.
// `most`: shares the scratch allows.
int prefill_splits_any(int B, int H_Q, int H_KV, int D, int Tq, int tiles, int units, int most) {
  const int PB = any_positions(D, H_Q / H_KV, Tq);
  const double wgs = (double)((Tq + PB - 1) / PB) * H_KV * B, merged = (double)B * Tq * H_Q * D * 4 / 12e6;
  int best = 1;
  double least = 0;
  for (int s = 1; s <= most && s <= 64 && (s == 1 || 2 * s <= tiles); ++s) {
    const double rounds = wgs * s / (2 * units), whole = ceil(rounds);
    const double cost = (whole <= 1 ? 1 : (whole + rounds) / 2) * ((tiles + s - 1) / s + 1) + (s > 1 ? merged * s : 0);
    if (s == 1 || cost < least) best = s, least = cost;
  }
  return without_empty_shares(D, tiles, best);
}

void launch_prefill_any(const kitty_kv_layer& L, const void* q, int64_t q_stride_b, int64_t q_stride_h,
                        int64_t q_stride_t, const void* k_new, const void* v_new, int64_t new_stride_b,
                        int64_t new_stride_h, int64_t new_stride_t, int B, int H_Q, int Tq, float scaling, void* out,
                        float* ws_ml, float* ws_acc, int num_splits, hipStream_t stream) {
  const int G = H_Q / L.H_KV, nt = prefill_tiles(L.D, G, Tq), PB = any_positions(L.D, G, Tq);
  const dim3 grid((Tq + PB - 1) / PB * num_splits, L.H_KV, B), block(256);
  const auto kernel = L.D == 256 ? attn_any_kernel<256, true, 1> : nt == 2 ? attn_any_kernel<64, true, 2> : attn_any_kernel<64, true, 3>;
  hipLaunchKernelGGL(kernel, grid, block, AnyLds(L.D, L.D_BOOSTED).with_q(L.D, nt), stream, L, (const uint8_t*)q, q_stride_b,
                     q_stride_h, q_stride_t, (const uint8_t*)k_new, (const uint8_t*)v_new, new_stride_b, new_stride_h,
                     new_stride_t, H_Q, Tq, scaling, ws_ml, ws_acc, num_splits, (__half*)out);
  if (num_splits > 1)
    launch_rows_merge(L.D, ws_ml, ws_acc, out, (int64_t)B * Tq * H_Q, num_splits, /* keep_nan */ false, stream);
}

}  // namespace kitty
