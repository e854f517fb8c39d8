// Chunked-prefill attention: T_q new tokens attend, causally among themselves, to everything the
// cache already holds (sink rows, packed pages, fp16 windows) and to the new chunk's own keys
// and values.  The reference has no such kernel (its prefill runs dense flash attention on an
// empty cache, benchmark_kitty.py:302, and kitty_attention.py:411 asserts t_query == 1); the
// arithmetic is the same as decode: softmax(q . k^ * scaling) . v^ with
// k^ = fp16(code) * scale + zero evaluated in fp16 (kitty_attention.py:162-165, 317-320).
//
// The work is a dense contraction (G * T_q query rows per KV head), so it runs on the matrix
// cores, flash-attention style.  One workgroup of 8 wavefronts, two per SIMD, owns 256 query rows of one
// (batch row, KV head): PB = 256 / G consecutive chunk positions times the G query heads of the
// group; wavefront w owns rows 32w .. 32w+31.  The workgroup walks the sequence in 128-token
// tiles.  Each tile is brought into LDS once, as fp16, by all 512 threads: packed pages are
// dequantized on the way (exactly the reference's two fp16 roundings), fp16 rows are copied.
// Two tile buffers alternate: while tile t is multiplied, tile t+1 is converted into the other
// buffer and the packed bytes of tile t+2 are in flight; one barrier per tile.
//
// Matrix-core formulation (v_mfma_f32_32x32x16_f16; lane = 32 kg + n holds A[n][8 k-slots],
// B[8 k-slots][n], C[8 (i / 4) + 4 kg + i % 4][n], i = 0 .. 15):
//   S^T[pos][row]  = sum_ch  K[pos][ch]  * Q[row][ch]      A = keys,   B = queries (registers)
//   O^T[cp][row]   = sum_pos V[pos][cp]  * P^T[pos][row]   A = values, B = probabilities
// The accumulator of the first product is, lane for lane, the B operand of the second: k-slot j
// of lane group kg stands for position 8 (j / 4) + 4 kg + j % 4 of 16.  A lane holds 16 logits of ONE row, so
// the running maximum and sum are one register each and a reduction over a row is one exchange between two lanes.
//
// LDS layouts, chosen so that dequantization writes 128-bit rows and the matrix-core operands
// come out of `ds_read_b64_tr_b16` (a 16-lane block reads 4 rows x 16 columns and lane i
// receives column i of the 4 rows):
//   K tile: [channel][position]       V tile: [position][channel slot]      row pitch 272 bytes
// "position" and "channel slot" are the order in which codes fall out of a plane word when it is
// masked with 0x00030003 << 2u: slot 2u + e of a 16-block is element u + 8e.  Keys and values use
// the same token permutation, the output undoes the channel permutation.
//
// What bounds it: power and the vector unit, in turn.  B = 4, 32 / 8 heads, 2048 positions over 30720 cached tokens: 4.4 to
// 5.0 ms by box, the card's power setting it (855 to 970 TFLOP/s; 5.13 to 5.29 before; the matrix instructions alone, on the same frame, take 3.1).  Per wave and tile, against
// v_mfma_f32_16x16x32 (two rows per lane, twice the matrix instructions) with 288-byte rows: 100 vector instructions,
// 60 scalar ones and a dependent load (the boost slot) less, and a quarter of the bank conflicts.
#include <type_traits>

#include "decode_common.h"

// wave priority while a wave issues the PV MFMAs (the other wave of the SIMD fills the gaps)
#define KITTY_PV_PRIO 2

namespace kitty {
// merge pass over independent rows (rows_merge.hip)
void launch_rows_merge(int D, const float* ws_ml, const float* ws_acc, void* out, int64_t rows, int num_splits,
                       bool keep_nan, hipStream_t stream);
namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float float4v __attribute__((ext_vector_type(4)));
typedef float float16v __attribute__((ext_vector_type(16)));
typedef short short4v __attribute__((ext_vector_type(4)));
typedef uint32_t uint4v __attribute__((ext_vector_type(4)));

constexpr int kPitch = 272;                   // bytes per LDS row: 128 fp16 + 16 bytes of padding
constexpr int kTile = kPage * kPitch;         // 34816 bytes, one K or V tile
constexpr int kLdsBytes = 4 * kTile;          // K and V, two buffers each
constexpr int kRows = 256;                    // query rows per workgroup
constexpr int kWaves = 8;                     // two per SIMD: one does vector work while the other feeds the matrix pipe
constexpr int kThreads = 64 * kWaves;
constexpr int kWaveRows = kRows / kWaves;     // 32: one column tile of the matrix instruction per wave
constexpr int kParts = 4;                     // threads that share one packed row of a tile while staging it
constexpr int kSubs = 2;                      // sub-tiles of 32 positions that share one look at the maxima
constexpr float kLog2e = 1.4426950408889634f;

// what issue() leaves in flight for a packed tile (fp16 rows are few and are copied by finish())
struct Stage {
  uint2 klo, khi, v;
  uint32_t kmeta, vmeta;
};

__device__ __forceinline__ int slot_of(int e) {   // element (token or channel) -> LDS slot
  return (e & ~15) | ((e & 7) << 1) | ((e >> 3) & 1);
}

__device__ __forceinline__ half4 lds_tr(const uint8_t* p) {
  short4v r = __builtin_amdgcn_ds_read_tr16_b64_v4i16((short4v __attribute__((address_space(3)))*)p);
  return __builtin_bit_cast(half4, r);
}

// matrix-core A operand: k-slots 0..3 from the 4 LDS rows at p, k-slots 4..7 from 8 rows further
__device__ __forceinline__ half8 load_a(const uint8_t* p) {
  const half4 a0 = lds_tr(p), a1 = lds_tr(p + 8 * kPitch);
  return __builtin_shufflevector(a0, a1, 0, 1, 2, 3, 4, 5, 6, 7);
}

// Maximum over lanes l and l^32 with the half-swap instruction of gfx950: two vector instructions, where a
// shuffle would be a round trip through LDS.
__device__ __forceinline__ float max_over_lane_halves(float v) {
  const unsigned b = __builtin_bit_cast(unsigned, v);
  const auto q = __builtin_amdgcn_permlane32_swap(b, b, false, false);
  const unsigned q0 = q[0], q1 = q[1];   // as scalars first: a bit_cast of q[1] itself reads element 0
  return vmax(__builtin_bit_cast(float, q0), __builtin_bit_cast(float, q1));
}

__device__ __forceinline__ float xor_lanes(float v, int mask) { return __shfl_xor(v, mask); }

// where the 16 tokens 16 g .. of a channel's row lie in a K tile: the two groups of a 32-token sub-tile 128 bytes apart
__device__ __forceinline__ int token_group_bytes(int g) { return 32 * (g >> 1) + 128 * (g & 1); }
// A 16-lane block of a transposing read takes every second row of eight, so that the rows of 272 bytes that two blocks
// read (16 positions of either 128-byte half) and the four rows of four 64-byte pieces that 16 lanes write
// meet each of the 64 banks once: row 8 a + 2 j + k is k-slot 4 k + j of its eight.
__device__ __forceinline__ int row_slot(int r) { return (r & ~7) | ((r & 1) << 2) | ((r >> 1) & 3); }

// fp16(code) * scale + zero with both roundings, for two codes at a time; `c` holds the codes as
// integers in its two halves.
__device__ __forceinline__ uint32_t dequant_pair(uint32_t c, half2v scale, half2v zero) {
#pragma clang fp contract(off)
  const half2v magic = {(_Float16)1024.f, (_Float16)1024.f};
  half2v f = __builtin_bit_cast(half2v, c | 0x64006400u) - magic;   // exact: 1024 + code - 1024
  half2v m = f * scale;
  half2v r = m + zero;
  return __builtin_bit_cast(uint32_t, r);
}

// The same for 4-bit codes at bit SHIFT of each half of x, taken where they lie: 1024 + code * 2^SHIFT is a number of
// fp16, and scaling it down and subtracting is exact.  `magic` is 1024 in both halves, in a register: with the mask as
// the instruction's only constant, masking and merging are one instruction.
template <int SHIFT>
__device__ __forceinline__ uint32_t dequant_code(uint32_t x, uint32_t magic, half2v scale, half2v zero) {
#pragma clang fp contract(off)
  constexpr _Float16 k = (_Float16)(1.0f / (1 << SHIFT)), o = (_Float16)(1024.0f / (1 << SHIFT));
  const half2v c = __builtin_bit_cast(half2v, (x & (0x000f000fu << SHIFT)) | magic);
  const half2v f = SHIFT == 0 ? c - half2v{o, o} : __builtin_elementwise_fma(c, half2v{k, k}, half2v{-o, -o});
  const half2v m = f * scale;
  const half2v r = m + zero;
  return __builtin_bit_cast(uint32_t, r);
}

template <bool BOOST, bool SPLIT>
struct Prefill {
  const kitty_kv_layer& L;
  const SeqCounts c;
  const int b, h, tid;
  const uint8_t* k_new;
  const uint8_t* v_new;
  int64_t new_stride_t;
  int kv_chunk;      // chunk tokens this workgroup can see
  int n_tiles;       // sink + body + chunk tiles actually walked
  int first_body, first_chunk;
  mutable int bad_page = 0;   // a page id outside the cache was met (checked_page)
  // Addresses reach issue() through LDS, checked: kChunk body tiles at a time, the K and V page ids are read by
  // one thread each, range-checked (checked_page) and turned into the addresses of this head's bytes and metadata,
  // in one half of a ring; the chunk after the current one is staged when the walk is half way through the
  // current one, and the barrier that ends every iteration of the walk publishes it.  (Reading and checking the ids where
  // they are used - a load whose value the next instructions need, in every iteration of every workgroup - cost this
  // kernel 10 %; multiplying ids by strides there, on every thread, some 70 of 640 vector instructions a tile.)
  // Body tiles are counted from id_base(), the first one of this workgroup's share.
  static constexpr int kChunk = 64;
  typedef const uint8_t* PageTable[4][2 * kChunk];   // [K, K metadata, V, V metadata][(body tile - id_base()) % (2 kChunk)]
  const uint8_t* (*pages)[2 * kChunk];
  int first_id = 0;
  __device__ __forceinline__ int id_base() const { return SPLIT ? first_id : 0; }

  __device__ __forceinline__ void stage_pages(int chunk) const {
    if (tid < 2 * kChunk) {
      const int side = tid / kChunk, i = id_base() + chunk * kChunk + tid % kChunk;
      if (i < (side ? c.pv : c.pk)) {
        const int64_t pg = side ? L.page_table_v[(int64_t)b * L.page_table_v_stride_b + i]
                                : L.page_table_k[(int64_t)b * L.page_table_k_stride_b + i];
        const int64_t ok = checked_page(pg, side ? L.cache_pages_v : L.cache_pages_k, bad_page);
        const uint8_t* at = side ? L.value_cache + ok * L.value_cache_stride_page + (int64_t)h * kVBytes
                                 : L.key_cache + ok * L.key_cache_stride_page + (int64_t)h * k_head_bytes(L.D_BOOSTED);
        const uint8_t* meta = side ? (const uint8_t*)L.value_meta + ok * L.value_meta_stride_page + (int64_t)h * kPage * 4
                                   : (const uint8_t*)L.key_meta + ok * L.key_meta_stride_page + (int64_t)h * kD * 4;
        const int r = (chunk & 1) * kChunk + tid % kChunk;
        pages[2 * side][r] = at;
        pages[2 * side + 1][r] = meta;
      }
    }
  }
  __device__ __forceinline__ const uint8_t* page(int which, int i) const {
    return pages[which][(i - id_base()) & (2 * kChunk - 1)];
  }

  __device__ __forceinline__ int body(int t) const { return t - first_body; }   // -1: the sink
  __device__ __forceinline__ bool k_packed(int t) const { return t >= first_body && t - first_body < c.pk && t < first_chunk; }
  __device__ __forceinline__ bool v_packed(int t) const { return t >= first_body && t - first_body < c.pv && t < first_chunk; }
  __device__ __forceinline__ int tokens(int t) const {
    return t < first_body ? c.sink : t < first_chunk ? min(kPage, c.nbody - body(t) * kPage) : min(kPage, kv_chunk - chunk_pos(t));
  }
  __device__ __forceinline__ int chunk_pos(int t) const { return (t - first_chunk) * kPage; }   // < 0: not a tile of the chunk

  // what a thread takes of packed rows: a K channel's tokens 32 part .., dealt so that 16 lanes write to 64 different banks; the
  // channels 32 part .. of the value row that belongs in LDS row tid / 4
  __device__ __forceinline__ int part() const { return tid % kParts; }
  __device__ __forceinline__ int key_channel() const {
    return (tid >> 6) * 16 + ((tid >> 4) & 3) * 2 + ((tid >> 2) & 1) + ((tid >> 3) & 1) * 8;
  }
  __device__ __forceinline__ int value_row() const { return tid / kParts; }
  __device__ __forceinline__ int value_token() const {   // slot 2u + e of a 16-block is token u + 8e
    const int m = row_slot(value_row());
    return (m & ~15) | ((m >> 1) & 7) | ((m & 1) << 3);
  }

  // The boost slot of this thread's channel in tile t.  The high plane's words lie where it says: asked for a tile before
  // issue(), or every wave would wait for one load in order to start the next.
  // (FULL, here and below: tile t is known to be a page on both sides)
  template <bool FULL>
  __device__ __forceinline__ int ask_slot(int t) const {
    return BOOST && (FULL || k_packed(t)) ? page(0, body(t))[kLoBytes + L.D_BOOSTED * kRowBytes + key_channel()] : 255;
  }

  // ---- stage 1: global loads of a packed tile into registers ----------------------------------
  template <bool FULL>
  __device__ __forceinline__ void issue(int t, int slot, Stage& g) const {
    if (FULL || k_packed(t)) {
      const uint8_t* at = page(0, body(t));
      g.klo = *(const uint2*)(at + key_channel() * kRowBytes + part() * 8);
      g.kmeta = *(const uint32_t*)(page(1, body(t)) + key_channel() * 4);
      g.khi = uint2{0u, 0u};
      if (BOOST && slot < L.D_BOOSTED) g.khi = *(const uint2*)(at + kLoBytes + slot * kRowBytes + part() * 8);
    }
    if (FULL || v_packed(t)) {
      g.v = *(const uint2*)(page(2, body(t)) + value_token() * kRowBytes + part() * 8);
      g.vmeta = *(const uint32_t*)(page(3, body(t)) + value_token() * 4);
    }
  }

  // ---- stage 2: registers -> fp16 tile in LDS -----------------------------------------------
  template <bool FULL>
  __device__ __forceinline__ void finish(int t, const Stage& g, uint8_t* kt, uint8_t* vt) const {
    const int64_t win = (int64_t)b * L.win_stride_b + (int64_t)h * L.win_stride_h;
    const int64_t sink = (int64_t)b * L.sink_stride_b + (int64_t)h * L.sink_stride_h;
    const bool in_sink = t < first_body, in_chunk = t >= first_chunk;
    // The values' fp16 rows, asked for in front of the keys' stores: one way to memory in a tile's chain, not two (10 tokens over 150 cached,
    // four layers: 117 -> 106 us; 300 over 1000, eight sequences: 623 -> 586; whole pages are not affected)
    uint4 rows_v[4];
    if (!FULL && !v_packed(t)) {   // dead rows must be finite
      int e = value_token();
      asm volatile("" : "+v"(e));
      const bool ok = e < tokens(t);
      const uint8_t* row = nullptr;
      if (ok)
        row = in_chunk ? v_new + (int64_t)(chunk_pos(t) + e) * new_stride_t
              : in_sink ? (const uint8_t*)L.sink_v + sink + (int64_t)e * (kD * 2)
                        : (const uint8_t*)v_tail_row(L, c, b, h, (body(t) - c.pv) * kPage + e);
      const uint4* src = (const uint4*)(row + part() * 64);
#pragma unroll
      for (int w = 0; w < 4; ++w) rows_v[w] = ok ? src[w] : uint4{0u, 0u, 0u, 0u};
    }
    if (FULL || k_packed(t)) {
      // thread = one channel, 32 tokens: plane words of 16 tokens each
      const half2v m2 = __builtin_bit_cast(half2v, g.kmeta);
      const half2v scale = {m2[0], m2[0]}, zero = {m2[1], m2[1]};
      const uint32_t k01 = dequant_pair(0x00010000u, scale, zero), k23 = dequant_pair(0x00030002u, scale, zero);
      uint8_t* row = kt + key_channel() * kPitch + part() * 32;
      uint32_t magic = 0x64006400u;
      asm volatile("" : "+v"(magic));
#pragma unroll
      for (int w = 0; w < 2; ++w) {
        const uint32_t lo = w ? g.klo.y : g.klo.x, hi = w ? g.khi.y : g.khi.x;
        uint32_t o[8];
        if (BOOST) {
          // even, odd: the four bits of tokens 2j and 2j + 1 of each half of the word in nibble j
          const uint32_t even = (lo & 0x33333333u) | ((hi << 2) & 0xccccccccu);
          const uint32_t odd = ((lo >> 2) & 0x33333333u) | (hi & 0xccccccccu);
#pragma unroll
          for (int j = 0; j < 4; j += 2) {
            const uint32_t x = even >> (4 * j), y = odd >> (4 * j);
            o[2 * j] = dequant_code<0>(x, magic, scale, zero);
            o[2 * j + 1] = dequant_code<0>(y, magic, scale, zero);
            o[2 * j + 2] = dequant_code<4>(x, magic, scale, zero);
            o[2 * j + 3] = dequant_code<4>(y, magic, scale, zero);
          }
        } else {   // four values per channel: the table of the V side below
#pragma unroll
          for (int u = 0; u < 8; ++u) {
            const uint32_t code = (lo >> (2 * u)) & 0x00030003u;
            o[u] = __builtin_amdgcn_perm(k23, k01, code * 0x0202u + 0x01000100u);
          }
        }
        uint8_t* dst = row + 128 * w;   // token_group_bytes(2 part + w)
        *(uint4*)dst = uint4{o[0], o[1], o[2], o[3]};
        *(uint4*)(dst + 16) = uint4{o[4], o[5], o[6], o[7]};
      }
    } else {
      // fp16 rows, transposed: a lane = tokens u and u + 8 of a 16-block (neighbours in LDS), a wave = 16 channels
      int id = tid;
      asm volatile("" : "+v"(id));   // formed here, not kept in registers over the packed tiles
      const int64_t stride = in_chunk ? new_stride_t : kD * 2;
      const uint8_t* rows = in_chunk ? k_new + (int64_t)chunk_pos(t) * new_stride_t
                            : in_sink ? (const uint8_t*)L.sink_k + sink : (const uint8_t*)L.qbuf_k + win;
      const int blk = (id & 63) >> 3, tok = blk * 16 + (id & 7), last = tokens(t) - 1, ch = (id >> 6) * 16;
      // (a row past the last one repeats it: its logits are masked)
      const uint4* s0 = (const uint4*)(rows + (int64_t)min(tok, last) * stride + ch * 2);
      const uint4* s1 = (const uint4*)(rows + (int64_t)min(tok + 8, last) * stride + ch * 2);
      uint8_t* col = kt + ch * kPitch + token_group_bytes(blk) + (id & 7) * 4;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const uint4 x = s0[i], y = s1[i];
        const uint32_t x4[4] = {x.x, x.y, x.z, x.w}, y4[4] = {y.x, y.y, y.z, y.w};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          *(uint32_t*)(col + (8 * i + 2 * j) * kPitch) = __builtin_amdgcn_perm(y4[j], x4[j], 0x05040100u);
          *(uint32_t*)(col + (8 * i + 2 * j + 1) * kPitch) = __builtin_amdgcn_perm(y4[j], x4[j], 0x07060302u);
        }
      }
    }
    uint8_t* vrow = vt + value_row() * kPitch + part() * 64;
    if (FULL || v_packed(t)) {
      // thread = one token, 32 channels: words of 16 channels each
      // All of a token's codes share one (scale, zero) and take four values: the four dequantized
      // numbers are computed once (same instructions as dequant_pair, so the same two roundings)
      // and every pair of codes picks its two with a byte permute, selector bytes (2c, 2c+1).
      const half2v m2 = __builtin_bit_cast(half2v, g.vmeta);
      const half2v scale = {m2[0], m2[0]}, zero = {m2[1], m2[1]};
      const uint32_t t01 = dequant_pair(0x00010000u, scale, zero), t23 = dequant_pair(0x00030002u, scale, zero);
#pragma unroll
      for (int w = 0; w < 2; ++w) {
        const uint32_t word = w ? g.v.y : g.v.x;
        uint32_t o[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          const uint32_t codes = (word >> (2 * u)) & 0x00030003u;
          o[u] = __builtin_amdgcn_perm(t23, t01, codes * 0x0202u + 0x01000100u);
        }
        *(uint4*)(vrow + w * 32) = uint4{o[0], o[1], o[2], o[3]};
        *(uint4*)(vrow + w * 32 + 16) = uint4{o[4], o[5], o[6], o[7]};
      }
    } else {
#pragma unroll
      for (int w = 0; w < 2; ++w) {
        // 16 channels at a time: slot 2u + e' takes channel u + 8e'
        const uint4 a = rows_v[2 * w], bb = rows_v[2 * w + 1];   // channels 0..7, 8..15
        const uint32_t a4[4] = {a.x, a.y, a.z, a.w}, b4[4] = {bb.x, bb.y, bb.z, bb.w};
        uint32_t o[8];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          o[2 * j] = __builtin_amdgcn_perm(b4[j], a4[j], 0x05040100u);
          o[2 * j + 1] = __builtin_amdgcn_perm(b4[j], a4[j], 0x07060302u);
        }
        *(uint4*)(vrow + w * 32) = uint4{o[0], o[1], o[2], o[3]};
        *(uint4*)(vrow + w * 32 + 16) = uint4{o[4], o[5], o[6], o[7]};
      }
    }
  }
};

// One wavefront's state: 32 query rows, one per lane pair (l, l + 32), against the tiles in LDS.
struct WaveAcc {
  float16v o[4];   // O^T: channel slots 16 ct .. 16 ct + 15 and 64 + 16 ct .. of the lane's row
  float m, l;      // running max (log2 units), per-lane partial sum
  bool first;
};

// One 128-token tile in (kt, vt) against this wavefront's rows, in groups of SUBS sub-tiles of 32 positions: logits,
// running maxima, probabilities, output.  A wave's matrix and vector phases follow one another; the other wave of the SIMD
// fills the pipe that this one leaves idle (issuing the next sub-tile's logits between a sub-tile's exponentials, as an
// earlier version did, costs 16 registers and gains nothing).  Two sub-tiles per group: when the maximum of any of
// the wave's 32 rows moves, all 64 output registers are scaled, and among the first few thousand tokens that is nearly every
// time (B = 2, 3001 tokens: 214 us with 32 positions per look, 204 with 64, 211 with 128, which spills; 189 if it
// never happened).
// limit: tokens of the tile with index < limit are visible to the lane's row.
// SPLIT: the walk starts anywhere in the sequence, so a row may see nothing of the first sub-tile (and
// then, causally, nothing at all of this share): its running maximum must stay a number.
// DENSE: tokens and channels lie in their natural order, and K as [token][channel] (see dense_attn_kernel).
template <bool SPLIT, bool DENSE>
struct TileAttend {
  const uint8_t* kb;   // K tile + this lane's corner of a transposing read; DENSE: + its row and channels
  const uint8_t* vb;   // V tile + the same corner
  const half8 (&q)[8];
  WaveAcc& A;
  const float sc2;     // not negative (the queries carry the sign)
  const int kg;

  __device__ __forceinline__ void qk(int sub, float16v& S) const {
    const uint8_t* kbase = kb + sub * (DENSE ? 32 * kPitch : 32);
    S = float16v{0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      const half8 a = DENSE ? *(const half8*)(kbase + 32 * c) : load_a(kbase + 16 * c * kPitch);
      S = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, q[c], S, 0, 0, 0);
    }
  }

  __device__ __forceinline__ void pv(int sub, const half8 (&p)[2]) const {
    const uint8_t* vbase = vb + (32 * sub) * kPitch;
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
#pragma unroll
      for (int ct = 0; ct < 4; ++ct)
        A.o[ct] = __builtin_amdgcn_mfma_f32_32x32x16_f16(load_a(vbase + 16 * kk * kPitch + ct * 32), p[kk], A.o[ct], 0, 0, 0);
  }

  static __device__ __forceinline__ float lane_max(const float16v& S) {
    const float x0 = vmax3(S[0], S[1], S[2]), x1 = vmax3(S[3], S[4], S[5]), x2 = vmax3(S[6], S[7], S[8]),
                x3 = vmax3(S[9], S[10], S[11]), x4 = vmax3(S[12], S[13], S[14]);
    return vmax3(vmax3(x0, x1, x2), vmax(x3, x4), S[15]);
  }

  // MASKED: a partial tile or one of the chunk's own
  template <int SUBS, bool MASKED>
  __device__ __forceinline__ void group(int sub, int limit) const {
    float16v S[SUBS];
    half8 p[SUBS][2];
#pragma unroll
    for (int s = 0; s < SUBS; ++s) {
      qk(sub + s, S[s]);
      if (MASKED) {   // scaled here (-inf times a scaling of 0 would be NaN)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int tok = 32 * (sub + s) + (DENSE ? 8 * (i >> 2) + 2 * (i & 3) + kg
                                                  : 16 * (i >> 3) + 4 * ((i >> 2) & 1) + 2 * kg + ((i >> 1) & 1) + 8 * (i & 1));
          S[s][i] = tok < limit ? S[s][i] * sc2 : -INFINITY;
        }
      }
    }
    // vmax3 is assembly, which the compiler's insertion of wait states between a matrix instruction and the first reader of its
    // result does not see into: 20 of them here, for the last product (16 passes: 19); the ones before it are done by then
    if (!MASKED) {
      if (SUBS == 1) asm volatile("s_nop 15\n\ts_nop 3" : "+v"(S[0]));
      else asm volatile("s_nop 15\n\ts_nop 3" : "+v"(S[0]), "+v"(S[SUBS - 1]));
    }
    // this lane's maximum; a logit above the running maximum of its row shows in the lane that holds it, so the maximum
    // over the two lane groups is only formed when some row's maximum really moves
    float mx = lane_max(S[0]);
#pragma unroll
    for (int s = 1; s < SUBS; ++s) mx = vmax(mx, lane_max(S[s]));
    if (!MASKED) mx *= sc2;
    if (__any(A.first || mx > A.m)) {
      const float col = max_over_lane_halves(mx);
      if (A.first) {
        A.m = SPLIT && col == -INFINITY ? 0.f : col;
        A.first = false;
      } else {
        const float m = vmax(A.m, col), alpha = __builtin_amdgcn_exp2f(A.m - m);
        A.l *= alpha;
#pragma unroll
        for (int ct = 0; ct < 4; ++ct) A.o[ct] *= alpha;
        A.m = m;
      }
    }
#pragma unroll
    for (int s = 0; s < SUBS; ++s) {
      float sum = 0.f;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        S[s][i] = __builtin_amdgcn_exp2f(MASKED ? S[s][i] - A.m : __builtin_fmaf(S[s][i], sc2, -A.m));
        sum += S[s][i];
      }
      A.l += sum;
#pragma unroll
      for (int kk = 0; kk < 2; ++kk)
#pragma unroll
        for (int j = 0; j < 8; ++j) p[s][kk][j] = (_Float16)S[s][8 * kk + j];
    }
    __builtin_amdgcn_s_setprio(KITTY_PV_PRIO);
#pragma unroll
    for (int s = 0; s < SUBS; ++s) pv(sub + s, p[s]);
    __builtin_amdgcn_s_setprio(0);
  }

  __device__ __forceinline__ void run_masked(int ntok, int limit) const {
    int sub = 0;
#pragma unroll 1
    for (; 32 * (sub + 1) < ntok; sub += 2) group<2, true>(sub, limit);
    if (32 * sub < ntok) group<1, true>(sub, limit);
  }
  // a whole tile that every row sees
  __device__ __forceinline__ void run_full() const {
#pragma unroll
    for (int sub = 0; sub < 4; sub += kSubs) group<kSubs, false>(sub, kPage);
  }
};

// Chunk positions per workgroup: the chunk cut into as few blocks as 256 rows allow, all of the same size
// (a chunk of 200 positions, four heads per group: 4 x 50 instead of 3 x 64 + 8), so that the rows are
// dense and a wavefront without rows has none of them to multiply.
__host__ __device__ inline int block_positions(int G, int Tq) {
  const int most = kRows / G;
  return c_div_up(Tq, c_div_up(Tq, most));
}

// SPLIT: blockIdx.x = block * num_splits + split; a workgroup walks its share of the tiles and leaves a
// partial per row (running maximum, running sum, un-normalised output) for rows_merge_kernel.  One
// workgroup fills a compute unit (143 KB of LDS), and a short chunk has few of them: 200 positions over
// 12k cached tokens, 32 / 8 heads, are 32 workgroups of 98 tiles on 256 units; in 8 shares they are 256 of 13
// tiles, and a layer (attention and append) takes 96 us instead of 520 (see prefill_splits).
template <bool BOOST, bool SPLIT>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(kWaves / 4, kWaves / 4))) void prefill_attn_kernel(
    kitty_kv_layer L, const uint8_t* __restrict__ q, int64_t q_stride_b, int64_t q_stride_h, int64_t q_stride_t,
    const uint8_t* __restrict__ k_new, const uint8_t* __restrict__ v_new, int64_t new_stride_b,
    int64_t new_stride_h, int64_t new_stride_t, int H_Q, int Tq, float scaling, __half* __restrict__ out,
    float* __restrict__ ws_ml, float* __restrict__ ws_acc, int num_splits) {
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  __shared__ typename Prefill<BOOST, SPLIT>::PageTable s_pages;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, kg = lane >> 5, n = lane & 31;
  const int b = blockIdx.z, h = blockIdx.y;
  const int G = H_Q / L.H_KV;
  const int PB = block_positions(G, Tq);                 // chunk positions per workgroup
  const int split = SPLIT ? (int)blockIdx.x % num_splits : 0;
  const int blk = SPLIT ? ((int)gridDim.x - 1 - (int)blockIdx.x) / num_splits
                        : (int)gridDim.x - 1 - (int)blockIdx.x;   // longest causal extent first
  const int p0 = blk * PB;

  SeqCounts cnt = load_counts(L, b);
  for (int* x : {&cnt.sink, &cnt.pk, &cnt.rk, &cnt.pv, &cnt.rv, &cnt.lv, &cnt.off, &cnt.nbody})   // the same in every lane
    *x = __builtin_amdgcn_readfirstlane(*x);
  Prefill<BOOST, SPLIT> P{L, cnt, b, h, tid,
                   k_new + (int64_t)b * new_stride_b + (int64_t)h * new_stride_h,
                   v_new + (int64_t)b * new_stride_b + (int64_t)h * new_stride_h,
                   new_stride_t, min(Tq, p0 + PB), 0, 0, 0};
  P.pages = s_pages;
  P.first_body = cnt.sink > 0 ? 1 : 0;
  P.first_chunk = P.first_body + c_div_up(cnt.nbody, kPage);
  P.n_tiles = P.first_chunk + c_div_up(P.kv_chunk, kPage);
  int t_begin = 0, t_end = P.n_tiles;
  if (SPLIT) {
    const int share = c_div_up(P.n_tiles, num_splits);
    t_begin = min(split * share, P.n_tiles);
    t_end = min(t_begin + share, P.n_tiles);
    P.first_id = max(t_begin - P.first_body, 0);
  }

  // this lane's query row: column n of the wave's tile is row 32 w + n
  half8 qreg[8];
  const uint32_t flip = scaling < 0.f ? 0x80008000u : 0u;   // the logits are scaled by a number that is not negative
  const int r = kWaveRows * w + n, g = r / PB, pos = p0 + r % PB;
  const bool ok = g < G && pos < Tq;
  const int qpos = ok ? pos : -1;
  {
    const uint8_t* row = q + (int64_t)b * q_stride_b + (int64_t)(h * G + (ok ? g : 0)) * q_stride_h +
                         (int64_t)(ok ? pos : 0) * q_stride_t;
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      // k-slots = channels 16c + kg, + 2, + 4, .. (row_slot)
      const uint4 x0 = *(const uint4*)(row + 32 * c), x1 = *(const uint4*)(row + 32 * c + 16);
      const uint32_t sel = kg ? 0x07060302u : 0x05040100u;
      uint4 x = uint4{__builtin_amdgcn_perm(x0.y, x0.x, sel), __builtin_amdgcn_perm(x0.w, x0.z, sel),
                      __builtin_amdgcn_perm(x1.y, x1.x, sel), __builtin_amdgcn_perm(x1.w, x1.z, sel)};
      if (!ok) x = uint4{0u, 0u, 0u, 0u};
      x.x ^= flip, x.y ^= flip, x.z ^= flip, x.w ^= flip;
      qreg[c] = __builtin_bit_cast(half8, x);
    }
  }

  WaveAcc A;
#pragma unroll
  for (int ct = 0; ct < 4; ++ct)
#pragma unroll
    for (int i = 0; i < 16; ++i) A.o[ct][i] = 0.f;
  A.m = A.l = 0.f;
  A.first = true;
  const float sc2 = fabsf(scaling) * kLog2e;

  // Software pipeline over tiles: tile t is multiplied from LDS buffer t & 1 while tile t+1 is
  // turned into fp16 in the other buffer from registers loaded one iteration earlier, and the
  // packed bytes of tile t+2 are on their way.  The waves of a SIMD take the two jobs in opposite
  // order (waves 0..3 convert first, waves 4..7 multiply first), so that one does vector work
  // while the other keeps the matrix pipe busy.  One barrier per tile.
  const bool convert_first = w < kWaves / 2;
  const bool has_rows = !SPLIT || kWaveRows * w < G * PB;   // (tested in full blocks it costs 2 %)
  Stage ga, gb;                       // tile t+1, tile t+2
  int slot = 255;                     // of tile t+2
  P.stage_pages(0);
  __syncthreads();
  if (!SPLIT || t_begin < t_end) {    // (the last splits of a short walk are empty)
    const int s0 = P.template ask_slot<false>(t_begin), s1 = t_begin + 1 < t_end ? P.template ask_slot<false>(t_begin + 1) : 255;
    P.template issue<false>(t_begin, s0, ga);
    if (t_begin + 1 < t_end) P.template issue<false>(t_begin + 1, s1, gb);
    if (t_begin + 2 < t_end) slot = P.template ask_slot<false>(t_begin + 2);
    P.template finish<false>(t_begin, ga, lds, lds + 2 * kTile);
    ga = gb;
  }
  __syncthreads();
  // FULL: tiles t .. t + 3 are whole pages on both sides - nearly all of a long walk, and a tile then costs 60 scalar
  // instructions (a wave issues one in 8 clocks) and the test for masks in each sub-tile less (loops of their own: in one loop
  // with a branch the output's registers are copied where the paths meet)
  auto step = [&](auto full, int t) {
    constexpr bool FULL = decltype(full)::value;
    const int buf = (t - t_begin) & 1;
    const bool more = FULL || t + 1 < t_end;
    if (FULL || t + 2 < t_end) P.template issue<FULL>(t + 2, slot, gb);
    if (FULL || t + 3 < t_end) slot = P.template ask_slot<FULL>(t + 3);
    {   // half way through a chunk of addresses: stage the next one (ask_slot() is at tile t + 3)
      constexpr int kChunk = Prefill<BOOST, SPLIT>::kChunk;
      const int i = P.body(t + 3) - P.id_base();
      if (i >= 0 && i % kChunk == kChunk / 2) P.stage_pages(i / kChunk + 1);
    }
    uint8_t* kn = lds + (buf ^ 1) * kTile;
    uint8_t* vn = lds + (2 + (buf ^ 1)) * kTile;
    if (more && convert_first) P.template finish<FULL>(t + 1, ga, kn, vn);
    if (has_rows) {
      // the lane's corner inside a 16-lane transposing read: row 2 j + kg of eight, j = n % 16 / 4 (row_slot), columns
      // 4 (n % 4) .., the upper 16 lanes of a half 128 bytes further; made opaque so that every read's offset stays a small immediate on these two bases
      uint32_t ok_ = buf * kTile + (kg + ((n >> 2) & 3) * 2) * kPitch + (n & 3) * 8 + (n >> 4) * 128;
      uint32_t ov_ = ok_ + 2 * kTile;
      asm volatile("" : "+v"(ok_), "+v"(ov_));
      const TileAttend<SPLIT, false> T{lds + ok_, lds + ov_, qreg, A, sc2, kg};
      const int ntok = FULL ? kPage : P.tokens(t), chunk_t0 = P.chunk_pos(t);
      // (a tile of the chunk that ends in front of the workgroup's first position is seen whole by every row)
      if (FULL || (ntok == kPage && chunk_t0 + kPage - 1 <= p0)) T.run_full();
      else T.run_masked(ntok, chunk_t0 >= 0 ? min(ntok, qpos - chunk_t0 + 1) : ntok);
    }
    if (more && !convert_first) P.template finish<FULL>(t + 1, ga, kn, vn);
    ga = gb;
    __syncthreads();
  };
  int t = t_begin;
  const int full_end = min(P.first_body + min(cnt.pk, cnt.pv), t_end) - 3;
#pragma unroll 1
  for (; t < min(P.first_body, t_end); ++t) step(std::false_type{}, t);
#pragma unroll 1
  for (; t < full_end; ++t) step(std::true_type{}, t);
#pragma unroll 1
  for (; t < t_end; ++t) step(std::false_type{}, t);

  // normalise and store: O^T[ct][i] is channel slot 64 (i / 8) + 16 ct + 8 (i / 4 % 2) + 4 kg + i % 4 of the lane's row;
  // slots 4x + {0, 2} of a 16-block are channels 2x, 2x + 1, slots 4x + {1, 3} are channels 2x + 8, 2x + 9
  const float l = A.l + xor_lanes(A.l, 32);
  if (ok) {
    const int64_t row = ((int64_t)b * Tq + qpos) * H_Q + (h * G + g);
    if (SPLIT) {
      const int64_t prow = row * num_splits + split;
      if (kg == 0) *(float2*)(ws_ml + prow * 2) = float2{l == 0.f ? -INFINITY : A.m, l};   // 0: this row saw nothing here
#pragma unroll
      for (int ct = 0; ct < 4; ++ct)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          float* o = ws_acc + prow * kD + 64 * (i >> 1) + 16 * ct + 4 * (i & 1) + 2 * kg;
          *(float2*)o = float2{A.o[ct][4 * i], A.o[ct][4 * i + 2]};
          *(float2*)(o + 8) = float2{A.o[ct][4 * i + 1], A.o[ct][4 * i + 3]};
        }
    } else {
      const float inv = 1.f / l;
#pragma unroll
      for (int ct = 0; ct < 4; ++ct)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          __half* o = out + row * kD + 64 * (i >> 1) + 16 * ct + 4 * (i & 1) + 2 * kg;
          *(__half2*)o = __floats2half2_rn(A.o[ct][4 * i] * inv, A.o[ct][4 * i + 2] * inv);
          *(__half2*)(o + 8) = __floats2half2_rn(A.o[ct][4 * i + 1] * inv, A.o[ct][4 * i + 3] * inv);
        }
    }
  }
  report_bad_page(L, b, P.bad_page);   // by whichever thread met one
}

// A chunk over a layer that holds nothing: dense causal attention.  The frame is that of the kernel above - 256
// rows a workgroup, two tile buffers, waves of a SIMD that stage and multiply in opposite order - but every tile is
// fp16 rows, so nothing has to be permuted to meet codes: a row is copied as it lies (16 lanes a row), loaded into registers
// while the tile before it is worked on.  K stays [token][channel] and is read 16 bytes a lane, its rows in the order of
// row_slot; V [token][channel] is read transposed.  On the kernel above such a tile costs twice a packed one: its rows are
// fetched when they are needed, K is transposed on its way in, every tile is masked.  Workgroups of one kv head share an XCD,
// whose L2 then serves its keys and values, longest first.  Bound, as the kernel above, by power and the vector unit.
// B = 2, 3001 tokens, 32 / 8 heads, with the packing of the prompt: 240 -> 204 us.
template <bool SPLIT>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(kWaves / 4, kWaves / 4))) void dense_attn_kernel(
    const uint8_t* __restrict__ q, int64_t q_stride_b, int64_t q_stride_h, int64_t q_stride_t,
    const uint8_t* __restrict__ k_new, const uint8_t* __restrict__ v_new, int64_t new_stride_b, int64_t new_stride_h,
    int64_t new_stride_t, int H_Q, int H_KV, int Tq, float scaling, __half* __restrict__ out, float* __restrict__ ws_ml,
    float* __restrict__ ws_acc, int num_splits, int heads) {
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, kg = lane >> 5, n = lane & 31;
  // blockIdx.x -> (kv head of a batch row, block x split): consecutive workgroups go to the XCDs in turn
  const int id = blockIdx.x;
  int head, item;
  if (heads % 8 == 0) {
    const int per_xcd = heads / 8, j = id / 8;
    head = (j % per_xcd) * 8 + id % 8, item = j / per_xcd;
  } else {
    head = id % heads, item = id / heads;
  }
  const int b = head / H_KV, h = head % H_KV;
  const int G = H_Q / H_KV;
  const int PB = block_positions(G, Tq);
  const int split = SPLIT ? item % num_splits : 0;
  const int blk = c_div_up(Tq, PB) - 1 - (SPLIT ? item / num_splits : item);   // longest causal extent first
  const int p0 = blk * PB, kv = min(Tq, p0 + PB);
  const int n_tiles = c_div_up(kv, kPage);
  int t_begin = 0, t_end = n_tiles;
  if (SPLIT) {
    const int share = c_div_up(n_tiles, num_splits);
    t_begin = min(split * share, n_tiles);
    t_end = min(t_begin + share, n_tiles);
  }
  const uint8_t* kc = k_new + (int64_t)b * new_stride_b + (int64_t)h * new_stride_h;
  const uint8_t* vc = v_new + (int64_t)b * new_stride_b + (int64_t)h * new_stride_h;

  // this lane's query row: column n of the wave's tile is row 32 w + n
  half8 qreg[8];
  const uint32_t flip = scaling < 0.f ? 0x80008000u : 0u;   // the logits are scaled by a number that is not negative
  const int r = kWaveRows * w + n, g = r / PB, pos = p0 + r % PB;
  const bool ok = g < G && pos < Tq;
  const int qpos = ok ? pos : -1;
  {
    const uint8_t* row = q + (int64_t)b * q_stride_b + (int64_t)(h * G + (ok ? g : 0)) * q_stride_h +
                         (int64_t)(ok ? pos : 0) * q_stride_t;
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      uint4 x = *(const uint4*)(row + (16 * c + 8 * kg) * 2);   // k-slots = channels 16c + 8kg ..
      if (!ok) x = uint4{0u, 0u, 0u, 0u};
      x.x ^= flip, x.y ^= flip, x.z ^= flip, x.w ^= flip;
      qreg[c] = __builtin_bit_cast(half8, x);
    }
  }

  WaveAcc A;
#pragma unroll
  for (int ct = 0; ct < 4; ++ct)
#pragma unroll
    for (int i = 0; i < 16; ++i) A.o[ct][i] = 0.f;
  A.m = A.l = 0.f;
  A.first = true;
  const float sc2 = fabsf(scaling) * kLog2e;

  // a thread stages 16-byte piece tid % 16 of tokens tid / 16, + 32, ..: 16 lanes write one row, 64 different banks
  const int e = tid >> 4, part = (tid & 15) * 16;
  uint4v kk[4], vv[4];
  auto issue = [&](int t) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int tok = t * kPage + e + 32 * i;
      const int64_t off = (int64_t)min(tok, kv - 1) * new_stride_t + part;
      kk[i] = *(const uint4v*)(kc + off);
      vv[i] = *(const uint4v*)(vc + off);
      if (tok >= kv) vv[i] = uint4v{0u, 0u, 0u, 0u};   // dead rows of V must be finite
    }
  };
  auto finish = [&](int buf) {
    uint8_t* kt = lds + buf * kTile + e * kPitch + part;
    uint8_t* vt = lds + (2 + buf) * kTile + e * kPitch + part;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      *(uint4v*)(kt + 32 * i * kPitch) = kk[i];
      *(uint4v*)(vt + 32 * i * kPitch) = vv[i];
    }
  };
  const bool stage_first = w < kWaves / 2;
  if (!SPLIT || t_begin < t_end) {
    issue(t_begin);
    finish(0);
    if (t_begin + 1 < t_end) issue(t_begin + 1);
  }
  __syncthreads();
  // FULL: a tile in front of the workgroup's first position, which every row sees whole
  auto step = [&](auto full, int t) {
    constexpr bool FULL = decltype(full)::value;
    const int buf = (t - t_begin) & 1;
    auto stage_next = [&] {
      if (t + 1 < t_end) finish(buf ^ 1);
      if (t + 2 < t_end) issue(t + 2);
    };
    if (stage_first) stage_next();
    {
      // K: the lane's logits are those of k-slots 4 kg .. of V's rows (row_slot)
      uint32_t ok_ = buf * kTile + ((n & ~7) + 2 * (n & 3) + ((n >> 2) & 1)) * kPitch + kg * 16;
      uint32_t ov_ = (2 + buf) * kTile + (kg + ((n >> 2) & 3) * 2) * kPitch + (n & 3) * 8 + (n >> 4) * 128;
      asm volatile("" : "+v"(ok_), "+v"(ov_));
      const int t0 = t * kPage, ntok = min(kPage, kv - t0);
      const TileAttend<SPLIT, true> T{lds + ok_, lds + ov_, qreg, A, sc2, kg};
      if (FULL) T.run_full();
      else T.run_masked(ntok, min(ntok, qpos - t0 + 1));
    }
    if (!stage_first) stage_next();
    __syncthreads();
  };
  int t = t_begin;
  const int full_end = min(p0 / kPage, t_end);
#pragma unroll 1
  for (; t < full_end; ++t) step(std::true_type{}, t);
#pragma unroll 1
  for (; t < t_end; ++t) step(std::false_type{}, t);

  const float l = A.l + xor_lanes(A.l, 32);
  if (!ok) return;
  const int64_t row = ((int64_t)b * Tq + qpos) * H_Q + (h * G + g);
  const int64_t prow = row * num_splits + split;
  if (SPLIT && kg == 0) *(float2*)(ws_ml + prow * 2) = float2{l == 0.f ? -INFINITY : A.m, l};   // 0: this row saw nothing here
  const float inv = 1.f / l;
#pragma unroll
  for (int ct = 0; ct < 4; ++ct)
#pragma unroll
    for (int i = 0; i < 4; ++i) {   // channels 64 (i / 2) + 16 ct + 8 (i % 2) + 4 kg ..
      const int ch = 64 * (i >> 1) + 16 * ct + 8 * (i & 1) + 4 * kg;
      const float4v o = {A.o[ct][4 * i], A.o[ct][4 * i + 1], A.o[ct][4 * i + 2], A.o[ct][4 * i + 3]};
      if (SPLIT) {
        *(float4v*)(ws_acc + prow * kD + ch) = o;
      } else {
        __half2 x[2] = {__floats2half2_rn(o[0] * inv, o[1] * inv), __floats2half2_rn(o[2] * inv, o[3] * inv)};
        *(uint2*)(out + row * kD + ch) = *(const uint2*)x;
      }
    }
}

}  // namespace

int prefill_lds_bytes() { return kLdsBytes; }

// How many shares the walk over the tiles is cut into.  A workgroup has a compute unit to itself, so a launch
// of W workgroups takes ceil(W / units) rounds of its longest walk; cutting the walk in s shortens the walk
// and multiplies the workgroups.  What a share costs besides its tiles is about three tiles' time (filling
// the pipeline, 128 KB of partials); the merge reads 512 bytes a row and share.  A tile is priced at 5.4 us, between
// a whole page (4.2 with all rows in use) and one of fp16 rows.  (At 4.2 short walks, which are mostly fp16 rows, get too few
// shares: 300 tokens over 1000 three, 144 us, where four take 129; long ones the same.)  The smallest total wins; ties go to
// fewer shares.
// `tiles`: 128-token tiles the layer holds (sink included) plus those of the chunk; `most`: shares the scratch allows.
int prefill_splits(int B, int H_Q, int H_KV, int Tq, int tiles, int units, int most) {
  const int G = H_Q / H_KV;
  if ((int64_t)B * Tq > 65535) return 1;   // more than a workgroup per compute unit for every query head: the device is full
  const int64_t wgs = (int64_t)c_div_up(Tq, block_positions(G, Tq)) * H_KV * B;
  const float rows = (float)B * (float)Tq * (float)H_Q;
  int best = 1;
  float best_us = 0.f;
  for (int s = 1; s <= most && (s == 1 || 2 * s <= tiles); ++s) {
    const int64_t rounds = (wgs * s + units - 1) / units;
    float us = 5.4f * (float)rounds * (float)(c_div_up(tiles, s) + 3);
    if (s > 1) us += 4.f + rows * (float)s * 3.5e-4f;   // write + read of 1 KB at about 3 TB/s
    if (s == 1 || us < 0.98f * best_us) best = s, best_us = us;
  }
  return best;
}

void launch_prefill_attn(const kitty_kv_layer& L, const void* q, int64_t q_stride_b, int64_t q_stride_h,
                         int64_t q_stride_t, const void* k_new, const void* v_new, int64_t new_stride_b,
                         int64_t new_stride_h, int64_t new_stride_t, int B, int H_Q, int Tq, float scaling,
                         void* out, float* ws_ml, float* ws_acc, int num_splits, hipStream_t stream) {
  const int G = H_Q / L.H_KV;
  const int blocks = c_div_up(Tq, block_positions(G, Tq));
  dim3 grid(blocks * num_splits, L.H_KV, B), block(kThreads);
  const int* c = L.counts;
  const int64_t dense_wgs = (int64_t)blocks * num_splits * L.H_KV * B;
  if (!L.seq_counts && c[KITTY_CNT_SINK] == 0 && c[KITTY_CNT_PAGES_K] + c[KITTY_CNT_QBUF_K] == 0 && dense_wgs <= (1 << 22)) {   // (grid limit)
    // (check_layer: as many values as keys)
#define KITTY_LAUNCH_DENSE(SPLIT)                                                                                \
  do {                                                                                                           \
    (void)hipFuncSetAttribute((const void*)dense_attn_kernel<SPLIT>, hipFuncAttributeMaxDynamicSharedMemorySize, kLdsBytes); \
    hipLaunchKernelGGL((dense_attn_kernel<SPLIT>), dim3((unsigned)dense_wgs), block, kLdsBytes, stream, (const uint8_t*)q, \
                       q_stride_b, q_stride_h, q_stride_t, (const uint8_t*)k_new, (const uint8_t*)v_new, new_stride_b, \
                       new_stride_h, new_stride_t, H_Q, L.H_KV, Tq, scaling, (__half*)out, ws_ml, ws_acc, num_splits,  \
                       L.H_KV * B);                                                                              \
  } while (0)
    if (num_splits > 1) {
      KITTY_LAUNCH_DENSE(true);
      launch_rows_merge(kD, ws_ml, ws_acc, out, (int64_t)B * Tq * H_Q, num_splits, /* keep_nan */ true, stream);
    } else {
      KITTY_LAUNCH_DENSE(false);
    }
#undef KITTY_LAUNCH_DENSE
    return;
  }
#define KITTY_LAUNCH_PREFILL(BOOST, SPLIT)                                                                       \
  do {                                                                                                           \
    /* more LDS than the default per-workgroup limit; per device, so set on every launch */                      \
    (void)hipFuncSetAttribute((const void*)prefill_attn_kernel<BOOST, SPLIT>,                                    \
                              hipFuncAttributeMaxDynamicSharedMemorySize, kLdsBytes);                            \
    hipLaunchKernelGGL((prefill_attn_kernel<BOOST, SPLIT>), grid, block, kLdsBytes, stream, L, (const uint8_t*)q, \
                       q_stride_b, q_stride_h, q_stride_t, (const uint8_t*)k_new, (const uint8_t*)v_new,         \
                       new_stride_b, new_stride_h, new_stride_t, H_Q, Tq, scaling, (__half*)out, ws_ml, ws_acc,  \
                       num_splits);                                                                              \
  } while (0)
  if (num_splits > 1) {
    if (L.D_BOOSTED > 0) KITTY_LAUNCH_PREFILL(true, true);
    else KITTY_LAUNCH_PREFILL(false, true);
    launch_rows_merge(kD, ws_ml, ws_acc, out, (int64_t)B * Tq * H_Q, num_splits, /* keep_nan */ true, stream);
  } else {
    if (L.D_BOOSTED > 0) KITTY_LAUNCH_PREFILL(true, false);
    else KITTY_LAUNCH_PREFILL(false, false);
  }
#undef KITTY_LAUNCH_PREFILL
}

}  // namespace kitty
