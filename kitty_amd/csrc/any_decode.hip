// Decode attention for head dimensions other than 128 (64 and 256): the split pass.
//
// The same arithmetic and storage format as any_dim.hip's chunk kernel (keys and values dequantized with the reference's two
// fp16 roundings, kitty_attention.py:162-165, 317-320; probabilities as fp32 numbers), with the rows of one decode
// step: the G query heads of a kv head.  What bounds it is turning codes into fp16 numbers, once per code and not per row, so
// a wavefront owns whole pages: it takes all 8 codes of every 16-bit piece that a transposing read hands it, four
// bits at a time, and shares nothing with the other wavefronts of its workgroup until the end.  No barrier in the walk; the
// packed bytes go from memory to LDS without passing registers, the next page's keys while this page's values are
// multiplied and its values while the next page's logits are formed.
//
//   S^T[token 8m + u][col] = sum_ch  K[token][ch] * Q[col][ch]       (A = K, row m; B = Q in registers), u = 0 .. 7
//   O^T[ch][col]           = sum_tok V[tok][ch]   * P^T[tok][col]    (A = V, B = P)
//
// Lane 16 kg + n holds S^T of tokens 32 kg + 8 j + u, j = 0 .. 3, of column n: tokens 32 kg + 8 c .. + 7 are the k-slots of lane
// group kg in the c-th product of 32 tokens.  A probability enters as three fp16 numbers that together are the fp32 number
// (p * 2^15, down to 2^-40 of the row's largest).  With at most five heads (COLS) the three sit in columns of their own - column
// n is part n / G of head n % G - so that one matrix instruction takes all of them and the columns are added once at the end.
//
// The version before it dealt every page's tokens to the four wavefronts, each of which took two of the 8 codes of a piece,
// behind two barriers a page: 553 vector and 147 scalar instructions per wavefront and page at D = 64, 1465 and 238 at D = 256,
// four times; now 880 (D = 64) and 2900 (D = 256) vector instructions a page in all.  A decode layer (append, this
// kernel, merge): D = 64, B = 8, 6100 tokens, 32 / 8 heads: 26 -> 22 us; D = 256, B = 2, 9000 tokens, 16 / 8: 39 -> 28.5.  Both
// passes alone: D = 64, B = 32, 8000 tokens, 24 / 8: 80 -> 45; D = 256, B = 4, 30000 tokens, 16 / 8: 110 -> 75.
#include <type_traits>

#include "any_dim.h"

namespace kitty {
// few tiles (any_dim.hip)
void launch_decode_by_tile(const kitty_kv_layer& L, const void* q, int B, int H_Q, float scaling, float* ws_ml, float* ws_acc,
                           int num_splits, hipStream_t stream);
namespace {

// LDS of one wavefront: the packed bytes of a page as they lie in memory
struct WaveLds {
  int zero_row, k_meta, v_raw, v_meta, bytes;
  __host__ __device__ WaveLds(int D, int DB) {
    zero_row = k_head_bytes_d(D, DB);          // 32 zero bytes: the high-plane row of a channel that has none
    k_meta = zero_row + kRowBytes;
    v_raw = k_meta + 4 * D;
    v_meta = v_raw + v_head_bytes_d(D);
    bytes = v_meta + 4 * kPage;
  }
};

template <int N>
__device__ __forceinline__ void wait_loads() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }
__device__ __forceinline__ void wait_reads() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

// 64 lanes x BYTES (4 or 16) from global memory to LDS; M0 reaches the instruction as an operand.  The s_nop is the wait state that the
// hardware needs between a scalar write of M0 and such a load, which the compiler does not put in front of assembly.  Every page is read once.
template <int BYTES>
__device__ __forceinline__ void to_lds(const uint8_t* src, uint32_t dst, int lane) {
  register uint32_t m0_lds asm("m0") = dst;
  const uint32_t off = lane * BYTES;
  if (BYTES == 16) asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, %1 nt" ::"v"(off), "s"(src), "s"(m0_lds) : "memory");
  else asm volatile("s_nop 0\n\tglobal_load_lds_dword %0, %1 nt" ::"v"(off), "s"(src), "s"(m0_lds) : "memory");
}
// `bytes` (a multiple of 16, at least 1024) in whole kilobytes, the last one ending with the data: bytes that two of them cover
// are the same
__device__ __forceinline__ void block_to_lds(const uint8_t* src, uint32_t dst, int bytes, int lane) {
#pragma unroll 1
  for (int at = 0; at < bytes; at += 1024) {
    const int from = __builtin_amdgcn_readfirstlane(min(at, bytes - 1024));
    to_lds<16>(src + from, dst + from, lane);
  }
}

// the infinite and NaN halves of a word, the others 0; `fin` is finite_word(x)
__device__ __forceinline__ uint32_t infinite_word(uint32_t x, uint32_t fin) {
  return __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2v, x) - __builtin_bit_cast(half2v, fin));
}

// fp16(code) * scale + zero, both operations rounded, for the codes at bit K of each half of x, in three instructions:
// 2^(10-K) + code is a number of fp16 whose bits are `magic` with the code in place, and multiplying it by the scale and
// subtracting 2^(10-K) * scale (`base`, exact while the scale is below 64) in one rounding is the rounded product.
template <int K>
constexpr uint32_t kMagic = (uint32_t)((25 - K) << 10) * 0x10001u;   // 2^(10-K) in both halves
template <int K>
__device__ __forceinline__ uint32_t scale_base(uint32_t scale) {
  constexpr _Float16 k = (_Float16)(-(float)(1 << (10 - K)));
  return __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2v, scale) * half2v{k, k});
}
__device__ __forceinline__ uint32_t dequant_fast(uint32_t x, uint32_t mask, uint32_t magic, uint32_t scale, uint32_t base, uint32_t zero) {
#pragma clang fp contract(off)
  const half2v c = __builtin_bit_cast(half2v, (x & mask) | magic);
  const half2v m = __builtin_elementwise_fma(c, __builtin_bit_cast(half2v, scale), __builtin_bit_cast(half2v, base));
  const half2v r = m + __builtin_bit_cast(half2v, zero);
  return __builtin_bit_cast(uint32_t, r);
}
// Of a (scale, zero) pair: bit 15 or 31 set unless |scale| < 64 (dequant_fast) and |zero| < 2^13 (with the former, a code up
// to 15 then cannot make the sum infinite)
__device__ __forceinline__ uint32_t out_of_range(uint32_t scale_zero) { return (scale_zero & 0x7fff7fffu) + 0x10002c00u; }

template <int D, bool COLS>
struct Step {
  static constexpr int kHalves = D == 256 ? 2 : 1;   // V rows in pieces of 128 channels
  static constexpr int kU = D == 256 ? 8 : 4;        // channels of a lane within a piece
  static constexpr int kOT = kHalves * kU;           // 16-channel tiles of the output
  float4v O[kOT];
  float m, l;            // running maximum (log2 units), this lane's sum
  float sel1, sel2;      // COLS: -1 if this column's part follows the first (second) one, else 0

  // Moves the running maximum if some lane's lies above it.
  __device__ __forceinline__ void settle(float mx) {
    if (__any(mx > m)) {
      const float col = max_over_lane_groups(mx);
      const float up = fmaxf(m, col);
      const float alpha = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - up);
      l *= alpha;
#pragma unroll
      for (int t = 0; t < kOT; ++t) O[t] *= alpha;
      m = up;
    }
  }
  __device__ __forceinline__ float shift() const { return m == -INFINITY ? 0.f : -m; }

  // eight probabilities (k-slots of one product) as operands: the column's part, or all three.  first: part 0 in every column
  __device__ __forceinline__ void parts(const float (&x)[8], uint32_t (&first)[4], uint32_t (&p1)[4], uint32_t (&p2)[4]) const {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float a = x[2 * i] * kProbScale, b = x[2 * i + 1] * kProbScale;
      const half2v h = {(_Float16)a, (_Float16)b};
      first[i] = __builtin_bit_cast(uint32_t, h);
      const float s1 = COLS ? sel1 : -1.f, s2 = COLS ? sel2 : -1.f;
      const float a1 = __builtin_fmaf((float)h[0], s1, a), b1 = __builtin_fmaf((float)h[1], s1, b);   // exact
      const half2v g = {(_Float16)a1, (_Float16)b1};
      p1[i] = __builtin_bit_cast(uint32_t, g);
      const half2v f = {(_Float16)__builtin_fmaf((float)g[0], s2, a1), (_Float16)__builtin_fmaf((float)g[1], s2, b1)};
      p2[i] = __builtin_bit_cast(uint32_t, f);
    }
  }
  // O[t] += values x probabilities.  WILD: some value may be infinite or NaN, and what is meets part 0 only (the others may be 0
  // or negative)
  template <bool WILD>
  __device__ __forceinline__ void weigh(const uint32_t (&a)[4], int t, const uint32_t (&first)[4], const uint32_t (&p1)[4],
                                        const uint32_t (&p2)[4]) {
    if (!WILD) {
      if (!COLS) O[t] = mfma16(a, first, O[t]), O[t] = mfma16(a, p1, O[t]);
      O[t] = mfma16(a, p2, O[t]);
      return;
    }
    uint32_t fin[4], inf[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) fin[i] = finite_word(a[i]), inf[i] = infinite_word(a[i], fin[i]);
    if (!COLS) O[t] = mfma16(fin, first, O[t]), O[t] = mfma16(fin, p1, O[t]);
    O[t] = mfma16(fin, p2, O[t]);
    O[t] = mfma16(inf, first, O[t]);
    __builtin_amdgcn_sched_barrier(0);   // (interleaved with its neighbours' this rare case would set the kernel's number of registers)
  }
};

// One workgroup of 4 wavefronts per (split, kv head, batch row).  Whole pages are dealt in turn: page i belongs to split
// i % dealt, wavefront i / dealt % 4.  The tiles with fp16 rows (sink, the end of the sequence) go to the splits from
// the last on, one each, and all four wavefronts share its tokens: wavefront w takes 8i + 2w and 8i + 2w + 1.  The partial
// (running maximum in log2 units, sum, un-normalised output) goes to the split-K workspace.
template <int D, bool COLS>
__global__ __launch_bounds__(256, D == 64 ? 4 : 2) void decode_any_kernel(kitty_kv_layer L, const uint8_t* __restrict__ q,
                                                                          int H_Q, float scaling, float* __restrict__ ws_ml,
                                                                          float* __restrict__ ws_acc, int num_splits) {
  static_assert(D == 64 || D == 256, "128 has kernels of its own");
  typedef Step<D, COLS> State;
  constexpr int kU = State::kU, kHalves = State::kHalves, kOT = State::kOT, kKC = D / 32;
  constexpr int kVLoads = 32 * D / 1024 + 2;
  const int split = blockIdx.x, h = blockIdx.y, b = blockIdx.z;
  const int tid = threadIdx.x, lane = tid & 63, kg = lane >> 4, n = lane & 15;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int G = H_Q / L.H_KV, DB = L.D_BOOSTED;
  SeqCounts c = load_counts(L, b);
  for (int* x : {&c.sink, &c.pk, &c.rk, &c.pv, &c.rv, &c.lv, &c.off, &c.nbody, &c.ntiles})   // the same in every lane
    *x = __builtin_amdgcn_readfirstlane(*x);
  const int n_full = min(min(c.pk, c.pv), c.nbody / kPage);
  const int has_sink = c.sink > 0 ? 1 : 0, n_special = has_sink + c.ntiles - 1 - n_full;
  int bad_page = 0;

  extern __shared__ __attribute__((aligned(16))) uint8_t lds_all[];
  __shared__ float s_m[4][16], s_l[4][16];
  __shared__ int s_left[4];
  const WaveLds at(D, DB);
  uint8_t* const lds = lds_all + w * at.bytes;
  const uint8_t* page_lds = lds;   // where a page's bytes are read
  const uint32_t lds_at = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)lds);
  if (lane < 2) ((uint4*)(lds + at.zero_row))[lane] = uint4{0u, 0u, 0u, 0u};

  // the query row of this column as operands: k-slots 0..3 of chunk kc are channels 32 kc + 4 kg .., 4..7 those 16 further
  auto load_query = [&](uint32_t (&qq)[kKC][4]) {
    int id = lane;
    asm volatile("" : "+v"(id));   // loaded where it is wanted, not kept in registers (32 at D = 256) from one use to the next
    const int g = COLS ? (id & 15) % G : id & 15;
    const uint32_t flip = scaling < 0.f ? 0x80008000u : 0u;   // the logits are scaled by a number that is not negative
    const uint8_t* row = q + ((int64_t)b * H_Q + h * G + (g < G ? g : 0)) * (D * 2) + (id >> 4) * 8;
#pragma unroll
    for (int kc = 0; kc < kKC; ++kc) {
      const uint2 x0 = *(const uint2*)(row + 64 * kc), x1 = *(const uint2*)(row + 64 * kc + 32);
      const uint32_t x[4] = {x0.x, x0.y, x1.x, x1.y};
#pragma unroll
      for (int i = 0; i < 4; ++i) qq[kc][i] = g < G ? x[i] ^ flip : 0u;
    }
  };
  State A;
#pragma unroll
  for (int t = 0; t < kOT; ++t) A.O[t] = float4v{0.f, 0.f, 0.f, 0.f};
  A.m = -INFINITY, A.l = 0.f;
  A.sel1 = n >= G ? -1.f : 0.f, A.sel2 = n >= 2 * G ? -1.f : 0.f;
  const float sc2 = fabsf(scaling) * kLog2e;
  uint32_t magic[5] = {kMagic<0>, kMagic<2>, kMagic<4>, kMagic<6>, kMagic<8>};
  static_assert(kMagic<0> == kCodeMagic, "the bits of 1024");
#pragma unroll
  for (int i = 0; i < 5; ++i) asm volatile("" : "+v"(magic[i]));   // in registers: with the mask as the instruction's constant, masking and merging are one

  // (a lane's offsets are formed here, not kept in registers from one fetch to the next: with more than five heads at D = 64 others then
  // spill, and a reload inside the page loop waits for the pages under way: B = 42, 4904 tokens, 14 / 2 heads: 25.0 us, 22.8 so)
  auto fetch_k = [&](int page) {
    int lane = tid & 63;
    asm volatile("" : "+v"(lane));
    const int64_t pg = checked_page(page_id(L.page_table_k, (int64_t)b * L.page_table_k_stride_b + page), L.cache_pages_k, bad_page);
    const uint8_t* src = L.key_cache + pg * L.key_cache_stride_page + (int64_t)h * k_head_bytes_d(D, DB);
    const uint8_t* meta = (const uint8_t*)L.key_meta + pg * L.key_meta_stride_page + (int64_t)h * D * 4;
    wait_reads();
    constexpr int kUsual = kRowBytes * (D + D / 4) + D;   // k_head_bytes_d with a quarter of the channels boosted
    if (DB == D / 4) {
#pragma unroll
      for (int i = 0; i < kUsual; i += 1024) to_lds<16>(src + min(i, kUsual - 1024), lds_at + min(i, kUsual - 1024), lane);
    } else {
      block_to_lds(src, lds_at, k_head_bytes_d(D, DB), lane);
    }
    to_lds<D == 64 ? 4 : 16>(meta, lds_at + at.k_meta, lane);
  };
  auto fetch_v = [&](int page) {
    int lane = tid & 63;
    asm volatile("" : "+v"(lane));
    const int64_t pg = checked_page(page_id(L.page_table_v, (int64_t)b * L.page_table_v_stride_b + page), L.cache_pages_v, bad_page);
    const uint8_t* src = L.value_cache + pg * L.value_cache_stride_page + (int64_t)h * v_head_bytes_d(D);
    const uint8_t* meta = (const uint8_t*)L.value_meta + pg * L.value_meta_stride_page + (int64_t)h * kPage * 4;
    wait_reads();
#pragma unroll
    for (int i = 0; i < 32 * D; i += 1024) to_lds<16>(src + i, lds_at + at.v_raw + i, lane);
    to_lds<4>(meta, lds_at + at.v_meta, lane);
    to_lds<4>(meta + 256, lds_at + at.v_meta + 256, lane);
  };
  // one 32-channel chunk of the keys: X = 8 codes of the low plane, H of the high one, of channels r and r + 1 in each
  // register, and their metadata.  The high plane's rows lie where the slot map says, read a chunk ahead.
  struct Chunk {
    uint32_t X[4], H[4];
    uint4 m0, m1;
  };
  // (a lane's corners, opaque: every read is one of them and a small immediate)
  struct Corner {
    uint32_t plane, quarter, slot, meta;
  };
  auto corner = [&](int kg, int n) {
    Corner k = {(uint32_t)((4 * kg + (n >> 2)) * kRowBytes + (n & 3) * 8), (uint32_t)((n & 3) * 8),
                (uint32_t)(kRowBytes * (D + DB) + 4 * kg + (n >> 2)), (uint32_t)(at.k_meta + 16 * kg)};
    asm volatile("" : "+v"(k.plane), "+v"(k.quarter), "+v"(k.slot), "+v"(k.meta));
    return k;
  };
  auto slots = [&](int kc, const Corner& at_) {
    const uint8_t* idx = page_lds + at_.slot + 32 * kc;
    return (int)idx[0] | (int)idx[16] << 8;
  };
  auto read_k = [&](int kc, int slot, Chunk& k, const Corner& at_) {
    const int s0 = slot & 255, s1 = slot >> 8;
    const uint8_t* p = page_lds + at_.plane + 32 * kc * kRowBytes;
    lds_tr(p, k.X[0], k.X[1]);
    lds_tr(p + 16 * kRowBytes, k.X[2], k.X[3]);
    lds_tr(page_lds + (s0 < DB ? (D + s0) * kRowBytes : at.zero_row) + at_.quarter, k.H[0], k.H[1]);
    lds_tr(page_lds + (s1 < DB ? (D + s1) * kRowBytes : at.zero_row) + at_.quarter, k.H[2], k.H[3]);
    const uint8_t* m = page_lds + at_.meta + 128 * kc;
    k.m0 = *(const uint4*)m;
    k.m1 = *(const uint4*)(m + 64);
  };
  auto scales = [&](const Chunk& k, uint32_t (&sc)[4], uint32_t (&zr)[4]) {
    sc[0] = low_halves(k.m0.x, k.m0.y), zr[0] = high_halves(k.m0.x, k.m0.y);
    sc[1] = low_halves(k.m0.z, k.m0.w), zr[1] = high_halves(k.m0.z, k.m0.w);
    sc[2] = low_halves(k.m1.x, k.m1.y), zr[2] = high_halves(k.m1.x, k.m1.y);
    sc[3] = low_halves(k.m1.z, k.m1.w), zr[3] = high_halves(k.m1.z, k.m1.w);
  };
  // ---- a whole page, by this wavefront alone -----------------------------------------------------------------------
  // every scale and zero in the range of dequant_fast
  auto logits = [&](const uint32_t (&qq)[kKC][4], float4v (&S)[8]) {
#pragma unroll
    for (int u = 0; u < 8; ++u) S[u] = float4v{0.f, 0.f, 0.f, 0.f};
    Chunk k;
    const Corner mine = corner(kg, n);
    int slot = slots(0, mine);
    read_k(0, slot, k, mine);
    if (kKC > 1) slot = slots(1, mine);
#pragma unroll
    for (int kc = 0; kc < kKC; ++kc) {
      uint32_t sc[4], zr[4], even[4], odd[4], b0[4], b4[4];
      scales(k, sc, zr);
#pragma unroll
      for (int i = 0; i < 4; ++i) {   // nibble j: the four bits of token 2j (even), 2j + 1 (odd)
        even[i] = (k.X[i] & 0x33333333u) | ((k.H[i] << 2) & 0xccccccccu);
        odd[i] = ((k.X[i] >> 2) & 0x33333333u) | (k.H[i] & 0xccccccccu);
        b0[i] = scale_base<0>(sc[i]), b4[i] = scale_base<4>(sc[i]);
      }
      if (kc + 1 < kKC) read_k(kc + 1, slot, k, mine);   // in flight while this chunk is unpacked
      if (kc + 2 < kKC) slot = slots(kc + 2, mine);
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        uint32_t a[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const uint32_t x = (u & 1 ? odd[i] : even[i]) >> (u >= 4 ? 8 : 0);
          a[i] = u & 2 ? dequant_fast(x, 0x00f000f0u, magic[2], sc[i], b4[i], zr[i]) : dequant_fast(x, 0x000f000fu, magic[0], sc[i], b0[i], zr[i]);
        }
        S[u] = mfma16(a, qq[kc], S[u]);
      }
    }
  };
  auto values = [&](float4v (&S)[8]) {
    constexpr bool kBase = D == 256;   // (at D = 64 four products share a scale's bases: nothing gained)
    // k-slots of product cj: tokens 32 kg + 8 cj .. + 7.  D = 64: a row has 8 pieces; lanes n and n + 8 both receive piece n % 8 and
    // take its lower and upper four codes
    uint32_t rows_at = at.v_raw + (32 * kg + (n >> 2)) * (D / 4) + (D == 64 ? n & 1 : n & 3) * 8, metas_at = at.v_meta + 32 * kg * 4;
    asm volatile("" : "+v"(rows_at), "+v"(metas_at));
    const uint8_t* const rows = page_lds + rows_at;
    const uint8_t* const metas = page_lds + metas_at;
    uint4 mm[2];
    uint32_t Y[4];
    auto read_meta = [&](int cj) { mm[0] = *(const uint4*)(metas + 32 * cj), mm[1] = *(const uint4*)(metas + 32 * cj + 16); };
    auto read_v = [&](int cj, int hf) {
      lds_tr(rows + 8 * cj * (D / 4) + hf * kRowBytes, Y[0], Y[1]);
      lds_tr(rows + (8 * cj + 4) * (D / 4) + hf * kRowBytes, Y[2], Y[3]);
    };
    auto product = [&](int cj) {
      const float x[8] = {S[0][0], S[1][0], S[2][0], S[3][0], S[4][0], S[5][0], S[6][0], S[7][0]};
#pragma unroll
      for (int u = 0; u < 8; ++u) S[u] = __builtin_shufflevector(S[u], S[u], 1, 2, 3, 0);
      uint32_t first[4], p1[4], p2[4], sc[4], zr[4], base[5][4];
      A.parts(x, first, p1, p2);
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        sc[2 * i] = low_halves(mm[i].x, mm[i].y), zr[2 * i] = high_halves(mm[i].x, mm[i].y);
        sc[2 * i + 1] = low_halves(mm[i].z, mm[i].w), zr[2 * i + 1] = high_halves(mm[i].z, mm[i].w);
      }
      if (kBase) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          base[0][j] = scale_base<0>(sc[j]), base[1][j] = scale_base<2>(sc[j]), base[2][j] = scale_base<4>(sc[j]);
          base[3][j] = scale_base<6>(sc[j]), base[4][j] = scale_base<8>(sc[j]);
        }
      }
#pragma unroll
      for (int hf = 0; hf < kHalves; ++hf) {
        uint32_t X[4], X10[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          X[j] = D == 64 ? Y[j] >> (n & 8) : Y[j];
          X10[j] = X[j] >> 10;
        }
        // in flight while these are unpacked (after the last product: once more the first)
        if (hf + 1 < kHalves) {
          read_v(cj, hf + 1);
        } else {
          read_v((cj + 1) & 3, 0);
          read_meta((cj + 1) & 3);
        }
        auto tile = [&](auto u_) {
          constexpr int u = decltype(u_)::value, k = u < 5 ? u : u - 5;
          uint32_t a[4];
#pragma unroll
          for (int j = 0; j < 4; ++j)
            a[j] = kBase ? dequant_fast(u < 5 ? X[j] : X10[j], 0x00030003u << (2 * k), magic[k], sc[j], base[k][j], zr[j])
                         : dequant_v<u>(X[j], X10[j], magic[0], sc[j], zr[j]);
          A.template weigh<false>(a, hf * kU + u, first, p1, p2);
        };
        tile(std::integral_constant<int, 0>{}), tile(std::integral_constant<int, 1>{});
        tile(std::integral_constant<int, 2>{}), tile(std::integral_constant<int, 3>{});
        if constexpr (kU == 8) {
          tile(std::integral_constant<int, 4>{}), tile(std::integral_constant<int, 5>{});
          tile(std::integral_constant<int, 6>{}), tile(std::integral_constant<int, 7>{});
        }
      }
    };
    read_v(0, 0);
    read_meta(0);
    if constexpr (D == 64) {
#pragma unroll
      for (int cj = 0; cj < 4; ++cj) product(cj);
    } else {   // (64 products of four instructions a word would be 24 KB of code)
#pragma unroll 1
      for (int cj = 0; cj < 4; ++cj) product(cj);
    }
  };

  // ---- any tile: tokens 8i + 2w + e, e = 0, 1 -------------------------------------------------------------------------------
  // there: its page lies at page_lds already
  auto special = [&](int tile, int w, bool there) {
    int id = lane;
    asm volatile("" : "+v"(id));   // as above
    const int kg = id >> 4, n = id & 15;
    const int body = tile - 1;   // -1: the sink
    const int ntok = tile == 0 ? c.sink : min(kPage, c.nbody - body * kPage);
    const bool k_packed = tile > 0 && body < c.pk, v_packed = tile > 0 && body < c.pv;
    const int64_t sink_base = (int64_t)b * L.sink_stride_b + (int64_t)h * L.sink_stride_h;
    const int64_t win_base = (int64_t)b * L.win_stride_b + (int64_t)h * L.win_stride_h;
    const int t0 = 32 * kg + 2 * w;   // operand register j of the second product: tokens t0 + 8 j, t0 + 8 j + 1
    uint32_t qq[kKC][4];
    if (k_packed && !there) fetch_k(body);
    if (v_packed && !there) fetch_v(body);
    load_query(qq);
    // fp16 values: rows u < lows of one tensor, then the ring's (the end of the sequence only); asked for before the logits
    typedef uint32_t words __attribute__((ext_vector_type(kU / 2)));
    words x8[kHalves][8];
    const uint8_t* rows[8];   // the rows of tokens t0 + 8 j + e
    auto read_rows = [&](int hf) {
      const int ch = D == 256 ? 128 * hf + 8 * n : 8 * (n & 7) + 4 * (n >> 3);
#pragma unroll
      for (int i = 0; i < 8; ++i) x8[hf][i] = *(const words*)(rows[i] + ch * 2);
    };
    if (!v_packed) {
      const int u0 = tile == 0 ? 0 : (body - c.pv) * kPage, lows = tile == 0 ? kPage : c.rv;
      const uint8_t* low = tile == 0 ? (const uint8_t*)L.sink_v + sink_base : (const uint8_t*)L.qbuf_v + win_base;
      const uint8_t* ring = (const uint8_t*)L.local_v + win_base;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int u = u0 + min(t0 + 8 * (i >> 1) + (i & 1), ntok - 1);
        rows[i] = u < lows ? low + (int64_t)u * (2 * D) : ring + (int64_t)((c.off + u - lows) & (kPage - 1)) * (2 * D);
      }
      read_rows(0);
    }
    if (k_packed) wait_loads<0>();
    float4v S[2] = {float4v{0.f, 0.f, 0.f, 0.f}, float4v{0.f, 0.f, 0.f, 0.f}};   // S[e][j]: token 32 kg + 8 j + 2 w + e
    if (k_packed) {
      const Corner mine = corner(kg, n);
#pragma unroll
      for (int kc = 0; kc < kKC; ++kc) {
        uint32_t sc[4], zr[4], a0[4], a1[4];
        Chunk k;
        read_k(kc, slots(kc, mine), k, mine);
        scales(k, sc, zr);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const uint32_t lo = k.X[i] >> (4 * w), hi = (k.H[i] >> (4 * w)) << 2;   // code e: bits 2e, 2e + 1 of lo, two further up in hi
          const uint32_t c0 = (lo & 0x00030003u) | (hi & ~0x00030003u), c1 = (lo & 0x000c000cu) | (hi & ~0x000c000cu);
          a0[i] = dequant_word<0>((c0 & 0x000f000fu) | kCodeMagic, sc[i], zr[i]);
          a1[i] = dequant_word<2>((c1 & 0x003c003cu) | kCodeMagic, sc[i], zr[i]);
        }
        S[0] = mfma16(a0, qq[kc], S[0]);
        S[1] = mfma16(a1, qq[kc], S[1]);
      }
    } else {
      const uint8_t* base = tile == 0 ? (const uint8_t*)L.sink_k + sink_base : (const uint8_t*)L.qbuf_k + win_base;
      const int first = 8 * n + 2 * w;
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        // a token past the end repeats the last one: its logits are masked below
        const uint8_t* row = base + (int64_t)min(first + e, ntok - 1) * (2 * D);
#pragma unroll
        for (int kc = 0; kc < kKC; ++kc) {
          const uint2 x0 = *(const uint2*)(row + (32 * kc + 4 * kg) * 2);
          const uint2 x1 = *(const uint2*)(row + (32 * kc + 16 + 4 * kg) * 2);
          const uint32_t a[4] = {x0.x, x0.y, x1.x, x1.y};
          S[e] = mfma16(a, qq[kc], S[e]);
        }
      }
    }
    if (!v_packed && kHalves == 2) read_rows(kHalves - 1);
    asm volatile("" ::: "memory");   // (in flight from here on)
#pragma unroll
    for (int e = 0; e < 2; ++e)
#pragma unroll
      for (int j = 0; j < 4; ++j) S[e][j] = 32 * kg + 8 * j + 2 * w + e < ntok ? S[e][j] * sc2 : -INFINITY;
    A.settle(fmaxf(fmaxf(fmaxf(S[0][0], S[0][1]), fmaxf(S[0][2], S[0][3])), fmaxf(fmaxf(S[1][0], S[1][1]), fmaxf(S[1][2], S[1][3]))));
    const float shift = A.shift();
    float x[8];   // operand register j: tokens t0 + 8 j, t0 + 8 j + 1
#pragma unroll
    for (int j = 0; j < 8; ++j) x[j] = __builtin_amdgcn_exp2f(S[j & 1][j >> 1] + shift);
#pragma unroll
    for (int j = 0; j < 8; ++j) A.l += x[j];
    uint32_t first[4], p1[4], p2[4];
    A.parts(x, first, p1, p2);
    if (v_packed) {
      wait_loads<0>();
      uint32_t sc[4], zr[4], big = 0u;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        uint2 mm = *(const uint2*)(page_lds + at.v_meta + (t0 + 8 * j) * 4);
        if (t0 + 8 * j >= ntok) mm.x = 0u;   // a token that does not count is 0, whatever its bytes say
        if (t0 + 8 * j + 1 >= ntok) mm.y = 0u;
        sc[j] = low_halves(mm.x, mm.y), zr[j] = high_halves(mm.x, mm.y);
        big |= out_of_range(mm.x) | out_of_range(mm.y);
      }
      const int rr = n >> 2, tok = t0 + (rr & 1) + 8 * (rr >> 1);
      auto weigh_page = [&](auto wild_) {
        constexpr bool WILD = decltype(wild_)::value;
#pragma unroll
        for (int hf = 0; hf < kHalves; ++hf) {
          const uint8_t* p = page_lds + at.v_raw + tok * (D / 4) + hf * kRowBytes + (D == 64 ? n & 1 : n & 3) * 8;
          uint32_t X[4], X10[4];
          lds_tr(p, X[0], X[1]);
          lds_tr(p + 16 * (D / 4), X[2], X[3]);
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            if (D == 64) X[j] >>= n & 8;
            X10[j] = X[j] >> 10;
          }
          auto vtile = [&](auto u_) {
            constexpr int u = decltype(u_)::value;
            uint32_t a[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) a[j] = dequant_v<u>(X[j], X10[j], kCodeMagic, sc[j], zr[j]);
            A.template weigh<WILD>(a, hf * kU + u, first, p1, p2);
          };
          vtile(std::integral_constant<int, 0>{}), vtile(std::integral_constant<int, 1>{});
          vtile(std::integral_constant<int, 2>{}), vtile(std::integral_constant<int, 3>{});
          if constexpr (kU == 8) {
            vtile(std::integral_constant<int, 4>{}), vtile(std::integral_constant<int, 5>{});
            vtile(std::integral_constant<int, 6>{}), vtile(std::integral_constant<int, 7>{});
          }
        }
      };
      if (__any((big & 0x80008000u) != 0u)) weigh_page(std::true_type{});
      else weigh_page(std::false_type{});
    } else {
#pragma unroll
      for (int hf = 0; hf < kHalves; ++hf) {
        uint32_t big = 0u;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          if (t0 + 8 * (i >> 1) + (i & 1) >= ntok) x8[hf][i] = words{};   // probability 0 times what a dead row may hold must be 0
#pragma unroll
          for (int k = 0; k < kU / 2; ++k) big |= (x8[hf][i][k] & 0x7fff7fffu) + 0x04000400u;
        }
        const bool wild = __any((big & 0x80008000u) != 0u);
        auto weigh_rows = [&](auto wild_) {
#pragma unroll
          for (int u = 0; u < kU; ++u) {
            uint32_t a[4];
#pragma unroll
            for (int j = 0; j < 4; ++j)
              a[j] = u & 1 ? high_halves(x8[hf][2 * j][u >> 1], x8[hf][2 * j + 1][u >> 1])
                           : low_halves(x8[hf][2 * j][u >> 1], x8[hf][2 * j + 1][u >> 1]);
            A.template weigh<decltype(wild_)::value>(a, hf * kU + u, first, p1, p2);
          }
        };
        if (wild) weigh_rows(std::true_type{});
        else weigh_rows(std::false_type{});
      }
    }
  };

  // whole pages first; the splits with a special tile take some only where there are few splits
  const int dealt = num_splits >= 3 * n_special ? num_splits - n_special : num_splits;
  const int first_page = split < dealt ? split + dealt * w : n_full;
  int page = first_page;
  const auto wide = [](uint32_t big) { return __any((big & 0x80008000u) != 0u); };
  uint32_t qq[kKC][4];
  if (page < n_full) fetch_k(page), fetch_v(page), load_query(qq);
#pragma unroll 1
  while (page < n_full) {
    const int next = page + 4 * dealt;
    float4v S[8];
    wait_loads<kVLoads>();   // (the query's loads, behind the first page's, have been waited for)
    uint32_t big = 0u;
#pragma unroll
    for (int i = 0; i < D / 64; ++i) big |= out_of_range(((const uint32_t*)(lds + at.k_meta))[64 * i + lane]);
    logits(qq, S);
    // vmax3 is assembly, which the compiler's wait states behind a matrix instruction do not see into
    asm volatile("s_nop 15" : "+v"(S[0]), "+v"(S[1]), "+v"(S[2]), "+v"(S[3]), "+v"(S[4]), "+v"(S[5]), "+v"(S[6]), "+v"(S[7]));
    wait_loads<0>();
    const uint2 mm = ((const uint2*)(lds + at.v_meta))[lane];
    big |= out_of_range(mm.x) | out_of_range(mm.y);
    if (wide(big)) break;
    if (next < n_full) fetch_k(next);
    float mx = vmax3(S[0][0], S[0][1], S[0][2]);
    mx = vmax(mx, S[0][3]);
#pragma unroll
    for (int u = 1; u < 8; ++u) mx = vmax3(mx, S[u][0], vmax3(S[u][1], S[u][2], S[u][3]));
    A.settle(mx * sc2);
    const float shift = A.shift();
    float sum = 0.f;
#pragma unroll
    for (int u = 0; u < 8; ++u)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        S[u][j] = __builtin_amdgcn_exp2f(__builtin_fmaf(S[u][j], sc2, shift));
        sum += S[u][j];
      }
    A.l += sum;
    values(S);
    if (next < n_full) fetch_v(next);
    page = next;
  }
  // A page with a scale or zero out of dequant_fast's range ends a wavefront's walk (a channel of large numbers is one in every page): that
  // page and those behind it are left to the four.  A decode layer with such a page per head / with nothing else (walking on and then
  // fetching every page again to find those passed over, four times the one found: in brackets; no such page: third): D = 64, B = 8, 6100
  // tokens, 32 / 8 heads: 25 / 33 us (29 / 36; 22); D = 256, B = 2, 9000 tokens, 16 / 8: 33 / 44 (49 / 69; 28); B = 4, 30000: 108 / 138 (107 /
  // 293; 74).
  if (lane == 0) s_left[w] = page;

  // then what is left, a quarter of a tile's tokens per wavefront: the special tiles, and the pages left, of which each wavefront
  // fetches one at a time
  int r = num_splits - 1 - split, owner = 3, ahead = -4 * dealt;
#pragma unroll 1
  while (true) {
    const bool there = r >= n_special;
    int tile;
    if (!there) {
      tile = r < has_sink ? 0 : n_full + 1 + r - has_sink;
      r += num_splits;
    } else {
      if (++owner == 4) {
        owner = 0, ahead += 4 * dealt;
        __syncthreads();   // everyone is done with the pages before
        const int first = min(min(s_left[0], s_left[1]), min(s_left[2], s_left[3]));
        if (__builtin_amdgcn_readfirstlane(first) + ahead >= n_full) break;
        if (page + ahead < n_full) fetch_k(page + ahead), fetch_v(page + ahead);
        wait_loads<0>();
        __syncthreads();
      }
      tile = __builtin_amdgcn_readfirstlane(s_left[owner]) + ahead + 1;
      if (tile > n_full) continue;
      page_lds = lds_all + owner * at.bytes;
    }
    special(tile, w, there);
  }

  if (lane == 0) report_bad_page(L, b, bad_page);
  // ---- the wavefronts' partials meet: a common maximum, then sums of four output tiles at a time -------------------
  float l = A.l;
  l += __shfl_xor(l, 16);
  l += __shfl_xor(l, 32);
  if (kg == 0) s_m[w][n] = A.m, s_l[w][n] = l;
  __syncthreads();
  float mm = -INFINITY;
#pragma unroll
  for (int i = 0; i < 4; ++i) mm = fmaxf(mm, s_m[i][n]);
  const float own = A.m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(A.m - mm) * (1.f / kProbScale);
  l = 0.f;
#pragma unroll
  for (int i = 0; i < 4; ++i)   // (a wavefront whose logits are all NaN has -inf for a maximum and NaN for a sum, which must stay)
    l += s_l[i][n] * (s_m[i][n] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(s_m[i][n] - mm));
  const int64_t row = ((int64_t)b * H_Q + h * G + n) * num_splits + split;
  // (a share of nothing but NaN counts: the merge passes over -inf)
  if (n < G && w == 0 && kg == 0) *(float2*)(ws_ml + row * 2) = float2{l != l ? 0.f : mm, l};
#pragma unroll
  for (int t4 = 0; t4 < kOT; t4 += 4) {
    __syncthreads();
#pragma unroll
    for (int t = 0; t < 4; ++t) ((float4v*)lds_all)[(w * 4 + t) * 64 + lane] = A.O[t4 + t] * own;
    __syncthreads();
    if (n < G) {
      float4v o = float4v{0.f, 0.f, 0.f, 0.f};   // tile t4 + w, summed over the wavefronts and the columns of the parts
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int part = 0; part < (COLS ? 3 : 1); ++part) o += ((const float4v*)lds_all)[(i * 4 + w) * 64 + lane + part * G];
      const int t = t4 + w;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int x = 4 * kg + j;
        ws_acc[row * D + (D == 256 ? 128 * (t >> 3) + 8 * x + (t & 7) : 8 * (x & 7) + 4 * (x >> 3) + t)] = o[j];
      }
    }
  }
}

template <int D>
void launch(const kitty_kv_layer& L, const void* q, int B, int H_Q, float scaling, float* ws_ml, float* ws_acc, int num_splits,
            hipStream_t stream) {
  const dim3 grid(num_splits, L.H_KV, B), block(256);
  const int lds = 4 * WaveLds(D, L.D_BOOSTED).bytes;
#define KITTY_LAUNCH(COLS)                                                                                                        \
  do {                                                                                                                            \
    /* more LDS than the default per-workgroup limit; per device, so set on every launch */                                      \
    if (lds > 65536) (void)hipFuncSetAttribute((const void*)decode_any_kernel<D, COLS>, hipFuncAttributeMaxDynamicSharedMemorySize, lds); \
    hipLaunchKernelGGL((decode_any_kernel<D, COLS>), grid, block, lds, stream, L, (const uint8_t*)q, H_Q, scaling, ws_ml, ws_acc, \
                       num_splits);                                                                                               \
  } while (0)
  if (H_Q / L.H_KV <= 5) KITTY_LAUNCH(true);
  else KITTY_LAUNCH(false);
#undef KITTY_LAUNCH
}

}  // namespace

namespace {
// Workgroups that fit the device at once: four per compute unit at D = 64, two at D = 256 (registers, LDS).
int64_t slots_any(int D, int units) { return (int64_t)(D == 64 ? 4 : 2) * units; }
// Few tiles: four wavefronts share one, and a tile takes a third of the time that one wavefront needs for it (8 us at D = 256, of which
// two are the way to memory).  The kernel that does only that holds its query operands in LDS.  It is the faster one with a tile or less
// a compute unit, and with two while a walk has not so many of them that the merge reads more than decode_any_kernel's fewer splits
// leave it.  Both passes in a graph, it and decode_any_kernel: D = 64, 8 walks of 4 tiles 7.8 and 8.4 us, 24 of 11 10.1 and 11.9, 16 of 32 10.7
// and 12.3, 8 of 63 10.8 and 11.5, 4 of 80 11.4 and 11.2, 2 of 200 12.9 and 11.4; D = 256, 8 of 17 13.8 and 17.6, 32 of 10 16.3 and 19.7, 24 of 21 17.2 and
// 21.9, 16 of 25 16.9 and 16.7, 16 of 32 19.1 and 16.4.
bool few_tiles(int D, int64_t walks, int tiles, int units) {
  return walks * tiles <= units || (walks * tiles <= 2 * units && tiles <= (D == 64 ? 64 : 24));
}
}  // namespace

void launch_decode_any(const kitty_kv_layer& L, const void* q, int B, int H_Q, float scaling, float* ws_ml, float* ws_acc,
                       int num_splits, int max_tiles, int units, hipStream_t stream) {
  if (few_tiles(L.D, (int64_t)B * L.H_KV, max_tiles, units)) launch_decode_by_tile(L, q, B, H_Q, scaling, ws_ml, ws_acc, num_splits, stream);
  else if (L.D == 64) launch<64>(L, q, B, H_Q, scaling, ws_ml, ws_acc, num_splits, stream);
  else launch<256>(L, q, B, H_Q, scaling, ws_ml, ws_acc, num_splits, stream);
}

// Splits of a decode walk.  Few tiles: one each.  Otherwise as many as give every wavefront a page at most, and the tiles with
// fp16 rows (three, as a rule) a split of their own, if the device holds them at once: D = 64, B = 8, 6100 tokens, 32 / 8
// heads: 19.1 us with 15 or 16 splits, 21.2 with 13, 21.9 with 22; D = 64, B = 1, 30000 tokens, 14 / 2: 12.4 with 78, 14.4 with 60;
// D = 256, B = 2, 9000 tokens, 16 / 8: 26.0 with 24, 32.6 with 18.  Else as many as fit (D = 64, B = 32, 8000 tokens, 24 / 8: 45.6
// us with 4, 49.1 with 8; D = 256, B = 4, 30000 tokens: 77 with 17, 84 with 29).  At D = 256 a count whose equal shares would leave one
// without a tile is moved to the next that does not, as for the kernel that cuts equal shares.  decode_any_kernel deals pages in turn and
// does not need that; it costs where the move leaves some wavefront a second page (B = 1, 49500 tokens, 8 / 4 heads: 35.2 us with 97, 29.5
// with 100) and gains a little where it adds splits (B = 2, 9000 tokens: 24.6 with 24, 25.5 with 21).
int decode_splits_any(int B, int H_KV, int D, int tiles, int units) {
  const int64_t walks = (int64_t)B * H_KV, slots = slots_any(D, units);
  int64_t s = tiles;
  if (!few_tiles(D, walks, tiles, units)) {
    s = (tiles + 1) / 4 + 3;
    if (s > slots / walks) s = slots / walks;
    if (s > tiles) s = tiles;
    if (s > 512) s = 512;
    if (s < 1) s = 1;
    if (D == 256) {
      const int64_t more = (tiles + tiles / s - 1) / (tiles / s), share = (tiles + s - 1) / s;
      s = more <= 512 && walks * more <= slots ? more : (tiles + share - 1) / share;
    }
  }
  return s > 512 ? 512 : (int)s;
}

}  // namespace kitty
