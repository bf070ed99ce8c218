// Causal attention of a prefill chunk straight off the 8-bit KV cache: the L query rows of each
// head are the chunk's positions n-L .. n-1, whose K/V are already the last L of the first n
// cache rows, and row i sees keys 0 .. n-L+i. Replaces, for prefill chunks, the reference's path
// of dequantizing the whole cache (laguna_mlx/cache.py:99-100) and running SDPA with the causal
// mask (laguna.py:107); tests/test_cache.py:79-93 is the reference's guard that the quantized
// prefill never materializes the score matrix, and neither does this kernel.
//
// Work: one workgroup of 8 waves per (sequence, KV head, block of 256 query rows), a KV head's rows
// being numbered position-major: row f is position f / G of query head f % G, so a block holds 256
// rows whatever G (any grouping fills the MFMA columns) and the rows of a wave lie at neighbouring
// positions. Wave w takes 32 rows (two MFMA N tiles of 16). The workgroup walks the 128-key tiles
// up to its last row's causal bound; each tile is brought into LDS once for all 8 waves and dequantized once:
//  * the raw tile (K and V codes, 128 B per key each, and the four bf16 word arrays) is copied
//    global -> LDS by DMA two tiles ahead (two raw slots, 5 copies per thread per tile);
//  * the tile is dequantized (scale * code + bias in fp32, rounded to fp16) into K [128 keys][128
//    dims] and V^T [128 dims][128 keys], both XOR-swizzled by 16-byte chunk so that the MFMA
//    operand reads are conflict-free;
//  * each wave runs Q.K^T (v_mfma_f32_16x16x32_f16: M = 16 keys, N = 16 rows, K = 32 dims; q
//    pre-scaled by scale * log2(e) in fp16; each K fragment read once for both N tiles), the
//    online softmax with lazy rescaling (a lane holds keys 16 mt + 4 q + r of one row; scores
//    relative to the running maximum, which the accumulators start from), and P.V (M = 16 dims,
//    N = 16 rows, K = 32 keys; the lane's own 8 probabilities are its k-slots: key 32 e + 16 h +
//    4 q + r of k-step e is slot 8 q + 4 h + r, and V^T stores the keys in that slot order).
// Ping-pong: a SIMD holds one wave of each half of the workgroup (waves 0-3: group A, 4-7: group
// B), and the two halves run the same per-tile phases one phase apart, so that one wave's matrix
// phase (Q.K^T or P.V: MFMA and LDS reads) overlaps the other's vector phase (softmax, or its
// share of the dequantization: K by group A, V by group B). Four barrier-separated slots per tile:
//
//   slot    group A                  group B
//   4t      Q.K^T(t)                 dequantize V(t)
//   4t+1    softmax(t)               Q.K^T(t)
//   4t+2    P.V(t)                   softmax(t)
//   4t+3    dequantize K(t+1)        P.V(t)
//
// K(t+1) overwrites K(t) after both halves' Q.K^T(t), V(t) overwrites V(t-1) after both halves'
// P.V(t-1), so one fp16 K and one V^T buffer suffice. The codes of raw tile t+2 and the words of
// t+3 go into t's slots once both dequantizations of t are done, from each half's softmax slot, and
// are waited for a tile later. Vector phases run at a raised wave priority: their instructions set
// the pace and the matrix phases' issue only every 16 cycles (2,048 rows at 82,671 keys, in four turns
// beside the kernel without it: 2,571-2,576 -> 2,549-2,551 us).
// Tiles past a wave's last row are skipped by that wave (it keeps its copy and dequantization
// duties); tiles straddling its rows' bounds are masked per row. Rows past the chunk (a ragged last
// block) read no q and store nothing. Keys past n-1 are never read: copies clamp their rows to n-1.
//
// Operands: with 1, 2, 4 or 8 query heads per KV head, K and V are dequantized to fp16 as above and
// have its range and rounding. The other groupings (CODES) keep the arithmetic of the verify kernel,
// which serves them in blocks of up to 16 positions: the operands are the exact codes, per quant
// group, and the affine terms are applied in fp32 after Q.K^T (s_g z_g + b_g Q_g with Q_g the sum of
// q over the group) and to P before P.V (P s_g in fp16, and sums of P b_g).
//  * K enters as c 2^-24, q times one 2^kq of the workgroup, so scores of any size stay exact to fp32;
//    V enters as c - 128 (P s_g is rounded, and the smaller the code the less of that shows: relative
//    error against 64 bits over scores of deviation 2 at 8,193 keys 0.001667, with c 0.00174, of the
//    verify kernel 0.001664), the sums take the value of code 128 instead of the bias.
//  * P.V: P s_g 2^kv in fp16, 2^kv per quant group and 64-key tile as in the verify kernel (attn_dev.h);
//    accumulators are rescaled when it changes.
//  * A NaN or infinity in a key's words reaches the rows that see that key: no factor is taken from
//    it, and masked tiles leave the terms of keys past a row's bound out.
// That is 350 VALU instructions more per 32 rows and 128 keys, and twice the registers for P, so the
// tiles are of 64 keys. Per 128 keys 7.0 us against 4.0 (clock 1.8-2.1 GHz), VALU-bound in the softmax
// slots and about half of the Q.K^T slots: 512 rows at 8,193 keys, 48/8 heads, 190 us (in blocks of 10
// positions through the verify kernel, each a launch that reads the whole cache and a merge, 1,010).
// Without the raised wave priority 197, without the order of MFMAs and sums in qk() 196; the terms
// from one register per lane by DPP broadcasts instead of LDS 204; the biases through a third product
// (Q_g as three bf16 values) 191.
#include "attn_dev.h"

namespace lq {
namespace {

using namespace attn;

// Codes 2 h, 2 h + 1 of a word as the fp16 pair 1024 + c (exponent 10: the code is the mantissa),
// one v_perm_b32; scale * (1024 + c) + (bias - 1024 scale) then dequantizes in one
// v_fma_mix (fp32 arithmetic, rounded once to fp16).
__device__ __forceinline__ half2_t codes_1024(uint32_t w, int h) {
  return __builtin_bit_cast(half2_t,
                            __builtin_amdgcn_perm(0x64646464u, w, h ? 0x04030402u : 0x04010400u));
}

// 4 codes as fp16 c - 128, exactly (1024 + c, then one packed subtraction per pair).
__device__ __forceinline__ uint2 codes_centred(uint32_t w) {
  const half2_t mid = {(_Float16)1152.0f, (_Float16)1152.0f};
  return make_uint2(__builtin_bit_cast(uint32_t, codes_1024(w, 0) - mid),
                    __builtin_bit_cast(uint32_t, codes_1024(w, 1) - mid));
}

constexpr int PW = 8;       // waves per workgroup
constexpr int PROWS = 256;  // query rows per workgroup
constexpr int SHARE_KEYS = 128;  // keys of the tiles that blocks and shares are counted in

// Largest over the wave, in every lane.
__device__ __forceinline__ uint32_t wave_max_u(uint32_t x) {
  x = max(x, (uint32_t)__builtin_amdgcn_mov_dpp((int)x, DPP_QUAD_XOR1, 0xF, 0xF, true));
  x = max(x, (uint32_t)__builtin_amdgcn_mov_dpp((int)x, DPP_QUAD_XOR2, 0xF, 0xF, true));
  x = max(x, (uint32_t)__builtin_amdgcn_mov_dpp((int)x, DPP_ROW_ROR4, 0xF, 0xF, true));
  x = max(x, (uint32_t)__builtin_amdgcn_mov_dpp((int)x, DPP_ROW_ROR8, 0xF, 0xF, true));
  const auto r = __builtin_amdgcn_permlane16_swap(x, x, false, false);
  x = max((uint32_t)r[0], (uint32_t)r[1]);
  const auto r2 = __builtin_amdgcn_permlane32_swap(x, x, false, false);
  return max((uint32_t)r2[0], (uint32_t)r2[1]);
}
// Exponent e of a finite bf16 value of bits b: its magnitude is below 2^e.
__device__ __forceinline__ int bound_exp(uint32_t b) { return (int)(b >> 7) - 126; }
typedef uint16_t us2_t __attribute__((ext_vector_type(2)));
// The magnitudes of a word's two bf16 halves as bits, 0 in place of an infinity or NaN.
__device__ __forceinline__ us2_t finite_bits(uint32_t w) {
  const us2_t m = __builtin_bit_cast(us2_t, w & 0x7fff7fffu);
  return us2_t{m.x < 0x7f80 ? m.x : (uint16_t)0, m.y < 0x7f80 ? m.y : (uint16_t)0};
}
// P.V exponent k of a quant group for keys whose largest |scale| has bf16 bits m: kept while it puts
// that scale in [2^-2, 2^7), else chosen to put it in [16, 32) (with P below 2^8, P times the scaled
// scale is a normal fp16 number down to 2^-18 of the tile's largest).
__device__ __forceinline__ int pv_exponent(int k, uint32_t m) {
  if (m == 0) return k;
  const int e = bound_exp(m);
  return k != VK_NONE && e + k >= -1 && e + k <= 7 ? k : min(max(5 - e, -40), 40);
}

template <int PT>
struct PrefillRaw {
  alignas(16) uint8_t k[PT * D];  // row-major [key][128 B]
  uint8_t v[PT * D];
};

template <int PT>
struct PrefillWords {
  alignas(16) uint32_t w[4][PT];  // K scale, K bias, V scale, V bias words (two bf16 groups each)
};

// Per key of a tile and quant group (CODES): the K scale times scale log2(e) 2^(24 - kq), the K bias,
// the V scale times 2^kv, the V value of code 128.
template <int PT>
struct PrefillTerms {
  alignas(16) float ks[2][PT];
  float ku[2][PT], vs[2][PT], vb[2][PT];
};

template <int PT>
struct PrefillSmem {
  PrefillRaw<PT> raw[2];           // codes of tiles t, t + 1
  PrefillWords<PT> wd[3];          // words of tiles t, t + 1, t + 2
  PrefillTerms<PT> tm;             // of tile t
  alignas(16) uint32_t qmax[PW];   // bf16 bits of the largest finite |q| of each wave's rows
  alignas(8) int vexp[2][2];       // tile t, t + 1: P.V exponent per group
  int lim[PROWS];                  // last key each row sees
  alignas(16) _Float16 k[PT * D];   // [key][dim], 16-byte chunk j of key r at chunk j ^ (r & 15)
  alignas(16) _Float16 vt[D * PT];  // [dim][slot], 16-byte chunk j of dim d at chunk j ^ vt_swz(d)
};

struct PrefillSplit {
  FastDiv g;        // division by G
  int shares;       // workgroups per KV head
  int tiles;        // tiles of a share; 0: every workgroup takes one whole block
  float* part_o;    // [2 x workgroups][PROWS][D] partial rows of shares (slot 2 x + 1: the part
  float2* part_ml;  // begins its block), normalized, and their (max in log2 units, sum)
};

// Key tiles of position block pb.
__host__ __device__ __forceinline__ int prefill_tiles(int pb, int R, FastDiv g, int base) {
  return (base + (int)fdiv_u((uint32_t)min(pb * PROWS + PROWS - 1, R - 1), g)) / SHARE_KEYS + 1;
}

template <bool CODES, bool SPLIT>
__global__ __launch_bounds__(64 * PW, 1) void q8_prefill_kernel(
    const uint16_t* __restrict__ q, const uint8_t* __restrict__ kc,
    const uint16_t* __restrict__ ks, const uint16_t* __restrict__ kb,
    const uint8_t* __restrict__ vc, const uint16_t* __restrict__ vs,
    const uint16_t* __restrict__ vb, uint16_t* __restrict__ out, int64_t cap, int n, int L,
    int Hkv, int G, int npb, PrefillSplit sp, float qk_scale_log2) {
  // keys per tile: 128, or 64 where a tile's P takes twice the registers (CODES)
  constexpr int PT = CODES ? 64 : 128;
  constexpr int PMT = PT / 16;  // M tiles (16 keys) per tile
  constexpr int PE = PT / 32;   // P.V k-steps (32 keys) per tile
  constexpr int U = SHARE_KEYS / PT;
  using PrefillRaw = lq::PrefillRaw<PT>;
  using PrefillWords = lq::PrefillWords<PT>;
  // 16-byte chunks of a V^T row are swizzled so that the 16 rows (dims) of a fragment read differ
  auto vt_swz = [](int d) { return PT == 128 ? d & 15 : (d >> 1) & 7; };
  __shared__ PrefillSmem<PT> sm;
  const int x = blockIdx.x;
  const int hk = x % Hkv;  // consecutive workgroups (consecutive XCDs) take consecutive KV heads
  const int share = (x / Hkv) % sp.shares;
  const int b = x / (Hkv * sp.shares);
  const int Hq = Hkv * G;
  const int R = L * G;       // rows of a KV head
  const int base = n - L;    // row i sees keys <= base + i

  const int64_t row0 = ((int64_t)b * Hkv + hk) * cap;
  const int last_row = n - 1;


  // This workgroup's segments, one after the other: with SPLIT the parts of the blocks that its
  // share of the KV head's tiles covers, else its one block whole (last position blocks first: they
  // see the most keys, so the dispatch order is longest first). A variant of its own for whole
  // blocks: the walk costs it 1.4% (2,048 rows at 82,671 keys, 2,486 -> 2,521 us).
  int pb = SPLIT ? 0 : npb - 1 - share;
  int u = sp.tiles * share;               // next tile, counted over the KV head's blocks in order
  const int u_end = u + sp.tiles;
  int u_blk = 0;                          // first tile of block pb in that count
  if (SPLIT) {
    int bt = prefill_tiles(pb, R, sp.g, base);
    while (u >= u_blk + bt && pb < npb) {
      u_blk += bt;
      bt = prefill_tiles(++pb, R, sp.g, base);
    }
  }
  for (bool more = !SPLIT || pb < npb; more;) {
  // re-read per segment, so that no lane value derived from it is kept in registers across them
  int tid = threadIdx.x;
  asm volatile("" : "+v"(tid));
  const int lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const bool grp_a = wv < PW / 2;  // wave-uniform
  const int lc = lane & 15;
  const int lq4 = lane >> 4;
  const int T_blk = prefill_tiles(pb, R, sp.g, base);  // tiles the block needs
  const int tb = SPLIT ? U * (u - u_blk) : 0;     // the segment: tiles tb .. tb + T - 1
  const bool last_part = !SPLIT || T_blk <= u_end - u_blk;
  int T = U * (last_part ? T_blk : u_end - u_blk) - tb;
  if (U > 1 && last_part)  // no tile past the block's last key
    T = (base + (int)fdiv_u((uint32_t)min(pb * PROWS + PROWS - 1, R - 1), sp.g)) / PT + 1 - tb;
  // this wave's rows f0 .. f0 + 31 (row 16 nt + lc of the wave: f0 + 16 nt + lc)
  const int f0 = pb * PROWS + 32 * wv;
  const int lim_lo = base + f0 / G;                                 // bound of its first row
  const int lim_hi = f0 < R ? base + min(f0 + 31, R - 1) / G : -1;  // of its last valid row

  // ---- raw tile copies, per thread, of 128 keys: two 16-byte K copies (wave wv: keys 16 wv ..
  // 16 wv + 15), two V copies, one word (wave wv: word array wv / 2, keys 64 (wv % 2) + lane); of 64
  // keys: one K and one V copy, and by group A a word (wave wv: array wv)
  const uint32_t lds_raw = lds_addr(&sm.raw[0]), lds_wd = lds_addr(&sm.wd[0]);
  const int ck = PT / 8 * wv + (lane >> 3);  // key of this lane's first K / V copy (second: + 8)
  const uint32_t cofs = 16u * (uint32_t)(lane & 7);
  // V: chunk c of row r at c ^ (bits 0, 1 and 4 of r): the 8 keys of a transposed read all differ
  const uint32_t cofs_v = 16u * (uint32_t)((lane & 7) ^ ((ck & 3) | ((ck >> 2) & 4)));
  const int wa = PT == 128 ? wv >> 1 : wv;
  const uint16_t* warr = wa == 0 ? ks : wa == 1 ? kb : wa == 2 ? vs : vb;
  const int wk0 = PT == 128 ? 64 * (wv & 1) : 0, wkey = wk0 + lane;
  auto issue_codes = [&](int t, int slot) {
    const int t0 = PT * (tb + min(t, T - 1));
    const uint32_t lb = lds_raw + (uint32_t)slot * (uint32_t)sizeof(PrefillRaw);
    // M0 operands: wave-uniform values, made explicit so that they live in SGPRs
    const uint32_t mk = __builtin_amdgcn_readfirstlane(lb + offsetof(PrefillRaw, k) + PT / 8u * D * wv);
    const uint32_t mv = __builtin_amdgcn_readfirstlane(lb + offsetof(PrefillRaw, v) + PT / 8u * D * wv);
    const int64_t kr0 = row0 + min(t0 + ck, last_row);
    const int64_t kr1 = row0 + min(t0 + ck + 8, last_row);
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off nt"
                 :: "v"(kc + kr0 * D + cofs), "s"(mk) : "memory");
    if constexpr (PT == 128)
      asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off nt"
                   :: "v"(kc + kr1 * D + cofs), "s"(mk + 1024u) : "memory");
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off nt"
                 :: "v"(vc + kr0 * D + cofs_v), "s"(mv) : "memory");
    if constexpr (PT == 128)
      asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off nt"
                   :: "v"(vc + kr1 * D + cofs_v), "s"(mv + 1024u) : "memory");
  };
  auto issue_words = [&](int t, int slot) {
    if (PT == 64 && !grp_a) return;  // wave-uniform
    const uint32_t mw = __builtin_amdgcn_readfirstlane(
        lds_wd + (uint32_t)slot * (uint32_t)sizeof(PrefillWords) +
        4u * (uint32_t)(PT * wa + wk0));
    const int64_t wr = row0 + min(PT * (tb + min(t, T - 1)) + wkey, last_row);
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %0, off nt"
                 :: "v"(warr + wr * 2), "s"(mw) : "memory");
  };

  // ---- dequantization (CODES: conversion) shares: K of a tile by group A (256 threads, a chunk of
  // 16 codes per 32 keys each), V^T by group B (a wave a k-step of 128 keys, or of 64 a group of it)
  const int ta = tid & 255;  // thread index within the group
  // (the thread index is re-read through an empty asm in each call, so that the compiler
  // recomputes these addresses in the slot instead of holding them in registers across the loop)
  auto dequant_k = [&](const PrefillRaw& rw, const PrefillWords& wd) {
    __builtin_amdgcn_s_setprio(2);
    int tr = ta;
    asm volatile("" : "+v"(tr));
    const int dc = tr & 7;  // 16 codes of key (tr >> 3) + 32 i, dims 16 dc .. 16 dc + 15
    const uint32_t gsel = (dc >> 2) ? SEL_HI : SEL_LO;
    uint4 c4[PT / 32];
    uint32_t sw[PT / 32], zw[PT / 32];
#pragma unroll
    for (int i = 0; i < PT / 32; ++i) {  // all reads first: one LDS round trip
      const int dk = (tr >> 3) + 32 * i;
      c4[i] = *reinterpret_cast<const uint4*>(rw.k + dk * D + 16 * dc);
      if (!CODES) {
        sw[i] = wd.w[0][dk];
        zw[i] = wd.w[1][dk];
      }
    }
#pragma unroll
    for (int i = 0; i < PT / 32; ++i) {
      const int dk = (tr >> 3) + 32 * i;
      const uint32_t cw[4] = {c4[i].x, c4[i].y, c4[i].z, c4[i].w};
      uint32_t h[8];
      if constexpr (CODES) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          h[2 * j] = codes_sub_w(cw[j], SUB_B01);
          h[2 * j + 1] = codes_sub_w(cw[j], SUB_B23);
        }
      } else {
        const float s = bf16_pick(sw[i], gsel);
        const float z = fmaf(-1024.0f, s, bf16_pick(zw[i], gsel));  // bias - 1024 scale
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const half2_t c01 = codes_1024(cw[j], 0), c23 = codes_1024(cw[j], 1);
          h[2 * j] = pack_h2(fmaf(s, (float)c01.x, z), fmaf(s, (float)c01.y, z));
          h[2 * j + 1] = pack_h2(fmaf(s, (float)c23.x, z), fmaf(s, (float)c23.y, z));
        }
      }
      uint4* kd = reinterpret_cast<uint4*>(sm.k + dk * D);
      kd[(2 * dc) ^ (dk & 15)] = make_uint4(h[0], h[1], h[2], h[3]);
      kd[(2 * dc + 1) ^ (dk & 15)] = make_uint4(h[4], h[5], h[6], h[7]);
    }
  };
  // V^T chunk (dim d, k-step e, lane group q) = the 8 keys T[j] = 32 e + 16 (j / 4) + 4 q + j % 4
  // of dim d, in that slot order. Group B wave e, lane group q: one transposed read
  // (ds_read_b64_tr_b8) per 16-dim window w gives lane (q, i) the codes of T[0..7] at dim 16 w + i
  // (source lane s addresses key T[s / 2], bytes 8 (s % 2) of the window; the raw V rows are
  // stored swizzled by 16-byte chunk, see the copies).
  auto dequant_v = [&](const PrefillRaw& rw, const PrefillWords& wd) {
    __builtin_amdgcn_s_setprio(2);
    int ln = lane;
    asm volatile("" : "+v"(ln));
    const int e = (wv - PW / 2) % PE, qg = ln >> 4, i = ln & 15;
    const int g0 = PE == 4 ? 0 : (wv - PW / 2) / PE, g1 = PE == 4 ? 2 : g0 + 1;  // groups of the wave
    const int k0 = 32 * e + 4 * qg;  // T[0..3] = k0 .. k0 + 3, T[4..7] = k0 + 16 .. k0 + 19
    const int skey = k0 + 16 * (i >> 3) + ((i >> 1) & 3);  // T[i / 2]: this lane's source key
    const uint8_t* src = rw.v + skey * D + 8 * (i & 1);
    const int ssw = (skey & 3) | ((skey >> 2) & 4);
    const uint4 s03 = *reinterpret_cast<const uint4*>(&wd.w[2][k0]);
    const uint4 s47 = *reinterpret_cast<const uint4*>(&wd.w[2][k0 + 16]);
    const uint4 z03 = *reinterpret_cast<const uint4*>(&wd.w[3][k0]);
    const uint4 z47 = *reinterpret_cast<const uint4*>(&wd.w[3][k0 + 16]);
    const uint32_t sw[8] = {s03.x, s03.y, s03.z, s03.w, s47.x, s47.y, s47.z, s47.w};
    const uint32_t zw[8] = {z03.x, z03.y, z03.z, z03.w, z47.x, z47.y, z47.z, z47.w};
#pragma unroll
    for (int g = g0; g < g1; ++g) {  // dims 64 g .. 64 g + 63: quant group g, windows 4 g .. 4 g + 3
      v2i_t raw[4];
#pragma unroll
      for (int w = 0; w < 4; ++w)
        raw[w] = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_v2i_t*)(src + 16 * ((4 * g + w) ^ ssw)));
      float sj[8], zj[8];  // scale and bias - 1024 scale of key T[j], group g
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        sj[j] = g ? bf16_hi(sw[j]) : bf16_lo(sw[j]);
        zj[j] = fmaf(-1024.0f, sj[j], g ? bf16_hi(zw[j]) : bf16_lo(zw[j]));
      }
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const int d = 16 * (4 * g + w) + i;
        uint4* vd = reinterpret_cast<uint4*>(sm.vt + d * PT) + ((4 * e + qg) ^ vt_swz(i));
        if constexpr (CODES) {
          const uint2 lo = codes_centred((uint32_t)raw[w].x), hi = codes_centred((uint32_t)raw[w].y);
          *vd = make_uint4(lo.x, lo.y, hi.x, hi.y);
          continue;
        }
        float v[8];
#pragma unroll
        for (int hw = 0; hw < 2; ++hw) {  // keys T[4 hw .. 4 hw + 3]
          const uint32_t word = hw ? (uint32_t)raw[w].y : (uint32_t)raw[w].x;
          const half2_t c01 = codes_1024(word, 0), c23 = codes_1024(word, 1);
          v[4 * hw + 0] = fmaf(sj[4 * hw + 0], (float)c01.x, zj[4 * hw + 0]);
          v[4 * hw + 1] = fmaf(sj[4 * hw + 1], (float)c01.y, zj[4 * hw + 1]);
          v[4 * hw + 2] = fmaf(sj[4 * hw + 2], (float)c23.x, zj[4 * hw + 2]);
          v[4 * hw + 3] = fmaf(sj[4 * hw + 3], (float)c23.y, zj[4 * hw + 3]);
        }
        *vd = make_uint4(pack_h2(v[0], v[1]), pack_h2(v[2], v[3]), pack_h2(v[4], v[5]),
                         pack_h2(v[6], v[7]));
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  // ---- CODES: a tile's P.V exponents, from the largest |V scale| of its keys per group: made by the
  // first wave of group B (a word per lane) beside group A's Q.K^T of the tile before
  int fk[2] = {VK_NONE, VK_NONE};  // of the tile, per group
  int ak[2] = {VK_NONE, VK_NONE};  // that the accumulators hold
  auto next_exponents = [&](int s, const PrefillWords& wd) {
    if (wv != PW / 2) return;  // wave-uniform
    const us2_t m = finite_bits(wd.w[2][lane]);
    const int k0 = pv_exponent(fk[0], __builtin_amdgcn_readfirstlane(wave_max_u(m.x)));
    const int k1 = pv_exponent(fk[1], __builtin_amdgcn_readfirstlane(wave_max_u(m.y)));
    if (lane == 0) *reinterpret_cast<int2*>(sm.vexp[s]) = make_int2(k0, k1);
  };
  auto take_exponents = [&](int2 k) __attribute__((always_inline)) {
    fk[0] = __builtin_amdgcn_readfirstlane(k.x);
    fk[1] = __builtin_amdgcn_readfirstlane(k.y);
  };
  // the tile's per-key terms, by group A: a word per lane, wave wv array wv
  float kscale = 0.0f;  // scale log2(e) 2^(24 - kq): codes enter as c 2^-24, q times 2^kq
  auto tile_terms = [&](const PrefillWords& wd) {
    const uint32_t w = wd.w[wv][lane];
    float x0 = bf16_lo(w), x1 = bf16_hi(w);
    if (wv == 0) {  // all wave-uniform
      x0 *= kscale;
      x1 *= kscale;
    } else if (wv == 2) {
      x0 *= fk[0] == VK_NONE ? 0.0f : pow2f(fk[0]);
      x1 *= fk[1] == VK_NONE ? 0.0f : pow2f(fk[1]);
    } else if (wv == 3) {  // the value of code 128
      const uint32_t sw = wd.w[2][lane];
      x0 = fmaf(128.0f, bf16_lo(sw), x0);
      x1 = fmaf(128.0f, bf16_hi(sw), x1);
    }
    float* dst = (wv == 0 ? sm.tm.ks : wv == 1 ? sm.tm.ku : wv == 2 ? sm.tm.vs : sm.tm.vb)[0] + lane;
    dst[0] = x0;
    dst[PT] = x1;
  };

  // outstanding copies allowed: a tile's codes and (of the waves that copy them) words
  auto wait_copies = [&]() {
    if constexpr (PT == 128)
      asm volatile("s_waitcnt vmcnt(5)" ::: "memory");
    else if (grp_a)
      asm volatile("s_waitcnt vmcnt(3)" ::: "memory");
    else
      asm volatile("s_waitcnt vmcnt(2)" ::: "memory");
  };
  issue_words(0, 0);
  issue_words(1, 1);
  issue_codes(0, 0);
  issue_codes(1, 1);
  issue_words(2, 2);

  // ---- q of the wave's rows as MFMA B operands: times scale log2(e) in fp16, or (CODES) its bf16
  // values, converted with the workgroup's factor 2^kq once that is known
  half8_t qb[2][4];
  // causal bounds of the wave's rows (-1: not a row of the chunk), read back where tiles are masked
  // and for the output
  if (lane < 32) sm.lim[32 * wv + lane] = f0 + lane < R ? base + (f0 + lane) / G : -1;
  const int* lim = sm.lim + 32 * wv + lc;  // row 16 nt + lc of the wave at lim[16 nt]
  us2_t qm = {0, 0};  // CODES: bf16 bits of the largest finite |q|
#pragma unroll
  for (int nt = 0; nt < 2; ++nt) {
    const int f = f0 + 16 * nt + lc;
    const bool valid = f < R;
    const int i = valid ? f / G : 0, head = valid ? f - i * G : 0;
    const uint16_t* qr = q + (((int64_t)b * Hq + hk * G + head) * L + i) * D + 8 * lq4;
    const float qs = valid ? qk_scale_log2 : 0.0f;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint4 u = *reinterpret_cast<const uint4*>(qr + 32 * j);
      if constexpr (CODES) {
        const uint32_t w[4] = {valid ? u.x : 0u, valid ? u.y : 0u, valid ? u.z : 0u, valid ? u.w : 0u};
#pragma unroll
        for (int r = 0; r < 4; ++r) qm = __builtin_elementwise_max(qm, finite_bits(w[r]));
        qb[nt][j] = words_as_h8(w[0], w[1], w[2], w[3]);
      } else {
        const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          qb[nt][j][2 * r] = (_Float16)(bf16_lo(w[r]) * qs);
          qb[nt][j][2 * r + 1] = (_Float16)(bf16_hi(w[r]) * qs);
        }
      }
    }
  }
  if (CODES) {
    const uint32_t x = wave_max_u(max((uint32_t)qm.x, (uint32_t)qm.y));
    if (lane == 0) sm.qmax[wv] = x;
  }

  f4_t oacc[2][8];
  f4_t lacc[2];  // row sums of P (MFMA layout: all four values of a lane hold its row's sum)
  // CODES: the lane's sums of P and of P times the V value of code 128, per group
  float lsum[2] = {0.0f, 0.0f}, bsum[2][2] = {};
  float qsum[2][2];  // CODES: sum of the row's q over group g, times scale log2(e)
  float m_run[2];
#pragma unroll
  for (int nt = 0; nt < 2; ++nt) {
#pragma unroll
    for (int dt = 0; dt < 8; ++dt) oacc[nt][dt] = f4_t{0.f, 0.f, 0.f, 0.f};
    lacc[nt] = f4_t{0.f, 0.f, 0.f, 0.f};
    m_run[nt] = -INFINITY;
  }
  half8_t ones8;
#pragma unroll
  for (int j = 0; j < 8; ++j) ones8[j] = (_Float16)1.0f;

  // ---- per-tile phases of one wave
  // MFMA A fragments: K key 16 mt + lc, dims 32 kk + 8 lq4 .. + 7 at kfrag[kk] + 256 mt (uint4
  // units); V^T dim 16 dt + lc, slots 32 e + 8 lq4 .. + 7 at vfrag[e] + 2 PT dt
  const uint4* kfrag[4];
  const uint4* vfrag[PE];  // chunks of 8 slots: PT / 8 per dim
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    kfrag[j] = reinterpret_cast<const uint4*>(sm.k) + 16 * lc + ((4 * j + lq4) ^ lc);
  }
#pragma unroll
  for (int e = 0; e < PE; ++e)
    vfrag[e] = reinterpret_cast<const uint4*>(sm.vt) + PT / 8 * lc + ((4 * e + lq4) ^ vt_swz(lc));
  f4_t c[2][PMT];     // scores, c[nt][mt]: keys 16 mt + 4 lq4 + r of row 16 nt + lc (log2 units)
  // P in fp16, per N tile and k-step (CODES: times the V scale of group g)
  uint32_t pwd[2][PE][CODES ? 2 : 1][4];
  // Q.K^T of both N tiles from one read of each K fragment, relative to the rows' running
  // maxima (0 before the first): the accumulators start at -mref
  auto qk = [&]() {
    __builtin_amdgcn_s_setprio(0);
    if constexpr (CODES) {
      // Per quant group the product with the codes, then in fp32 s_0 z_0 + s_1 z_1 + b_1 Q_1 + b_0 Q_0
      float off[2];
#pragma unroll
      for (int nt = 0; nt < 2; ++nt) off[nt] = m_run[nt] == -INFINITY ? 0.0f : -m_run[nt];
      // The terms and sums of M tile mt - 1 between the MFMAs of M tile mt, their reads and those of the
      // next fragments ahead of them (the scheduling groups and barriers keep this order).
      uint4 fa[2][4];
      f4_t z[2][2][2], tu[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) fa[0][j] = kfrag[j][0];
#pragma unroll
      for (int mt = 0; mt <= PMT; ++mt) {
        __builtin_amdgcn_sched_barrier(0);
        if (mt > 0) {
          const int k0 = 16 * (mt - 1) + 4 * lq4;
          tu[0] = *reinterpret_cast<const f4_t*>(sm.tm.ku[0] + k0);
          tu[1] = *reinterpret_cast<const f4_t*>(sm.tm.ku[1] + k0);
          tu[2] = *reinterpret_cast<const f4_t*>(sm.tm.ks[0] + k0);
          tu[3] = *reinterpret_cast<const f4_t*>(sm.tm.ks[1] + k0);
        }
        if (mt + 1 < PMT) {
#pragma unroll
          for (int j = 0; j < 4; ++j) fa[(mt + 1) & 1][j] = kfrag[j][256 * (mt + 1)];
        }
        __builtin_amdgcn_sched_barrier(0);
        if (mt < PMT) {
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const int g = j & 1, e = j >> 1;  // k-step e of group g: dims 64 g + 32 e ..
            const uint4 a = fa[mt & 1][2 * g + e];
            const half8_t ah = words_as_h8(a.x, a.y, a.z, a.w);
#pragma unroll
            for (int nt = 0; nt < 2; ++nt)
              z[mt & 1][nt][g] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                  ah, qb[nt][2 * g + e], e == 0 ? f4_t{0.f, 0.f, 0.f, 0.f} : z[mt & 1][nt][g], 0, 0, 0);
          }
        }
        if (mt > 0) {
#pragma unroll
          for (int nt = 0; nt < 2; ++nt)
#pragma unroll
            for (int r = 0; r < 4; ++r)
              c[nt][mt - 1][r] = fmaf(tu[2][r], z[(mt - 1) & 1][nt][0][r],
                                      fmaf(tu[3][r], z[(mt - 1) & 1][nt][1][r],
                                           fmaf(tu[1][r], qsum[nt][1],
                                                fmaf(tu[0][r], qsum[nt][0], off[nt]))));
        }
        if (mt > 0 && mt < PMT) {
          __builtin_amdgcn_sched_group_barrier(0x008, 4, 0);  // MFMA
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            __builtin_amdgcn_sched_group_barrier(0x002, 8, 0);  // VALU
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
        if (mt > 0) asm volatile("" : "+v"(c[0][mt - 1]), "+v"(c[1][mt - 1]));
      }
      return;
    }
    f4_t cinit[2];
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) {
      const float mref = m_run[nt] == -INFINITY ? 0.0f : m_run[nt];
      cinit[nt] = f4_t{-mref, -mref, -mref, -mref};
    }
    // fragments one M tile ahead of the MFMAs that use them (the scheduling barriers keep the
    // reads of M tile mt + 1 issued before the MFMAs of M tile mt)
    uint4 fa[2][4];
#pragma unroll
    for (int j = 0; j < 4; ++j) fa[0][j] = kfrag[j][0];
#pragma unroll
    for (int mt = 0; mt < PMT; ++mt) {
      if (mt + 1 < PMT) {
#pragma unroll
        for (int j = 0; j < 4; ++j) fa[(mt + 1) & 1][j] = kfrag[j][256 * (mt + 1)];
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint4 a = fa[mt & 1][j];  // key 16 mt + lc
        const half8_t ah = words_as_h8(a.x, a.y, a.z, a.w);
#pragma unroll
        for (int nt = 0; nt < 2; ++nt)  // each chain starts from the shared -mref tuple
          c[nt][mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah, qb[nt][j],
                                                             j == 0 ? cinit[nt] : c[nt][mt], 0, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // P of a tile (CODES) as the operands of both groups, and the lane's sums, in fp32 as the verify
  // kernel takes them. In a tile that is masked (FULL false) keys past a row's bound are left out, so
  // that their terms (an infinity or NaN among them) do not reach it.
  auto weights = [&](int t0, auto full) __attribute__((always_inline)) {
    constexpr bool FULL = decltype(full)::value;
#pragma unroll
    for (int mt = 0; mt < PMT; ++mt) {
      __builtin_amdgcn_sched_barrier(0);
      const int k0 = 16 * mt + 4 * lq4;
      const f4_t s0 = *reinterpret_cast<const f4_t*>(sm.tm.vs[0] + k0);
      const f4_t s1 = *reinterpret_cast<const f4_t*>(sm.tm.vs[1] + k0);
      const f4_t z0 = *reinterpret_cast<const f4_t*>(sm.tm.vb[0] + k0);
      const f4_t z1 = *reinterpret_cast<const f4_t*>(sm.tm.vb[1] + k0);
#pragma unroll
      for (int nt = 0; nt < 2; ++nt) {
        const int last = FULL ? 0 : lim[16 * nt];
        float ls = 0.0f, b0 = 0.0f, b1 = 0.0f, w0[4], w1[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float p = __builtin_amdgcn_exp2f(c[nt][mt][r]);
          const bool seen = FULL || t0 + k0 + r <= last;
          ls += p;
          b0 = fmaf(p, seen ? z0[r] : 0.0f, b0);
          b1 = fmaf(p, seen ? z1[r] : 0.0f, b1);
          w0[r] = p * (seen ? s0[r] : 0.0f);
          w1[r] = p * (seen ? s1[r] : 0.0f);
        }
        lsum[nt] += ls;
        bsum[nt][0] += b0;
        bsum[nt][1] += b1;
        uint32_t* d0 = pwd[nt][mt >> 1][0] + 2 * (mt & 1);
        uint32_t* d1 = pwd[nt][mt >> 1][CODES ? 1 : 0] + 2 * (mt & 1);
        d0[0] = pack_h2(w0[0], w0[1]);
        d0[1] = pack_h2(w0[2], w0[3]);
        d1[0] = pack_h2(w1[0], w1[1]);
        d1[1] = pack_h2(w1[2], w1[3]);
        // made here, so that neither the terms nor P live on
        asm volatile("" : "+v"(d0[0]), "+v"(d0[1]), "+v"(d1[0]), "+v"(d1[1]), "+v"(lsum[nt]),
                     "+v"(bsum[nt][0]), "+v"(bsum[nt][1]));
      }
    }
  };
  // softmax per N tile: masking, lazy rescale, P in fp16 (its row sums are taken by P.V)
  auto softmax = [&](int t0, bool full) {
    __builtin_amdgcn_s_setprio(2);
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) {
      if (!full) {
        const int last = lim[16 * nt];
#pragma unroll
        for (int mt = 0; mt < PMT; ++mt)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            c[nt][mt][r] = t0 + 16 * mt + 4 * lq4 + r <= last ? c[nt][mt][r] : -INFINITY;
      }
      float tmax = -INFINITY;
#pragma unroll
      for (int mt = 0; mt < PMT; ++mt)
#pragma unroll
        for (int r = 0; r < 4; ++r) tmax = fmaxf(tmax, c[nt][mt][r]);
      tmax = max_xor16(tmax);
      tmax = max_xor32(tmax);
      // a new running maximum: the tile's exceeds it by more than RESCALE_LOG2 (any finite one
      // the first time)
      const bool bump = tmax > (m_run[nt] == -INFINITY ? -INFINITY : RESCALE_LOG2);
      if (__builtin_amdgcn_ballot_w64(bump)) {
        const float mref = m_run[nt] == -INFINITY ? 0.0f : m_run[nt];
        const float mn = bump ? mref + tmax : m_run[nt];
        const float alpha = m_run[nt] == -INFINITY ? 0.0f : exp2_nonpos(m_run[nt] - mn);
        m_run[nt] = mn;
        lacc[nt] *= alpha;
        lsum[nt] *= alpha;
        bsum[nt][0] *= alpha;
        bsum[nt][1] *= alpha;
#pragma unroll
        for (int dt = 0; dt < 8; ++dt) oacc[nt][dt] *= alpha;
        const float shift = bump ? tmax : 0.0f;  // new reference minus the one the scores hold
#pragma unroll
        for (int mt = 0; mt < PMT; ++mt) c[nt][mt] -= shift;
      }
      if constexpr (CODES) continue;
#pragma unroll
      for (int e = 0; e < PE; ++e) {
        half2_t ph[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int hh = j >> 1, r = 2 * (j & 1);
          ph[j] = half2_t{(_Float16)__builtin_amdgcn_exp2f(c[nt][2 * e + hh][r]),
                          (_Float16)__builtin_amdgcn_exp2f(c[nt][2 * e + hh][r + 1])};
        }
        uint32_t* pd = pwd[nt][e][0];
#pragma unroll
        for (int j = 0; j < 4; ++j) pd[j] = __builtin_bit_cast(uint32_t, ph[j]);
        // P is made in this slot, not sunk into P.V's
        asm volatile("" : "+v"(pd[0]), "+v"(pd[1]), "+v"(pd[2]), "+v"(pd[3]));
      }
    }
    if constexpr (CODES) {
      if (full)
        weights(t0, std::true_type{});
      else
        weights(t0, std::false_type{});
    }
  };
  // P.V of both N tiles from one read of each V^T fragment, and the rows' sums of P:
  // out^T[16 dt + 4 lq4 + r][row 16 nt + lc] += V^T[dims][slots] P^T[slots][rows]
  // CODES: the accumulators go over to the tile's exponents
  auto refactor = [&]() __attribute__((always_inline)) {
    if (fk[0] != ak[0] || fk[1] != ak[1]) {  // wave-uniform; the first tile, then rare
      const float r0 = ak[0] == VK_NONE ? 1.0f : pow2f(fk[0] - ak[0]);
      const float r1 = ak[1] == VK_NONE ? 1.0f : pow2f(fk[1] - ak[1]);
#pragma unroll
      for (int nt = 0; nt < 2; ++nt)
#pragma unroll
        for (int dt = 0; dt < 8; ++dt) oacc[nt][dt] *= dt < 4 ? r0 : r1;
      ak[0] = fk[0];
      ak[1] = fk[1];
    }
  };
  auto pw = [&](int nt, int e, int g) __attribute__((always_inline)) {
    const uint32_t* w = pwd[nt][e][g];
    return words_as_h8(w[0], w[1], w[2], w[3]);
  };
  auto pv = [&](int snext) {  // CODES: ends with the exponents of the next tile (sm.vexp[snext])
    __builtin_amdgcn_s_setprio(0);
    int2 knext;
    if (CODES) knext = *reinterpret_cast<const int2*>(sm.vexp[snext]);
    // fragments four dims tiles ahead (half a k-step), as in qk: step u = (k-step u / 2, dim
    // tiles 4 (u % 2) .. + 3)
    uint4 fv[2][4];
    if (CODES) refactor();
#pragma unroll
    for (int j = 0; j < 4; ++j) fv[0][j] = vfrag[0][2 * PT * j];
#pragma unroll
    for (int u = 0; u < 2 * PE; ++u) {
      if (u + 1 < 2 * PE) {
        const int e1 = (u + 1) >> 1, d1 = 4 * ((u + 1) & 1);
#pragma unroll
        for (int j = 0; j < 4; ++j) fv[(u + 1) & 1][j] = vfrag[e1][2 * PT * (d1 + j)];
      }
      __builtin_amdgcn_sched_barrier(0);
      const int e = u >> 1, d0 = 4 * (u & 1);
      if (!CODES && (u & 1)) {  // row sums of this k-step's P: a ones A operand (every output row the sum)
#pragma unroll
        for (int nt = 0; nt < 2; ++nt)
          lacc[nt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ones8, pw(nt, e, 0), lacc[nt], 0, 0, 0);
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint4 a = fv[u & 1][j];  // dim 16 (d0 + j) + lc
        const half8_t ah = words_as_h8(a.x, a.y, a.z, a.w);
#pragma unroll
        for (int nt = 0; nt < 2; ++nt)
          oacc[nt][d0 + j] =
              __builtin_amdgcn_mfma_f32_16x16x32_f16(ah, pw(nt, e, CODES ? u & 1 : 0),
                                                     oacc[nt][d0 + j], 0, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if (CODES) take_exponents(knext);
  };

  // ---- prologue: tile 0 and the words of tile 1 landed (outstanding: tile 1's codes, tile 2's
  // words), K(0) in fp16; CODES: tile 0's exponents and terms, q in fp16
  wait_copies();
  __syncthreads();
  if (CODES) {
    next_exponents(0, sm.wd[0]);
    // one factor for the workgroup's rows: the largest finite |q| in [2^14, 2^15) (exact for values
    // down to 2^-31 of it); rows with an infinity or NaN leave the others' factor alone
    const uint4 a = *reinterpret_cast<const uint4*>(sm.qmax);
    const uint4 e = *reinterpret_cast<const uint4*>(sm.qmax + 4);
    const uint32_t m = __builtin_amdgcn_readfirstlane(
        max(max(max(a.x, a.y), max(a.z, a.w)), max(max(e.x, e.y), max(e.z, e.w))));
    const int kq = m == 0 ? 0 : min(max(15 - bound_exp(m), -100), 100);
    const float qf = pow2f(kq);
    kscale = qk_scale_log2 * pow2f(24 - kq);
#pragma unroll
    for (int nt = 0; nt < 2; ++nt)
#pragma unroll
      for (int g = 0; g < 2; ++g) {
        float x = 0.0f;
#pragma unroll
        for (int j = 2 * g; j < 2 * g + 2; ++j) {
          const uint4 u = __builtin_bit_cast(uint4, qb[nt][j]);
          const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            x += bf16_lo(w[r]) + bf16_hi(w[r]);
            qb[nt][j][2 * r] = (_Float16)(bf16_lo(w[r]) * qf);
            qb[nt][j][2 * r + 1] = (_Float16)(bf16_hi(w[r]) * qf);
          }
        }
        qsum[nt][g] = sum_xor32(sum_xor16(x)) * qk_scale_log2;
      }
    __syncthreads();
    take_exponents(*reinterpret_cast<const int2*>(sm.vexp[0]));
  }
  if (grp_a) {
    dequant_k(sm.raw[0], sm.wd[0]);
    if (CODES) tile_terms(sm.wd[0]);
  }
  __syncthreads();

  // The two halves run their own loops (wave-uniform branch): each wave passes the same four
  // barriers per tile. Tiles 0 .. Tact - 1 hold keys visible to the wave's rows; past them the
  // wave keeps only its copy, exponent and dequantization duties. (Two loops rather than a condition
  // per phase, so that the scores and P are not live across the loop's back edge.) The words run
  // a tile ahead of the codes, so that a tile's exponents are made beside the Q.K^T of the tile before
  // it, which outlasts that half's V.
  const int Tact = lim_hi < 0 ? 0 : max(0, min(T, lim_hi / PT + 1 - tb));
  int w0 = 0, w1 = 1;  // word slots of tiles t and t + 1
  auto next_words = [&]() {
    w0 = w1;
    w1 = w1 == 2 ? 0 : w1 + 1;
  };
  if (grp_a) {
    int t = 0;
    for (; t < Tact; ++t) {
      const int t0 = PT * (tb + t);
      qk();                                             // slot 4t
      __syncthreads();
      issue_codes(t + 2, t & 1);                        // slot 4t + 1: into t's slots
      issue_words(t + 3, w0);
      softmax(t0, t0 + PT - 1 <= lim_lo);
      __syncthreads();
      pv((t + 1) & 1);                                  // slot 4t + 2
      wait_copies();  // codes of t + 1, words of t + 2 landed
      __syncthreads();
      if (t + 1 < T) {                                  // slot 4t + 3
        if (CODES) tile_terms(sm.wd[w1]);
        dequant_k(sm.raw[(t + 1) & 1], sm.wd[w1]);
      }
      next_words();
      __syncthreads();
    }
    for (; t < T; ++t) {
      __syncthreads();
      issue_codes(t + 2, t & 1);
      issue_words(t + 3, w0);
      __syncthreads();
      if (CODES) take_exponents(*reinterpret_cast<const int2*>(sm.vexp[(t + 1) & 1]));
      wait_copies();
      __syncthreads();
      if (t + 1 < T) {
        if (CODES) tile_terms(sm.wd[w1]);
        dequant_k(sm.raw[(t + 1) & 1], sm.wd[w1]);
      }
      next_words();
      __syncthreads();
    }
  } else {
    int t = 0;
    for (; t < Tact; ++t) {
      const int t0 = PT * (tb + t);
      dequant_v(sm.raw[t & 1], sm.wd[w0]);              // slot 4t
      if (CODES) next_exponents((t + 1) & 1, sm.wd[w1]);
      __syncthreads();
      qk();                                             // slot 4t + 1
      __syncthreads();
      issue_codes(t + 2, t & 1);                        // slot 4t + 2
      issue_words(t + 3, w0);
      softmax(t0, t0 + PT - 1 <= lim_lo);
      wait_copies();
      __syncthreads();
      pv((t + 1) & 1);                                  // slot 4t + 3
      next_words();
      __syncthreads();
    }
    for (; t < T; ++t) {
      dequant_v(sm.raw[t & 1], sm.wd[w0]);
      if (CODES) next_exponents((t + 1) & 1, sm.wd[w1]);
      __syncthreads();
      __syncthreads();
      issue_codes(t + 2, t & 1);
      issue_words(t + 3, w0);
      wait_copies();
      __syncthreads();
      if (CODES) take_exponents(*reinterpret_cast<const int2*>(sm.vexp[(t + 1) & 1]));
      next_words();
      __syncthreads();
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the clamped copies past the end

  // ---- output rows: acc / l (CODES: with the factors taken out and the bias sums added); of a part
  // of the block's tiles in fp32, with the row's (m, l), for prefill_merge_kernel
  const bool whole = !SPLIT || (last_part && tb == 0);
  const int64_t slot = 2 * (int64_t)x + (tb == 0);
#pragma unroll
  for (int nt = 0; nt < 2; ++nt) {
    const float l = CODES ? sum_xor32(sum_xor16(lsum[nt])) : lacc[nt][0];
    float osc[2], ob[2];  // CODES: the groups' factor out of the accumulators, and bias sums
    if (CODES) {
#pragma unroll
      for (int g = 0; g < 2; ++g) {
        osc[g] = ak[g] == VK_NONE ? 1.0f : pow2f(-ak[g]);
        ob[g] = sum_xor32(sum_xor16(bsum[nt][g]));
      }
    }
    const int last = lim[16 * nt];
    if (last >= 0) {
      const float inv = l > 0.0f ? 1.0f / l : 0.0f;
      const int wrow = 32 * wv + 16 * nt + lc;
      const int i = last - base, head = pb * PROWS + wrow - i * G;
      uint16_t* orow = out + (((int64_t)b * Hq + hk * G + head) * L + i) * D;
      float* prow = sp.part_o + (slot * PROWS + wrow) * D;
#pragma unroll
      for (int dt = 0; dt < 8; ++dt) {
        f4_t o = oacc[nt][dt];
        if (CODES) {
#pragma unroll
          for (int r = 0; r < 4; ++r) o[r] = fmaf(o[r], osc[dt >> 2], ob[dt >> 2]);
        }
        o *= inv;
        if (whole) {
          const uint32_t lo = (uint32_t)f32_to_bf16(o[0]) | ((uint32_t)f32_to_bf16(o[1]) << 16);
          const uint32_t hi = (uint32_t)f32_to_bf16(o[2]) | ((uint32_t)f32_to_bf16(o[3]) << 16);
          *reinterpret_cast<uint2*>(orow + 16 * dt + 4 * lq4) = make_uint2(lo, hi);
        } else {
          *reinterpret_cast<f4_t*>(prow + 16 * dt + 4 * lq4) = o;
        }
      }
      if (!whole && lq4 == 0) sp.part_ml[slot * PROWS + wrow] = make_float2(m_run[nt], l);
    }
  }

  more = SPLIT && u_blk + T_blk < u_end && pb + 1 < npb;
  u_blk += T_blk;
  u = u_blk;
  ++pb;
  if (more) __syncthreads();  // the LDS is the next segment's
  }
}

// Rows of split blocks: the shares' partial rows weighted by their sums (log-sum-exp). One
// workgroup per 2 rows of a block; a row's parts (those of consecutive shares) are dealt to four
// groups of 32 lanes (4 dims each), which combine through LDS. Blocks that one share covered whole
// are written already. Bound by the loads' latency: 33 MB of parts (64 rows at 82,735 keys, 32/8
// heads, 31 parts per row) took 20.4 us with one group per row and 8 rows per workgroup. The tiles
// before the block are summed by all threads: in a loop of each, that was most of the launch where
// blocks are many (3,072 rows behind 2,000 keys, 32/8 heads, split into parts: 336 us in all, now 243).
__global__ __launch_bounds__(256) void prefill_merge_kernel(uint16_t* __restrict__ out, int n, int L,
                                                            int Hkv, int G, PrefillSplit sp) {
  __shared__ f4_t sh_acc[2][4][32];
  __shared__ float2 sh_ml[2][4];
  __shared__ int sh_u[4];
  const int hk = blockIdx.y % Hkv, b = blockIdx.y / Hkv;
  const int R = L * G, base = n - L;
  const int pb = blockIdx.x / (PROWS / 2);
  const int tr = threadIdx.x >> 7, grp = (threadIdx.x >> 5) & 3, ln = threadIdx.x & 31;
  const int wrow = 2 * (blockIdx.x % (PROWS / 2)) + tr;
  // tiles of the blocks before this one, over the workgroup's threads
  int part = 0;
  for (int j = threadIdx.x; j < pb; j += 256) part += prefill_tiles(j, R, sp.g, base);
#pragma unroll
  for (int m = 1; m < 64; m *= 2) part += __shfl_xor(part, m);
  if ((threadIdx.x & 63) == 0) sh_u[threadIdx.x >> 6] = part;
  __syncthreads();
  const int u0 = sh_u[0] + sh_u[1] + sh_u[2] + sh_u[3];
  const int u1 = u0 + prefill_tiles(pb, R, sp.g, base);
  const int j0 = u0 / sp.tiles, j1 = (u1 - 1) / sp.tiles;
  const int f = pb * PROWS + wrow;
  if (j0 == j1 || f - tr >= R) return;  // workgroup-uniform
  const bool valid = f < R;
  auto row = [&](int j) {  // row of share j's part of this block
    const int64_t x = hk + (int64_t)Hkv * (j + (int64_t)sp.shares * b);
    return (2 * x + (j == j0)) * PROWS + wrow;
  };
  float M = -INFINITY;
  f4_t acc = {0.f, 0.f, 0.f, 0.f};
  float den = 0.0f;
  if (valid) {
#pragma unroll 4
    for (int j = j0 + grp; j <= j1; j += 4) M = fmaxf(M, sp.part_ml[row(j)].x);
#pragma unroll 4
    for (int j = j0 + grp; j <= j1; j += 4) {
      const int64_t r = row(j);
      const float2 ml = sp.part_ml[r];
      const f4_t o = *reinterpret_cast<const f4_t*>(sp.part_o + r * D + 4 * ln);
      if (ml.y != 0.0f) {  // a part that saw keys; a NaN sum goes into the row's
        const float w = exp2_nonpos(ml.x - M) * ml.y;
        acc += o * w;
        den += w;
      }
    }
  }
  sh_acc[tr][grp][ln] = acc;
  if (ln == 0) sh_ml[tr][grp] = make_float2(M, den);
  __syncthreads();
  if (grp != 0 || !valid) return;
  float mx = -INFINITY;
#pragma unroll
  for (int g = 0; g < 4; ++g) mx = fmaxf(mx, sh_ml[tr][g].x);
  acc = f4_t{0.f, 0.f, 0.f, 0.f};
  den = 0.0f;
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    const float2 ml = sh_ml[tr][g];
    if (ml.y != 0.0f) {
      const float w = exp2_nonpos(ml.x - mx);
      acc += sh_acc[tr][g][ln] * w;
      den += w * ml.y;
    }
  }
  const f4_t o = acc * (den != 0.0f ? 1.0f / den : 0.0f);
  const int i = (int)fdiv_u((uint32_t)f, sp.g), head = f - i * G;
  const uint32_t lo = (uint32_t)f32_to_bf16(o[0]) | ((uint32_t)f32_to_bf16(o[1]) << 16);
  const uint32_t hi = (uint32_t)f32_to_bf16(o[2]) | ((uint32_t)f32_to_bf16(o[3]) << 16);
  *reinterpret_cast<uint2*>(out + (((int64_t)b * Hkv * G + hk * G + head) * L + i) * D + 4 * ln) =
      make_uint2(lo, hi);
}

// How the blocks of a chunk are dealt to workgroups: whole, one block each (tiles 0), or each KV
// head's tiles, block after block, in equal shares of `tiles` for as many workgroups as fill the
// CUs. Whole blocks go round by round, longest first: their time follows the tiles of each round's
// longest block. A share's time follows its tiles, the blocks that it touches (q, the first copies,
// the output rows) and the partial rows that are written and merged. Costs fitted to 190 chunks timed
// both ways (G 1 to 8, 17 to 4,096 rows behind 64 to 32,000 keys; within 15% from 40 us on); split where
// they say 3% or more. us, whole / split: 32/8 heads, 64 rows behind 32,000 keys 790 / 56, 512 behind
// 1,000 48 / 53 and 2,000 73 / 60, 1,536 behind 2,000 100 / 115, 3,072 behind 2,000 190 / 242; 16/2,
// 2,048 behind 500 74 / 80 and 2,000 111 / 95; 48/8, 512 behind 500 61 / 65 and 8,000 419 / 196, 2,048
// behind 2,000 293 / 312 and 16,000 1,628 / 1,305.
struct SplitCosts {  // in 10 ns
  int tile, segment, block, split;  // of a share per tile and touched block, of all blocks each, constant
  int whole_tile, whole;            // of whole blocks per tile, constant
};
constexpr SplitCosts FP16_COSTS = {390, 900, 17, 900, 308, 990};
constexpr SplitCosts CODES_COSTS = {600, 700, 27, 500, 564, 920};
constexpr int MIN_SHARE = 2;

// Groupings that the verify kernel served before keep its arithmetic (see the top of the file).
bool codes_variant(int64_t G) { return !(G == 1 || G == 2 || G == 4 || G == 8); }

PrefillSplit plan_split(int64_t B, int64_t Hkv, int64_t G, int64_t L, int64_t n, int cus) {
  const int R = (int)(L * G), base = (int)(n - L), npb = (R + PROWS - 1) / PROWS;
  PrefillSplit sp{make_fastdiv((uint32_t)G), npb, 0, nullptr, nullptr};
  const int64_t S = cus / (B * Hkv);
  if (S < 2 || npb > 4 * S) return sp;  // no CUs to spare; the last round matters little
  int64_t total = 0, rounds = 0;
  for (int i = 0, r = -1; i < npb; ++i) {  // longest blocks first, B Hkv of each length
    const int t = prefill_tiles(npb - 1 - i, R, sp.g, base);
    total += t;
    if ((int)(((i + 1) * B * Hkv - 1) / cus) > r) {
      rounds += t;
      ++r;
    }
  }
  const int64_t tiles = std::max<int64_t>(MIN_SHARE, (total + S - 1) / S);
  const int64_t touched = 2 + (tiles - 2) / prefill_tiles(0, R, sp.g, base);  // block 0: shortest
  const SplitCosts c = codes_variant(G) ? CODES_COSTS : FP16_COSTS;
  const int64_t split = c.tile * tiles + c.segment * touched + c.block * npb * B * Hkv + c.split;
  if (tiles >= rounds || 103 * split > 100 * (c.whole_tile * rounds + c.whole)) return sp;
  sp.tiles = (int)tiles;
  sp.shares = (int)((total + tiles - 1) / tiles);
  return sp;
}

int64_t split_bytes(const PrefillSplit& sp, int64_t B, int64_t Hkv) {
  return sp.tiles ? 2 * B * Hkv * sp.shares * PROWS * (int64_t)(D * sizeof(float) + sizeof(float2))
                  : 0;
}

int prefill_attn(const uint16_t* q, const uint8_t* kc, const uint16_t* ks, const uint16_t* kb,
                 const uint8_t* vc, const uint16_t* vs, const uint16_t* vb, int64_t B, int64_t Hq,
                 int64_t Hkv, int64_t L, int64_t D, int64_t cap, int64_t n, float scale,
                 uint16_t* out, bool split, void* workspace, int64_t workspace_bytes,
                 hipStream_t st) {
  LQ_CHECK_ARG(D == 128, "head_dim must be 128 (got %lld)", (long long)D);
  LQ_CHECK_ARG(Hkv >= 1 && Hq >= Hkv && Hq % Hkv == 0, "Hq=%lld must be a multiple of Hkv=%lld",
               (long long)Hq, (long long)Hkv);
  const int64_t G = Hq / Hkv;
  LQ_CHECK_ARG(G <= 64, "%lld query heads per KV head exceed 64", (long long)G);
  LQ_CHECK_ARG(B >= 1 && L >= 1 && L <= n && n <= cap && cap <= (1 << 24),
               "need 1 <= L=%lld <= n=%lld <= cap=%lld <= 2^24", (long long)L, (long long)n,
               (long long)cap);
  LQ_CHECK_ARG(q && kc && ks && kb && vc && vs && vb && out, "null pointer");
  const int64_t npb = (L * G + PROWS - 1) / PROWS;
  LQ_CHECK_ARG(B * Hkv * npb <= (int64_t)INT32_MAX, "too many workgroups");
  PrefillSplit sp{make_fastdiv((uint32_t)G), (int)npb, 0, nullptr, nullptr};
  if (split) {
    sp = plan_split(B, Hkv, G, L, n, device_cu_count());
    const int64_t need = split_bytes(sp, B, Hkv);
    if (need > 0 && (!workspace || workspace_bytes < need)) {
      set_error("workspace of %lld bytes is smaller than the %lld needed",
                (long long)workspace_bytes, (long long)need);
      return LQ_EWORKSPACE;
    }
    sp.part_o = (float*)workspace;
    sp.part_ml = (float2*)(sp.part_o + 2 * B * Hkv * sp.shares * PROWS * D);
  }
  const int64_t wgs = B * Hkv * sp.shares;
  const bool codes = codes_variant(G);
  auto* kern = codes ? (sp.tiles ? q8_prefill_kernel<true, true> : q8_prefill_kernel<true, false>)
                     : (sp.tiles ? q8_prefill_kernel<false, true> : q8_prefill_kernel<false, false>);
  kern<<<dim3((unsigned)wgs), dim3(64 * PW), 0, st>>>(
      q, kc, ks, kb, vc, vs, vb, out, cap, (int)n, (int)L, (int)Hkv, (int)G, (int)npb, sp,
      scale * 1.4426950408889634f);
  LQ_CHECK_LAUNCH("q8_prefill_kernel");
  if (sp.tiles) {
    prefill_merge_kernel<<<dim3((unsigned)(npb * (PROWS / 2)), (unsigned)(B * Hkv)), dim3(256), 0,
                           st>>>(out, (int)n, (int)L, (int)Hkv, (int)G, sp);
    LQ_CHECK_LAUNCH("prefill_merge_kernel");
  }
  return LQ_OK;
}

}  // namespace
}  // namespace lq

extern "C" int lq_q8_prefill_attn(const uint16_t* q, const uint8_t* kc, const uint16_t* ks,
                                  const uint16_t* kb, const uint8_t* vc, const uint16_t* vs,
                                  const uint16_t* vb, int64_t B, int64_t Hq, int64_t Hkv,
                                  int64_t L, int64_t D, int64_t cap, int64_t n, float scale,
                                  uint16_t* out, void* stream) {
  using namespace lq;
  clear_error();
  LQ_CHECK_ARG(Hkv < 1 || Hq % Hkv || Hq / Hkv == 1 || Hq / Hkv == 2 || Hq / Hkv == 4 ||
                   Hq / Hkv == 8,
               "this entry takes 1, 2, 4 or 8 query heads per KV head (got %lld)",
               (long long)(Hq / Hkv));
  return prefill_attn(q, kc, ks, kb, vc, vs, vb, B, Hq, Hkv, L, D, cap, n, scale, out, false,
                      nullptr, 0, (hipStream_t)stream);
}

extern "C" int64_t lq_prefill_workspace_bytes(int64_t B, int64_t Hq, int64_t Hkv, int64_t L,
                                              int64_t n) {
  using namespace lq;
  clear_error();
  if (B < 1 || Hkv < 1 || Hq < Hkv || Hq % Hkv || Hq / Hkv > 64 || L < 1 || L > n ||
      n > (1 << 24)) {
    set_error("bad prefill shape B=%lld Hq=%lld Hkv=%lld L=%lld n=%lld", (long long)B,
              (long long)Hq, (long long)Hkv, (long long)L, (long long)n);
    return -1;
  }
  return split_bytes(plan_split(B, Hkv, Hq / Hkv, L, n, device_cu_count()), B, Hkv);
}

extern "C" int lq_q8_prefill_attn_grouped(const uint16_t* q, const uint8_t* kc, const uint16_t* ks,
                                          const uint16_t* kb, const uint8_t* vc,
                                          const uint16_t* vs, const uint16_t* vb, int64_t B,
                                          int64_t Hq, int64_t Hkv, int64_t L, int64_t D,
                                          int64_t cap, int64_t n, float scale, uint16_t* out,
                                          void* workspace, int64_t workspace_bytes,
                                          void* stream) {
  lq::clear_error();
  return lq::prefill_attn(q, kc, ks, kb, vc, vs, vb, B, Hq, Hkv, L, D, cap, n, scale, out, true,
                          workspace, workspace_bytes, (hipStream_t)stream);
}
