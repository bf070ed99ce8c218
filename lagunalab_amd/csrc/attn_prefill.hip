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
// up to its last row's
// causal bound; each tile is brought into LDS once for all 8 waves and dequantized once:
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
// the pace and the matrix phases' issue only every 16 cycles (2,048 rows at 82,671 keys: 2,437 ->
// 2,407 us against 2,429 and 2,414 of an unchanged kernel beside them).
// Tiles past a wave's last row are skipped by that wave (it keeps its copy and dequantization
// duties); tiles straddling its rows' bounds are masked per row. Rows past the chunk (a ragged last
// block) read no q and store nothing. Keys past n-1 are never read: copies clamp their rows to n-1.
//
// fp16 operand range: q, K and V enter the MFMAs in fp16. In the RANGE variant out-of-range data
// carries power-of-two factors that are taken out again exactly: 2^-kk on a tile's K with 2^kk on
// q, and 2^-kv on a tile's V (the accumulators are rescaled when it changes). Group A takes bounds
// of the largest |K| and |V| of tile t+1 from its scale and bias words in slot 4t, every wave the
// factors from them at the end of its P.V(t). Data of ordinary size (WIN_LO .. WIN_HI) has all
// factors at 0, and the paths that apply them are wave-uniform branches not taken; they still cost
// 2-3% (2,048 rows at 82,671 keys, 32/8 heads: 2.43 -> 2.48 ms), so groupings of 1, 2, 4 and 8,
// whose range has always been that of fp16, run without. The other groupings went through the
// verify kernel in blocks of 64 / G positions (each block a launch that reads the whole cache, and
// a merge), whose operands have such factors: 512 rows at 8,193 keys, 48/8 heads, 1,026 -> 237 us.
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

constexpr int PW = 8;       // waves per workgroup
constexpr int PROWS = 256;  // query rows per workgroup
constexpr int PT = 128;     // keys per tile
constexpr int PMT = PT / 16;  // M tiles (16 keys) per tile
constexpr int PE = PT / 32;   // P.V k-steps (32 keys) per tile

// Exponent window of the fp16 operands: a bound M < 2^e needs no factor for WIN_LO <= e <= WIN_HI,
// else the factor brings e to WIN_HI - 1. |K| and |V| are below 2 M (M = max(|bias|, 256 |scale|)),
// so WIN_HI = 14 keeps them below 2^15.
constexpr int WIN_LO = -2, WIN_HI = 14;
// A V factor that falls again (smaller values after larger ones) multiplies the accumulators: by at
// most 2^KV_FALL below the largest factor so far, so that they stay finite (they are below 2^41 in
// that factor's units); values 2^KV_FALL smaller than others of the head lose bits instead.
constexpr int KV_FALL = 60;
constexpr uint32_t IN_WINDOW = 126u << 7;  // a bound in the window, whatever it is (exponent 0)

__device__ __forceinline__ bool in_window(int e) {
  return (unsigned)(e - WIN_LO) <= (unsigned)(WIN_HI - WIN_LO);
}
__device__ __forceinline__ float exp2_int(int k) { return __uint_as_float((uint32_t)(127 + k) << 23); }
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
// Exponent e of the bound: the value of bf16 bits b is below 2^e.
__device__ __forceinline__ int bound_exp(uint32_t b) { return (int)(b >> 7) - 126; }
typedef uint16_t us2_t __attribute__((ext_vector_type(2)));
// Both bf16 halves of a word times f (a power of two: exact but for underflow).
__device__ __forceinline__ uint32_t scale_word(uint32_t w, float f) {
  return (__float_as_uint(bf16_lo(w) * f) >> 16) | (__float_as_uint(bf16_hi(w) * f) & 0xffff0000u);
}

struct PrefillRaw {
  alignas(16) uint8_t k[PT * D];  // row-major [key][128 B]
  uint8_t v[PT * D];
};

struct PrefillWords {
  alignas(16) uint32_t w[4][PT];  // K scale, K bias, V scale, V bias words (two bf16 groups each)
};

struct PrefillSmem {
  PrefillRaw raw[2];               // codes of tiles t, t + 1
  PrefillWords wd[3];              // words of tiles t, t + 1, t + 2
  alignas(16) uint32_t rng[2][4];  // tile t, t + 1: bf16 bits of the tile's largest |K| (waves 0, 1)
                                   // and |V| (waves 2, 3) bound
  uint32_t qmax[PW];               // bf16 bits of the largest |q| of each wave's rows
  int lim[PROWS];                  // last key each row sees
  alignas(16) _Float16 k[PT * D];   // [key][dim], 16-byte chunk j of key r at chunk j ^ (r & 15)
  alignas(16) _Float16 vt[D * PT];  // [dim][slot], 16-byte chunk j of dim d at chunk j ^ (d & 15)
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
  return (base + (int)fdiv_u((uint32_t)min(pb * PROWS + PROWS - 1, R - 1), g)) / PT + 1;
}

template <bool RANGE, bool SPLIT>
__global__ __launch_bounds__(64 * PW, 1) void q8_prefill_kernel(
    const uint16_t* __restrict__ q, const uint8_t* __restrict__ kc,
    const uint16_t* __restrict__ ks, const uint16_t* __restrict__ kb,
    const uint8_t* __restrict__ vc, const uint16_t* __restrict__ vs,
    const uint16_t* __restrict__ vb, uint16_t* __restrict__ out, int64_t cap, int n, int L,
    int Hkv, int G, int npb, PrefillSplit sp, float q_scale, float k_scale) {
  __shared__ PrefillSmem sm;
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
  const int tb = SPLIT ? u - u_blk : 0;           // the segment: tiles tb .. tb + T - 1
  const int T = SPLIT ? min(T_blk, u_end - u_blk) - tb : T_blk;
  // this wave's rows f0 .. f0 + 31 (row 16 nt + lc of the wave: f0 + 16 nt + lc)
  const int f0 = pb * PROWS + 32 * wv;
  const int lim_lo = base + f0 / G;                                 // bound of its first row
  const int lim_hi = f0 < R ? base + min(f0 + 31, R - 1) / G : -1;  // of its last valid row

  // ---- raw tile copies, per thread: two 16-byte K copies (wave wv: keys 16 wv .. 16 wv + 15),
  // two V copies, one word (wave wv: word array wv / 2, keys 64 (wv % 2) + lane)
  const uint32_t lds_raw = lds_addr(&sm.raw[0]), lds_wd = lds_addr(&sm.wd[0]);
  const int ck = 16 * wv + (lane >> 3);  // key of this lane's first K / V copy (second: + 8)
  const uint32_t cofs = 16u * (uint32_t)(lane & 7);
  // V: chunk c of row r at c ^ (bits 0, 1 and 4 of r): the 8 keys of a transposed read all differ
  const uint32_t cofs_v = 16u * (uint32_t)((lane & 7) ^ (((lane >> 3) & 3) | ((wv & 1) << 2)));
  const int wa = wv >> 1;
  const uint16_t* warr = wa == 0 ? ks : wa == 1 ? kb : wa == 2 ? vs : vb;
  const int wkey = 64 * (wv & 1) + lane;
  auto issue_codes = [&](int t, int slot) {
    const int t0 = PT * (tb + min(t, T - 1));
    const uint32_t lb = lds_raw + (uint32_t)slot * (uint32_t)sizeof(PrefillRaw);
    // M0 operands: wave-uniform values, made explicit so that they live in SGPRs
    const uint32_t mk = __builtin_amdgcn_readfirstlane(lb + offsetof(PrefillRaw, k) + 2048u * wv);
    const uint32_t mv = __builtin_amdgcn_readfirstlane(lb + offsetof(PrefillRaw, v) + 2048u * wv);
    const int64_t kr0 = row0 + min(t0 + ck, last_row);
    const int64_t kr1 = row0 + min(t0 + ck + 8, last_row);
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off nt"
                 :: "v"(kc + kr0 * D + cofs), "s"(mk) : "memory");
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off nt"
                 :: "v"(kc + kr1 * D + cofs), "s"(mk + 1024u) : "memory");
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off nt"
                 :: "v"(vc + kr0 * D + cofs_v), "s"(mv) : "memory");
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off nt"
                 :: "v"(vc + kr1 * D + cofs_v), "s"(mv + 1024u) : "memory");
  };
  auto issue_words = [&](int t, int slot) {
    const uint32_t mw = __builtin_amdgcn_readfirstlane(
        lds_wd + (uint32_t)slot * (uint32_t)sizeof(PrefillWords) +
        4u * (uint32_t)(PT * wa + 64 * (wv & 1)));
    const int64_t wr = row0 + min(PT * (tb + min(t, T - 1)) + wkey, last_row);
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %0, off nt"
                 :: "v"(warr + wr * 2), "s"(mw) : "memory");
  };

  // ---- dequantization shares: K of a tile by group A (256 threads, 4 chunks of 16 codes each),
  // V^T by group B (16 slot groups, 4 per wave)
  const int ta = tid & 255;  // thread index within the group
  // (the thread index is re-read through an empty asm in each call, so that the compiler
  // recomputes these addresses in the slot instead of holding them in registers across the loop)
  auto dequant_k = [&](const PrefillRaw& rw, const PrefillWords& wd, int kk) {
    __builtin_amdgcn_s_setprio(2);
    int tr = ta;
    asm volatile("" : "+v"(tr));
    const int dc = tr & 7;  // 16 codes of key (tr >> 3) + 32 i, dims 16 dc .. 16 dc + 15
    const uint32_t gsel = (dc >> 2) ? SEL_HI : SEL_LO;
    uint4 c4[4];
    uint32_t sw[4], zw[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {  // all reads first: one LDS round trip
      const int dk = (tr >> 3) + 32 * i;
      c4[i] = *reinterpret_cast<const uint4*>(rw.k + dk * D + 16 * dc);
      sw[i] = wd.w[0][dk];
      zw[i] = wd.w[1][dk];
    }
    if (RANGE && kk != 0) {  // wave-uniform, rare
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        sw[i] = scale_word(sw[i], exp2_int(-kk));
        zw[i] = scale_word(zw[i], exp2_int(-kk));
      }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int dk = (tr >> 3) + 32 * i;
      const float s = RANGE ? bf16_pick(sw[i], gsel) * k_scale : bf16_pick(sw[i], gsel);
      const float b = RANGE ? bf16_pick(zw[i], gsel) * k_scale : bf16_pick(zw[i], gsel);
      const float z = fmaf(-1024.0f, s, b);  // bias - 1024 scale
      const uint32_t cw[4] = {c4[i].x, c4[i].y, c4[i].z, c4[i].w};
      uint32_t h[8];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const half2_t c01 = codes_1024(cw[j], 0), c23 = codes_1024(cw[j], 1);
        h[2 * j] = pack_h2(fmaf(s, (float)c01.x, z), fmaf(s, (float)c01.y, z));
        h[2 * j + 1] = pack_h2(fmaf(s, (float)c23.x, z), fmaf(s, (float)c23.y, z));
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
  auto dequant_v = [&](const PrefillRaw& rw, const PrefillWords& wd, int kv) {
    __builtin_amdgcn_s_setprio(2);
    int ln = lane;
    asm volatile("" : "+v"(ln));
    const int e = wv - PW / 2, qg = ln >> 4, i = ln & 15;
    const int k0 = 32 * e + 4 * qg;  // T[0..3] = k0 .. k0 + 3, T[4..7] = k0 + 16 .. k0 + 19
    const int skey = k0 + 16 * (i >> 3) + ((i >> 1) & 3);  // T[i / 2]: this lane's source key
    const uint8_t* src = rw.v + skey * D + 8 * (i & 1);
    const int ssw = (skey & 3) | ((skey >> 2) & 4);
    const uint4 s03 = *reinterpret_cast<const uint4*>(&wd.w[2][k0]);
    const uint4 s47 = *reinterpret_cast<const uint4*>(&wd.w[2][k0 + 16]);
    const uint4 z03 = *reinterpret_cast<const uint4*>(&wd.w[3][k0]);
    const uint4 z47 = *reinterpret_cast<const uint4*>(&wd.w[3][k0 + 16]);
    uint32_t sw[8] = {s03.x, s03.y, s03.z, s03.w, s47.x, s47.y, s47.z, s47.w};
    uint32_t zw[8] = {z03.x, z03.y, z03.z, z03.w, z47.x, z47.y, z47.z, z47.w};
    if (RANGE && kv != 0) {  // wave-uniform, rare
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        sw[j] = scale_word(sw[j], exp2_int(-kv));
        zw[j] = scale_word(zw[j], exp2_int(-kv));
      }
    }
#pragma unroll
    for (int g = 0; g < 2; ++g) {  // dims 64 g .. 64 g + 63: quant group g, windows 4 g .. 4 g + 3
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
        reinterpret_cast<uint4*>(sm.vt + d * PT)[(4 * e + qg) ^ i] =
            make_uint4(pack_h2(v[0], v[1]), pack_h2(v[2], v[3]), pack_h2(v[4], v[5]),
                       pack_h2(v[6], v[7]));
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  // ---- operand range of a tile, by group A (256 threads: one scale and one bias word each, waves
  // 0-1 K, 2-3 V), read back by every wave two slots later. A wave whose words put the bound in the
  // window writes IN_WINDOW (two compares and their ballots instead of a reduction over the wave),
  // unless a factor in use (!plain) needs the bound itself.
  int eq = 0;                // exponent of the workgroup's |q| q_scale bound
  int kk = 0, kv = 0;        // K times 2^-kk (q times 2^kk), V times 2^-kv
  int kv_hi = -1000;         // largest kv so far
  int kv_step = 0;           // the accumulators take 2^kv_step
  bool plain = false;        // all of them 0, and 0 for a tile with bounds in the window
  auto range_words = [&](const PrefillWords& wd) {
    const int kv2 = 2 * (wv >> 1);
    return make_uint2(wd.w[kv2][ta & 127], wd.w[kv2 + 1][ta & 127]);
  };
  auto tile_range = [&](int s, uint2 w) {
    const us2_t sc = __builtin_bit_cast(us2_t, w.x & 0x7fff7fffu);
    const us2_t bi = __builtin_bit_cast(us2_t, w.y & 0x7fff7fffu);
    const us2_t m = __builtin_elementwise_max(bi, (us2_t)(sc + (uint16_t)(8 << 7)));  // 256 |scale|
    uint32_t x = max((uint32_t)m.x, (uint32_t)m.y);
    const bool low = !__builtin_amdgcn_ballot_w64(x >= (uint32_t)((126 + WIN_LO) << 7));
    const bool high = __builtin_amdgcn_ballot_w64(x >= (uint32_t)((127 + WIN_HI) << 7));
    if (low || high || !plain)
      x = wave_max_u(x);
    else
      x = IN_WINDOW;
    if (lane == 0) sm.rng[s][wv] = x;
  };
  // A tile's factors, from its bounds r (each kept at 0, or as it is, while the window allows it).
  // While `plain`, a tile with its bounds in the window (in_range) changes nothing: the ordinary
  // tile costs two readlanes and a compare each.
  auto in_range = [&](uint4 r) {
    return in_window(bound_exp(__builtin_amdgcn_readfirstlane(max(r.x, r.y)))) &&
           in_window(bound_exp(__builtin_amdgcn_readfirstlane(max(r.z, r.w))));
  };
  auto tile_factors = [&](uint4 r) __attribute__((always_inline)) {
    const int ek = bound_exp(__builtin_amdgcn_readfirstlane(max(r.x, r.y)));
    const int ev = bound_exp(__builtin_amdgcn_readfirstlane(max(r.z, r.w)));
    // 0 if K's window has it, else K's bound at its near end; then as far down as q's bound
    // asks (never so far that K leaves fp16: |q K| stays below 2^29 in log2 units)
    kk = min(max(0, ek - WIN_HI), max(ek - WIN_LO, -100));
    kk = min(max(min(kk, WIN_HI + 1 - eq), ek - WIN_HI), 100);
    const int was = kv;
    if (!in_window(ev - kv))
      kv = max(in_window(ev) ? 0 : min(max(ev - (WIN_HI - 1), -100), 120), kv_hi - KV_FALL);
    kv_step = kv_hi == -1000 ? 0 : was - kv;  // nothing accumulated before the first tile
    kv_hi = max(kv_hi, kv);
    plain = kk == 0 && kv == 0 && kv_step == 0 && eq <= WIN_HI + 1;
  };

  issue_words(0, 0);
  issue_words(1, 1);
  issue_codes(0, 0);
  issue_codes(1, 1);
  issue_words(2, 2);

  // ---- q of the wave's rows as MFMA B operands, times q_scale 2^kk in fp16
  half8_t qb[2][4];
  // causal bounds of the wave's rows (-1: not a row of the chunk), read back where tiles are masked
  // and for the output
  if (lane < 32) sm.lim[32 * wv + lane] = f0 + lane < R ? base + (f0 + lane) / G : -1;
  const int* lim = sm.lim + 32 * wv + lc;  // row 16 nt + lc of the wave at lim[16 nt]
  // this lane's first q element of N tile nt (row 0 for a row past the chunk); ln is the lane,
  // re-read through an empty asm where the loop reloads q, so that no address lives across it
  auto q_row = [&](int nt, int ln) __attribute__((always_inline)) {
    const int f = f0 + 16 * nt + (ln & 15);
    const int i = f < R ? f / G : 0, head = f < R ? f - i * G : 0;
    return q + (((int64_t)b * Hq + hk * G + head) * L + i) * D + 8 * (ln >> 4);
  };
  us2_t qm = {0, 0};  // bf16 bits of the largest |q|
  auto load_q = [&](int ln, float qs) __attribute__((always_inline)) {
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) {
      const uint16_t* qr = q_row(nt, ln);
      const float f = f0 + 16 * nt + (ln & 15) < R ? qs : 0.0f;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint4 u = *reinterpret_cast<const uint4*>(qr + 32 * j);
        const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          if (RANGE) qm = __builtin_elementwise_max(qm, __builtin_bit_cast(us2_t, w[r] & 0x7fff7fffu));
          qb[nt][j][2 * r] = (_Float16)(bf16_lo(w[r]) * f);
          qb[nt][j][2 * r + 1] = (_Float16)(bf16_hi(w[r]) * f);
        }
      }
    }
  };
  load_q(lane, q_scale);
  if (RANGE) {
    const uint32_t x = wave_max_u(max((uint32_t)qm.x, (uint32_t)qm.y));
    if (lane == 0) sm.qmax[wv] = x;
  }

  f4_t oacc[2][8];
  f4_t lacc[2];  // row sums of P (MFMA layout: all four values of a lane hold its row's sum)
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
  // units); V^T dim 16 dt + lc, slots 32 e + 8 lq4 .. + 7 at vfrag[e] + 256 dt
  const uint4* kfrag[4];
  const uint4* vfrag[PE];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    kfrag[j] = reinterpret_cast<const uint4*>(sm.k) + 16 * lc + ((4 * j + lq4) ^ lc);
    vfrag[j] = reinterpret_cast<const uint4*>(sm.vt) + 16 * lc + ((4 * j + lq4) ^ lc);
  }
  f4_t c[2][PMT];     // scores, c[nt][mt]: keys 16 mt + 4 lq4 + r of row 16 nt + lc (log2 units)
  half8_t pw[2][PE];  // P in fp16, per N tile and k-step
  // Q.K^T of both N tiles from one read of each K fragment, relative to the rows' running
  // maxima (0 before the first): the accumulators start at -mref
  int kq = 0;  // the factor 2^kq that qb holds
  auto qk = [&]() {
    __builtin_amdgcn_s_setprio(0);
    if (RANGE && kk != kq) {  // wave-uniform, rare: this tile's K has another factor
      kq = kk;
      int ln = lane;
      asm volatile("" : "+v"(ln));
      load_q(ln, q_scale * exp2_int(kq));
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
#pragma unroll
        for (int dt = 0; dt < 8; ++dt) oacc[nt][dt] *= alpha;
        const float shift = bump ? tmax : 0.0f;  // new reference minus the one the scores hold
#pragma unroll
        for (int mt = 0; mt < PMT; ++mt) c[nt][mt] -= shift;
      }
#pragma unroll
      for (int e = 0; e < PE; ++e) {
        half2_t ph[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int hh = j >> 1, r = 2 * (j & 1);
          ph[j] = half2_t{(_Float16)__builtin_amdgcn_exp2f(c[nt][2 * e + hh][r]),
                          (_Float16)__builtin_amdgcn_exp2f(c[nt][2 * e + hh][r + 1])};
        }
        pw[nt][e] = __builtin_bit_cast(half8_t, ph);
        asm volatile("" : "+v"(pw[nt][e]));  // P is made in this slot, not sunk into P.V's
      }
    }
  };
  // P.V of both N tiles from one read of each V^T fragment, and the rows' sums of P:
  // out^T[16 dt + 4 lq4 + r][row 16 nt + lc] += V^T[dims][slots] P^T[slots][rows]
  int kv_acc = 0;  // the factor 2^-kv_acc that the accumulators hold
  auto pv = [&](int snext) {  // ends with the factors of the next tile (its range in sm.rng[snext])
    __builtin_amdgcn_s_setprio(0);
    kv_acc = kv;
    uint4 rnext;
    if (RANGE) rnext = *reinterpret_cast<const uint4*>(sm.rng[snext]);
    bool ordinary = false;
    // fragments four dims tiles ahead (half a k-step), as in qk: step u = (k-step u / 2, dim
    // tiles 4 (u % 2) .. + 3)
    uint4 fv[2][4];
    if (RANGE && kv_step != 0) {  // wave-uniform, rare: the tile's V has another factor
#pragma unroll
      for (int nt = 0; nt < 2; ++nt)
#pragma unroll
        for (int dt = 0; dt < 8; ++dt)
#pragma unroll
          for (int r = 0; r < 4; ++r) oacc[nt][dt][r] = ldexpf(oacc[nt][dt][r], kv_step);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) fv[0][j] = vfrag[0][256 * j];
#pragma unroll
    for (int u = 0; u < 2 * PE; ++u) {
      if (u + 1 < 2 * PE) {
        const int e1 = (u + 1) >> 1, d1 = 4 * ((u + 1) & 1);
#pragma unroll
        for (int j = 0; j < 4; ++j) fv[(u + 1) & 1][j] = vfrag[e1][256 * (d1 + j)];
      }
      __builtin_amdgcn_sched_barrier(0);
      const int e = u >> 1, d0 = 4 * (u & 1);
      if (RANGE && u == 3) ordinary = in_range(rnext);  // beside the MFMAs in flight
      if (u & 1) {  // row sums of this k-step's P: a ones A operand (every output row the sum)
#pragma unroll
        for (int nt = 0; nt < 2; ++nt)
          lacc[nt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ones8, pw[nt][e], lacc[nt], 0, 0, 0);
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint4 a = fv[u & 1][j];  // dim 16 (d0 + j) + lc
        const half8_t ah = words_as_h8(a.x, a.y, a.z, a.w);
#pragma unroll
        for (int nt = 0; nt < 2; ++nt)
          oacc[nt][d0 + j] =
              __builtin_amdgcn_mfma_f32_16x16x32_f16(ah, pw[nt][e], oacc[nt][d0 + j], 0, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if (RANGE && !(ordinary && plain)) tile_factors(rnext);
  };

  // ---- prologue: tile 0 and the words of tile 1 landed (outstanding: tile 1's codes, tile 2's
  // words), tile 0's range, K(0) dequantized
  asm volatile("s_waitcnt vmcnt(5)" ::: "memory");
  __syncthreads();
  if (RANGE) {
    if (grp_a) tile_range(0, range_words(sm.wd[0]));
    __syncthreads();
    const uint4 a = *reinterpret_cast<const uint4*>(sm.qmax);
    const uint4 e = *reinterpret_cast<const uint4*>(sm.qmax + 4);
    const uint32_t m = max(max(max(a.x, a.y), max(a.z, a.w)), max(max(e.x, e.y), max(e.z, e.w)));
    // a product of two values below 2^a and 2^b is below 2^(a + b)
    eq = bound_exp(__builtin_amdgcn_readfirstlane(m)) +
         bound_exp((__float_as_uint(q_scale) & 0x7fffffffu) >> 16);
    tile_factors(*reinterpret_cast<const uint4*>(sm.rng[0]));
  }
  if (grp_a) dequant_k(sm.raw[0], sm.wd[0], kk);
  __syncthreads();

  // The two halves run their own loops (wave-uniform branch): each wave passes the same four
  // barriers per tile. Tiles 0 .. Tact - 1 hold keys visible to the wave's rows; past them the
  // wave keeps only its copy, range and dequantization duties. (Two loops rather than a condition
  // per phase, so that the scores and P are not live across the loop's back edge.) The words run
  // a tile ahead of the codes, so that a tile's range and factors are taken at the ends of the
  // matrix slots before it is dequantized (which the other half's vector phase outlasts) and not
  // in the dequantization slots, which set the pace: those made the loop 8% slower.
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
      uint2 rw;                                         // slot 4t
      if (RANGE) rw = range_words(sm.wd[w1]);
      qk();
      if (RANGE) tile_range((t + 1) & 1, rw);
      __syncthreads();
      issue_codes(t + 2, t & 1);                        // slot 4t + 1: into t's slots
      issue_words(t + 3, w0);
      softmax(t0, t0 + PT - 1 <= lim_lo);
      __syncthreads();
      pv((t + 1) & 1);                                  // slot 4t + 2
      asm volatile("s_waitcnt vmcnt(5)" ::: "memory");  // codes of t + 1, words of t + 2 landed
      __syncthreads();
      if (t + 1 < T) dequant_k(sm.raw[(t + 1) & 1], sm.wd[w1], kk);  // slot 4t + 3
      next_words();
      __syncthreads();
    }
    for (; t < T; ++t) {
      if (RANGE) tile_range((t + 1) & 1, range_words(sm.wd[w1]));
      __syncthreads();
      issue_codes(t + 2, t & 1);
      issue_words(t + 3, w0);
      __syncthreads();
      if (RANGE) tile_factors(*reinterpret_cast<const uint4*>(sm.rng[(t + 1) & 1]));
      asm volatile("s_waitcnt vmcnt(5)" ::: "memory");
      __syncthreads();
      if (t + 1 < T) dequant_k(sm.raw[(t + 1) & 1], sm.wd[w1], kk);
      next_words();
      __syncthreads();
    }
  } else {
    int t = 0;
    for (; t < Tact; ++t) {
      const int t0 = PT * (tb + t);
      dequant_v(sm.raw[t & 1], sm.wd[w0], kv);          // slot 4t
      __syncthreads();
      qk();                                             // slot 4t + 1
      __syncthreads();
      issue_codes(t + 2, t & 1);                        // slot 4t + 2
      issue_words(t + 3, w0);
      softmax(t0, t0 + PT - 1 <= lim_lo);
      asm volatile("s_waitcnt vmcnt(5)" ::: "memory");
      __syncthreads();
      pv((t + 1) & 1);                                  // slot 4t + 3
      next_words();
      __syncthreads();
    }
    for (; t < T; ++t) {
      dequant_v(sm.raw[t & 1], sm.wd[w0], kv);
      __syncthreads();
      __syncthreads();
      issue_codes(t + 2, t & 1);
      issue_words(t + 3, w0);
      asm volatile("s_waitcnt vmcnt(5)" ::: "memory");
      __syncthreads();
      if (RANGE) tile_factors(*reinterpret_cast<const uint4*>(sm.rng[(t + 1) & 1]));
      next_words();
      __syncthreads();
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the clamped copies past the end

  // ---- output rows: acc / l, V's factor taken out; of a part of the block's tiles in fp32, with
  // the row's (m, l), for prefill_merge_kernel
  const bool whole = !SPLIT || T == T_blk;
  const int64_t slot = 2 * (int64_t)x + (tb == 0);
#pragma unroll
  for (int nt = 0; nt < 2; ++nt) {
    const float l = lacc[nt][0];
    const int last = lim[16 * nt];
    if (last >= 0) {
      const float inv = l > 0.0f ? 1.0f / l : 0.0f;
      const int wrow = 32 * wv + 16 * nt + lc;
      const int i = last - base, head = pb * PROWS + wrow - i * G;
      uint16_t* orow = out + (((int64_t)b * Hq + hk * G + head) * L + i) * D;
      float* prow = sp.part_o + (slot * PROWS + wrow) * D;
#pragma unroll
      for (int dt = 0; dt < 8; ++dt) {
        f4_t o = oacc[nt][dt] * inv;
        if (RANGE && kv_acc != 0) {  // wave-uniform, rare
#pragma unroll
          for (int r = 0; r < 4; ++r) o[r] = ldexpf(o[r], kv_acc);
        }
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
// heads, 21 parts per row) took 20.4 us with one group per row and 8 rows per workgroup.
__global__ __launch_bounds__(256) void prefill_merge_kernel(uint16_t* __restrict__ out, int n, int L,
                                                            int Hkv, int G, PrefillSplit sp) {
  __shared__ f4_t sh_acc[2][4][32];
  __shared__ float2 sh_ml[2][4];
  const int hk = blockIdx.y % Hkv, b = blockIdx.y / Hkv;
  const int R = L * G, base = n - L;
  const int pb = blockIdx.x / (PROWS / 2);
  const int tr = threadIdx.x >> 7, grp = (threadIdx.x >> 5) & 3, ln = threadIdx.x & 31;
  const int wrow = 2 * (blockIdx.x % (PROWS / 2)) + tr;
  int u0 = 0;
  for (int j = 0; j < pb; ++j) u0 += prefill_tiles(j, R, sp.g, base);
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
      const float w = ml.y > 0.0f ? exp2_nonpos(ml.x - M) * ml.y : 0.0f;
      if (w > 0.0f) acc += o * w;
      den += w;
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
    const float w = ml.y > 0.0f ? exp2_nonpos(ml.x - mx) : 0.0f;
    if (w > 0.0f) acc += sh_acc[tr][g][ln] * w;
    den += w * ml.y;
  }
  const f4_t o = acc * (den > 0.0f ? 1.0f / den : 0.0f);
  const int i = (int)fdiv_u((uint32_t)f, sp.g), head = f - i * G;
  const uint32_t lo = (uint32_t)f32_to_bf16(o[0]) | ((uint32_t)f32_to_bf16(o[1]) << 16);
  const uint32_t hi = (uint32_t)f32_to_bf16(o[2]) | ((uint32_t)f32_to_bf16(o[3]) << 16);
  *reinterpret_cast<uint2*>(out + (((int64_t)b * Hkv * G + hk * G + head) * L + i) * D + 4 * ln) =
      make_uint2(lo, hi);
}

// How the blocks of a chunk are dealt to workgroups: whole, one block each (tiles 0), or each KV
// head's tiles, block after block, in equal shares of `tiles` for as many workgroups as fill the
// CUs. Costs in tiles (3.7-4.2 us each, by clock): whole blocks go round by round, longest first;
// a share pays about two per block that it touches (q, the first copies, the output rows) and the
// partial rows with their merge launch about six. Measured, us per 32/8 chunk, whole against
// split: 64 rows at 82,735 keys 2,068 / 137, 1,024 rows at 83,695 keys 2,138 / 1,440; 48/8, 512
// rows at 8,193 keys, 237 / 147, 2,048 rows at 62,048 keys (1.5 rounds whole) 3,908 / 3,255; and
// where whole stays better, 2,048 rows at 2,112 keys (17 tiles at most) 79 / 120.
constexpr int SEGMENT_TILES = 2;
constexpr int MERGE_TILES = 6;
constexpr int MIN_SHARE = 4;
PrefillSplit plan_split(int64_t B, int64_t Hkv, int64_t G, int64_t L, int64_t n, int cus) {
  const int R = (int)(L * G), base = (int)(n - L), npb = (R + PROWS - 1) / PROWS;
  PrefillSplit sp{make_fastdiv((uint32_t)G), npb, 0, nullptr, nullptr};
  const int64_t S = cus / (B * Hkv);
  if (S < 2 || npb > 4 * S) return sp;  // no CUs to spare; the last round matters little
  int64_t total = 0, rounds = 0;
  for (int pb = 0; pb < npb; ++pb) {
    const int t = prefill_tiles(pb, R, sp.g, base);
    total += t;
    if ((npb - 1 - pb) % S == 0) rounds += t;
  }
  const int64_t tiles = std::max<int64_t>(MIN_SHARE, (total + S - 1) / S);
  const int64_t touched = 2 + (tiles - 2) / prefill_tiles(0, R, sp.g, base);  // block 0: shortest
  if (33 * (tiles + SEGMENT_TILES * touched + MERGE_TILES) > 32 * rounds) return sp;  // 3% or more
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
  // scores in log2 units; the range variant leaves q exact (bf16 times a power of two) and gives K,
  // which is rounded to fp16 anyway, the scale's mantissa in [0.5, 1)
  const float qk = scale * 1.4426950408889634f;
  int se = 0;
  const float sm = std::frexp(qk, &se);
  // groupings that the verify kernel served before keep its range (see the top of the file)
  const bool range = !(G == 1 || G == 2 || G == 4 || G == 8);
  auto* kern = range ? (sp.tiles ? q8_prefill_kernel<true, true> : q8_prefill_kernel<true, false>)
                     : (sp.tiles ? q8_prefill_kernel<false, true> : q8_prefill_kernel<false, false>);
  kern<<<dim3((unsigned)wgs), dim3(64 * PW), 0, st>>>(
      q, kc, ks, kb, vc, vs, vb, out, cap, (int)n, (int)L, (int)Hkv, (int)G, (int)npb,
      sp, range ? ldexpf(1.0f, se) : qk, range ? sm : 1.0f);
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
