// Decode step (one new token per sequence) against a static KV cache: RoPE + cache append, and
// grouped-query attention of the new token over the cached positions.  Both are HBM-bound: the
// attention kernel reads every cached K and V element of a sequence exactly once.
//
// Cache layout (bf16, head_dim 128, `capacity` positions per sequence slot, capacity % 32 == 0):
//   K cache [slots][kv_heads][capacity][128]        - a position's 128 dims are contiguous
//   V cache [slots][kv_heads][capacity/8][128][8]   - 8 consecutive positions of one dim are contiguous
// Both layouts are what the 16x16x32 MFMA operands want as 16-byte per-lane loads straight from
// global memory (no LDS staging, no transposes):
//   scores^T = K Q^T : A = K rows (lane: one position, 8 consecutive dims)
//   out      = P V   : B = V     (lane: one dim, 8 consecutive positions)
#include "dfhip_pairs.h"

namespace {

constexpr int HD = 128;           // head dim
constexpr int DEC_THREADS = 256;  // 4 waves
constexpr int CHUNK = 32;         // positions per softmax step of a wave
constexpr int COMPUTE_UNITS = 256;
constexpr int MAX_GROUP = 16;     // query heads per kv head (rows of the MFMA tile)

DFHIP_DEVICE f32x4 mfma16(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// The rotation of one pair (x[i], x[i + 64]) of a head by the angle of its position: the one formula of both kernels
// below, so that they round alike.
// (The fused multiply-adds are spelt out: left to the compiler the two kernels could contract the expressions
// differently.)
DFHIP_DEVICE void rotate_pair(float lo, float hi, float c, float s, bf16_t& out_lo, bf16_t& out_hi) {
  out_lo = static_cast<bf16_t>(__builtin_fmaf(lo, c, -(hi * s)));
  out_hi = static_cast<bf16_t>(__builtin_fmaf(hi, c, lo * s));
}
DFHIP_DEVICE uint16_t bits_of(bf16_t v) { return __builtin_bit_cast(uint16_t, v); }

struct KVFrags {
  bf16x8 k[2][4];   // [set][k-step]
  bf16x8 v[8];      // [dim block]
};

// Four dims of a head of the output: item `it` is head it / 32, dims 4 (it % 32) .. + 3.
DFHIP_DEVICE void store_row(uint16_t* out_row, int it, f32x4 num, float den) {
#pragma unroll
  for (int e = 0; e < 4; ++e) out_row[4 * it + e] = static_cast<uint16_t>(f32_to_bf16_bits(num[e] / den));
}

// 16-byte words of a part's block in the workspace: the sums of `group` heads, then one word (maximum, sum) per head.
__host__ __device__ constexpr int part_block(int group) { return group * (HD / 4 + 1); }

// Parts of a sequence of `len` positions where the launch has `parts` workgroups for each: at least 256 positions (two
// chunks per wave) a part, and at least three parts, since the meeting costs about 3 us.  Shorter sequences stay whole:
// the bits and the time of an uncut launch.  [us, uncut / cut by the
// capacity alone / by the length: 2 sequences in a cache of 8192 positions, of 33 6.4 / 13.4 / 6.5, of 512 9.8 / 14.3 /
// 9.9, of 2048 27 - 31 / 16.8 / 11.6, of 8192 111 / 21.9 / 20.8]
DFHIP_DEVICE int sequence_parts(int len, int parts) {
  if (len < 3 * 256) return 1;
  return len / 256 < parts ? len / 256 : parts;
}

// What a workgroup is to work on.
struct Share { int token, kvh, part, slot, len; };

// Workgroup `block` of a launch.  Of more workgroups than compute units the longest sequences come first (ties in the order of the
// tokens), all parts of one before the next sequence, so that what runs at the end is short and what shares a unit differs.
// A wave ranks the sequences by itself: the length of the `rank`-th longest is the largest that more than `rank` tokens reach,
// found bit by bit, then the token is counted off among those of that length.  Up to 64 J tokens.
// Sequences of one length, launches of few workgroups and of many tokens (whose workgroups even out by themselves) keep the order
// of the tokens, and the first parts of all tokens come before the second ones, so that the parts that every sequence uses lie
// on all XCDs; so do those whose number of kv heads is no multiple of the XCDs.  (The parts of a token first, the only
// workgroups with work of 8 short sequences are every eighth one, on one XCD: 512 positions 20.2 us, so 12.2.)
// [us, order of the tokens -> longest first, sequences of 1/4 .. 1 of the capacity in any order: 20 of 4096 positions 47 -> 43, 36
// of 4096 72 -> 70, 24 of 4096 55 -> 51, 16 of 8192 67 -> 63; whole ones: 40 of 4096 79 -> 76, 64 of 2048 67 -> 62, 128 of 2048 125 -> 107,
// 100 of 1024 59 -> 50; all of one length, level (200 of 1024 140 -> 142).  Ranked with fewer workgroups than units: 12 of 512
// 11.9 -> 12.8; the first parts of all tokens first, ranked: 16 of 8192 68, 24 of 4096 54]
template <bool SPLIT, int J>
DFHIP_DEVICE Share share_of(int block, const int32_t* __restrict__ slots, const int32_t* __restrict__ lengths, int tokens,
                            int kv_heads, int parts, int capacity) {
  const int lane = threadIdx.x & 63;
  int own[J], own_slot[J], len[J];
  bool same = true;
#pragma unroll
  for (int j = 0; j < J; ++j) {
    const int t = 64 * j + lane < tokens ? 64 * j + lane : 0;
    own[j] = lengths[t];
    own_slot[j] = slots[t];
  }
  const int first = __builtin_amdgcn_readfirstlane(own[0]);
#pragma unroll
  for (int j = 0; j < J; ++j) {
    same &= own[j] == first;
    len[j] = 64 * j + lane >= tokens ? -1 : own[j] < 0 ? 0 : own[j] < capacity ? own[j] : capacity;
  }
  same = __all(same);
  const bool together = SPLIT && !same && kv_heads % 8 == 0;    // the parts of a token
  const int per_part = together ? kv_heads : tokens * kv_heads;
  int rank = 0;
  if (together) {
    rank = block / (kv_heads * parts);
    block -= rank * kv_heads * parts;
  }
  const int part = SPLIT ? block / per_part : 0;
  block -= part * per_part;
  if (!together) rank = block / kv_heads;
  const int kvh = together ? block : block - rank * kv_heads;
  int token = rank;
  if (!same) {
    auto reach = [&](int least) {              // tokens of at least this length
      int n = 0;
#pragma unroll
      for (int j = 0; j < J; ++j) n += __popcll(__ballot(len[j] >= least));
      return n;
    };
    int length = 0;
    for (int bit = 31 - __clz(capacity); bit >= 0; --bit)
      if (reach(length | 1 << bit) > rank) length |= 1 << bit;
    int before = rank - reach(length + 1);     // tokens of this length that come first
#pragma unroll
    for (int j = 0; j < J; ++j) {
      const uint64_t equal = __ballot(len[j] == length);
      const int n = __popcll(equal);
      const int at = __builtin_amdgcn_mbcnt_hi((uint32_t)(equal >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)equal, 0));
      const uint64_t found = __ballot(len[j] == length && at == before);
      if (before >= 0 && before < n) token = 64 * j + __builtin_ctzll(found);
      before -= n;
    }
    token = __builtin_amdgcn_readfirstlane(token);
  }
  int slot_of = own_slot[0], len_of = own[0];
#pragma unroll
  for (int j = 1; j < J; ++j)
    if (token >= 64 * j) slot_of = own_slot[j], len_of = own[j];
  return {token, kvh, part, __builtin_amdgcn_readlane(slot_of, token & 63), __builtin_amdgcn_readlane(len_of, token & 63)};
}

// One workgroup per (token, kv head).  Wave w takes the chunks w, w+4, ... of 32 positions.
// MFMA row i of a score tile is mapped to position 8*(i/4) + i%4 (+4 for the second tile of the
// chunk), so that after the two tiles lane (head = lane%16, g = lane/16) holds the scores of its
// head for positions 8g .. 8g+7 - which is exactly the A-operand fragment of P for the P V product.
//
// APPEND: the workgroup first does what rope_kv_append_kernel does for its share of the token - `q` is the
// token's row of the q / k / v product, the group's query heads are rotated in registers, the kv head's new key
// is rotated and, with the new value, written to the caches at position lengths[t] - 1 - and then attends.  The
// wave whose chunks include that position does the append and keeps the new key and value in LDS for its own
// fragments of that position, which it patches when it gets there (no read of what was just written and no
// barrier: the wave that wrote the LDS words is the one that reads them; the other three waves only rotate their
// copies of the query heads).
//
// SPLIT: a (token, kv head) pair has `parts` workgroups, for launches with too few pairs to fill the chip (attention_parts
// says when), of which the token's length takes as many as pay (sequence_parts); the others end at once.  A part leaves
// its unnormalised sums, maximum and sum of exponentials in `partials` ([pair][part][part_block(group)] words of 16
// bytes), counts itself in and is done; the part that arrives last combines them, in the same order whoever that is.
template <bool APPEND, bool SPLIT>
DFHIP_DEVICE void decode_attention(int block, bool ordered, int tokens, const uint16_t* __restrict__ q, int64_t ld_q, uint16_t* __restrict__ kc,
                                   uint16_t* __restrict__ vc, const int32_t* __restrict__ slots,
                                   const int32_t* __restrict__ lengths, uint16_t* __restrict__ out, int64_t ld_out,
                                   int kv_heads, int group, int num_slots, int capacity, float scale_log2,
                                   const float* __restrict__ cos_t, const float* __restrict__ sin_t, int table_rows,
                                   int parts, float* __restrict__ partials, int* __restrict__ arrivals) {
  // partial results of the four waves, sized by the launch for the real group (a workgroup that asks for
  // little LDS leaves room for a GEMM workgroup of the other nano-batch on the same CU)
  extern __shared__ __attribute__((aligned(16))) float combine_lds[];
  float* const o_lds = combine_lds;                       // [4][group][HD]
  float* const m_lds = combine_lds + 4 * group * HD;      // [4][group]
  float* const l_lds = m_lds + 4 * group;                 // [4][group]
  Share my;
  if (ordered && tokens > 1 && tokens <= 64) {
    my = share_of<SPLIT, 1>(block, slots, lengths, tokens, kv_heads, parts, capacity);
  } else if (ordered && tokens > 1 && tokens <= 256) {
    my = share_of<SPLIT, 4>(block, slots, lengths, tokens, kv_heads, parts, capacity);
  } else {
    my.part = SPLIT ? block / (tokens * kv_heads) : 0;
    block -= my.part * tokens * kv_heads;
    my.token = block / kv_heads;
    my.kvh = block - my.token * kv_heads;
    my.slot = slots[my.token];
    my.len = lengths[my.token];
  }
  const int part = my.part, t = my.token, kvh = my.kvh, pair = t * kv_heads + kvh;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int hq = lane & 15, g = lane >> 4;
  const int slot = my.slot;
  int len = my.len;
  uint16_t* out_row = out + (int64_t)t * ld_out + (int64_t)kvh * group * HD;
  if (slot < 0 || slot >= num_slots || len < 1) {   // nothing to attend to: defined output, no access
    if (part == 0)
      for (int idx = tid; idx < group * HD; idx += DEC_THREADS) out_row[idx] = 0;
    return;
  }
  const int pos = len - 1;                     // APPEND: the new token's position (before the clamp below)
  const bool append = APPEND && pos < capacity;
  len = len < capacity ? len : capacity;
  const int used = SPLIT ? sequence_parts(len, parts) : 1;   // workgroups that share this pair
  if (SPLIT && part >= used) return;
  const int64_t head_base = ((int64_t)slot * kv_heads + kvh) * capacity * HD;
  uint16_t* kbase = kc + head_base;
  uint16_t* vbase = vc + head_base;
  const int trow = pos < table_rows ? pos : table_rows - 1;
  const uint16_t* const token_row = q + (int64_t)t * ld_q;                  // APPEND: q | k | v of the token
  uint16_t* const new_k = reinterpret_cast<uint16_t*>(l_lds + 4 * group);   // [HD], APPEND only
  uint16_t* const new_v = new_k + HD;                                        // [HD]

  bf16x8 qf[4];
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) {
    if (hq < group) {
      qf[ks] = *reinterpret_cast<const bf16x8*>(q + (int64_t)t * ld_q + (int64_t)(kvh * group + hq) * HD + 32 * ks + 8 * g);
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) qf[ks][e] = static_cast<bf16_t>(0.0f);
    }
  }
  // SPLIT: a K load takes eight whole 128-byte lines, two neighbouring lanes 32 bytes of one; bits 0, 5, 4 of the lane are the
  // 16-byte chunk of the line, 1, 2, 3 bits 1, 3, 4 of the row, and load (a, s, half) gives bits 0 and 2 of it and the half.
  // With a row per lane, as the fragments have it, a compute unit takes in 34 GB/s of keys at most, which is what few
  // workgroups with a part each wait for [us, 2 x 20 sequences of 1/4 .. 1 of 4096 positions: 92 -> 83].  Whole sequences keep
  // every unit busy at the rate of the memory, and are 1 % slower that way (2 x 128 of 2048).
  const int krow = 8 * (hq >> 2) + (hq & (SPLIT ? 2 : 3));
  const uint16_t* k_lane = kbase + (int64_t)krow * HD + 8 * (SPLIT ? (lane & 1) + 4 * (g & 1) + 2 * (g >> 1) : g);
  const uint16_t* v_lane = vbase + ((int64_t)g * HD + hq) * 8;

  // every cached element is read once per step and by nobody else: non-temporal loads, which do not displace
  // what the caches hold for the kernels that run beside this one (128 sequences x 2048 positions: 187 -> 158 us)
  auto load = [&](KVFrags& f, int chunk) {
    const uint16_t* kp = k_lane + (int64_t)chunk * (CHUNK * HD);
    const uint16_t* vp = v_lane + (int64_t)chunk * (CHUNK * HD);
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int ks = 0; ks < 4; ++ks)
        f.k[s][ks] = __builtin_nontemporal_load(reinterpret_cast<const bf16x8*>(
            SPLIT ? kp + (4 * s + (ks & 1)) * HD + 64 * (ks >> 1) : kp + s * 4 * HD + 32 * ks));
#pragma unroll
    for (int nb = 0; nb < 8; ++nb) f.v[nb] = __builtin_nontemporal_load(reinterpret_cast<const bf16x8*>(vp + nb * 16 * 8));
  };

  // SPLIT: two loads -> two fragments (lane: row hq, chunk 4 ks + g): neighbouring lanes exchange one of their two pieces, then
  // lanes 16 apart
  auto deal = [&](bf16x8& first, bf16x8& second) {
    u32x4 x = __builtin_bit_cast(u32x4, first), y = __builtin_bit_cast(u32x4, second);
    const bool odd = lane & 1;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      constexpr int SWAP = 0xB1;                 // quad_perm [1, 0, 3, 2]
      const int from_x = __builtin_amdgcn_update_dpp((int)x[e], (int)x[e], SWAP, 0xF, 0xF, true);
      const int from_y = __builtin_amdgcn_update_dpp((int)y[e], (int)y[e], SWAP, 0xF, 0xF, true);
      const auto both = __builtin_amdgcn_permlane16_swap(odd ? (uint32_t)from_y : x[e], odd ? y[e] : (uint32_t)from_x, false, false);
      x[e] = both[0];
      y[e] = both[1];
    }
    first = __builtin_bit_cast(bf16x8, x);
    second = __builtin_bit_cast(bf16x8, y);
  };

  float m = -INFINITY, l = 0.0f;
  f32x4 o[8];
#pragma unroll
  for (int nb = 0; nb < 8; ++nb) o[nb] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

  auto step = [&](KVFrags& f, int c) {
    if constexpr (SPLIT)
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int ks = 0; ks < 4; ks += 2) deal(f.k[s][ks], f.k[s][ks + 1]);
    if (APPEND && append && c == pos / CHUNK) {
      // the chunk of the new token: its key row and value column come from LDS, whatever the loads returned
      const int krow_pos = c * CHUNK + 8 * (hq >> 2) + (hq & 3);
#pragma unroll
      for (int s = 0; s < 2; ++s)
        if (krow_pos + 4 * s == pos) {
#pragma unroll
          for (int ks = 0; ks < 4; ++ks) f.k[s][ks] = *reinterpret_cast<const bf16x8*>(new_k + 32 * ks + 8 * g);
        }
      if (pos / 8 == c * (CHUNK / 8) + g) {
#pragma unroll
        for (int nb = 0; nb < 8; ++nb) {
          const uint16_t v = new_v[nb * 16 + hq];
#pragma unroll
          for (int e = 0; e < 8; ++e)
            if (e == (pos & 7)) f.v[nb][e] = __builtin_bit_cast(bf16_t, v);
        }
      }
    }
    if ((c + 1) * CHUNK > len) {
      // the last chunk of the sequence: positions from len on may hold anything (a cache that was never
      // written there, NaN bit patterns included) and their probability 0 would not silence a NaN in the
      // product, so their V elements are zeroed.  Their K rows need nothing: their scores are replaced below.
#pragma unroll
      for (int nb = 0; nb < 8; ++nb)
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (c * CHUNK + 8 * g + e >= len) f.v[nb][e] = static_cast<bf16_t>(0.0f);
    }
    f32x4 s1 = {0.0f, 0.0f, 0.0f, 0.0f}, s2 = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      s1 = mfma16(f.k[0][ks], qf[ks], s1);
      s2 = mfma16(f.k[1][ks], qf[ks], s2);
    }
    // this lane: head hq, positions c*32 + 8g + 0..7
    const int p_first = c * CHUNK + 8 * g;
    float sc[8];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      sc[r] = (p_first + r < len) ? s1[r] * scale_log2 : -INFINITY;
      sc[4 + r] = (p_first + 4 + r < len) ? s2[r] * scale_log2 : -INFINITY;
    }
    float cmax = sc[0];
#pragma unroll
    for (int r = 1; r < 8; ++r) cmax = fmaxf(cmax, sc[r]);
    cmax = fmaxf(cmax, __shfl_xor(cmax, 16, 64));
    cmax = fmaxf(cmax, __shfl_xor(cmax, 32, 64));
    const float m_new = fmaxf(m, cmax);       // finite: every chunk has at least one valid position
    const float alpha = exp2f(m - m_new);
    float psum = 0.0f;
    bf16x8 pf;
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      const float p = exp2f(sc[r] - m_new);
      psum += p;
      pf[r] = static_cast<bf16_t>(p);
    }
    psum += __shfl_xor(psum, 16, 64);
    psum += __shfl_xor(psum, 32, 64);
    l = l * alpha + psum;
    m = m_new;
    // the accumulators of this lane belong to heads 4g + r: their factors live in lanes 4g + r
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float a = __shfl(alpha, 4 * g + r, 64);
#pragma unroll
      for (int nb = 0; nb < 8; ++nb) o[nb][r] *= a;
    }
#pragma unroll
    for (int nb = 0; nb < 8; ++nb) o[nb] = mfma16(pf, f.v[nb], o[nb]);
  };

  // two fragment sets in turn: the loads of the next chunk are in flight while one is multiplied
  const int all_chunks = (len + CHUNK - 1) / CHUNK;
  const int chunk0 = SPLIT ? (int)((int64_t)all_chunks * part / used) : 0;
  const int chunks = SPLIT ? (int)((int64_t)all_chunks * (part + 1) / used) : all_chunks;   // end of this part's
  KVFrags fa, fb;
  if (chunk0 + wave < chunks) load(fa, chunk0 + wave);
  // (the first chunk's loads are on their way while the query heads are rotated)
  if (APPEND) {
    // the lane's fragments ks and ks + 2 hold the two halves of the pairs i = 32 ks + 8 g + e, ks = 0, 1
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int i = 32 * ks + 8 * g + e;
        const float c = cos_t[trow * (HD / 2) + i], s = sin_t[trow * (HD / 2) + i];
        bf16_t lo, hi;
        rotate_pair(static_cast<float>(qf[ks][e]), static_cast<float>(qf[ks + 2][e]), c, s, lo, hi);
        qf[ks][e] = lo;
        qf[ks + 2][e] = hi;
      }
    // The wave whose chunks include the new position appends: lane i rotates the pair (i, i + 64) of the new key
    // and copies two elements of the new value - to the caches for the later steps, to LDS for this wave's own
    // fragments of that position (the same wave writes and reads them: no barrier).
    const int pos_chunk = pos / CHUNK;
    if (append && pos_chunk >= chunk0 && pos_chunk < chunks && wave == (pos_chunk - chunk0) % 4) {
      const int q_heads = kv_heads * group;
      const uint16_t* k_in = token_row + (int64_t)(q_heads + kvh) * HD;
      const uint16_t* v_in = token_row + (int64_t)(q_heads + kv_heads + kvh) * HD;
      bf16_t lo, hi;
      rotate_pair(bf16_bits_to_f32(k_in[lane]), bf16_bits_to_f32(k_in[lane + 64]), cos_t[trow * (HD / 2) + lane],
                  sin_t[trow * (HD / 2) + lane], lo, hi);
      new_k[lane] = bits_of(lo);
      new_k[lane + 64] = bits_of(hi);
      kbase[(int64_t)pos * HD + lane] = bits_of(lo);
      kbase[(int64_t)pos * HD + lane + 64] = bits_of(hi);
#pragma unroll
      for (int d = lane; d < HD; d += 64) {
        const uint16_t v = v_in[d];
        new_v[d] = v;
        vbase[((int64_t)(pos >> 3) * HD + d) * 8 + (pos & 7)] = v;
      }
    }
  }
  for (int c = chunk0 + wave; c < chunks; c += 8) {
    if (c + 4 < chunks) load(fb, c + 4);
    step(fa, c);
    if (c + 4 < chunks) {
      if (c + 8 < chunks) load(fa, c + 8);
      step(fb, c + 4);
    }
  }

  // combine the four waves
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int h = 4 * g + r;
    if (h < group) {
#pragma unroll
      for (int nb = 0; nb < 8; ++nb) o_lds[(wave * group + h) * HD + nb * 16 + hq] = o[nb][r];
    }
  }
  if (g == 0 && hq < group) {
    m_lds[wave * group + hq] = m;
    l_lds[wave * group + hq] = l;
  }
  __syncthreads();
  // a thread combines four dims of a head: items (head, dims 4 d .. 4 d + 3)
  const int items = group * (HD / 4);
  f32x4* const blocks = SPLIT ? reinterpret_cast<f32x4*>(partials) + (int64_t)pair * parts * part_block(group) : nullptr;
  for (int it = tid; it < items; it += DEC_THREADS) {
    const int h = it >> 5;
    float mm = m_lds[h];
#pragma unroll
    for (int w = 1; w < 4; ++w) mm = fmaxf(mm, m_lds[w * group + h]);
    f32x4 num = {0.0f, 0.0f, 0.0f, 0.0f};
    float den = 0.0f;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const float f = exp2f(m_lds[w * group + h] - mm);   // 0 for a wave that had no chunk (m = -inf)
      const f32x4 v = reinterpret_cast<const f32x4*>(o_lds)[w * items + it];
#pragma unroll
      for (int e = 0; e < 4; ++e) num[e] += v[e] * f;
      den += l_lds[w * group + h] * f;
    }
    if (SPLIT && used > 1) {
      f32x4* const mine = blocks + part * part_block(group);
      store_f32x4_device_coherent(mine + it, num);
      if ((it & 31) == 0) store_f32x4_device_coherent(mine + items + h, f32x4{mm, den, 0.0f, 0.0f});
    } else {
      store_row(out_row, it, num, den);
    }
  }
  if constexpr (SPLIT) {
    if (used == 1) return;
    wait_vmcnt<0>();
    __syncthreads();
    int* const ticket_cell = reinterpret_cast<int*>(combine_lds);
    if (tid == 0) *ticket_cell = atomicAdd(arrivals + pair, 1);
    __syncthreads();
    const int ticket = *ticket_cell;
    __syncthreads();
    if (ticket != used - 1) return;
    if (tid == 0) atomicExch(arrivals + pair, 0);
    const auto left = coherent_blocks(blocks, used * part_block(group) * 16);
    // Two threads share an item's parts (part q: thread q % 2) where there are threads enough; their sums meet in LDS,
    // in the room of the waves' partial results.
    const int lanes = 2 * items <= DEC_THREADS ? 2 : 1;
    const int share = lanes > 1 ? tid / items : 0;
    const int it0 = lanes > 1 ? tid - share * items : tid;
    f32x4* const sums = reinterpret_cast<f32x4*>(combine_lds);          // [lanes][items] sums, then [lanes][items] (m, l)
    if (share < lanes)
      for (int it = it0; it < items; it += lanes > 1 ? items : DEC_THREADS) {
        f32x4 num = {0.0f, 0.0f, 0.0f, 0.0f};
        float mm = -INFINITY, den = 0.0f;
        for (int q0 = share; q0 < used; q0 += 4 * lanes) {
          f32x4 v[4], ml[4];
#pragma unroll
          for (int c = 0; c < 4; ++c) {
            const int q = q0 + c * lanes < used ? q0 + c * lanes : q0;
            const int at = (q * part_block(group) + it) * 16, head_at = (q * part_block(group) + items + (it >> 5)) * 16;
            v[c] = load_f32x4_device_coherent(left, at, 0);
            ml[c] = load_f32x4_device_coherent(left, head_at, 0);
          }
          DFHIP_PIN;
#pragma unroll
          for (int c = 0; c < 4; ++c) {
            if (q0 + c * lanes >= used) continue;
            const float m_new = fmaxf(mm, ml[c][0]);
            const float keep = exp2f(mm - m_new), add = exp2f(ml[c][0] - m_new);
#pragma unroll
            for (int e = 0; e < 4; ++e) num[e] = num[e] * keep + v[c][e] * add;
            den = den * keep + ml[c][1] * add;
            mm = m_new;
          }
        }
        if (lanes > 1) {
          sums[share * items + it] = num;
          sums[(lanes + share) * items + it] = f32x4{mm, den, 0.0f, 0.0f};
        } else {
          store_row(out_row, it, num, den);
        }
      }
    if (lanes > 1) {
      __syncthreads();
      if (tid < items) {
        float mm = -INFINITY, den = 0.0f;
        for (int c = 0; c < lanes; ++c) mm = fmaxf(mm, sums[(lanes + c) * items + tid][0]);
        f32x4 num = {0.0f, 0.0f, 0.0f, 0.0f};
        for (int c = 0; c < lanes; ++c) {
          const f32x4 v = sums[c * items + tid], ml = sums[(lanes + c) * items + tid];
          const float f = exp2f(ml[0] - mm);
#pragma unroll
          for (int e = 0; e < 4; ++e) num[e] += v[e] * f;
          den += ml[1] * f;
        }
        store_row(out_row, tid, num, den);
      }
    }
  }
}

struct DecodeAttention {
  const uint16_t* q;
  uint16_t *kc, *vc;
  const int32_t *slots, *lengths;
  uint16_t* out;
  const float *cos_t, *sin_t;
  float* partials;
  int* arrivals;
  int64_t ld_q, ld_out;
  int tokens, kv_heads, group, num_slots, capacity, table_rows, parts;
  float scale_log2;
};
template <bool APPEND, bool SPLIT>
struct DecodeAttentionOf : DecodeAttention {
  static constexpr int THREADS = DEC_THREADS;
  __host__ __device__ int blocks() const { return tokens * kv_heads * parts; }
  DFHIP_DEVICE void run(int block, bool ordered) const {
    decode_attention<APPEND, SPLIT>(block, ordered, tokens, q, ld_q, kc, vc, slots, lengths, out, ld_out, kv_heads, group, num_slots, capacity,
                                    scale_log2, cos_t, sin_t, table_rows, parts, partials, arrivals);
  }
  bool beside(const DecodeAttentionOf& other) const {
    return kc == other.kc && vc == other.vc && out != other.out && (!SPLIT || arrivals != other.arrivals);
  }
};
template <bool APPEND, bool SPLIT>
__global__ void __launch_bounds__(DEC_THREADS) decode_attention_kernel(const DecodeAttentionOf<APPEND, SPLIT> p) {
  p.run(blockIdx.y * gridDim.x + blockIdx.x, p.blocks() > COMPUTE_UNITS);
}
// The launches of two nano-batches as one: eight workgroups of each in turn, so that the long sequences of both come first.
template <class K>
__global__ void __launch_bounds__(DEC_THREADS) decode_attention_pair_kernel(const DfhipBoth<K> p) {
  const int block = blockIdx.y * gridDim.x + blockIdx.x;
  const int first = p.side[0].blocks(), second = p.side[1].blocks(), both = (first < second ? first : second) & ~7;
  int side = (block >> 3) & 1, own = (block >> 4) * 8 + (block & 7);
  if (block >= 2 * both) {
    own = block - both;                        // what the longer launch has left
    side = own >= first;
    if (side) own -= first - both;
  }
  if (own < (side ? second : first)) p.side[side].run(own, first + second > COMPUTE_UNITS);
}
template <class K>
bool join_attention(const void* a, const void* b, dim3 ga, dim3 gb, void* both, DfhipJoined* joined) {
  return dfhip_join_as<K>(reinterpret_cast<const void*>(decode_attention_pair_kernel<K>), a, b, ga, gb, both, joined);
}
template <bool APPEND, bool SPLIT>
int launch_attention(const DecodeAttention& args, size_t lds_bytes, hipStream_t stream) {
  using K = DecodeAttentionOf<APPEND, SPLIT>;
  const auto kernel = decode_attention_kernel<APPEND, SPLIT>;
  static const bool known = (dfhip_pairable(reinterpret_cast<const void*>(kernel), join_attention<K>, DFHIP_SHORT_BLOCKS), true);
  (void)known;
  hipLaunchKernelGGL(kernel, dim3(args.tokens * args.kv_heads, args.parts), dim3(DEC_THREADS), lds_bytes, stream, K{args});
  return dfhip_check_launch();
}

// One workgroup per token: rotate q and k of the new token (position lengths[t] - 1), store q,
// append k and v to the caches of slot slots[t].
__global__ void __launch_bounds__(256)
rope_kv_append_kernel(const uint16_t* __restrict__ qkv, int64_t ld_qkv, uint16_t* __restrict__ q_out, int64_t ld_q,
                      uint16_t* __restrict__ kc, uint16_t* __restrict__ vc, const int32_t* __restrict__ slots,
                      const int32_t* __restrict__ lengths, const float* __restrict__ cos_t,
                      const float* __restrict__ sin_t, int q_heads, int kv_heads, int num_slots, int capacity,
                      int table_rows) {
  const int t = blockIdx.x, tid = threadIdx.x;
  const int slot = slots[t], pos = lengths[t] - 1;
  const bool cache_ok = slot >= 0 && slot < num_slots && pos >= 0 && pos < capacity;
  const int trow = pos < 0 ? 0 : (pos < table_rows ? pos : table_rows - 1);
  const uint16_t* row = qkv + (int64_t)t * ld_qkv;
  const int64_t slot_base = (int64_t)slot * kv_heads;
  for (int idx = tid; idx < (q_heads + kv_heads) * (HD / 2); idx += 256) {
    const int head = idx >> 6, i = idx & 63;
    const float lo = bf16_bits_to_f32(row[head * HD + i]), hi = bf16_bits_to_f32(row[head * HD + i + 64]);
    const float c = cos_t[trow * (HD / 2) + i], s = sin_t[trow * (HD / 2) + i];
    bf16_t olo, ohi;
    rotate_pair(lo, hi, c, s, olo, ohi);
    if (head < q_heads) {
      uint16_t* dst = q_out + (int64_t)t * ld_q + head * HD + i;
      dst[0] = bits_of(olo);
      dst[64] = bits_of(ohi);
    } else if (cache_ok) {
      uint16_t* dst = kc + ((slot_base + (head - q_heads)) * capacity + pos) * HD + i;
      dst[0] = bits_of(olo);
      dst[64] = bits_of(ohi);
    }
  }
  if (!cache_ok) return;
  const uint16_t* vrow = row + (q_heads + kv_heads) * HD;
  for (int idx = tid; idx < kv_heads * HD; idx += 256) {
    const int kh = idx >> 7, dim = idx & (HD - 1);
    vc[(((slot_base + kh) * (capacity / 8) + (pos >> 3)) * HD + dim) * 8 + (pos & 7)] = vrow[idx];
  }
}

}  // namespace

extern "C" int dfhip_rope_kv_append_bf16(const void* qkv, int64_t ld_qkv, void* q_out, int64_t ld_q, void* k_cache,
                                         void* v_cache, const int32_t* slots, const int32_t* lengths,
                                         const float* cos_table, const float* sin_table, int T, int q_heads,
                                         int kv_heads, int head_dim, int num_slots, int capacity, int table_rows,
                                         dfhip_stream_t stream) {
  if (!qkv || !q_out || !k_cache || !v_cache || !slots || !lengths || !cos_table || !sin_table)
    return DFHIP_ERR_NULL_POINTER;
  if (T < 1 || q_heads < 1 || kv_heads < 1 || head_dim != HD || num_slots < 1 || capacity < CHUNK ||
      capacity % CHUNK != 0 || table_rows < 1)
    return DFHIP_ERR_BAD_SHAPE;
  if (ld_qkv < (int64_t)(q_heads + 2 * kv_heads) * HD || ld_q < (int64_t)q_heads * HD) return DFHIP_ERR_BAD_STRIDE;
  hipLaunchKernelGGL(rope_kv_append_kernel, dim3(T), dim3(256), 0, static_cast<hipStream_t>(stream),
                     static_cast<const uint16_t*>(qkv), ld_qkv, static_cast<uint16_t*>(q_out), ld_q,
                     static_cast<uint16_t*>(k_cache), static_cast<uint16_t*>(v_cache), slots, lengths, cos_table,
                     sin_table, q_heads, kv_heads, num_slots, capacity, table_rows);
  return dfhip_check_launch();
}

extern "C" int dfhip_decode_attention_bf16(const void* q, int64_t ld_q, const void* k_cache, const void* v_cache,
                                           const int32_t* slots, const int32_t* lengths, void* out, int64_t ld_out,
                                           int T, int q_heads, int kv_heads, int head_dim, int num_slots,
                                           int capacity, float scale, dfhip_stream_t stream) {
  if (!q || !k_cache || !v_cache || !slots || !lengths || !out) return DFHIP_ERR_NULL_POINTER;
  if (T < 1 || q_heads < 1 || kv_heads < 1 || q_heads % kv_heads != 0 || q_heads / kv_heads > MAX_GROUP ||
      head_dim != HD || num_slots < 1 || capacity < CHUNK || capacity % CHUNK != 0 ||
      (int64_t)T * kv_heads >= (int64_t)1 << 31)
    return DFHIP_ERR_BAD_SHAPE;
  if (ld_q < (int64_t)q_heads * HD || ld_out < (int64_t)q_heads * HD) return DFHIP_ERR_BAD_STRIDE;
  if (ld_q % 8 || !dfhip_aligned16(q) || !dfhip_aligned16(k_cache) || !dfhip_aligned16(v_cache))
    return DFHIP_ERR_BAD_ALIGNMENT;
  const float scale_log2 = scale * 1.4426950408889634f;
  const int group = q_heads / kv_heads;
  const size_t combine_bytes = (size_t)4 * group * (HD + 2) * sizeof(float);
  const DecodeAttention args{static_cast<const uint16_t*>(q), static_cast<uint16_t*>(const_cast<void*>(k_cache)),
                             static_cast<uint16_t*>(const_cast<void*>(v_cache)), slots, lengths, static_cast<uint16_t*>(out),
                             nullptr, nullptr, nullptr, nullptr, ld_q, ld_out, T, kv_heads, group, num_slots, capacity, 1, 1,
                             scale_log2};
  return launch_attention<false, false>(args, combine_bytes, static_cast<hipStream_t>(stream));
}

// Workgroups per (token, kv head) pair: two to a compute unit in all (what fits at once), with at least 256 positions of a full
// cache each (two chunks per wave).  The lengths are on the device: the launch is sized for full caches and each sequence takes
// its share of it (sequence_parts).  A launch with fewer than MIN_PARTS of them, from 171 pairs on but for those below, cuts
// nothing.  [us, uncut / cut, 8 kv heads, all full: 2 sequences of 8192 positions 111 / 21.5 (their bytes at 6.7 TB/s: 10), 8 of 2048
// 33 / 16.8 (10), 20 of 4096 69 / 57 (50); in two parts, not taken: 32 of 512, 2048 and 4096 14.6 / 16.5, 42.9 / 46.0, 79 / 84]
// One workgroup to a unit up to 32 pairs, not taken: 2 of 8192 21.5 -> 18.8, 3 of 8192 24.7 -> 23.7, 4 of 4096 18.2 -> 17.1, 4 of
// 16384 47.7 -> 46.6, but further from float64.  A probability is rounded to bf16 relative to its wave's largest, which is exact:
// half as many waves round more of the large ones.  [distance, 2-norm, mean of 16 draws, 2 of 8192 2.650e-3 -> 2.672e-3, 4 of 8192
// 2.682e-3 -> 2.713e-3, 4 of 16384 2.706e-3 -> 2.738e-3, each +- 0.15 %]
// While every compute unit loads, each gets 26 GB/s, its share of what the memory gives (one by itself takes in 50 and more), so a few
// pairs more than units take up to twice the time, most units idle in the second half: 257 .. 384 of them are cut in four where the cache has room for 2048 positions, and so are 171 .. 192, which leave a quarter of the units idle, where it
// has room for 4096.  [us, uncut / four parts, 8 kv heads, all full: 33 sequences of 2048 68 / 53, 48 of 2048 73 / 69, 36 of 4096 133 / 100,
// 36 of 8192 266 / 190, 24 of 4096 70 / 65, of 8192 134 / 126; of 1/4 .. 1 of the capacity, longest first: 33 of 2048 45 / 41, 48 of 2048
// 56 / 57, 36 of 4096 90 / 71, 48 of 4096 106 / 91, 24 of 4096 65 / 51, of 8192 124 / 90; not taken, for the sake of full caches: 32 of
// 4096 79 / 86, 69 / 62, 64 of 4096 160 / 169, 121 / 117, 56 of 2048 77 / 80, 61 / 66]
constexpr int MIN_PARTS = 3;
static int attention_parts(int T, int kv_heads, int capacity) {
  const int64_t pairs = (int64_t)T * kv_heads;
  if ((pairs > 256 && pairs <= 384 && capacity >= 2048) || (pairs > 170 && pairs <= 192 && capacity >= 4096)) return 4;
  int64_t parts = 512 / pairs;
  if (parts > capacity / 256) parts = capacity / 256;
  if (parts > 32) parts = 32;
  return parts < 1 ? 1 : (int)parts;
}
// The arrival counters at the start of the workspace: a launch that splits has at most 384 pairs, and the area is the same
// for every shape, so that no launch's partial sums lie where another's counters are expected to be zero.
constexpr size_t ATTENTION_COUNTER_BYTES = 4096;

static int decode_attention_append(const void* qkv, int64_t ld_qkv, void* k_cache, void* v_cache, const int32_t* slots,
                                   const int32_t* lengths, const float* cos_table, const float* sin_table, void* out,
                                   int64_t ld_out, int T, int q_heads, int kv_heads, int head_dim, int num_slots,
                                   int capacity, int table_rows, float scale, int parts, void* workspace,
                                   dfhip_stream_t stream) {
  if (!qkv || !k_cache || !v_cache || !slots || !lengths || !cos_table || !sin_table || !out)
    return DFHIP_ERR_NULL_POINTER;
  if (T < 1 || q_heads < 1 || kv_heads < 1 || q_heads % kv_heads != 0 || q_heads / kv_heads > MAX_GROUP ||
      head_dim != HD || num_slots < 1 || capacity < CHUNK || capacity % CHUNK != 0 || table_rows < 1 ||
      (int64_t)T * kv_heads >= (int64_t)1 << 31)
    return DFHIP_ERR_BAD_SHAPE;
  if (ld_qkv < (int64_t)(q_heads + 2 * kv_heads) * HD || ld_out < (int64_t)q_heads * HD) return DFHIP_ERR_BAD_STRIDE;
  if (ld_qkv % 8 || !dfhip_aligned16(qkv) || !dfhip_aligned16(k_cache) || !dfhip_aligned16(v_cache))
    return DFHIP_ERR_BAD_ALIGNMENT;
  const int group = q_heads / kv_heads;
  const size_t lds_bytes = (size_t)4 * group * (HD + 2) * sizeof(float) + 2 * HD * sizeof(uint16_t);
  if (parts < MIN_PARTS) parts = 1;
  float* partials = reinterpret_cast<float*>(static_cast<uint8_t*>(workspace) + ATTENTION_COUNTER_BYTES);
  const DecodeAttention args{static_cast<const uint16_t*>(qkv), static_cast<uint16_t*>(k_cache), static_cast<uint16_t*>(v_cache),
                             slots, lengths, static_cast<uint16_t*>(out), cos_table, sin_table, parts > 1 ? partials : nullptr,
                             static_cast<int*>(workspace), ld_qkv, ld_out, T, kv_heads, group, num_slots, capacity, table_rows,
                             parts, scale * 1.4426950408889634f};
  const auto launch = parts > 1 ? launch_attention<true, true> : launch_attention<true, false>;
  return launch(args, lds_bytes, static_cast<hipStream_t>(stream));
}

extern "C" int dfhip_decode_attention_append_bf16(const void* qkv, int64_t ld_qkv, void* k_cache, void* v_cache,
                                                  const int32_t* slots, const int32_t* lengths,
                                                  const float* cos_table, const float* sin_table, void* out,
                                                  int64_t ld_out, int T, int q_heads, int kv_heads, int head_dim,
                                                  int num_slots, int capacity, int table_rows, float scale,
                                                  dfhip_stream_t stream) {
  return decode_attention_append(qkv, ld_qkv, k_cache, v_cache, slots, lengths, cos_table, sin_table, out, ld_out, T,
                                 q_heads, kv_heads, head_dim, num_slots, capacity, table_rows, scale, 1, nullptr, stream);
}

extern "C" size_t dfhip_decode_attention_workspace_bytes(int T, int q_heads, int kv_heads, int capacity) {
  if (T < 1 || kv_heads < 1 || q_heads < kv_heads || capacity < 1) return 0;
  const int parts = attention_parts(T, kv_heads, capacity);
  if (parts < 2) return 0;
  return ATTENTION_COUNTER_BYTES +
         (size_t)T * kv_heads * parts * part_block(q_heads / kv_heads) * 16;
}

extern "C" int dfhip_decode_attention_append_split_bf16(
    const void* qkv, int64_t ld_qkv, void* k_cache, void* v_cache, const int32_t* slots, const int32_t* lengths,
    const float* cos_table, const float* sin_table, void* out, int64_t ld_out, int T, int q_heads, int kv_heads,
    int head_dim, int num_slots, int capacity, int table_rows, float scale, void* workspace, size_t workspace_bytes,
    dfhip_stream_t stream) {
  const size_t need = dfhip_decode_attention_workspace_bytes(T, q_heads, kv_heads, capacity);
  if (need > 0) {
    if (!workspace) return DFHIP_ERR_NULL_POINTER;
    if (!dfhip_aligned16(workspace)) return DFHIP_ERR_BAD_ALIGNMENT;
    if (workspace_bytes < need) return DFHIP_ERR_BAD_ARGUMENT;
  }
  const int parts = need > 0 ? attention_parts(T, kv_heads, capacity) : 1;
  return decode_attention_append(qkv, ld_qkv, k_cache, v_cache, slots, lengths, cos_table, sin_table, out, ld_out, T,
                                 q_heads, kv_heads, head_dim, num_slots, capacity, table_rows, scale, parts, workspace,
                                 stream);
}
