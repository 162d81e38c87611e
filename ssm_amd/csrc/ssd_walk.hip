// Mamba-2 SSD forward of 16-bit calls as one pass over the sequence: a workgroup owns the 64 channels of one (batch, head),
// or of two neighbouring heads, and walks their steps in blocks of 32 with the running state in matrix-core accumulators,
// so that x, z and y are all that travels between HBM and the chip.  Per block, with cs the running sum of dt A since the
// block's first step:
//
//   y_l = exp(cs_l) C_l.S + sum_{s<=l} (C_l.B_s) exp(cs_l - cs_s) dt_s x_s  (+ D x_l, gate)
//   S  <- exp(cs_31) S + sum_s exp(cs_31 - cs_s) dt_s x_s (x) B_s
//
// Four waves multiply: wave (pt, nh) holds the states of 32 channels and half of the state dimension, S^T as tiles [n][p].
// A tile is the left operand of C.S as it stands - lane = channel, registers = states - once the fragments of C hold the
// states in the order of the accumulators' rows (prep_pack_role), so the state is rounded to 16 bits in registers and never
// goes through LDS.  Four more waves per head do what is element by element: they weight x for the block after the one being
// multiplied, add what the two halves of the state gave to the block before it, gate that and store it as whole rows.
// One barrier per block.  x is read from LDS with transposing reads (ds_read_b64_tr_b16); 16-byte pieces of a row are
// XOR-swizzled by the row.
//
// Decays.  Where a block decays by no more than 2^-160, they factor at its middle, r = cs_31 / 2: with x~_s = exp(r - cs_s)
// dt_s x_s and the state held at the middle of its block, S~ = exp(r) S,
//   y_l = exp(cs_l - r) (C_l.S~ + sum_{s<=l} (C_l.B_s) x~_s),      S~ <- exp(..) (S~ + sum_s x~_s (x) B_s),
// no element of C.B needs a factor, and C.B goes from memory to the matrix cores as it is.  What rounding to bfloat16 takes
// from x~ joins the products inside the block as an operand of its own, so that these lose nothing beyond the rounding of
// C.B.  Heads of which a block goes beyond that range, and float16 calls (whose exponents hold no such x~), form
// exp(cs_l - cs_s) dt_s (C_l.B_s) per element instead, x weighted towards the block's end for the state.
// The factors r - cs_s reach 2^80: where dt x is so large that x~, or what it is summed into, leaves bfloat16, a y or a state
// comes out infinite or not a number, and the workgroup does its heads again per element, whose factors are at most 1.
// In float16 the same is done where a state goes beyond 65504: the second time it is rounded to float16 scaled by a power of two.
// Calls that write y over x or z, which are not there a second time, go that way at once.
//
// A growing head (A > 0): decays between steps of one of the call's chunks are bounded by 1, the factors on the state entering
// the chunk are not (the published kernels evaluate exp(min(x, 0)) and exp(x) there).  Such a head goes per element and keeps
// that state apart from what the chunk has added so far.
//
// Which of the three ways a workgroup goes is told from A and the blocks' sums on the device; each has a loop of its own.
// Choosing block by block inside one loop cost every call 0.05 to 0.1 us a block.  4 x 80 heads of 4096 steps, 128 states, us
// a call with all heads factoring, one in eight not, none, all growing: 174, 187, 186, 309; 4 x 64 heads 139, 143, 139, 168; 24
// heads of 512 steps 21.0, 22.4, 22.7, 25.8.  (With workgroups of their own for the heads that do not factor, behind the others:
// 180, 250, 250, 671; 182, 229, 142, 330; 21.4, 21.3, 21.6, 43.  Before this walk: 274; 203; 21.9, whatever the decays.)
//
// What bounds it: a CU takes in x and z at no more than about 20 (one head's rows of 128 bytes) to 27 (two heads') bytes per
// ns whatever is in flight - a kernel that only streams them this way takes 88 us for 256 heads x 4096 steps on 256 CUs, 148
// us for 320 heads, as a CU with two workgroups takes twice as long, and 114 us for these as 160 pairs - and the vector ALU
// issues behind the matrix cores, not beside them.  So: a head per workgroup while every workgroup has a CU of its own,
// two neighbours beyond; and the fragments of B and C into LDS once per workgroup.  4 x 4096 steps, 128 states, 64 / 80 heads:
// 139 / 174 us a call.  Before (half a head per workgroup, 64-byte rows, chunks of 256 steps): 203 / 274.
// With fragments loaded by each wave it was 135 / 200 when this was 137 / 195.
#include "ssd_common.hpp"
#include "ssd_walk.hpp"
#include <type_traits>

namespace ssm {

constexpr int WK = SSD_WALK_BLOCK, WK_TILE = WK * SSD_P * 2;             // steps of a block; bytes of its 64 channels
constexpr int WALK_SINGLES = 256;                                        // heads that get a workgroup each: the CUs

// FACTORS: heads whose decays factor; ELEMENTS: element by element; GROWS: the same, and the state that enters a chunk of the
// call apart.
enum WalkMode { FACTORS, ELEMENTS, GROWS };
template <WalkMode M> using walk_mode = std::integral_constant<WalkMode, M>;

// Byte offsets into LDS.  Twice each: 32 rows of x per head, weighted (X ..), and what their rounding lost, or x itself
// (NH tiles on); part sums [head][nh][pt][step][32 channels] of float32; per head cs, log2 dt - cs and log2 dt of a block taken
// element by element.  Fragments of three blocks.  A word: whether something left the range.
template <int NH, int N> struct WalkLds {
  static constexpr int KN = N / 16, X = 2 * NH * WK_TILE, PARTS = NH * 4 * 4096, STEPS = 3 * WK * 4;
  static constexpr int PART = 2 * X, C = PART + 2 * PARTS, B = C + 3 * KN * 1024, CB = B + 3 * KN * 1024, STEP = CB + 3 * 2048;
  static constexpr int AGAIN = STEP + 2 * NH * STEPS, BYTES = AGAIN + 16;
};
static_assert(WalkLds<2, 128>::BYTES <= 160 * 1024, "one pair per CU");

typedef __amdgpu_buffer_rsrc_t rsrc_t;
typedef __attribute__((__vector_size__(4 * sizeof(unsigned)))) unsigned u32x4_t;
typedef const __attribute__((address_space(4))) float *scalar_floats;

// The barrier without the wait for accesses to memory that a fence would bring.
__device__ __forceinline__ void walk_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}
template <int N>
__device__ __forceinline__ void wait_memory() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }

// 16 bytes per lane from memory to LDS, lane i to byte `at` + 16 i.  Written out, because the compiler would make every
// later read of LDS wait for it; the waits are walk_products'.  `at` is asked for in m0, so that the compiler knows who has it.
__device__ __forceinline__ void to_lds16(const void *base, unsigned off, unsigned at) {
  asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"{m0}"(at), "v"(off), "s"(base) : "memory");
}

typedef __attribute__((__vector_size__(4 * sizeof(short)))) short i16x4_t;
// Operand fragment from rows in LDS: lane (m, g2) gets steps 8 g2 .. + 7 of its channel; `a0` and `a1` are the lane's byte
// addresses for the first and the last four of them.
template <typename E>
__device__ __forceinline__ V8<E> transposed_frag(const unsigned char *lds, int a0, int a1) {
  typedef __attribute__((address_space(3))) i16x4_t *ptr;
  struct { i16x4_t a, b; } r = {__builtin_amdgcn_ds_read_tr16_b64_v4i16((ptr)(lds + a0)), __builtin_amdgcn_ds_read_tr16_b64_v4i16((ptr)(lds + a1))};
  return __builtin_bit_cast(V8<E>, r);
}

template <typename E>
__device__ __forceinline__ V8<E> state_frag(const f32x16_t &s, int t) {
  V8<E> r;
#pragma unroll
  for (int j = 0; j < 8; ++j) r[j] = (E)s[8 * t + j];
  return r;
}

// The larger of `most` and the sizes of two values, no number if one of them is none.
__device__ __forceinline__ void note_size(float &most, float a, float b) { asm("v_maximum3_f32 %0, |%1|, |%2|, %0" : "+v"(most) : "v"(a), "v"(b)); }

// What the running sums of a block that factors are relative to: the sum at its middle.
template <typename E>
__device__ __forceinline__ float walk_middle(float end) { return std::is_same<E, __bf16>::value && walk_factors(end) ? 0.5f * end : 0.0f; }

// Keeps in `seen` that one of eight values stored was infinite or no number.  bfloat16: read as float16 these bits are no
// number, nor are those from 2^121 on, and a maximum that passes on what is no number costs half an instruction a word.
__device__ __forceinline__ void note_overflow(unsigned &seen, const V8<__bf16> &v) {
  const u32x4_t w = __builtin_bit_cast(u32x4_t, v);
  asm("v_pk_maximum3_f16 %0, %1, %2, %0" : "+v"(seen) : "v"(w[0]), "v"(w[1]));
  asm("v_pk_maximum3_f16 %0, %1, %2, %0" : "+v"(seen) : "v"(w[2]), "v"(w[3]));
}
__device__ __forceinline__ void note_overflow(unsigned &seen, const V8<_Float16> &v) {
  const u32x4_t w = __builtin_bit_cast(u32x4_t, v);
#pragma unroll
  for (int i = 0; i < 4; ++i) asm("v_pk_fma_f16 %0, %1, 0, %0" : "+v"(seen) : "v"(w[i]));
}
__device__ __forceinline__ bool noted_overflow(unsigned seen) { return (seen & 0x7fffu) > 0x7c00u || (seen >> 16 & 0x7fffu) > 0x7c00u; }

// One head, or two neighbouring heads of a group (the last of an odd number alone: it is computed twice and written once).
template <int NH>
struct WalkHeads {
  int b, g, h0, h1;
  bool two;
  __device__ __forceinline__ WalkHeads(const SsdWalkParams &p, int id) {
    const int per_group = p.heads / p.groups, sets = (per_group + NH - 1) / NH;
    const int i = id % sets;
    g = id / sets % p.groups;
    b = id / sets / p.groups;
    h0 = g * per_group + NH * i;
    two = NH == 2 && 2 * i + 1 < per_group;
    h1 = two ? h0 + 1 : h0;
  }
  __device__ __forceinline__ WalkHeads(int b_, int g_, int h) : b(b_), g(g_), h0(h), h1(h), two(false) {}
  // Running sums at the ends of a head's blocks, read through the scalar cache.
  __device__ __forceinline__ scalar_floats ends(const SsdWalkParams &p, int second) const {
    return (scalar_floats)(size_t)(p.ends + ((size_t)b * p.heads + (second ? h1 : h0)) * p.turns);
  }
  // The pair's stretch of x, z or y as a buffer: reads past the last row give zero, stores there are dropped.
  __device__ __forceinline__ rsrc_t rsrc(const void *base, const SsdWalkParams &p) const {
    const unsigned pitch = (unsigned)p.heads * SSD_P * 2;
    const unsigned char *at = reinterpret_cast<const unsigned char *>(base) + ((size_t)b * p.len * p.heads + h0) * SSD_P * 2;
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<unsigned char *>(at), 0, (int)((unsigned)(p.len - 1) * pitch + (two ? 2 : 1) * SSD_P * 2), 0x00020000);
  }
};

// Whether all of the heads' blocks factor.
template <int NH>
__device__ __forceinline__ bool heads_factor(const SsdWalkParams &p, const WalkHeads<NH> &hp) {
  const float *e0 = p.ends + ((size_t)hp.b * p.heads + hp.h0) * p.turns, *e1 = p.ends + ((size_t)hp.b * p.heads + hp.h1) * p.turns;
  bool ok = true;
  for (int c0 = 0; c0 < p.turns; c0 += WAVE) {
    const int c = min(c0 + lane_id(), p.turns - 1);
    const float a = e0[c], b = NH == 2 ? e1[c] : a;
    ok = ok && walk_factors(a) && walk_factors(b);
  }
  return __all(ok);
}

// The waves of rows.  Turn c: gate and store block c - 1, stage block c + 1.  Each thread has eight channels of one row of
// every block; what it takes from memory of them is requested four turns ahead.  Whether a y left the range.
template <typename E, int NH, int N, int DMODE, bool HAS_Z, typename InMode>
__device__ __forceinline__ bool walk_rows(const SsdWalkParams &p, unsigned char *lds, const WalkHeads<NH> &hp, const InMode &in_mode) {
  using L = WalkLds<NH, N>;
  constexpr bool F16 = std::is_same<E, _Float16>::value;
  const int wave = wave_id_uniform() - 4, lane = lane_id(), tid = wave * WAVE + lane;
  const int row = tid / (8 * NH), second = NH == 2 ? tid >> 3 & 1 : 0, piece = tid & 7;
  const unsigned pitch = (unsigned)p.heads * SSD_P * 2, block = WK * pitch;
  const rsrc_t rx = hp.rsrc(p.x, p), rz = hp.rsrc(HAS_Z ? p.z : p.x, p), ry = hp.rsrc(p.y, p);
  const unsigned mine = (unsigned)row * pitch + (hp.two ? second : 0) * (SSD_P * 2) + piece * 16;
  const bool drop = second && !hp.two;
  const float2 *steps = reinterpret_cast<const float2 *>(p.steps) + ((size_t)hp.b * p.heads + hp.h0) * p.turns * WK;
  const unsigned step_at = ((hp.two ? second : 0) * (unsigned)p.turns * WK + row) * 8;
  const int h = second ? hp.h1 : hp.h0;
  float D8[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) D8[j] = DMODE == 0 ? 0.0f : p.Dk[DMODE == 2 ? h * SSD_P + 8 * piece + j : h];
  const scalar_floats ends[2] = {hp.ends(p, 0), hp.ends(p, NH - 1)};

  unsigned seen = 0;
  const int at16 = second * WK_TILE + row * 128 + ((piece ^ (row & 7)) << 4);
  const int half_at = L::PART + second * 16384 + (piece >> 2) * 4096 + row * 128;
  const int q0 = half_at + (((2 * (piece & 3)) ^ (row & 7)) << 4), q1 = half_at + (((2 * (piece & 3) + 1) ^ (row & 7)) << 4);

  const auto rows = [&](auto mode) __attribute__((always_inline)) {
    constexpr WalkMode MODE = decltype(mode)::value;
    V8<E> x[4], z[4];
    float2 step[4];
    float skip[2][8], grow[2];
    // A ring's place is loaded again once `after` is there: a load in front of the last use of what the place held would take
    // another register, and the copy back at the end of the loop would wait for it.
    const auto load_rows = [&](rsrc_t r, int c, const V8<E> &after) {
      unsigned off = mine + (unsigned)c * block;
      asm volatile("" : "+v"(off) : "v"(after));
      return __builtin_bit_cast(V8<E>, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
    };
    const auto load_step = [&](int c, const V8<E> &after) {
      unsigned off = step_at;
      asm volatile("" : "+v"(off) : "v"(after));
      return *at_bytes<const float2>(steps + (size_t)min(c, p.turns - 1) * WK, off);
    };
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      x[u] = load_rows(rx, u, V8<E>{});
      if (HAS_Z) z[u] = load_rows(rz, u, V8<E>{});
      step[u] = load_step(u, V8<E>{});
    }
    const auto stage = [&](int c, int u, const float (&end)[2]) __attribute__((always_inline)) {
      // first looked at here: the scheduler would start on blocks ahead, and wait for reads that are still on their way
      asm volatile("" : "+v"(x[u]), "+v"(step[u].x), "+v"(step[u].y));
      float v[8], lost[8];
      unpack8(x[u], v);
      if (DMODE != 0) {
#pragma unroll
        for (int j = 0; j < 8; ++j) skip[u & 1][j] = D8[j] * v[j];
      }
      V8<E> rounded, rest;
      const float to_end = NH == 2 && second ? end[1] : end[0], cs = step[u].x + (MODE == FACTORS ? 0.0f : walk_middle<E>(to_end));
      const float w = step[u].y * exp2_hw(MODE == FACTORS ? -cs : fminf(to_end - cs, 0.0f));
      rest = x[u];
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] *= w;
      rounded = pack8_e<E>(v);
      if constexpr (MODE == FACTORS) {
        grow[u & 1] = exp2_hw(cs);
        unpack8(rounded, lost);
#pragma unroll
        for (int j = 0; j < 8; ++j) lost[j] = v[j] - lost[j];
        rest = pack8_e<E>(lost);
      } else if (piece == 0) {
        float *st = reinterpret_cast<float *>(lds + L::STEP + ((u & 1) * NH + second) * L::STEPS);
        const float l2 = log2_hw(step[u].y);                 // dt = 0: -inf, a weight of zero
        st[row] = cs;
        st[WK + row] = l2 - cs;
        st[2 * WK + row] = l2;
      }
      unsigned char *to = lds + (u & 1) * L::X + at16;
      *reinterpret_cast<V8<E> *>(to) = rounded;
      *reinterpret_cast<V8<E> *>(to + NH * WK_TILE) = rest;
      x[u] = load_rows(rx, c + 4, rest);
      step[u] = load_step(c + 4, rest);
    };
    struct Parts { float4 a0, a1, b0, b1; };
    const auto read_parts = [&](int u) __attribute__((always_inline)) {
      const unsigned char *half = lds + (u & 1) * L::PARTS;
      return Parts{*reinterpret_cast<const float4 *>(half + q0), *reinterpret_cast<const float4 *>(half + q1),
                   *reinterpret_cast<const float4 *>(half + 8192 + q0), *reinterpret_cast<const float4 *>(half + 8192 + q1)};
    };
    const auto gate = [&](int c, int u, const Parts &r, float up, const float (&dx)[8]) __attribute__((always_inline)) {
      float v[8] = {r.a0.x + r.b0.x, r.a0.y + r.b0.y, r.a0.z + r.b0.z, r.a0.w + r.b0.w, r.a1.x + r.b1.x, r.a1.y + r.b1.y, r.a1.z + r.b1.z, r.a1.w + r.b1.w};
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        if (MODE == FACTORS) v[j] = DMODE == 0 ? v[j] * up : __builtin_fmaf(v[j], up, dx[j]);
        else if (DMODE != 0) v[j] += dx[j];
      }
      if (HAS_Z) {
        float zf[8];
        asm volatile("" : "+v"(z[u]));
        unpack8(z[u], zf);
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] *= silu_f32(zf[j]);
      }
      const V8<E> out = pack8_e<E>(v);
      if (MODE == FACTORS || (F16 && MODE == ELEMENTS))
        if (c >= 0) note_overflow(seen, out);
      if (HAS_Z) z[u] = load_rows(rz, c + 4, out);
      // The scalar offset stays the constant 0: a 16-byte store reads its data some cycles after it issues, and only for that
      // form does the compiler keep what rewrites those registers away from it.  With the offset in a scalar register wrong
      // words have been seen under load.
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, out), ry, drop ? 1u << 31 : mine + (unsigned)c * block, 0, 0);
    };
    // Ends of blocks are asked for a turn before they are looked at, and not looked at behind reads of LDS.
    float end[2] = {};
    const auto next_ends = [&](int c) __attribute__((always_inline)) {
      if (MODE == FACTORS) return;
      asm volatile("" ::: "memory");
      end[0] = ends[0][min(c, p.turns - 1)];
      end[1] = NH == 2 ? ends[1][min(c, p.turns - 1)] : end[0];
    };
    next_ends(0);
    walk_barrier();                                          // (the products' first fragments)
    stage(0, 0, end);
    next_ends(1);
    walk_barrier();
    for (int c0 = 0; c0 < p.turns; c0 += 4) {
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int c = c0 + u, before = (u + 3) & 3;
        const float to[2] = {end[0], end[1]};
        if (MODE != FACTORS) asm volatile("" ::"s"(to[0]), "s"(to[1]) : "memory");
        next_ends(c + 2);
        const Parts parts = read_parts(before);              // of block c - 1 (before the first: values whose store is dropped)
        const float up = grow[before & 1];
        float dx[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) dx[j] = skip[before & 1][j];
        stage(c + 1, (u + 1) & 3, to);                       // of the block after the last: values that nothing reads
        gate(c - 1, before, parts, up, dx);
        walk_barrier();
      }
    }
    gate(p.turns - 1, 3, read_parts(3), grow[1], skip[1]);
  };
  in_mode(rows);
  return __any(noted_overflow(seen));
}

// The four waves of products.  Turn c: block c.  Final states are written once `settled` (asked when this wave's share of the
// heads is done, with whether it left the range) has said that they stand.
template <typename E, int NH, int N, typename InMode, typename Settled>
__device__ __forceinline__ void walk_products(const SsdWalkParams &p, unsigned char *lds, const WalkHeads<NH> &hp, const InMode &in_mode, const Settled &settled) {
  using L = WalkLds<NH, N>;
  constexpr bool F16 = std::is_same<E, _Float16>::value;
  constexpr int NT = N / 32, TPW = NT / 2, KN = N / 16, SHARE = KN / 4;
  const int wave = wave_id_uniform(), lane = lane_id();
  const int m = lane & 31, g2 = lane >> 5, pt = wave & 1, nh = wave >> 1;
  const int k = lane & 15, tr_row = 8 * g2 + (k >> 2), tr_piece = 4 * pt + 2 * (lane >> 4 & 1) + ((k & 3) >> 1);
  const int tr0 = tr_row * 128 + ((tr_piece ^ (k >> 2)) << 4) + (k & 1) * 8, tr1 = (tr0 + 512) ^ 64;
  unsigned char *const part = lds + L::PART + (2 * nh + pt) * 4096 + m * 128;
  const scalar_floats ends[2] = {hp.ends(p, 0), hp.ends(p, NH - 1)};
  const unsigned lds0 = (unsigned)(size_t)(__attribute__((address_space(3))) unsigned char *)lds;
  const unsigned lane16 = (unsigned)lane * 16;

  // Fragments go from memory into LDS, a quarter by each wave, so that a workgroup reads each once: those of C three blocks
  // ahead, of B and C.B two.
  const size_t unit0 = (size_t)hp.b * p.nblocks * p.groups + hp.g;
  const auto unit = [&](int c) { return unit0 + (size_t)min(c, p.nblocks - 1) * p.groups; };
  const auto request_c = [&](int c, int slot) {
    const E *from = reinterpret_cast<const E *>(p.Cblk) + (unit(c) * KN + SHARE * wave) * SSD_FRAG;
#pragma unroll
    for (int i = 0; i < SHARE; ++i) to_lds16(from + i * SSD_FRAG, lane16, lds0 + L::C + (slot * KN + SHARE * wave + i) * 1024);
  };
  const auto request_b = [&](int c, int slot) {
    const E *from = reinterpret_cast<const E *>(p.Btblk) + (unit(c) * KN + SHARE * wave) * SSD_FRAG;
#pragma unroll
    for (int i = 0; i < SHARE; ++i) to_lds16(from + i * SSD_FRAG, lane16, lds0 + L::B + (slot * KN + SHARE * wave + i) * 1024);
    if (wave < 2) to_lds16(reinterpret_cast<const E *>(p.CBblk) + (unit(c) * 2 + wave) * SSD_FRAG, lane16, lds0 + L::CB + slot * 2048 + wave * 1024);
  };
  const auto frag = [&](int at) { return load_frag_e<E>(lds + at + lane16); };

  request_c(1, 1);
  request_c(2, 2);
  request_b(0, 0);
  request_b(1, 1);
  if (p.init) {
    request_c(0, 0);
  } else {
    // without a state to start from the first block's product with it is zero whatever C holds
#pragma unroll
    for (int i = 0; i < SHARE; ++i) *reinterpret_cast<V8<E> *>(lds + L::C + (SHARE * wave + i) * 1024 + lane16) = V8<E>{};
  }
  const auto products = [&](auto mode) __attribute__((always_inline)) {
    constexpr WalkMode MODE = decltype(mode)::value;
    static_assert(MODE != GROWS || NH == 1 || N == 64);      // (registers)
    f32x16_t S[NH][TPW];
    size_t state0[NH];
#pragma unroll
    for (int hd = 0; hd < NH; ++hd) {
      state0[hd] = (((size_t)hp.b * p.heads + (hd ? hp.h1 : hp.h0)) * SSD_P + 32 * pt + m) * N + 32 * nh * TPW;
#pragma unroll
      for (int i = 0; i < TPW; ++i) {
        S[hd][i] = (f32x16_t){0};
        if (p.init) {
#pragma unroll
          for (int r = 0; r < 16; ++r) S[hd][i][r] = p.init[state0[hd] + 32 * i + crow(r, g2)];
        }
      }
    }
    wait_memory<0>();
#pragma unroll
    for (int hd = 0; hd < NH; ++hd) {                        // (said to the compiler too: it would wait inside the loop)
#pragma unroll
      for (int i = 0; i < TPW; ++i) asm volatile("" : "+v"(S[hd][i]));
    }
    walk_barrier();
    __builtin_amdgcn_s_setprio(1);
    f32x16_t entered[MODE == GROWS ? NH : 1][TPW];           // the state entering the chunk,
    float base[NH] = {};                                     // and the running sum up to the block, from the chunk's first step
    float held[NH] = {}, next[NH];                           // from the block's middle, where the state is held, to its end
#pragma unroll
    for (int hd = 0; hd < NH; ++hd) next[hd] = ends[hd][0];
    for (int c = 0, t3 = 0; c < p.turns; ++c) {              // turns past the last block: steps of size zero
      const int last3 = t3 == 0 ? 2 : t3 - 1;
      float end[NH];
#pragma unroll
      for (int hd = 0; hd < NH; ++hd) end[hd] = next[hd];
      // in the turn of the block before, c - 1: the state, brought from the middle of that block to the middle of this one
      f32x16_t acc[NH], acc_entered[MODE == GROWS ? NH : 1];
      const bool any_entered = c >= p.chunk_blocks || p.init;
      if (MODE == GROWS && c % p.chunk_blocks == 0) {
#pragma unroll
        for (int hd = 0; hd < NH; ++hd) {
#pragma unroll
          for (int i = 0; i < TPW; ++i) {
            entered[hd][i] = S[hd][i];
            S[hd][i] = (f32x16_t){0};
          }
          base[hd] = 0.0f;
        }
      }
#pragma unroll
      for (int hd = 0; hd < NH; ++hd) {
        if (MODE == FACTORS) {
          const float here = 0.5f * end[hd];
          float to_here = held[hd] + here;
          if (to_here < -120.0f) {                           // a factor that float32 does not hold, in two that it does
            const float g = exp2_hw(held[hd]);
#pragma unroll
            for (int i = 0; i < TPW; ++i) {
#pragma unroll
              for (int r = 0; r < 16; ++r) S[hd][i][r] *= g;
            }
            to_here = here;
          }
          const float g = exp2_hw(to_here);
          held[hd] = here;
#pragma unroll
          for (int i = 0; i < TPW; ++i) {
#pragma unroll
            for (int r = 0; r < 16; ++r) S[hd][i][r] *= g;
          }
        }
        float up = 1.0f;
        const auto scale_states = [&](float by) __attribute__((always_inline)) {
#pragma unroll
          for (int i = 0; i < TPW; ++i) {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
              S[hd][i][r] *= by;
              if (MODE == GROWS) entered[hd][i][r] *= by;
            }
          }
        };
        if (F16 && MODE == GROWS) {                          // a state that float16 does not hold
          float most2[2] = {};
#pragma unroll
          for (int i = 0; i < TPW; ++i) {
#pragma unroll
            for (int r = 0; r < 16; ++r) note_size(most2[r & 1], S[hd][i][r], entered[hd][i][r]);
          }
          float most = fmaxf(most2[0], most2[1]);
          if (__any(most >= 32768.0f)) {
#pragma unroll
            for (int other = 1; other < WAVE; other <<= 1) most = fmaxf(most, __shfl_xor(most, other, WAVE));
            const int above = (int)(__float_as_uint(most) >> 23) - (127 + 14);
            up = exp2_hw((float)above);
            scale_states(exp2_hw((float)-above));
          }
        }
        acc[hd] = (f32x16_t){0};
#pragma unroll
        for (int i = 0; i < TPW; ++i) {
#pragma unroll
          for (int t = 0; t < 2; ++t) acc[hd] = mma(state_frag<E>(S[hd][i], t), frag(L::C + (t3 * KN + 2 * (nh * TPW + i) + t) * 1024), acc[hd]);
        }
        if (MODE == GROWS) {
          acc_entered[hd] = (f32x16_t){0};
          if ((N == 64 && NH == 1) || any_entered) {
#pragma unroll
            for (int i = 0; i < TPW; ++i) {
#pragma unroll
              for (int t = 0; t < 2; ++t)
                acc_entered[hd] = mma(state_frag<E>(entered[hd][i], t), frag(L::C + (t3 * KN + 2 * (nh * TPW + i) + t) * 1024), acc_entered[hd]);
            }
          }
          if (F16 && up != 1.0f) {
            scale_states(up);
#pragma unroll
            for (int r = 0; r < 16; ++r) {
              acc[hd][r] *= up;
              acc_entered[hd][r] *= up;
            }
          }
        }
      }
      if (wave < 2) wait_memory<2 * SHARE + 1>();            // what turn c - 1 requested may be under way, no more
      else wait_memory<2 * SHARE>();
      walk_barrier();
      request_c(c + 3, t3);
      request_b(c + 2, last3);
#pragma unroll
      for (int hd = 0; hd < NH; ++hd) next[hd] = ends[hd][min(c + 1, p.turns - 1)];
      const V8<E> cb = frag(L::CB + t3 * 2048 + nh * 1024);
      V8<E> w[NH];
#pragma unroll
      for (int hd = 0; hd < NH; ++hd) {
        w[hd] = cb;
        if (MODE == FACTORS) continue;
        const float *st = reinterpret_cast<const float *>(lds + L::STEP + ((c & 1) * NH + hd) * L::STEPS), own = st[m];
        const float f = exp2_hw(MODE == GROWS ? fminf(own, 0.0f) : own);
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[hd][r] *= f;
        if (MODE == GROWS) {
          const float fh = fminf(exp2_hw(base[hd] + own), 3.0e38f);    // (finite: what is zero stays zero)
#pragma unroll
          for (int r = 0; r < 16; ++r) acc[hd][r] = __builtin_fmaf(acc_entered[hd][r], fh, acc[hd][r]);
        }
        // dt_s exp(min(cs_l - cs_s, 0)) as one exponential: min(a, 0) + b = min(a + b, b) with b = log2 dt_s.  The bound is
        // inactive on and below the diagonal of a decaying head, is the clamp of a growing one, and keeps the places above
        // the diagonal (zeros of C.B) finite.
#pragma unroll
        for (int k4 = 0; k4 < 2; ++k4) {
          const float4 e4 = *reinterpret_cast<const float4 *>(st + WK + 16 * nh + 8 * g2 + 4 * k4);
          const float4 l4 = *reinterpret_cast<const float4 *>(st + 2 * WK + 16 * nh + 8 * g2 + 4 * k4);
          const float e[4] = {e4.x, e4.y, e4.z, e4.w}, l2[4] = {l4.x, l4.y, l4.z, l4.w};
#pragma unroll
          for (int j = 0; j < 4; ++j) w[hd][4 * k4 + j] = (E)((float)cb[4 * k4 + j] * exp2_hw(fminf(own + e[j], l2[j])));
        }
        const float gs = exp2_hw(MODE == GROWS ? fminf(end[hd], 0.0f) : end[hd]);
#pragma unroll
        for (int i = 0; i < TPW; ++i) {
#pragma unroll
          for (int r = 0; r < 16; ++r) S[hd][i][r] *= gs;
        }
      }
#pragma unroll
      for (int hd = 0; hd < NH; ++hd) {
        const unsigned char *xt = lds + (c & 1) * L::X + hd * WK_TILE;
        const V8<E> xf[2] = {transposed_frag<E>(xt, tr0, tr1), transposed_frag<E>(xt, tr0 + 2048, tr1 + 2048)};
        if (MODE == FACTORS) acc[hd] = mma(nh ? xf[1] : xf[0], cb, acc[hd]);
        acc[hd] = mma(transposed_frag<E>(xt + NH * WK_TILE, tr0 + 2048 * nh, tr1 + 2048 * nh), w[hd], acc[hd]);
#pragma unroll
        for (int i = 0; i < TPW; ++i) {
#pragma unroll
          for (int ks = 0; ks < 2; ++ks) S[hd][i] = mma(frag(L::B + (t3 * KN + ks * NT + nh * TPW + i) * 1024), xf[ks], S[hd][i]);
        }
#pragma unroll
        for (int q = 0; q < 4; ++q)
          *reinterpret_cast<float4 *>(part + (c & 1) * L::PARTS + hd * 16384 + (((2 * q + g2) ^ (m & 7)) << 4)) =
              make_float4(acc[hd][4 * q], acc[hd][4 * q + 1], acc[hd][4 * q + 2], acc[hd][4 * q + 3]);
      }
      if (MODE == GROWS) {
        const bool last = (c + 1) % p.chunk_blocks == 0 || c + 1 == p.turns;
#pragma unroll
        for (int hd = 0; hd < NH; ++hd) {
          base[hd] += end[hd];
          if (last) {
            const float gh = fminf(exp2_hw(base[hd]), 3.0e38f);
#pragma unroll
            for (int i = 0; i < TPW; ++i) {
#pragma unroll
              for (int r = 0; r < 16; ++r) S[hd][i][r] = __builtin_fmaf(entered[hd][i][r], gh, S[hd][i][r]);
            }
          }
        }
      }
      t3 = t3 == 2 ? 0 : t3 + 1;
    }
    walk_barrier();
    wait_memory<0>();                                        // nothing may land in LDS that is others' by then
    // (a walk after this one writes what was not good once more, and may take the state it starts from out of the same place)
    const auto write_states = [&] {
#pragma unroll
      for (int hd = 0; hd < NH; ++hd) {
        const float g = MODE == FACTORS ? exp2_hw(held[hd]) : 1.0f;
        if (hd && !hp.two) break;
#pragma unroll
        for (int i = 0; i < TPW; ++i) {
#pragma unroll
          for (int q = 0; q < 4; ++q)
            *reinterpret_cast<float4 *>(p.final_states + state0[hd] + 32 * i + 8 * q + 4 * g2) =
                make_float4(S[hd][i][4 * q] * g, S[hd][i][4 * q + 1] * g, S[hd][i][4 * q + 2] * g, S[hd][i][4 * q + 3] * g);
        }
      }
    };
    const bool in_place = p.final_states == p.init;          // (or neither)
    if (!in_place && p.final_states) write_states();
    bool left = false;
    if (MODE == FACTORS && p.final_states) {                 // (a state that no y has seen)
      float most[2] = {};
#pragma unroll
      for (int hd = 0; hd < NH; ++hd) {
#pragma unroll
        for (int i = 0; i < TPW; ++i) {
#pragma unroll
          for (int r = 0; r < 16; r += 2) note_size(most[r >> 1 & 1], S[hd][i][r], S[hd][i][r + 1]);
        }
      }
      left = !__all(most[0] < __builtin_inff() && most[1] < __builtin_inff());
    }
    if (settled(left) && in_place && p.final_states) write_states();
  };
  in_mode(products);
}

// One walk over the heads; whether what it wrote stands.
template <typename E, int NH, int N, int DMODE, bool HAS_Z, bool KEEP_ENTERED>
__device__ __forceinline__ bool walk(const SsdWalkParams &p, unsigned char *lds, const WalkHeads<NH> &hp, bool factor = false) {
  int *again = reinterpret_cast<int *>(lds + WalkLds<NH, N>::AGAIN);
  if (threadIdx.x == 0) *again = 0;
  bool stands;
  const auto settled = [&](bool left_range) {
    if (left_range) *again = 1;
    walk_barrier();
    stands = __builtin_amdgcn_readfirstlane(*again) == 0;
    walk_barrier();                                        // LDS is others' to write
    return stands;
  };
  const auto in_mode = [&](const auto &part) __attribute__((always_inline)) {
    if constexpr (KEEP_ENTERED) part(walk_mode<GROWS>{});
    else if constexpr (std::is_same<E, _Float16>::value) part(walk_mode<ELEMENTS>{});
    else if (factor) part(walk_mode<FACTORS>{});
    else part(walk_mode<ELEMENTS>{});
  };
  if (wave_id_uniform() >= 4) settled(walk_rows<E, NH, N, DMODE, HAS_Z>(p, lds, hp, in_mode));
  else walk_products<E, NH, N>(p, lds, hp, in_mode, settled);
  return stands;
}

constexpr int walk_threads(int nh) { return nh == 2 ? 768 : 512; }

// (xcd_order: neighbouring heads of a batch row, which read the same fragments, go to one XCD.)
template <typename E, int NH, int N, int DMODE, bool HAS_Z>
__global__ __launch_bounds__(walk_threads(NH)) __attribute__((amdgpu_waves_per_eu(NH + 1)))
void ssd_walk_kernel(const SsdWalkParams p) {
  extern __shared__ __align__(16) unsigned char lds[];
  const WalkHeads<NH> all(p, (int)xcd_order(blockIdx.x, p.sets));
  const float A0 = p.A[all.h0], A1 = p.A[all.h1];          // (asked for together with what heads_factor reads)
  constexpr bool F16 = std::is_same<E, _Float16>::value;
  const bool factor = !F16 && !p.in_place && heads_factor(p, all);
  const bool grows0 = A0 > 0.0f, grows1 = A1 > 0.0f;
  const WalkHeads<NH> one(all.b, all.g, grows0 ? all.h1 : all.h0);
  bool stands = !(F16 && p.in_place);
  if (stands && (!grows0 || !grows1)) stands = walk<E, NH, N, DMODE, HAS_Z, false>(p, lds, grows0 == grows1 ? all : one, factor);
  // those that grow, or left the range
  if (stands && !grows0 && !grows1) return;
  wait_memory<0>();                                        // what is written again is written after this
  walk_barrier();
  if constexpr (NH == 1 || N == 64) {
    walk<E, NH, N, DMODE, HAS_Z, true>(p, lds, !stands || grows0 == grows1 ? all : WalkHeads<NH>(all.b, all.g, grows0 ? all.h0 : all.h1));
  } else {
    if (wave_id_uniform() >= walk_threads(1) / WAVE) return;
#pragma nounroll
    for (int second = 0; second < (all.two ? 2 : 1); ++second)
      if (!stands || (second ? grows1 : grows0)) walk<E, 1, N, DMODE, HAS_Z, true>(p, lds, WalkHeads<1>(all.b, all.g, second ? all.h1 : all.h0));
  }
}

template <typename E, int NH, int N>
static int launch_walk(const SsdWalkParams &p, int dmode, hipStream_t s) {
  constexpr int LDS = WalkLds<NH, N>::BYTES;
  const unsigned grid = (unsigned)p.sets;
#define SSM_WALK(DM, HZ)                                                                              \
  {                                                                                                   \
    const auto kernel = ssd_walk_kernel<E, NH, N, DM, HZ>;                                            \
    if (allow_dynamic_lds(kernel, LDS) != hipSuccess) {                                               \
      set_error("ssm_ssd_combined_fwd: cannot reserve %d bytes of LDS", LDS);                         \
      return SSM_ERR_LAUNCH;                                                                          \
    }                                                                                                 \
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(walk_threads(NH)), LDS, s, p);                        \
  }
  if (p.z) {
    if (dmode == 0) SSM_WALK(0, true)
    else if (dmode == 1) SSM_WALK(1, true)
    else SSM_WALK(2, true)
  } else {
    if (dmode == 0) SSM_WALK(0, false)
    else if (dmode == 1) SSM_WALK(1, false)
    else SSM_WALK(2, false)
  }
#undef SSM_WALK
  SSM_CHECK_LAUNCH("ssm_ssd_combined_fwd");
  return SSM_OK;
}

int ssd_walk_forward(SsdWalkParams p, int dmode, bool f16, int nstate, hipStream_t s) {
  p.in_place = p.y == p.x || p.y == p.z;
  const int per_group = p.heads / p.groups;
  // One head per workgroup while every workgroup has a CU of its own, or where heads share nothing: a group of one head is no
  // pair, and 320 or 384 such heads take, two by two (each twice) / one by one, 4 x 4096 steps, 128 states 795 / 753 us, 64
  // states 535 / 510, 4 x 512 101 / 89, chunks of 64 and 64 states 73 / 58, float16 108 / 89 (the preparation of B and C per
  // head with it).  Groups of three, whose third head is done twice: 324 heads x 4096 357 / 369, x 512 49 / 55, 516 x 2048
  // 322 / 304, 768 x 2048 386 / 382.
  const int nh = p.batch * p.heads <= WALK_SINGLES || per_group == 1 ? 1 : 2;
  p.sets = p.batch * p.groups * ((per_group + nh - 1) / nh);
#define SSM_WALK_N(E, NN) return nh == 1 ? launch_walk<E, 1, NN>(p, dmode, s) : launch_walk<E, 2, NN>(p, dmode, s);
  if (f16) {
    if (nstate == 128) SSM_WALK_N(_Float16, 128)
    SSM_WALK_N(_Float16, 64)
  }
  if (nstate == 128) SSM_WALK_N(__bf16, 128)
  SSM_WALK_N(__bf16, 64)
#undef SSM_WALK_N
}

}  // namespace ssm
