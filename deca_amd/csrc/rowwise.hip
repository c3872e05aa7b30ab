// Row-wise softmax / RMSNorm over an [M, N] row-major 16-bit tensor, gfx950.
//
// One code object per (op, shape, dtype, config): every DECA_* macro below is
// a compile-time constant supplied by kernels/rowwise_hip.py, as the reference
// bakes shape and RowConfig into each generated kernel
// (src/kernels/rowwise_tir.py:99-127).
//
//   DECA_OP      0 softmax, 1 rmsnorm
//   DECA_M/N     rows / reduced dimension
//   DECA_BF16    0 float16, 1 bfloat16
//   DECA_TPR     lanes cooperating on one row (16, 32, 64, ... 1024)
//   DECA_RPB     rows per workgroup
//   DECA_VEC     elements per vector access (8 -> 16 B, 4 -> 8 B)
//   DECA_MODE    0 reg (row cached in VGPRs), 1 twopass (row streamed twice)
//   DECA_UNROLL  chunks in flight per twopass iteration
//   DECA_HINT    1: non-temporal loads of read-once data and non-temporal stores
//   DECA_LEAN    1 (reg mode): nothing but the packed row stays in registers between
//                the reduction and the stores -- the fp32 values are computed again
//   DECA_HALF    1 (reg mode, VEC = 8): N is an odd multiple of 4.  Rows then start on 8-byte
//                boundaries only; the accesses are 16 bytes all the same (the hardware asks
//                for 4-byte alignment) but for the last half vector of a row.  RMSNorm fp16
//                3001 x 5124: 14.3 us with 8-byte accesses and 128 lanes a row, 11.4 us with
//                these and a wave a row (3001 x 5120, whose rows are aligned: 10.6); softmax
//                bf16 777 x 65532: 52.0 and 45.9 us
//   DECA_ONLINE  1 (reg mode, VEC = 8, whole waves a row): the first pass takes the chunks of a
//                row as they arrive (see there)
//   DECA_LINES   1 (reg mode, VEC = 8, whole waves a row): the lanes' chunks start at the memory line
//                that the row starts in, so that a wave's accesses are whole lines however the rows
//                lie.  Rows off the lines had every wave touch one more and share it with the next,
//                for 3-12 % of the time: softmax bf16 2048 x 84936 135 us (5.15 TB/s) -> 124, where
//                84992 takes 123; RMSNorm bf16 3001 x 5128 12.3 -> 10.8, 16384 x 4104 46.3 -> 44.6.
//                The weight is read across lines instead, which the L1 serves.
//   DECA_EPS     RMSNorm epsilon
//
// Lane t of a row owns the VEC-element chunks (c * TPR + t) * VEC, so one wave
// touches 64 * VEC * 2 contiguous bytes per access (1 KiB at VEC = 8).
// Reductions: DPP butterflies inside a wave (quad_perm, row_half_mirror,
// row_mirror), v_permlane16_swap / v_permlane32_swap across the 16- and 32-lane
// halves (register exchanges, no LDS pipe), then an LDS exchange between the waves
// of a row.  All math is fp32.
//
// Numerics follow src/kernels/rowwise_tir.py:278-389:
//   softmax: m2 = max(x) * log2e; y = exp2(x * log2e - m2) * (1 / sum)
//   rmsnorm: r = rsqrt(sum(x^2) / N + eps); y = dtype(f32(dtype(x * r)) * f32(w))
#include <hip/hip_runtime.h>

#ifndef DECA_OP
#error "rowwise.hip is a template: define the DECA_* macros"
#endif

#ifndef DECA_HALF
#define DECA_HALF 0
#endif
#define TPR DECA_TPR
#define RPB DECA_RPB
#define VEC DECA_VEC
#define NT (TPR * RPB)
#define SPAN (TPR * VEC)
#ifndef DECA_LINES
#define DECA_LINES 0
#endif
#define LINE 128  // bytes
// elements by which a row may start behind its line
#define LINE_PAD (DECA_LINES ? (DECA_HALF ? 60 : 56) : 0)
#define NCHUNK ((DECA_N + LINE_PAD + SPAN - 1) / SPAN)
#define C_FULL (DECA_N / SPAN)
#define RED_LANES (TPR < 64 ? TPR : 64)
#define NW (TPR / 64 > 0 ? TPR / 64 : 1)

static_assert(DECA_HALF ? (VEC == 8 && DECA_N % 8 == 4 && DECA_MODE == 0) : DECA_N % VEC == 0,
              "N must be a multiple of the vector width, or of half of it (DECA_HALF)");
static_assert(DECA_M % RPB == 0, "M must be a multiple of rows_per_block");
static_assert(NT % 64 == 0 && NT <= 1024, "workgroup must be whole waves");
static_assert(VEC == 8 || VEC == 4 || VEC == 2, "vec");

#if DECA_BF16
typedef __bf16 elem_t;
#else
typedef _Float16 elem_t;
#endif
typedef elem_t vec_t __attribute__((ext_vector_type(VEC)));
#if DECA_HALF
typedef elem_t half_t __attribute__((ext_vector_type(4)));
typedef vec_t mem_t __attribute__((aligned(8)));  // a vector as it lies in memory
#else
typedef vec_t mem_t;
#endif

#ifndef DECA_LEAN
#define DECA_LEAN 0
#endif
#ifndef DECA_ONLINE
#define DECA_ONLINE 0
#endif
// Rows are read and written through a buffer descriptor
#define BUFFER (DECA_ONLINE || DECA_LINES)
static_assert(!BUFFER || (DECA_MODE == 0 && VEC == 8 && TPR % 64 == 0),
              "online, lines: reg mode, 16-byte accesses, whole waves a row");
static_assert(!DECA_ONLINE || DECA_OP == 0, "online: softmax");

#define LOG2E 1.4426950408889634f
#define NEG_INF (-1e30f)

// ---------------------------------------------------------------------------
// cross-lane helpers
// ---------------------------------------------------------------------------
template <int CTRL>
__device__ __forceinline__ float dpp_f(float v) {
  int r = __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true);
  return __builtin_bit_cast(float, r);
}

struct MaxOp {
  __device__ __forceinline__ float operator()(float a, float b) const { return fmaxf(a, b); }
};
struct AddOp {
  __device__ __forceinline__ float operator()(float a, float b) const { return a + b; }
};

// All-reduce over groups of LANES consecutive lanes of a wave64.  Steps 4 and 8
// use mirrors instead of xor: every quad (then every 8 lanes) already holds one
// value, so the mirrored partner supplies the other half's value.
template <int LANES, class Op>
__device__ __forceinline__ float wave_allreduce(float v, Op op) {
  if (LANES >= 2) v = op(v, dpp_f<0xB1>(v));   // quad_perm [1,0,3,2]
  if (LANES >= 4) v = op(v, dpp_f<0x4E>(v));   // quad_perm [2,3,0,1]
  if (LANES >= 8) v = op(v, dpp_f<0x141>(v));  // row_half_mirror
  if (LANES >= 16) v = op(v, dpp_f<0x140>(v)); // row_mirror
  // The last two steps pair 16-lane rows, then the 32-lane halves, with the row
  // swaps of gfx950 (v_permlane16_swap / v_permlane32_swap on two copies of v:
  // one copy ends up with the even rows' values in both rows of a pair, the other
  // with the odd rows'), which stay in the vector ALU instead of going through LDS.
  typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
  if (LANES >= 32) {
    const unsigned u = __builtin_bit_cast(unsigned, v);
    const u32x2 r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    const unsigned even = r.x, odd = r.y;
    v = op(__builtin_bit_cast(float, even), __builtin_bit_cast(float, odd));
  }
  if (LANES >= 64) {
    const unsigned u = __builtin_bit_cast(unsigned, v);
    const u32x2 r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    const unsigned lo = r.x, hi = r.y;
    v = op(__builtin_bit_cast(float, lo), __builtin_bit_cast(float, hi));
  }
  return v;
}

// Reduction of `v` over all TPR lanes of a row.  `red` holds one float per
// wave of the workgroup; with one wave per row it is never touched.
template <class Op>
__device__ __forceinline__ float row_reduce(float v, Op op, float* red, int row_in_block,
                                            int wave_in_row, int lane) {
  v = wave_allreduce<RED_LANES>(v, op);
#if NW > 1
  float* slot = red + row_in_block * NW;
  if (lane == 0) slot[wave_in_row] = v;
  __syncthreads();
  float r = slot[0];
#pragma unroll
  for (int i = 1; i < NW; ++i) r = op(r, slot[i]);
  v = r;
#endif
  return v;
}

// ---------------------------------------------------------------------------
// memory helpers
// ---------------------------------------------------------------------------
// (ONCE is a template parameter: as an argument, the two loads are merged before it is known
// and the non-temporal hint is lost)
template <bool ONCE>
__device__ __forceinline__ vec_t load_vec(const elem_t* p) {
#if DECA_HINT
  if constexpr (ONCE) return __builtin_nontemporal_load(reinterpret_cast<const mem_t*>(p));
#endif
  return *reinterpret_cast<const mem_t*>(p);
}

__device__ __forceinline__ void store_vec(elem_t* p, vec_t v) {
#if DECA_HINT
  __builtin_nontemporal_store(v, reinterpret_cast<mem_t*>(p));
#else
  *reinterpret_cast<mem_t*>(p) = v;
#endif
}

__device__ __forceinline__ float fast_exp2(float v) { return __builtin_amdgcn_exp2f(v); }

// Exponential of an element against the row's max, m2 = max * log2(e).  One rounding of the exponent
// in every pass: the sum and the stores must agree, or the difference of x * log2(e) from its rounded
// product, half a unit of a number as large as the elements, is left in the quotient.  So a pass
// selects behind it what lies in the row: with the select in front, the product is rounded by
// itself there (rows of 50000.0 in fp16: 1.6e-3 instead of 5e-4).
__device__ __forceinline__ float exp2_of(float x, float m2) { return fast_exp2(__builtin_fmaf(x, LOG2E, -m2)); }

template <int AUX>
struct aux_t {
  static constexpr int value = AUX;
};

// ---------------------------------------------------------------------------
// kernel
// ---------------------------------------------------------------------------
extern "C" __global__ void __launch_bounds__(NT)
deca_main(const elem_t* __restrict__ x,
#if DECA_OP == 1
          const elem_t* __restrict__ w,
#endif
          elem_t* __restrict__ y) {
#if NW > 1
  __shared__ float red_lds[2 * RPB * NW];
  float* red0 = red_lds;
  float* red1 = red_lds + RPB * NW;
#else
  float* red0 = nullptr;
  float* red1 = nullptr;
#endif
  const int tid = threadIdx.x;
  const int t = tid % TPR;
  const int rb = tid / TPR;
  const int lane = tid % 64;
  const int wr = t / 64;
  const size_t row_base = (static_cast<size_t>(blockIdx.x) * RPB + rb) * DECA_N;
  const elem_t* xr = x + row_base;
  elem_t* yr = y + row_base;

#if BUFFER
  // All accesses go through a buffer descriptor of the row: a lane offset and a constant per chunk
  // instead of 64-bit addresses, and the range check takes the place of branches: what lies before
  // (offsets that wrap) or behind the row is read as 0 and not written.
  typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
  typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
  constexpr int AUX = DECA_HINT ? 2 : 0;  // non-temporal
  const size_t row_u = (static_cast<size_t>(blockIdx.x) * RPB + __builtin_amdgcn_readfirstlane(rb)) * DECA_N;
  auto row_of = [&](const elem_t* p) __attribute__((always_inline)) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<elem_t*>(p), 0, DECA_N * 2, 0x00027000);
  };
  const auto src = row_of(x + row_u), dst = row_of(y + row_u);
#if DECA_LINES
  // Bytes of the first line before the row, a multiple of a vector (or of a half one), so that only
  // rows of an odd number of halves have vectors that reach over an end.
  const unsigned skip = static_cast<unsigned>(reinterpret_cast<size_t>(x + row_u)) & (LINE - (DECA_HALF ? 8 : 16));
  constexpr int C_FIRST = 1;
#else
  constexpr unsigned skip = 0;
  constexpr int C_FIRST = 0;
#endif
  // chunks that lie in the row for every lane
  auto inner = [&](int c) __attribute__((always_inline)) { return c >= C_FIRST && c < C_FULL; };
  const unsigned lane_off = t * (VEC * 2) - skip;
  unsigned inner_off = lane_off + C_FIRST * (SPAN * 2);
#if DECA_LINES
  asm volatile("" : "+v"(inner_off));  // (opaque, as below)
#endif
  const unsigned wave_off = __builtin_amdgcn_readfirstlane(wr) * (64 * VEC * 2) - skip;
  // Offset of a vector of a chunk at an end of the row.  (Opaque: a sum that wraps does so in the
  // register.  Split, the instruction's own offset would be added to a register that lies before the
  // row; what the range check makes of that is not relied on.)
  auto end_off = [&](int c) __attribute__((always_inline)) {
    unsigned off = lane_off + c * (SPAN * 2);
    asm volatile("" : "+v"(off));
    return off;
  };
  // The vectors that reach over an end of the row (DECA_HALF): the half inside is accessed by itself.
  constexpr unsigned NOWHERE = 0xfffffff0u, LAST_HALF = DECA_N * 2u - 8u;
  auto over_start = [&](int c) __attribute__((always_inline)) {
    return DECA_HALF && DECA_LINES && c == 0 && lane_off == 0u - 8u;
  };
  auto over_end = [&](int c) __attribute__((always_inline)) {
    return DECA_HALF && c >= C_FULL && lane_off + c * (SPAN * 2) == LAST_HALF;
  };
  struct ends_t {
    u32x2 start, end;
  };
  auto ends_of = [&](auto rsrc, auto aux) __attribute__((always_inline)) {
    ends_t e = {};
#if DECA_HALF
    // (by all lanes of the waves that hold an end: a branch of some lanes would wait for the others)
    constexpr int HINT = decltype(aux)::value;
    if (DECA_LINES && wave_off == 0u - skip)
      e.start = __builtin_amdgcn_raw_buffer_load_b64(rsrc, over_start(0) ? 0u : NOWHERE, 0, HINT);
    bool lane_end = false, wave_end = false;
#pragma unroll
    for (int c = C_FULL; c < NCHUNK; ++c) {
      lane_end |= over_end(c);
      wave_end |= LAST_HALF - (wave_off + c * (SPAN * 2)) < 64u * VEC * 2;
    }
    if (wave_end) e.end = __builtin_amdgcn_raw_buffer_load_b64(rsrc, lane_end ? LAST_HALF : NOWHERE, 0, HINT);
#endif
    return e;
  };
  auto elem_ok = [&](int c, int i) __attribute__((always_inline)) {
    return inner(c) || lane_off + c * (SPAN * 2) + (DECA_HALF && i >= 4 ? 8 : 0) < DECA_N * 2u;
  };
  auto fetch = [&](auto rsrc, int c, auto aux) __attribute__((always_inline)) {
    constexpr int HINT = decltype(aux)::value;
    if (inner(c))
      return __builtin_bit_cast(
          vec_t, __builtin_amdgcn_raw_buffer_load_b128(rsrc, inner_off, (c - C_FIRST) * (SPAN * 2), HINT));
    const unsigned off = end_off(c);
    return __builtin_bit_cast(
        vec_t, __builtin_amdgcn_raw_buffer_load_b128(rsrc, over_end(c) ? NOWHERE : off, 0, HINT));
  };
  auto join = [&](vec_t x, const ends_t& e, int c) __attribute__((always_inline)) {
    u32x4 v = __builtin_bit_cast(u32x4, x);
    if (over_start(c)) v = u32x4{0, 0, e.start.x, e.start.y};
    if (over_end(c)) v = u32x4{e.end.x, e.end.y, 0, 0};
    return __builtin_bit_cast(vec_t, v);
  };
  // (of a wave: whether any of its lanes holds elements of the chunk)
  auto in_row = [&](int c) __attribute__((always_inline)) {
    return c < C_FULL || static_cast<int>(wave_off + c * (SPAN * 2)) < DECA_N * 2;
  };
  const ends_t x_ends = ends_of(src, aux_t<AUX>());
  auto load_x = [&](int c) __attribute__((always_inline)) { return fetch(src, c, aux_t<AUX>()); };
  // (behind all loads: what has to wait for one ends where another is conditional)
  auto join_x = [&](vec_t(&row)[NCHUNK]) __attribute__((always_inline)) {
#pragma unroll
    for (int c = 0; c < NCHUNK; ++c) row[c] = join(row[c], x_ends, c);
  };
#if DECA_OP == 1
  const auto weights = row_of(w);  // (as long as a row)
  const ends_t w_ends = ends_of(weights, aux_t<0>());
  auto load_w = [&](const elem_t*, int c) __attribute__((always_inline)) {
    return join(fetch(weights, c, aux_t<0>()), w_ends, c);
  };
#endif
  // (Stores carry all of their offset in the lane's address: after one with an offset in a scalar
  // register the compiler leaves out the wait that its data needs before they are overwritten.)
  ends_t y_ends = {};
  auto store_row = [&](int c, vec_t v) __attribute__((always_inline)) {
    const u32x4 u = __builtin_bit_cast(u32x4, v);
    if (inner(c)) {
      __builtin_amdgcn_raw_buffer_store_b128(u, dst, inner_off + (c - C_FIRST) * (SPAN * 2), 0, AUX);
      return;
    }
    const unsigned off = end_off(c);
    __builtin_amdgcn_raw_buffer_store_b128(u, dst, over_end(c) ? NOWHERE : off, 0, AUX);
    if (DECA_LINES && c == 0) y_ends.start = u32x2{u.z, u.w};
    if (over_end(c)) y_ends.end = u32x2{u.x, u.y};
  };
  auto store_ends = [&]() __attribute__((always_inline)) {
#if DECA_HALF
    if (over_start(0)) __builtin_amdgcn_raw_buffer_store_b64(y_ends.start, dst, 0, 0, AUX);
    bool lane_end = false;
#pragma unroll
    for (int c = C_FULL; c < NCHUNK; ++c) lane_end |= over_end(c);
    if (lane_end) __builtin_amdgcn_raw_buffer_store_b64(y_ends.end, dst, LAST_HALF, 0, AUX);
#endif
  };
#else
  auto col = [&](int c) { return (c * TPR + t) * VEC; };
  // Chunks >= C_FULL are out of the row for the upper lanes.
  auto in_row = [&](int c) { return c < C_FULL || col(c) < DECA_N; };
#if DECA_HALF
  // The last vector of a row: its upper half is beyond the end.
  auto whole = [&](int c) { return c < C_FULL || col(c) + VEC <= DECA_N; };
  auto elem_ok = [&](int c, int i) { return i < 4 ? in_row(c) : whole(c); };
  auto load_half = [&](const elem_t* base, int c) {
    const half_t h = *reinterpret_cast<const half_t*>(base + col(c));
    const half_t none = {};
    return __builtin_shufflevector(h, none, 0, 1, 2, 3, 4, 5, 6, 7);
  };
  auto load_x = [&](int c) { return whole(c) ? load_vec<true>(xr + col(c)) : load_half(xr, c); };
  auto load_w = [&](const elem_t* w, int c) { return whole(c) ? load_vec<false>(w + col(c)) : load_half(w, c); };
  auto store_row = [&](int c, vec_t v) {
    if (whole(c))
      store_vec(yr + col(c), v);
    else
      *reinterpret_cast<half_t*>(yr + col(c)) = __builtin_shufflevector(v, v, 0, 1, 2, 3);
  };
#else
  auto elem_ok = [&](int c, int) { return in_row(c); };
  auto load_x = [&](int c) { return load_vec<true>(xr + col(c)); };
  auto load_w = [&](const elem_t* w, int c) { return load_vec<false>(w + col(c)); };
  auto store_row = [&](int c, vec_t v) { store_vec(yr + col(c), v); };
#endif

#endif  // BUFFER

#if DECA_ONLINE
  // ------------------------- reg mode, chunks as they arrive -------------------------
  // Softmax: exponentials against the lane's max so far, whose sum is rescaled when that grows,
  // so that behind the last chunk only the reduction is left, of max and sum in one exchange.  A
  // row whose workgroup has a CU (nearly) to itself otherwise adds two passes of vector work over
  // the row to the time of its loads and stores, with the memory idle (bf16, 1024 lanes a row:
  // 1024 x 128256 105.6 -> 96.4 us, 5.45 TB/s; 2020 x 63956 99.1 -> 94.6; 275 x 118396 41.7 -> 34.8).
  // Bound then: the last exchange, the exponentials of the stores and the next workgroup's start,
  // which other rows of the CU only hide in part (a copy of the same size runs at 6.4 TB/s).
  vec_t xh[NCHUNK];
#pragma unroll
  for (int c = 0; c < NCHUNK; ++c) xh[c] = in_row(c) ? load_x(c) : vec_t{};
  // (all requests first: the scheduler would put off the later ones until the first pass is under
  // way, 91.5 -> 93.6 us for 2048 x 65536 bf16)
  __builtin_amdgcn_sched_barrier(0);
  join_x(xh);
  // The sums are rescaled by the difference of the rounded products max * log2(e) that the
  // exponents were formed with, not of the maxima: as in the two-pass form, that rounding then
  // cancels in the quotient, however large the elements are.  Beyond 1e9 it makes exponentials of
  // the largest elements themselves infinite, and a lane may hold no other ones (masked by a large
  // negative number): held finite, so that the rescale makes them 0 and not NaN.  (Opaque to the
  // optimiser, which would put the product back into the exponents and knows no infinities.)
  auto scaled = [&](float v) __attribute__((always_inline)) {
    float p = v * LOG2E;
    asm volatile("" : "+v"(p));
    return p;
  };
  auto finite = [&](float v) __attribute__((always_inline)) {
    unsigned u = __builtin_bit_cast(unsigned, v);
    asm volatile("" : "+v"(u));
    return __builtin_bit_cast(float, u == 0x7f800000u ? 0x7f7fffffu : u);
  };
  float m = NEG_INF, m2 = NEG_INF * LOG2E, sum = 0.0f;
  constexpr int AT_ONCE = 2;  // chunks per rescale of the sum
#pragma unroll
  for (int c0 = 0; c0 < NCHUNK; c0 += AT_ONCE) {
#pragma unroll
    for (int c = c0; c < c0 + AT_ONCE && c < NCHUNK; ++c)
#pragma unroll
      for (int i = 0; i < VEC; ++i) m = fmaxf(m, elem_ok(c, i) ? static_cast<float>(xh[c][i]) : NEG_INF);
    const float before = m2;
    m2 = scaled(m);
    float acc = 0.0f;
#pragma unroll
    for (int c = c0; c < c0 + AT_ONCE && c < NCHUNK; ++c)
#pragma unroll
      for (int i = 0; i < VEC; ++i) {
        const float e = exp2_of(static_cast<float>(xh[c][i]), m2);
        acc += elem_ok(c, i) ? e : 0.0f;
      }
    sum = finite(sum * fast_exp2(before - m2) + acc);
  }
  const float top2 = wave_allreduce<RED_LANES>(m2, MaxOp());
  sum = wave_allreduce<RED_LANES>(sum * fast_exp2(m2 - top2), AddOp());
  m2 = top2;
#if NW > 1
  float* tops = red0 + rb * NW;
  float* sums = red1 + rb * NW;
  if (lane == 0) {
    tops[wr] = m2;
    sums[wr] = finite(sum);
  }
  __syncthreads();
  float tops2[NW];
#pragma unroll
  for (int i = 0; i < NW; ++i) {
    tops2[i] = tops[i];
    m2 = fmaxf(m2, tops2[i]);
  }
  sum = 0.0f;
#pragma unroll
  for (int i = 0; i < NW; ++i) sum += sums[i] * fast_exp2(tops2[i] - m2);
#endif
  const float inv = __builtin_amdgcn_rcpf(sum);
  // (nothing but the packed row is kept from the first pass)
#pragma unroll
  for (int c = 0; c < NCHUNK; ++c) asm volatile("" : "+v"(xh[c]));
#pragma unroll
  for (int c = 0; c < NCHUNK; ++c) {
    vec_t o;
#pragma unroll
    for (int i = 0; i < VEC; ++i)
      o[i] = static_cast<elem_t>(exp2_of(static_cast<float>(xh[c][i]), m2) * inv);
    if (in_row(c)) store_row(c, o);
  }
  store_ends();

#elif DECA_MODE == 0
  // ------------------------------ reg mode ------------------------------
  vec_t xh[NCHUNK];
#pragma unroll
  for (int c = 0; c < NCHUNK; ++c) {
    if (in_row(c)) xh[c] = load_x(c);
#if BUFFER
    else xh[c] = vec_t{};
#endif
  }
#if BUFFER
  join_x(xh);
#endif

#if DECA_OP == 0
  float m = NEG_INF;
#pragma unroll
  for (int c = 0; c < NCHUNK; ++c) {
#pragma unroll
    for (int i = 0; i < VEC; ++i) m = fmaxf(m, elem_ok(c, i) ? static_cast<float>(xh[c][i]) : NEG_INF);
  }
  const float m2 = row_reduce(m, MaxOp(), red0, rb, wr, lane) * LOG2E;
#if DECA_LEAN
  // (see below: the fp32 conversions of the max pass are not kept for the sum)
#pragma unroll
  for (int c = 0; c < NCHUNK; ++c) asm volatile("" : "+v"(xh[c]));
#endif
  float s = 0.0f;
#pragma unroll
  for (int c = 0; c < NCHUNK; ++c) {
#pragma unroll
    for (int i = 0; i < VEC; ++i) {
      const float e = exp2_of(static_cast<float>(xh[c][i]), m2);
      s += elem_ok(c, i) ? e : 0.0f;
    }
  }
  const float inv = __builtin_amdgcn_rcpf(row_reduce(s, AddOp(), red1, rb, wr, lane));
#if DECA_LEAN
  // The optimiser would keep the exponentials of the sum alive for the stores
  // (2 VGPRs per element on top of the packed row).  Reading the row through an
  // opaque copy makes it compute them again from the same bits instead.
#pragma unroll
  for (int c = 0; c < NCHUNK; ++c) asm volatile("" : "+v"(xh[c]));
#elif BUFFER
  // The same for the chunks at the ends of the row: the chunks between are stored meanwhile.  (All
  // kept, the row leaves in one burst: bf16 22303 x 6008 84.7 -> 89.7 us, 10520 x 18824 127.8 -> 132.9;
  // level on half of 28 shapes.)
#pragma unroll
  for (int c = 0; c < NCHUNK; ++c)
    if (!inner(c)) asm volatile("" : "+v"(xh[c]));
#endif
#pragma unroll
  for (int c = 0; c < NCHUNK; ++c) {
    if (in_row(c)) {
      vec_t o;
#pragma unroll
      for (int i = 0; i < VEC; ++i)
        o[i] = static_cast<elem_t>(exp2_of(static_cast<float>(xh[c][i]), m2) * inv);
      store_row(c, o);
    }
  }
#else
  float ss = 0.0f;
#pragma unroll
  for (int c = 0; c < NCHUNK; ++c) {
#pragma unroll
    for (int i = 0; i < VEC; ++i) {
      // (a buffer load beyond the row returns 0)
      const float v = BUFFER || elem_ok(c, i) ? static_cast<float>(xh[c][i]) : 0.0f;
      ss += v * v;
    }
  }
  ss = row_reduce(ss, AddOp(), red0, rb, wr, lane);
  const float r = __builtin_amdgcn_rsqf(ss * (1.0f / DECA_N) + static_cast<float>(DECA_EPS));
#if DECA_LEAN
  // as above: the fp32 conversions of the row are made again, not kept
#pragma unroll
  for (int c = 0; c < NCHUNK; ++c) asm volatile("" : "+v"(xh[c]));
#endif
#pragma unroll
  for (int c = 0; c < NCHUNK; ++c) {
    if (in_row(c)) {
      const vec_t wv = load_w(w, c);
      vec_t o;
#pragma unroll
      for (int i = 0; i < VEC; ++i) {
        const float normed = static_cast<float>(static_cast<elem_t>(static_cast<float>(xh[c][i]) * r));
        o[i] = static_cast<elem_t>(normed * static_cast<float>(wv[i]));
      }
      store_row(c, o);
    }
  }
#endif
#if BUFFER
  store_ends();
#endif

#else
  // ----------------------------- twopass mode -----------------------------
  constexpr int U = DECA_UNROLL;
  constexpr int N_LOOP = C_FULL / U;  // iterations whose U chunks are all in the row

#if DECA_OP == 0
  float run_m = NEG_INF;  // running max, already scaled by log2e
  float run_s = 0.0f;
  auto online = [&](const vec_t* v, const bool* ok, int n) {
    float mx = run_m;
#pragma unroll
    for (int u = 0; u < n; ++u)
#pragma unroll
      for (int i = 0; i < VEC; ++i)
        mx = fmaxf(mx, ok[u] ? static_cast<float>(v[u][i]) * LOG2E : NEG_INF);
    float acc = 0.0f;
#pragma unroll
    for (int u = 0; u < n; ++u)
#pragma unroll
      for (int i = 0; i < VEC; ++i)
        acc += fast_exp2((ok[u] ? static_cast<float>(v[u][i]) * LOG2E : NEG_INF) - mx);
    run_s = run_s * fast_exp2(run_m - mx) + acc;
    run_m = mx;
  };
#else
  float run_ss = 0.0f;
  auto online = [&](const vec_t* v, const bool* ok, int n) {
    float acc = 0.0f;
#pragma unroll
    for (int u = 0; u < n; ++u)
#pragma unroll
      for (int i = 0; i < VEC; ++i) {
        const float f = ok[u] ? static_cast<float>(v[u][i]) : 0.0f;
        acc += f * f;
      }
    run_ss += acc;
  };
#endif

  // pass 1: the row is read again soon, so it is loaded with the default policy
  for (int g = 0; g < N_LOOP; ++g) {
    vec_t v[U];
    bool ok[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      v[u] = load_vec<false>(xr + col(g * U + u));
      ok[u] = true;
    }
    online(v, ok, U);
  }
#pragma unroll
  for (int c = N_LOOP * U; c < NCHUNK; ++c) {
    vec_t v[1];
    bool ok[1];
    ok[0] = in_row(c);
    if (ok[0]) v[0] = load_vec<false>(xr + col(c));
    online(v, ok, 1);
  }

#if DECA_OP == 0
  const float m2 = row_reduce(run_m, MaxOp(), red0, rb, wr, lane);
  const float tot = row_reduce(run_s * fast_exp2(run_m - m2), AddOp(), red1, rb, wr, lane);
  const float inv = __builtin_amdgcn_rcpf(tot);
  auto emit = [&](int c, vec_t v) {
    vec_t o;
#pragma unroll
    for (int i = 0; i < VEC; ++i)
      o[i] = static_cast<elem_t>(fast_exp2(static_cast<float>(v[i]) * LOG2E - m2) * inv);
    store_vec(yr + col(c), o);
  };
#else
  const float tot = row_reduce(run_ss, AddOp(), red0, rb, wr, lane);
  const float r = __builtin_amdgcn_rsqf(tot * (1.0f / DECA_N) + static_cast<float>(DECA_EPS));
  auto emit = [&](int c, vec_t v) {
    const vec_t wv = *reinterpret_cast<const vec_t*>(w + col(c));
    vec_t o;
#pragma unroll
    for (int i = 0; i < VEC; ++i) {
      const float normed = static_cast<float>(static_cast<elem_t>(static_cast<float>(v[i]) * r));
      o[i] = static_cast<elem_t>(normed * static_cast<float>(wv[i]));
    }
    store_vec(yr + col(c), o);
  };
#endif

  // pass 2: last use of the row
  for (int g = 0; g < N_LOOP; ++g) {
    vec_t v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] = load_vec<true>(xr + col(g * U + u));
#pragma unroll
    for (int u = 0; u < U; ++u) emit(g * U + u, v[u]);
  }
#pragma unroll
  for (int c = N_LOOP * U; c < NCHUNK; ++c) {
    if (in_row(c)) emit(c, load_vec<true>(xr + col(c)));
  }
#endif
}
