// Float-activation products (Q8_0 / Q5_0 weights, fp32 activations) of 2..128 rows on the bf16
// matrix cores.
//
// A weight is an int8 code times its 32-column block's f16 scale d. A code (at most 8 significant
// bits) is a bf16 exactly, and an fp32 activation is the sum of three bf16 parts (8 significant bits
// each, fx_split), exactly down to |x| = 2^-110, so one block's sum over code * x takes three
// v_mfma_f32_16x16x32_bf16 into one fp32 accumulator with every product exact, and the row then
// takes acc = fma(d, sum, acc): the arithmetic of the per-lane kernels (quant.rs:48-161,
// quant_multi.rs:168-190) in an order of its own. Against float64 its error is the fp32 matrix
// cores' (v_mfma_f32_16x16x4f32, eight a block, the form before this one) or less, at 48 matrix-core
// cycles a block and 16 x 16 outputs instead of 256. Below 2^-110 the third part would need steps
// finer than bf16's smallest, 2^-133, and an infinity has no parts: a part of a row that met either
// walks its blocks again with a split that takes them whole (looked for once a part, not once a
// block: 3072 -> 1024 by 9 rows 8.2 -> 7.6 us, Qwen3-0.6B's 128-row layers 680 -> 646 us for eight).
//
// Order of a row's sum, the same for every number of rows in the pass (2..128) and every tile
// shape: its blocks are cut in P contiguous parts (fx_parts of the blocks a row), each part's
// blocks in order, then the parts in order. So a prefill pass of 128 rows gives the bits of its
// rows in passes of 2..16.
//
// Loads. In the operand layout consecutive lanes hold different rows, so a load straight into it is
// 64 separate requests of 8 or 16 bytes, and one CU's address unit takes about one a cycle: with
// such loads Qwen3-0.6B's 3072 -> 1024 product of 128 rows took 19.3 us whatever its occupancy and
// prefetch depth. So a wavefront loads two blocks at a time along the rows (64 bytes of codes, 256
// of x a row: 16 or fewer requests an instruction), parks them in its own LDS (swizzled, no
// barrier) and reads the operands there, the next stage's loads (one tile: the next two's) in flight meanwhile. What
// bounds the kernels then is the arrival of the weights at 2..16 rows (a launch moves 2-6 MB) and
// the vector instructions: the split of x (48 of ~71 a block when a wavefront has one tile) and the
// int8 -> bf16 conversion, so in prefill passes a wavefront takes NT tiles of 16 rows x NV groups of
// 16 vectors and pays each once per NT x NV products.
#include "decode_dev.h"
#include "fx.h"
#include "norm_dev.h"

namespace spx {

typedef __bf16 bf8v __attribute__((ext_vector_type(8)));
template <int P>
constexpr int FX_NW = P > 8 ? P : 8;  // wavefronts a workgroup: FX_NW / P row groups of P parts
// Wavefronts a SIMD that the registers are held to (no spills but four registers in Q5_0's four-tile form).
template <int P, int NT, int NV>
constexpr int FX_WPE = P > 8 || NT * NV <= 2 || NV == 1 ? 4 : 2;

__device__ __forceinline__ f4v fx_mfma(uint4 a, uint4 b, f4v c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf8v, a), __builtin_bit_cast(bf8v, b), c, 0, 0, 0);
}
// The high halves of two words: (hi16(b) << 16) | hi16(a).
__device__ __forceinline__ uint32_t fx_hi2(uint32_t a, uint32_t b) { return __builtin_amdgcn_perm(b, a, 0x07060302u); }

struct FxX {
  uint4 hi, mid, lo;
};
// Eight fp32 values as three bf16 parts each: the top 16 bits of x, of the rest r = x - hi (exact,
// at most 16 significant bits) and of r - mid (at most 8). Two kinds of value come out wrong: of an
// infinite x the rest is a NaN, and below |x| = 2^-110 the last part can need steps finer than
// bf16's smallest, 2^-133; such bits are left in the low half of cut, and FIX (rest: 2^100 times what
// was cut off, at most 16 significant bits) splits both kinds whole. All others have the same parts
// either way.
template <bool FIX>
__device__ __forceinline__ FxX fx_split(float4 a, float4 b, uint32_t &cut, FxX *rest = nullptr) {
  const float x[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
  uint32_t h[8], m[8], l[8];
#pragma unroll
  for (int i = 0; i < 8; i++) {
    h[i] = __float_as_uint(x[i]);
    float r = x[i] - __uint_as_float(h[i] & 0xffff0000u);
    if (FIX) r = fabsf(x[i]) == INFINITY ? 0.0f : r;
    m[i] = __float_as_uint(r);
    l[i] = __float_as_uint(r - __uint_as_float(m[i] & 0xffff0000u));
    cut |= l[i];
  }
  auto pack = [](const uint32_t (&v)[8]) { return make_uint4(fx_hi2(v[0], v[1]), fx_hi2(v[2], v[3]), fx_hi2(v[4], v[5]), fx_hi2(v[6], v[7])); };
  const FxX o{pack(h), pack(m), pack(l)};
  if (FIX) {
#pragma unroll
    for (int i = 0; i < 8; i++) {
      const float t = fabsf(x[i]) < 0x1p-100f ? (__uint_as_float(l[i]) - __uint_as_float(l[i] & 0xffff0000u)) * 0x1p100f : 0.0f;
      h[i] = __float_as_uint(t);
      m[i] = __float_as_uint(t - __uint_as_float(h[i] & 0xffff0000u));
    }
    rest->hi = pack(h);
    rest->mid = pack(m);
  }
  return o;
}

// Eight codes as bf16: the floats of small integers, whose low halves are zero.
template <class F>
__device__ __forceinline__ uint4 fx_codes(F code) {
  uint32_t f[8];
#pragma unroll
  for (int i = 0; i < 8; i++) f[i] = __float_as_uint((float)code(i));
  return make_uint4(fx_hi2(f[0], f[1]), fx_hi2(f[2], f[3]), fx_hi2(f[4], f[5]), fx_hi2(f[6], f[7]));
}

// Two blocks (u = 0, 1) of one 16-row tile: as a wavefront loads them (lane: block (lane >> 1) & 1 of
// row lane >> 2; g: its index, relative to block g0 of the planes), in its LDS, and as operands:
// row j = lane & 15, columns 8 kq .. + 7, kq = lane >> 4.
template <int T> struct FxW;
template <> struct FxW<T_Q8_0> {
  static constexpr int BYTES = 1024 + 64;  // codes [row][4 pieces of 16 bytes, piece c at c ^ (row >> 2)], d [row][u]
  uint4 c;
  uint16_t d;
  __device__ __forceinline__ void load(const Planes &pl, int64_t g0, uint32_t g) {
    const int lane = threadIdx.x & 63;
    c = gld<uint4>(pl.p0 + g0 * 32 + (size_t)(g * 32 + 16 * (lane & 1)));
    d = gld<uint16_t>(pl.p3 + g0 * 2 + (size_t)(g * 2));
  }
  __device__ __forceinline__ void park(SPX_L uint8_t *s) const {
    const int lane = threadIdx.x & 63;
    lst<uint4>(s + (lane >> 2) * 64 + (((lane & 3) ^ (lane >> 4)) * 16), c);
    lst<uint16_t>(s + 1024 + (lane >> 1) * 2, d);
  }
  static __device__ __forceinline__ uint4 codes(const SPX_L uint8_t *s, int u, int j, int kq) {
    const uint2 w = lld<uint2>(s + j * 64 + (((2 * u + (kq >> 1)) ^ (j >> 2)) * 16) + 8 * (kq & 1));
    return fx_codes([&](int i) { return (int8_t)((i < 4 ? w.x : w.y) >> (8 * (i & 3))); });
  }
  static __device__ __forceinline__ float scale(const SPX_L uint8_t *s, int u, int j) { return h2f(lld<uint16_t>(s + 1024 + (2 * j + u) * 2)); }
};
template <> struct FxW<T_Q5_0> {  // columns 0..15: low nibbles, 16..31: high nibbles of the 16 bytes; bit e of the high-bit word is column e's
  static constexpr int BYTES = 512 + 128 + 64;  // nibbles [row][2 x 16 bytes], high bits [row][u], d [row][u]
  uint2 c;
  uint32_t qh;
  uint16_t d;
  __device__ __forceinline__ void load(const Planes &pl, int64_t g0, uint32_t g) {
    const int lane = threadIdx.x & 63;
    c = gld<uint2>(pl.p0 + g0 * 16 + (size_t)(g * 16 + 8 * (lane & 1)));
    qh = gld<uint32_t>(pl.p1 + g0 * 4 + (size_t)(g * 4));
    d = gld<uint16_t>(pl.p3 + g0 * 2 + (size_t)(g * 2));
  }
  __device__ __forceinline__ void park(SPX_L uint8_t *s) const {
    const int lane = threadIdx.x & 63;
    lst<uint2>(s + lane * 8, c);
    lst<uint32_t>(s + 512 + (lane >> 1) * 4, qh);
    lst<uint16_t>(s + 640 + (lane >> 1) * 2, d);
  }
  static __device__ __forceinline__ uint4 codes(const SPX_L uint8_t *s, int u, int j, int kq) {
    const uint2 w = lld<uint2>(s + j * 32 + 16 * u + 8 * (kq & 1));
    const uint32_t b = lld<uint32_t>(s + 512 + (2 * j + u) * 4) >> (8 * kq), sh = 4 * (kq >> 1);
    // bits 0..3 (4..7) of b to bit 4 of bytes 0..3: bit i of a nibble times 1 + 2^7 + 2^14 + 2^21
    const uint32_t q[2] = {((w.x >> sh) & 0x0f0f0f0fu) | ((((b & 15u) * 0x00204081u) & 0x01010101u) << 4),
                           ((w.y >> sh) & 0x0f0f0f0fu) | (((((b >> 4) & 15u) * 0x00204081u) & 0x01010101u) << 4)};
    return fx_codes([&](int i) { return (int)((q[i >> 2] >> (8 * (i & 3))) & 0xffu) - 16; });
  }
  static __device__ __forceinline__ float scale(const SPX_L uint8_t *s, int u, int j) { return h2f(lld<uint16_t>(s + 640 + (2 * j + u) * 2)); }
};

// LDS of one wavefront's two blocks: NT tiles, then NV groups of 16 vectors x 64 floats (row r's
// 16-byte pieces c at c ^ r).
template <int T, int NT, int NV>
constexpr int FX_STAGE = NT * FxW<T>::BYTES + NV * 4096;

// Where a wavefront's loads of x start: vector 4 i + (lane >> 4) of group v, i = 0..3 (byte offsets
// from x); row(k) = the row of x that vector k of the workgroup is.
template <int NV, class F>
__device__ __forceinline__ void fx_xrows(uint32_t (&xo)[NV][4], F row, int ld) {
#pragma unroll
  for (int v = 0; v < NV; v++)
#pragma unroll
    for (int i = 0; i < 4; i++) xo[v][i] = (uint32_t)row(16 * v + 4 * i + (int)((threadIdx.x & 63) >> 4)) * (uint32_t)ld * 4u;
}
// The first block of lane's row of a tile (FxW::load's g less the block), the rows r0 .. r0 + 15 of at most
// rows, blocks counted from row rf.
__device__ __forceinline__ uint32_t fx_wrows(int r0, int rows, int rf, int nb) {
  return (uint32_t)(min(r0 + (int)((threadIdx.x & 63) >> 2), rows - 1) - rf) * (uint32_t)nb;
}

// One wavefront's part: blocks [b0, b1) of NT 16-row tiles against NV groups of 16 vectors.
// Tile t's planes are pl[t / TB], counted from block g0[t / TB] (both wave-uniform). s: the
// wavefront's LDS (FX_STAGE bytes). acc[t][v][q]: row lane & 15 of vector 4 (lane >> 4) + q.
template <int T, int NT, int NV, int TB>
__device__ __forceinline__ void fx_part(SPX_L uint8_t *s, const Planes *pl, const int64_t *g0, const uint32_t (&go)[NT], const float *x,
                                        const uint32_t (&xo)[NV][4], int b0, int b1, f4v (&acc)[NT][NV]) {
  struct Raw {
    FxW<T> w[NT];
    float4 x[NV][4];
  };
  const int lane = threadIdx.x & 63, j = lane & 15, kq = lane >> 4;
  SPX_L uint8_t *sx = s + NT * FxW<T>::BYTES;
  auto clear = [&]() {
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
      for (int v = 0; v < NV; v++) acc[t][v] = f4v{0.0f, 0.0f, 0.0f, 0.0f};
  };
  clear();
  const uint8_t *xb = reinterpret_cast<const uint8_t *>(x);
  auto load = [&](Raw &r, int b) {
    const uint32_t c = (uint32_t)min(b + 1, b1 - 1), bw = (lane & 2) ? c : (uint32_t)b;
#pragma unroll
    for (int t = 0; t < NT; t++) r.w[t].load(pl[t / TB], g0[t / TB], go[t] + bw);
    const uint32_t xc = ((lane & 8) ? c : (uint32_t)b) * 128u + 16u * (lane & 7);
#pragma unroll
    for (int v = 0; v < NV; v++)
#pragma unroll
      for (int i = 0; i < 4; i++) r.x[v][i] = gld<float4>(xb + (size_t)(xo[v][i] + xc));
  };
  auto park = [&](const Raw &r) {
    __builtin_amdgcn_wave_barrier();  // (one wavefront's LDS accesses run in order)
#pragma unroll
    for (int t = 0; t < NT; t++) r.w[t].park(s + t * FxW<T>::BYTES);
#pragma unroll
    for (int v = 0; v < NV; v++)
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const int row = 4 * i + (lane >> 4);
        lst<float4>(sx + v * 4096 + row * 256 + ((lane & 15) ^ row) * 16, r.x[v][i]);
      }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  };
  uint32_t cut = 0;
  auto work = [&](int u) {
    FxX xs[NV];
#pragma unroll
    for (int v = 0; v < NV; v++) {
      const SPX_L uint8_t *xr = sx + v * 4096 + j * 256;
      xs[v] = fx_split<false>(lld<float4>(xr + (((8 * u + 2 * kq) ^ j) * 16)), lld<float4>(xr + (((8 * u + 2 * kq + 1) ^ j) * 16)), cut);
    }
#pragma unroll
    for (int t = 0; t < NT; t++) {
      const SPX_L uint8_t *st = s + t * FxW<T>::BYTES;
      const uint4 w = FxW<T>::codes(st, u, j, kq);
      const float d = FxW<T>::scale(st, u, j);
#pragma unroll
      for (int v = 0; v < NV; v++) {
        f4v m = fx_mfma(xs[v].lo, w, f4v{0.0f, 0.0f, 0.0f, 0.0f});
        m = fx_mfma(xs[v].mid, w, m);
        m = fx_mfma(xs[v].hi, w, m);
#pragma unroll
        for (int q = 0; q < 4; q++) acc[t][v][q] = fmaf(d, m[q], acc[t][v][q]);
      }
    }
  };
  // The same with the values that it gets wrong whole: the bits of work for a vector without any.
  auto work_fix = [&](int u) {
#pragma unroll
    for (int v = 0; v < NV; v++) {
      const SPX_L uint8_t *xr = sx + v * 4096 + j * 256;
      FxX xr2;
      const FxX xs = fx_split<true>(lld<float4>(xr + (((8 * u + 2 * kq) ^ j) * 16)), lld<float4>(xr + (((8 * u + 2 * kq + 1) ^ j) * 16)), cut, &xr2);
#pragma unroll
      for (int t = 0; t < NT; t++) {
        __builtin_amdgcn_sched_barrier(0);  // (one tile's registers at a time)
        const SPX_L uint8_t *st = s + t * FxW<T>::BYTES;
        const uint4 w = FxW<T>::codes(st, u, j, kq);
        const float d = FxW<T>::scale(st, u, j);
        const f4v z{0.0f, 0.0f, 0.0f, 0.0f}, m = fx_mfma(xs.hi, w, fx_mfma(xs.mid, w, fx_mfma(xs.lo, w, z))), c = fx_mfma(xr2.hi, w, fx_mfma(xr2.mid, w, z));
#pragma unroll
        for (int q = 0; q < 4; q++) {
          acc[t][v][q] = fmaf(d, m[q], acc[t][v][q]);
          if (c[q] != 0.0f) acc[t][v][q] = fmaf(d, c[q] * 0x1p-100f, acc[t][v][q]);
        }
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  if (b0 >= b1) return;
  if constexpr (NT * NV > 1) {  // the next stage's loads cover this one's products (other wavefronts' too)
    Raw r;
    load(r, b0);
    for (int b = b0; b < b1; b += 2) {
      park(r);
      if (b + 2 < b1) load(r, b + 2);
      work(0);
      if (b + 1 < b1) work(1);
    }
  } else {  // one tile: two stages ahead
    Raw ra, rb;
    load(ra, b0);
    if (b0 + 2 < b1) load(rb, b0 + 2);
    for (int b = b0;;) {
      park(ra);
      if (b + 4 < b1) load(ra, b + 4);
      work(0);
      if (b + 1 < b1) work(1);
      b += 2;
      if (b >= b1) break;
      park(rb);
      if (b + 4 < b1) load(rb, b + 4);
      work(0);
      if (b + 1 < b1) work(1);
      b += 2;
      if (b >= b1) break;
    }
  }
  // an infinity or a NaN in x is a NaN in its vector's sums
  float sum = 0.0f;
#pragma unroll
  for (int t = 0; t < NT; t++)
#pragma unroll
    for (int v = 0; v < NV; v++) sum = sum + ((acc[t][v][0] + acc[t][v][1]) + (acc[t][v][2] + acc[t][v][3]));
  if (__builtin_expect(__builtin_amdgcn_ballot_w64((cut & 0xffffu) != 0 || sum != sum) != 0, 0)) {
    clear();
#pragma unroll 1
    for (int b = b0; b < b1; b += 2) {
      Raw r;
      load(r, b);
      park(r);
#pragma unroll 1
      for (int u = 0; u < min(2, b1 - b); u++) work_fix(u);
    }
  }
}

// The parts in LDS, [wave][tile][group][q][lane], and the sum over the P parts of wavefront group
// g's tile t: row j of vector v (0..16 NV).
template <int NT, int NV>
__device__ __forceinline__ void fx_park(float *part, const f4v (&acc)[NT][NV]) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
#pragma unroll
  for (int t = 0; t < NT; t++)
#pragma unroll
    for (int v = 0; v < NV; v++)
#pragma unroll
      for (int q = 0; q < 4; q++) part[(((wave * NT + t) * NV + v) * 4 + q) * 64 + lane] = acc[t][v][q];
}
template <int P, int NT, int NV>
__device__ __forceinline__ float fx_sum(const float *part, int g, int t, int v, int j) {
  const int i = ((t * NV + (v >> 4)) * 4 + (v & 3)) * 64 + j + 16 * ((v >> 2) & 3);
  float s = part[g * P * NT * NV * 256 + i];
#pragma unroll
  for (int p = 1; p < P; p++) s = s + part[(g * P + p) * NT * NV * 256 + i];
  return s;
}

// ------------------------------------------------------------------ matvec
// Up to three segments; a workgroup takes 16 NT (8 / P) rows of one of them (tasks stride over
// the grid) x 16 NV vectors (blockIdx.y): wavefront w part w mod P of row group w / P.
template <int T, int P, int NT, int NV>
__global__ __launch_bounds__(FX_NW<P> * 64) __attribute__((amdgpu_waves_per_eu(FX_WPE<P, NT, NV>))) void k_fx_mv(const MVArgs a, const StepRec *st) {
  constexpr int NW = FX_NW<P>, RG = 16 * NT, RW = RG * (NW / P), NO = RW * 16 * NV;
  extern __shared__ __align__(16) uint8_t smem[];
  float *part = reinterpret_cast<float *>(smem);
  __shared__ unsigned long long sbest[16 * NV];
  const int m = st ? st->m : a.m;
  const bool coh = a.tail.nw != nullptr;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), j = threadIdx.x & 15;
  const int g = wave / P, p = wave % P, v0 = blockIdx.y * 16 * NV;
  if (a.best) {
    if (threadIdx.x < 16 * NV) sbest[threadIdx.x] = 0;
    __syncthreads();
  }
  auto tasks = [&](int i) { return i < a.nseg ? (int)((a.seg[i].r1 - a.seg[i].r0 + RW - 1) / RW) : 0; };
  const int s0 = tasks(0), s1 = tasks(1), total = s0 + s1 + tasks(2);
  const int nb = (int)a.seg[0].w.nb, b0 = p * nb / P, b1 = (p + 1) * nb / P;
  uint32_t xo[NV][4];
  fx_xrows<NV>(xo, [&](int k) { return min(v0 + k, m - 1); }, (int)a.ld_x);
  SPX_L uint8_t *stage = (SPX_L uint8_t *)smem + wave * FX_STAGE<T, NT, NV>;
  for (int t = blockIdx.x; t < total; t += gridDim.x) {
    const int si = __builtin_amdgcn_readfirstlane(t >= s0 ? (t >= s0 + s1 ? 2 : 1) : 0);
    const int wg = t - (si > 0 ? s0 : 0) - (si > 1 ? s1 : 0);
    const Seg &sg = a.seg[si];
    const int r1 = (int)sg.r1, r0 = (int)sg.r0 + wg * RW, rg = r0 + g * RG, rf = min(rg, r1 - 1);
    const Planes pl = sg.w.pl;
    const int64_t g0 = ((int64_t)sg.expert * sg.w.rows + rf) * nb;
    uint32_t go[NT];
#pragma unroll
    for (int u = 0; u < NT; u++) go[u] = fx_wrows(rg + 16 * u, r1, rf, nb);
    f4v acc[NT][NV];
    fx_part<T, NT, NV, NT>(stage, &pl, &g0, go, a.x, xo, b0, b1, acc);
    __syncthreads();  // the stages' LDS takes the parts
    fx_park<NT, NV>(part, acc);
    __syncthreads();
    for (int i = threadIdx.x; i < NO; i += NW * 64) {
      const int r = i % RW, v = i / RW, vec = v0 + v;
      const int row = r0 + r;
      const float res = fx_sum<P, NT, NV>(part, r / RG, (r % RG) >> 4, v, r & 15);
      unsigned long long key = 0;
      if (vec < m && row < r1) {
        out_store(sg.out + (int64_t)vec * sg.ld_out + row, res, coh);
        key = pick_key(res, a.lscale, row);
      }
      if (a.best) {  // the best key of 16 rows of vector v, then one LDS atomic
#pragma unroll
        for (int o = 1; o < 16; o <<= 1) {
          const unsigned long long k2 = __shfl_xor(key, o, 64);
          key = k2 > key ? k2 : key;
        }
        if (j == 0 && vec < m) atomicMax(&sbest[v], key);
      }
    }
    __syncthreads();
  }
  if (a.best && threadIdx.x < 16 * NV && v0 + (int)threadIdx.x < m) a.best[(int64_t)(v0 + threadIdx.x) * a.nbest + blockIdx.x] = sbest[threadIdx.x];
  if (coh && arrive_last(a.tail.counter, gridDim.x)) norm_rows<NW>(a.tail, 0, m);
}

// ------------------------------------------------------------------ gate / up + SwiGLU
// h = silu(gate x) * (up x): a workgroup takes 16 NH (8 / P) rows of h (NH gate tiles and the same
// up tiles a wavefront) x 16 NV vectors: of the pass's rows (blockIdx.y, no jobs), or of job
// blockIdx.y's users (at most 16; NV = 1): vector k is row vec[k] of x, its h row out[k].
template <int T, int P, int NH, int NV>
__global__ __launch_bounds__(FX_NW<P> * 64) __attribute__((amdgpu_waves_per_eu(FX_WPE<P, 2 * NH, NV>))) void k_fx_gateup(const GUArgs a, const StepRec *st) {
  constexpr int NW = FX_NW<P>, NT = 2 * NH, RG = 16 * NH, RW = RG * (NW / P), NO = RW * 16 * NV;
  extern __shared__ __align__(16) uint8_t smem[];
  float *part = reinterpret_cast<float *>(smem);
  __shared__ int sv[16], so[16];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = wave / P, p = wave % P;
  int m = st->m, e = 0;
  const int v0 = a.jobs ? 0 : blockIdx.y * 16 * NV;
  if (a.jobs) {
    // (the job record is always addressable: requested together with the job count)
    const Job &J = a.jobs[blockIdx.y];
    const int nj = *a.njobs, jm = J.nvec, je = J.expert, jv = J.vec[threadIdx.x & 15], jo = J.out[threadIdx.x & 15];
    if ((int)blockIdx.y >= nj) return;
    m = jm;
    e = je;
    if (threadIdx.x < 16) { sv[threadIdx.x] = jv; so[threadIdx.x] = jo; }
    __syncthreads();
  }
  const int nb = (int)a.gate.nb, cols = (int)a.gate.cols, n_ff = a.n_ff, b0 = p * nb / P, b1 = (p + 1) * nb / P;
  uint32_t xo[NV][4];
  fx_xrows<NV>(xo, [&](int k) { const int i = min(v0 + k, m - 1); return a.jobs ? sv[i] : i; }, cols);
  const int r0 = blockIdx.x * RW, rg = r0 + g * RG, rf = min(rg, n_ff - 1);
  const Planes pl[2] = {a.gate.pl, a.up.pl};
  const int64_t gb = ((int64_t)e * n_ff + rf) * nb, g0[2] = {gb, gb};
  uint32_t go[NT];
#pragma unroll
  for (int u = 0; u < NT; u++) go[u] = fx_wrows(rg + 16 * (u % NH), n_ff, rf, nb);
  f4v acc[NT][NV];
  fx_part<T, NT, NV, NH>((SPX_L uint8_t *)smem + wave * FX_STAGE<T, NT, NV>, pl, g0, go, a.x, xo, b0, b1, acc);
  __syncthreads();  // the stages' LDS takes the parts
  fx_park<NT, NV>(part, acc);
  __syncthreads();
  for (int i = threadIdx.x; i < NO; i += NW * 64) {
    const int r = i % RW, v = i / RW, vec = v0 + v, row = r0 + r, t = (r % RG) >> 4;
    const float gv = fx_sum<P, NT, NV>(part, r / RG, t, v, r & 15), uv = fx_sum<P, NT, NV>(part, r / RG, NH + t, v, r & 15);
    if (vec < m && row < n_ff) a.h[(int64_t)(a.jobs ? so[v] : vec) * n_ff + row] = gv / (1.0f + expf(-gv)) * uv;
  }
}

// ------------------------------------------------------------------ routed down
// y of (user, row) to yd for job blockIdx.y's users (at most 16; user k's h row out[k]): a
// workgroup takes 16 NT (8 / P) rows of the expert's down matrix.
template <int T, int P, int NT>
__global__ __launch_bounds__(FX_NW<P> * 64) __attribute__((amdgpu_waves_per_eu(FX_WPE<P, NT, 1>))) void k_fx_down(const DownArgs a) {
  constexpr int NW = FX_NW<P>, RG = 16 * NT, RW = RG * (NW / P), NO = RW * 16;
  extern __shared__ __align__(16) uint8_t smem[];
  float *part = reinterpret_cast<float *>(smem);
  __shared__ int so[16];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = wave / P, p = wave % P;
  const Job &J = a.jobs[blockIdx.y];
  const int nj = *a.njobs, nv = J.nvec, e = J.expert, jo = J.out[threadIdx.x & 15];
  if ((int)blockIdx.y >= nj) return;
  const int dim = (int)a.w.rows, nb = (int)a.w.nb, n_ff = (int)a.w.cols;
  if (threadIdx.x < 16) so[threadIdx.x] = jo;
  __syncthreads();
  const int b0 = p * nb / P, b1 = (p + 1) * nb / P;
  uint32_t xo[1][4];
  fx_xrows<1>(xo, [&](int k) { return so[min(k, nv - 1)]; }, n_ff);
  const int r0 = blockIdx.x * RW, rg = r0 + g * RG, rf = min(rg, dim - 1);
  const Planes pl = a.w.pl;
  const int64_t g0 = ((int64_t)e * dim + rf) * nb;
  uint32_t go[NT];
#pragma unroll
  for (int u = 0; u < NT; u++) go[u] = fx_wrows(rg + 16 * u, dim, rf, nb);
  f4v acc[NT][1];
  fx_part<T, NT, 1, NT>((SPX_L uint8_t *)smem + wave * FX_STAGE<T, NT, 1>, &pl, &g0, go, a.x, xo, b0, b1, acc);
  __syncthreads();  // the stages' LDS takes the parts
  fx_park<NT, 1>(part, acc);
  __syncthreads();
  for (int i = threadIdx.x; i < NO; i += NW * 64) {
    const int r = i % RW, v = i / RW, row = r0 + r;
    const float y = fx_sum<P, NT, 1>(part, r / RG, (r % RG) >> 4, v, r & 15);
    if (v < nv && row < dim) a.yd[(int64_t)so[v] * dim + row] = y;
  }
}

// ------------------------------------------------------------------ launchers
static int cu_count_fx() {
  static const int n = [] {
    int dev = 0, c = 0;
    return hipGetDevice(&dev) == hipSuccess && hipDeviceGetAttribute(&c, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && c > 0 ? c : 256;
  }();
  return n;
}

// Parts a row of nb blocks is summed in (a rule on the width alone: the bits depend on it), so
// that a part is four to eight blocks at the usual widths and its loads go out in one round: 4 below
// 32 blocks (1024 columns), 8 below 64, 16 above.
static int fx_parts(int nb) { return nb >= 64 ? 16 : nb >= 32 ? 8 : 4; }
// f(format, parts) for a format and a width
template <class F>
static hipError_t with_parts(int dtype, int nb, F &&f) {
  using std::integral_constant;
  auto by_p = [&](auto Tc) {
    switch (fx_parts(nb)) {
    case 16: return f(Tc, integral_constant<int, 16>{});
    case 8: return f(Tc, integral_constant<int, 8>{});
    default: return f(Tc, integral_constant<int, 4>{});
    }
  };
  return dtype == T_Q8_0 ? by_p(integral_constant<int, T_Q8_0>{}) : by_p(integral_constant<int, T_Q5_0>{});
}

bool fx_type(int dtype) { return dtype == T_Q8_0 || dtype == T_Q5_0; }

template <int P, class K, class... A>
static hipError_t fx_go(K kern, dim3 grid, size_t sm, hipStream_t s, A... args) {
  if (sm > 61440)  // (the static part comes on top)
    if (hipError_t e = hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)sm); e != hipSuccess) return e;
  hipLaunchKernelGGL(kern, grid, dim3(FX_NW<P> * 64), sm, s, args...);
  return hipGetLastError();
}
template <int T, int P, int NT, int NV>  // the wavefronts' stages, then their parts
static constexpr size_t fx_lds() {
  constexpr size_t n = (size_t)FX_NW<P> * (FX_STAGE<T, NT, NV> > NT * NV * 1024 ? FX_STAGE<T, NT, NV> : NT * NV * 1024);
  static_assert(n + 512 <= 160 * 1024, "more than a CU's LDS (the kernels' static part is at most 512 bytes)");
  return n;
}

// Workgroups of a launch over one matrix of at most 16 vectors (with greedy keys: its slots).
static bool fx_wide(int64_t rows, int wg) { return (rows + 64 * wg - 1) / (64 * wg) >= 2 * cu_count_fx(); }
int fx_mv_wgs(const TensorView &w, int m) {
  const int P = fx_parts((int)w.nb), wg = P > 8 ? 1 : 8 / P;
  const int64_t rw = 16 * wg * (m <= MAX_M && fx_wide(w.rows, wg) ? 4 : 1);
  return (int)((w.rows + rw - 1) / rw);
}

// Tile shapes: up to 16 rows, one tile a wavefront, more where the tiles alone fill the CUs four
// times (the LM head: the split of x paid once for four tiles). More rows: the largest shape that
// still gives every CU a workgroup.
hipError_t launch_fx_mv(const MVArgs &a, int m, const StepRec *st, int grid_cap, hipStream_t s) {
  const int DT = a.seg[0].w.dtype, nb = (int)a.seg[0].w.nb, cu = cu_count_fx();
  int64_t rows = 0;
  for (int i = 0; i < a.nseg; i++) {
    if (a.seg[i].w.dtype != DT || a.seg[i].w.nb != nb) return hipErrorInvalidValue;
    rows += a.seg[i].r1 - a.seg[i].r0;
  }
  if (!fx_type(DT) || m < 1 || m > PMAX || a.nseg < 1 || rows < 1 || rows > 0x3fffffff || a.pro.nw || a.res_out || (a.tail.nw && m > MAX_M) ||
      (int64_t)m * a.ld_x * 4 > 0x7fffffffll)
    return hipErrorInvalidValue;
  auto go = [&](auto Tc, auto Pc, auto NTc, auto NVc) {
    constexpr int T = decltype(Tc)::value, PP = decltype(Pc)::value, NT = decltype(NTc)::value, NV = decltype(NVc)::value, RW = 16 * NT * (FX_NW<PP> / PP);
    int64_t t = 0;
    for (int i = 0; i < a.nseg; i++) t += (a.seg[i].r1 - a.seg[i].r0 + RW - 1) / RW;
    if (grid_cap > 0) t = a.best ? grid_cap : std::min<int64_t>(t, grid_cap);  // (a slot of best a workgroup)
    return fx_go<PP>(k_fx_mv<T, PP, NT, NV>, dim3((unsigned)t, (unsigned)((m + 16 * NV - 1) / (16 * NV))), fx_lds<T, PP, NT, NV>(), s, a, st);
  };
  auto shape = [&](auto Tc, auto Pc) {
    constexpr int PP = decltype(Pc)::value, WG = FX_NW<PP> / PP;
    using std::integral_constant;
    const int64_t tiles = (rows + 15) / 16;
    auto wgs = [&](int NT, int NV) { return (tiles + NT * WG - 1) / (NT * WG) * ((m + 16 * NV - 1) / (16 * NV)); };
    if (m <= MAX_M) {
      if (!a.tail.nw && fx_wide(rows, WG)) return go(Tc, Pc, integral_constant<int, 4>{}, integral_constant<int, 1>{});
      return go(Tc, Pc, integral_constant<int, 1>{}, integral_constant<int, 1>{});
    }
    if constexpr (PP <= 8) {
      if (wgs(4, 2) >= cu) return go(Tc, Pc, integral_constant<int, 4>{}, integral_constant<int, 2>{});
      if (wgs(2, 2) >= cu) return go(Tc, Pc, integral_constant<int, 2>{}, integral_constant<int, 2>{});
    } else {  // sixteen wavefronts: 128 registers each, one vector group
      if (wgs(4, 1) >= 2 * cu) return go(Tc, Pc, integral_constant<int, 4>{}, integral_constant<int, 1>{});
    }
    if (wgs(2, 1) >= cu) return go(Tc, Pc, integral_constant<int, 2>{}, integral_constant<int, 1>{});
    return go(Tc, Pc, integral_constant<int, 1>{}, integral_constant<int, 1>{});
  };
  return with_parts(DT, nb, shape);
}

hipError_t launch_fx_gateup(const GUArgs &a, int m, const StepRec *st, int max_jobs, hipStream_t s) {
  const int DT = a.gate.dtype, nb = (int)a.gate.nb, cu = cu_count_fx();
  if (!fx_type(DT) || a.up.dtype != a.gate.dtype || a.up.nb != nb || a.hq.q || a.pro.nw || m < 1 || m > PMAX) return hipErrorInvalidValue;
  auto go = [&](auto Tc, auto Pc, auto NHc, auto NVc) {
    constexpr int T = decltype(Tc)::value, PP = decltype(Pc)::value, NH = decltype(NHc)::value, NV = decltype(NVc)::value, RW = 16 * NH * (FX_NW<PP> / PP);
    return fx_go<PP>(k_fx_gateup<T, PP, NH, NV>, dim3((unsigned)((a.n_ff + RW - 1) / RW), (unsigned)(a.jobs ? max_jobs : (m + 16 * NV - 1) / (16 * NV))),
                 fx_lds<T, PP, 2 * NH, NV>(), s, a, st);
  };
  auto shape = [&](auto Tc, auto Pc) {
    constexpr int PP = decltype(Pc)::value, WG = FX_NW<PP> / PP;
    using std::integral_constant;
    const int tiles = (a.n_ff + 15) / 16;
    if (a.jobs) return go(Tc, Pc, integral_constant<int, 2>{}, integral_constant<int, 1>{});
    if (m <= MAX_M) return go(Tc, Pc, integral_constant<int, 1>{}, integral_constant<int, 1>{});
    if constexpr (PP <= 8) {
      if ((tiles + 2 * WG - 1) / (2 * WG) * ((m + 31) / 32) >= cu) return go(Tc, Pc, integral_constant<int, 2>{}, integral_constant<int, 2>{});
      return go(Tc, Pc, integral_constant<int, 1>{}, integral_constant<int, 2>{});
    } else {
      // sixteen wavefronts: one vector group (two need more LDS than a CU has). Two row tiles from a
      // workgroup a CU on: 4 layers of dim 2048, us a pass with two / one, 128 rows of n_ff 4096 572 / 613,
      // 64 rows of 2048 (256 workgroups) 339 / 347, 64 rows of 1024 (128) 328 / 314.
      if ((tiles + 1) / 2 * ((m + 15) / 16) >= cu) return go(Tc, Pc, integral_constant<int, 2>{}, integral_constant<int, 1>{});
      return go(Tc, Pc, integral_constant<int, 1>{}, integral_constant<int, 1>{});
    }
  };
  return with_parts(DT, nb, shape);
}

hipError_t launch_fx_down(const DownArgs &a, int max_jobs, hipStream_t s) {
  const int DT = a.w.dtype, nb = (int)a.w.nb;
  if (!fx_type(DT) || !a.yd || max_jobs < 1) return hipErrorInvalidValue;
  auto go = [&](auto Tc, auto Pc) {
    constexpr int T = decltype(Tc)::value, PP = decltype(Pc)::value, NT = 2, RW = 16 * NT * (FX_NW<PP> / PP);
    return fx_go<PP>(k_fx_down<T, PP, NT>, dim3((unsigned)((a.w.rows + RW - 1) / RW), (unsigned)max_jobs), fx_lds<T, PP, NT, 1>(), s, a);
  };
  return with_parts(DT, nb, go);
}

}  // namespace spx
