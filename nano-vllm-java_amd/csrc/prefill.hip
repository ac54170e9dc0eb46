// Kernel (c): varlen causal prefill on the fp16 matrix units at fp32 precision, over dense K/V or
// the paged KV cache.  (Small steps: prefill_fp32.hip.)
//
// Semantics (layers/Attention.java:245-280 prefillDense / prefillWithCache, :328-396
// attendJobs): query qi of a sequence with qLen queries and kLen keys sits at absolute
// position aq = kLen - qLen + qi and sees keys [max(0, aq - W + 1) (window W > 0, else 0),
// aq]; KV head kvh = h / rep; score = dot(q, k) * scale; out = softmax-weighted sum of v.
//
// Each fp32 operand (q, k, v and the probabilities) is split into two scaled fp16 parts and each
// product taken as three fp16 ones with fp32 sums (split_f16.h), at 5.3 times the rate of
// v_mfma_f32.
//
// Mapping onto CDNA4.  The grid is exactly as many workgroups per head group as can be resident
// at once; each runs the segments of its slot of a stream-K schedule (equal numbers of 32-key
// tiles per slot; a query tile whose keys straddle slots is split and its partials merged).  A
// segment is a tile of 32 * NW / HPW queries of one sequence for HPW query heads of one KV head;
// each wave owns 32 queries of one head, so one LDS read of a K or V operand (two parts, 32 bytes
// a lane) feeds three 32 x 32 x 16 products.
//   * Key tiles of 32 rows: each wave loads a share of the next tile's K and V rows into
//     registers (8 floats of each per lane at a time) while the current tile is computed, then
//     splits them and writes the parts to LDS, double-buffered, one barrier per tile.  K parts
//     lie [key][dim], V parts [dim][key] in the key order of the PV contraction, so that both
//     are read as 16-byte operands; 16-byte chunks are XOR-swizzled by the row (k_pos, part_pos) so
//     that any 16 rows read at one column touch every bank once.
//   * Scales: q per query; K and V per tile, from the tile's largest magnitude, which the waves
//     exchange through LDS ahead of the barrier that the split waits for anyway.  A K tile's
//     scale goes into the factor of its scores.  O^T is kept in the units of V's scale, which
//     stays for tiles down to 2^-3 of it.
//   * S^T[key][query] = K Q^T, then O^T[dim][query] += V^T P^T: S^T leaves 16 keys of one query
//     in each lane, which are the lane's B operand of PV once the contraction takes its keys in
//     that order, so P never leaves registers.
//   * Softmax in the log2 domain, relative to a reference that moves, and O with it, only when a
//     tile's max exceeds it by more than 2^4 or lies more than 2^10 below it.  Only tiles that
//     cross the causal diagonal, the window edge or the end of the keys are masked.
//   * Every query adds up what the steps of the split can have done to its sums.  A wave with a
//     query where that is more than 2^-19 of its largest result, whose sums are not finite
//     (infinities in the inputs), in whose scores the steps could show, or in whose V tiles
//     one dim lies far below the others takes the segment's 32 queries again on fp32 matrix
//     instructions, after all segments (fp32_segment).  Where every query sees an infinity a call
//     takes 3 to 5 times as long (a 2048-token chunk after 12289 tokens 7.1 ms, 3.4 on the fp32
//     tiles); with the keys taken one by one it was 7 to 19 times.
//   * Operands are read from LDS two steps ahead of their products and the next tile is split
//     and stored after QK: 14% fewer cycles than in source order, 4% less time.
//
// Bound by the board's power where steps are large: at d = 128 the matrix units are 47% busy at
// 1.96 GHz, and splitting the waves into early and late ones, raising their priority around QK or
// interleaving the split with the products changed nothing.  At d = 512 reloads of spilled
// registers wait for the V loads in flight.  Measured per layer call, against fp32 matrix
// instructions: a 2048-token chunk after 12289 cached tokens, 32 q / 8 KV heads, d = 128: 3.32 ->
// 1.37 ms; prompts of 512-2048 tokens: 16 q / 8 KV heads, d = 128, 273 -> 158 us; 4 q / 1 KV, d =
// 256, window 512, 127 -> 105 us; 8 q / 1 KV, d = 512, 687 -> 484 us; seven prompts of 5-333
// tokens, 32 q / 8 KV, d = 64: 36.8 -> 31.1 us.  (The checks and the moving units cost 1-3% of
// these.)  Error against float64 (rel-L2): 1.7e-6 -> 1.3e-6, 7.1e-7 -> 4.8e-7, 9.7e-7 -> 4.6e-7,
// 1.0e-6 -> 5.9e-7, 2.1e-7 -> 1.65e-7.
#include "nva_internal.h"
#include "nva_device.h"
#include "split_f16.h"

namespace nva {

namespace {

constexpr float kLog2e = 1.4426950408889634f;
// Probabilities, at most 2^kRaise, are split as 2^11 p <= 2^15.  (The factor is not taken in the
// exponential: beside 11, the argument of a probability near 1 is rounded to 2^-21.)
constexpr int kProbExp = 11;
// Log2 units.  The reference that a query's probabilities are relative to moves up to a tile's max
// that exceeds it by more than kRaise, and down to kMargin above one that lies kLower further below,
// but no more than kRefSpan below the largest max so far.
constexpr float kRaise = 4.0f, kMargin = 4.0f, kLower = 6.0f, kRefSpan = 40.0f;
// Largest factor from products of scaled q and k to scores.  The steps of the split put such a
// product off by at most about 2^-7 (both operands at their largest in every dim, when fp32 sums are
// off by more), by about 2^-10 beside a K row or channel far above the others: 2^-23 of a score at
// this factor.  Rows of such steps move away from float64 from 2^-11 on.
constexpr float kMaxScoreUnit = 0x1p-13f;
// The exponent of V's scale stays for tiles of up to kUnitSlack below it and within kUnitSpan of the
// largest one's.
constexpr int kUnitSlack = 3, kUnitSpan = 32;
// Eight keys of a V dim are held to 2^-22 of the largest of them, or better, if that is at least
// 2^-kDimBits of the most that the scale takes: 2^-14 (a tile at the low end of kUnitSlack) to 2^-18
// of the tile's largest |v|.  A segment with a smaller chunk (a channel far above the others) is not
// for the split: the row as a whole would not show what those dims lose.
constexpr int kDimBits = 18;
constexpr int KT = 32;                // keys per tile
constexpr int kAhead = 2;             // operand reads in flight ahead of their products
constexpr int kKeepReads = 0x6;       // sched_barrier: only VALU and SALU move across
constexpr int QW = 32;                // queries per wave

// Offset (in fp16) of 16-byte chunk c of K row r of one part: 16 rows at any one column lie in
// 16 different 16-byte columns of the 256-byte bank period (a row of 64 dims is half of one).
template <int D>
__device__ __forceinline__ int k_pos(int r, int c) {
  const int x = D == 64 ? (r >> 1) & 7 : r & 15;
  return r * D + ((c ^ x) << 3);
}
// Key (within the tile) at element j of V chunk c, step c / 2 and lane half c % 2 of the PV
// contraction: the key of S^T register 8 (c / 2) + j.
__device__ __forceinline__ int v_key(int c, int j) {
  return 16 * (c >> 1) + 4 * (c & 1) + 8 * (j >> 2) + (j & 3);
}

// Row of key t: dense rows follow kbase; paged rows go through the LDS copy of the block
// table, which starts at page blk0.
__device__ __forceinline__ int64_t key_row(const KvView &kv, const int32_t *stab, int blk0,
                                           int kbase, int t) {
  if (!kv.paged) return (int64_t)kbase + t;
  int blk, off;
  if (kv.bs_shift >= 0) {
    blk = t >> kv.bs_shift;
    off = t & (kv.block_size - 1);
  } else {
    blk = t / kv.block_size;
    off = t - blk * kv.block_size;
  }
  return (int64_t)stab[blk - blk0] * kv.block_size + off;
}

__device__ __forceinline__ float4 ld4(const float *p) { return *reinterpret_cast<const float4 *>(p); }

// Where a query's results go: the output row, or the partial of one key chunk (rows of the tile
// are laid out query-major, chunk-minor).
struct Dest {
  float *row;
  size_t pidx;
  bool partial;
};
__device__ __forceinline__ Dest destination(const TileLaunch &a, const TileItem &it, int qi, int h,
                                            int D) {
  Dest d;
  d.partial = it.part >= 0;
  d.pidx = 0;
  if (!d.partial) {
    d.row = a.out + ((size_t)(it.qstart + qi) * a.hq + h) * D;
  } else {
    d.pidx = ((size_t)it.part + (size_t)(qi - it.q0) * it.nsplit + it.split) * a.hq + h;
    d.row = a.part_acc + d.pidx * D;
  }
  return d;
}

// The segment's result for a wave's 32 queries (from tile query q0 on) and dims [v0, v0 + 32 NB) of V
// on fp32 matrix instructions, operands straight from memory: for segments that the split does not
// fit.  Lanes and registers of S^T and O^T are those of the split products; a step of PV contracts
// the keys of one S^T register.  Scores are added up over sums of 64 dims and O^T over the tiles' own,
// which leaves 2.2e-7 of a row where the split leaves 2.2e-7 to 2.9e-7.
template <int D, int NB>
__device__ void fp32_segment(const TileLaunch &a, const TileItem &it, int kvh, int h, int q0, int v0) {
  const int lane = threadIdx.x & 63;
  const int i = lane & 31, half = lane >> 5;
  const int W = a.window;
  const int off = it.klen - it.qlen;
  const int qi = q0 + i;
  const bool qvalid = qi < it.qlen;
  const int aq = off + (qvalid ? qi : it.qlen - 1);
  const int vis_lo = W > 0 ? max(0, aq - W + 1) : 0;
  const int q1 = min(q0 + QW, it.qlen) - 1;
  const int all_lo = W > 0 ? max(0, off + q1 - W + 1) : 0;  // keys that every query sees
  const int all_hi = off + q0 + 1;
  const int any_lo = W > 0 ? max(0, off + q0 - W + 1) : 0;
  const int any_hi = min(it.ke, off + q1 + 1);
  const int32_t *table = a.kv.table + (size_t)it.seq * a.kv.bt_stride;
  const float sl2 = a.scale * kLog2e;
  const size_t rs = (size_t)a.hkv * D;
  const float *qp = a.q + ((size_t)(it.qstart + aq - off) * a.hq + h) * D + 4 * half;
  const float *kbase = a.kv.k + (size_t)kvh * D + 4 * half;
  const float *vbase = a.kv.v + (size_t)kvh * D + v0;
  f32x16 o[NB];
#pragma unroll
  for (int b = 0; b < NB; b++)
#pragma unroll
    for (int r = 0; r < 16; r++) o[b][r] = 0.0f;
  float m = -INFINITY, l = 0.0f;
#pragma unroll 1
  for (int kt = it.ks; kt < any_hi; kt += KT) {
    if (kt + KT <= any_lo) continue;
    const bool full = kt >= all_lo && kt + KT <= min(all_hi, it.ke);
    const int64_t row = key_row(a.kv, table, 0, it.kbase, min(kt + i, it.ke - 1));
    const float *kp = kbase + (size_t)row * rs;
    f32x16 st;
#pragma unroll
    for (int r = 0; r < 16; r++) st[r] = 0.0f;
#pragma unroll 1
    for (int c = 0; c < D; c += 64) {  // 64 dims a sum, in two chains
      f32x16 sa, sb;
#pragma unroll
      for (int r = 0; r < 16; r++) sa[r] = sb[r] = 0.0f;
#pragma unroll 2
      for (int s = c; s < c + 64; s += 16) {
        const float4 x = ld4(kp + s), y = ld4(qp + s), z = ld4(kp + s + 8), w = ld4(qp + s + 8);
        sa = __builtin_amdgcn_mfma_f32_32x32x2f32(x.x, y.x, sa, 0, 0, 0);
        sb = __builtin_amdgcn_mfma_f32_32x32x2f32(z.x, w.x, sb, 0, 0, 0);
        sa = __builtin_amdgcn_mfma_f32_32x32x2f32(x.y, y.y, sa, 0, 0, 0);
        sb = __builtin_amdgcn_mfma_f32_32x32x2f32(z.y, w.y, sb, 0, 0, 0);
        sa = __builtin_amdgcn_mfma_f32_32x32x2f32(x.z, y.z, sa, 0, 0, 0);
        sb = __builtin_amdgcn_mfma_f32_32x32x2f32(z.z, w.z, sb, 0, 0, 0);
        sa = __builtin_amdgcn_mfma_f32_32x32x2f32(x.w, y.w, sa, 0, 0, 0);
        sb = __builtin_amdgcn_mfma_f32_32x32x2f32(z.w, w.w, sb, 0, 0, 0);
      }
      st += sa + sb;
    }
    float mx = -INFINITY;
#pragma unroll
    for (int r = 0; r < 16; r++) {
      const int key = kt + 8 * (r >> 2) + 4 * half + (r & 3);
      st[r] = full || (key >= vis_lo && key <= aq && key < it.ke) ? st[r] * sl2 : -INFINITY;
      mx = fmaxf(mx, st[r]);
    }
    const float mn = fmaxf(m, max_halves(mx));
    const float alpha = m == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m - mn);
    const float ms = mn == -INFINITY ? 0.0f : mn;
    m = mn;
    float lt[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int r = 0; r < 16; r++) {
      st[r] = __builtin_amdgcn_exp2f(st[r] - ms);
      lt[r >> 2] += st[r];
    }
    l = fmaf(l, alpha, (lt[0] + lt[1]) + (lt[2] + lt[3]));
    f32x16 t[NB];
#pragma unroll
    for (int b = 0; b < NB; b++)
#pragma unroll
      for (int r = 0; r < 16; r++) t[b][r] = 0.0f;
    bool odd = false;  // an infinity or NaN in V: no product with the 0 of a query that does not see it
#pragma unroll
    for (int r = 0; r < 16; r++) {
      if (r % 4 == 0) __builtin_amdgcn_sched_barrier(0);  // four steps' loads in flight
      const int64_t vrow = __shfl((long long)row, 8 * (r >> 2) + 4 * half + (r & 3), 64);
      const float *vp = vbase + (size_t)vrow * rs + i;
#pragma unroll
      for (int b = 0; b < NB; b++) {
        const float v = vp[32 * b];
        odd |= !(fabsf(v) < INFINITY);
        t[b] = __builtin_amdgcn_mfma_f32_32x32x2f32(v, st[r], t[b], 0, 0, 0);
      }
    }
    if (!full && __any(odd)) {
#pragma unroll
      for (int b = 0; b < NB; b++)
#pragma unroll
        for (int r = 0; r < 16; r++) t[b][r] = 0.0f;
#pragma unroll 1
      for (int k = 0; k < min(KT, any_hi - kt); k++) {
        float p = st[0];  // of key k, in the lanes that hold it, then in both halves
#pragma unroll
        for (int r = 1; r < 16; r++) p = r == 4 * (k >> 3) + (k & 3) ? st[r] : p;
        p = __shfl(p, i + 32 * ((k >> 2) & 1), 64);
        const float *vp = vbase + (size_t)__shfl((long long)row, k, 64) * rs + 4 * half;
        const bool seen = kt + k >= vis_lo && kt + k <= aq;
#pragma unroll
        for (int b = 0; b < NB; b++)
#pragma unroll
          for (int r = 0; r < 16; r += 4) {
            if (r == 0) __builtin_amdgcn_sched_barrier(0);
            const float4 v = ld4(vp + 32 * b + 2 * r);
            t[b][r] = seen ? fmaf(p, v.x, t[b][r]) : t[b][r];
            t[b][r + 1] = seen ? fmaf(p, v.y, t[b][r + 1]) : t[b][r + 1];
            t[b][r + 2] = seen ? fmaf(p, v.z, t[b][r + 2]) : t[b][r + 2];
            t[b][r + 3] = seen ? fmaf(p, v.w, t[b][r + 3]) : t[b][r + 3];
          }
      }
    }
#pragma unroll
    for (int b = 0; b < NB; b++)
#pragma unroll
      for (int r = 0; r < 16; r++) o[b][r] = fmaf(o[b][r], alpha, t[b][r]);
  }
  l = sum_halves(l);
  if (!qvalid) return;
  const Dest d = destination(a, it, qi, h, D);
  const float f = d.partial ? 1.0f : l == 0.0f ? 0.0f : 1.0f / l;
#pragma unroll
  for (int b = 0; b < NB; b++)
#pragma unroll
    for (int r = 0; r < 16; r += 4)
      *reinterpret_cast<float4 *>(d.row + v0 + 32 * b + 2 * r + 4 * half) =
          make_float4(o[b][r] * f, o[b][r + 1] * f, o[b][r + 2] * f, o[b][r + 3] * f);
  if (d.partial && half == 0 && v0 == 0) {
    a.part_m[d.pidx] = m;
    a.part_l[d.pidx] = l;
  }
}

// The reference of a query's probabilities from a tile of this max on; its sums are to be
// multiplied by exp2(m - result).  It follows the tiles' maxima both ways: the probabilities are
// split beside 2^kProbExp, and in tiles far below the largest max (where one key of little or no V
// has most of the weight, all others) the split's steps would show.  A whole number, so that the
// factors of the sums are exact.  top: the largest max so far, rounded up.
__device__ __forceinline__ float reference(float mx, float m, float &top) {
  const float up = ceilf(mx);
  top = fmaxf(top, up);
  const float low = fmaxf(up + kMargin, top - kRefSpan);
  const bool down = mx > -INFINITY && m > low + kLower;
  return mx > m + kRaise ? up : down ? low : m;
}

// The exponent of V's scale, in which O is kept, for a tile of exponent e.  It follows the tiles both
// ways, so that neither V nor the probabilities lose bits to a larger V before or after them.  top:
// the largest e so far.  (Tiles of zeros leave it as it is.)
__device__ __forceinline__ int value_unit(int e, int unit, int &top) {
  top = max(top, e);
  return e > unit                                      ? e
         : e > kMinExp && e < unit - kUnitSlack ? max(e, top - kUnitSpan)
                                                : unit;
}

// The segments of a slot that a wave takes again, after all of them (in the loop over the segments
// that code would take registers from the tiles).  From the 64th on they share a bit: some may be
// taken again for nothing.
struct Again {
  int first;
  uint64_t bits;
  __device__ void add(int seg) { bits |= 1ull << min(seg - first, 63); }
  __device__ int next(int seg, int end) const {
    while (seg < end && !(bits >> min(seg - first, 63) & 1)) seg++;
    return seg;
  }
};

// The size below which a dim's keys are too small for a V scale of this exponent.
__device__ __forceinline__ float dim_limit(int unit) {
  return __uint_as_float((uint32_t)max(unit + 1 - kDimBits, 0) << 23);
}

// What the steps of the split add to the error of a query's o in one tile, p being the sum of the
// lane's probabilities: half a step of lo, 2^-25 and 2^-25.8 on average, in each of 16 (scaled)
// probabilities beside |v| of up to 2^15, and in each v.  (Added up over the tiles by squares: the
// roundings are independent.)
__device__ __forceinline__ float split_steps(float p) {
  constexpr float scale = 1 << kProbExp;
  return fmaf(p, scale * 0x1p-26f, fminf(p * (scale * 0x1p15f), 0x1p-9f));
}

// A query's largest result over a wave's dims; -INFINITY if one of them is not finite.
template <int NB>
__device__ __forceinline__ float largest_result(const f32x16 (&o)[NB], float l) {
  float zero = 0.0f * l, top = 0.0f;
#pragma unroll
  for (int b = 0; b < NB; b++)
#pragma unroll
    for (int r = 0; r < 16; r++) {
      zero = fmaf(0.0f, o[b][r], zero);  // NaN if any is not finite
      top = fmaxf(top, fabsf(o[b][r]));
    }
  const float x = zero == 0.0f ? top : -INFINITY;
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false,
                                                  false);
  const float y = __uint_as_float(r[0]), z = __uint_as_float(r[1]);
  return fminf(y, z) < 0.0f ? -INFINITY : fmaxf(y, z);
}

// Whether a query's sums (o in units of 2^kProbExp and the V scale) cannot stand: one is not finite,
// or the split's steps, e their squares, are more than 2^-19 of the largest result: with |v| at its
// bound; usually a quarter of that, as |v| mostly lies at a sixth of it.  (At the smallest scale, V
// holds nothing but zeros and values below 2^-105.)
__device__ __forceinline__ bool unsound(float result, float e, int v_top) {
  return result < 0.0f || (result < __builtin_sqrtf(e) * 0x1p19f && v_top > kMinExp);
}

// The factor of a query's sums in its result: 1 / l or, in a partial, to the largest max.
__device__ __forceinline__ float result_factor(const Dest &d, float l, float m, float top) {
  if (d.partial) return m == -INFINITY ? 1.0f : __builtin_amdgcn_exp2f(m - top);
  return l == 0.0f ? 0.0f : 1.0f / l;
}
__device__ __forceinline__ float4 result4(const f32x16 &o, int r, float f, int o_exp) {
  const int e = o_exp - 141 - kProbExp;  // the scales of V and of the probabilities
  return make_float4(__builtin_ldexpf(o[r] * f, e), __builtin_ldexpf(o[r + 1] * f, e),
                     __builtin_ldexpf(o[r + 2] * f, e), __builtin_ldexpf(o[r + 3] * f, e));
}

// A wave's share of the workgroup's tiles: UW units of 64 lanes x 8 floats of K (RPU whole rows
// each, a lane eight dims of one) and of V (one V chunk of 64 dims, a lane eight keys of one).
template <int D, int NW>
struct TileShare {
  static constexpr int RPU = 64 / (D / 8);
  static constexpr int UW = D / 16 / NW;
  static_assert(RPU >= 1 && UW >= 1 && UW * NW * 16 == D, "tile does not split evenly over the waves");
  const KvView &kv;
  const float *k, *v;  // of this KV head
  size_t rs;           // floats per token
  const int32_t *stab;
  int blk0, kbase, ks, ke;
  int wave, lane;
  int cur_page, cur_id;  // page whose block id cur_id holds (wave-uniform)

  __device__ int krow() const { return lane / (D / 8); }
  __device__ int kchunk() const { return lane % (D / 8); }
  __device__ int unit(int u) const { return u * NW + wave; }
  // Row of key t, wave-uniform.
  __device__ int64_t uniform_row(int t) {
    const int pg = t >> kv.bs_shift;
    if (pg != cur_page) {
      cur_id = __builtin_amdgcn_readfirstlane(stab[pg - blk0]);
      cur_page = pg;
    }
    return (int64_t)cur_id * kv.block_size + (t - (pg << kv.bs_shift));
  }
  // A full tile inside one page, or of dense rows: 32 consecutive rows.
  __device__ bool one_run(int kt) const {
    return kt + KT <= ke &&
           (!kv.paged ||
            (kv.bs_shift >= 0 && (kt >> kv.bs_shift) == ((kt + KT - 1) >> kv.bs_shift)));
  }
  // A full tile that starts at a multiple of 8 keys, over pages of at least 8: a K unit and each
  // 4-key run of a V unit lie in one page.
  __device__ bool short_runs(int kt) const {
    return kt + KT <= ke && kv.bs_shift >= 3 && (kt & 7) == 0;
  }
  __device__ f32x8 load_krow(const float *row) const {
    const float4 x = ld4(row + 8 * kchunk()), y = ld4(row + 8 * kchunk() + 4);
    return f32x8{x.x, x.y, x.z, x.w, y.x, y.y, y.z, y.w};
  }

  __device__ void load_k(int kt, f32x8 (&r)[UW]) {
    const size_t lane_row = (size_t)krow() * rs;
    if (one_run(kt)) {
      const float *g = k + (kv.paged ? uniform_row(kt) : (int64_t)kbase + kt) * (int64_t)rs;
#pragma unroll
      for (int u = 0; u < UW; u++) r[u] = load_krow(g + (size_t)(unit(u) * RPU) * rs + lane_row);
    } else if (short_runs(kt)) {
#pragma unroll
      for (int u = 0; u < UW; u++)
        r[u] = load_krow(k + uniform_row(kt + unit(u) * RPU) * (int64_t)rs + lane_row);
    } else {  // per-row addresses, rows past the chunk clamped to its last key (and masked)
#pragma unroll
      for (int u = 0; u < UW; u++) {
        const int t = min(kt + unit(u) * RPU + krow(), ke - 1);
        r[u] = load_krow(k + (size_t)key_row(kv, stab, blk0, kbase, t) * rs);
      }
    }
  }
  __device__ void load_v(int kt, f32x8 (&r)[UW]) {
    if (one_run(kt)) {
      const float *g = v + (kv.paged ? uniform_row(kt) : (int64_t)kbase + kt) * (int64_t)rs;
#pragma unroll
      for (int u = 0; u < UW; u++)
#pragma unroll
        for (int j = 0; j < 8; j++)
          r[u][j] = (g + (size_t)v_key(unit(u) & 3, j) * rs + 64 * (unit(u) >> 2))[lane];
    } else if (short_runs(kt)) {
#pragma unroll
      for (int u = 0; u < UW; u++)
#pragma unroll
        for (int j = 0; j < 8; j += 4) {
          const float *g = v + uniform_row(kt + v_key(unit(u) & 3, j)) * (int64_t)rs +
                           64 * (unit(u) >> 2);
#pragma unroll
          for (int jj = 0; jj < 4; jj++) r[u][j + jj] = (g + (size_t)jj * rs)[lane];
        }
    } else {
#pragma unroll
      for (int u = 0; u < UW; u++) {
        // One lane per row looks up the V rows; each lane then takes them in turn.
        const int t = min(kt + v_key(unit(u) & 3, lane & 7), ke - 1);
        const int64_t row = key_row(kv, stab, blk0, kbase, t);
#pragma unroll
        for (int j = 0; j < 8; j++) {
          const uint64_t x =
              (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)row, j) |
              (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(row >> 32), j) << 32;
          r[u][j] = (v + (size_t)x * rs + 64 * (unit(u) >> 2))[lane];
        }
      }
    }
  }

  // The share's parts to LDS; the second part lies KT * D further on.
  __device__ void store_k(const f32x8 (&r)[UW], float scale, _Float16 *dst) const {
#pragma unroll
    for (int u = 0; u < UW; u++) {
      const Split8 x = split8(r[u], scale);
      _Float16 *d = dst + k_pos<D>(unit(u) * RPU + krow(), kchunk());
      *reinterpret_cast<f16x8 *>(d) = x.hi;
      *reinterpret_cast<f16x8 *>(d + KT * D) = x.lo;
    }
  }
  __device__ void store_v(const f32x8 (&r)[UW], float scale, _Float16 *dst) const {
#pragma unroll
    for (int u = 0; u < UW; u++) {
      const Split8 x = split8(r[u], scale);
      _Float16 *d = dst + part_pos(64 * (unit(u) >> 2) + lane, unit(u) & 3);
      *reinterpret_cast<f16x8 *>(d) = x.hi;
      *reinterpret_cast<f16x8 *>(d + KT * D) = x.lo;
    }
  }
  static __device__ float largest(const f32x8 (&r)[UW]) {
    float m = 0.0f;
#pragma unroll
    for (int u = 0; u < UW; u++) m = abs_max(m, r[u]);
    return m;
  }
  // Of how many lanes' dims least_chunk() has to be too small in the segment's tile t.  One of eight
  // keys is; where rows past the end repeat the last key, a chunk may be one value, which is small
  // now and then, but not in many dims at once.
  __device__ int dims_needed(int t) const { return ks + (t + 1) * KT <= ke ? 1 : 8; }
  // The smallest of the lane's V chunks (eight keys of one dim), by the largest value of each; chunks
  // of zeros don't count.
  static __device__ float least_chunk(const f32x8 (&r)[UW]) {
    float m = INFINITY;
#pragma unroll
    for (int u = 0; u < UW; u++) {
      const float x = abs_max(0.0f, r[u]);
      m = fminf(m, x > 0.0f ? x : INFINITY);
    }
    return m;
  }
};

// Stages a segment's block ids in LDS, so that the tile loads never wait on a global load;
// returns the first page.  Every wave of the workgroup calls it.
__device__ __forceinline__ int stage_table(const TileLaunch &a, const TileItem &it, int32_t *stab) {
  if (!a.kv.paged) return 0;
  const int bs = a.kv.block_size;
  const int blk0 = it.ks / bs;
  const int npages = (it.ke - 1) / bs - blk0 + 1;
  const int32_t *table = a.kv.table + (size_t)it.seq * a.kv.bt_stride + blk0;
  for (int j = threadIdx.x; j < npages; j += blockDim.x) stab[j] = table[j];
  __syncthreads();
  return blk0;
}

}  // namespace

// NW waves per workgroup.  At most 256 registers and two waves per SIMD at d = 128, 168 and three
// at d = 64.
template <int D, int HPW, int NW>
__global__ void __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(D == 64 ? 3 : 2)))
prefill_split_kernel(TileLaunch a) {
  constexpr int KS = D / 16;         // contraction steps of QK
  constexpr int NB = D / 32;         // O^T blocks of 32 dims
  constexpr int PART = KT * D;       // fp16 values of one part of a K (or V) tile
  constexpr int UW = TileShare<D, NW>::UW;
  __shared__ __attribute__((aligned(16))) _Float16 sk[2][2 * PART];
  __shared__ __attribute__((aligned(16))) _Float16 sv[2][2 * PART];
  __shared__ __attribute__((aligned(16))) float smax[2][2][NW];  // each wave's largest |k|, |v|
  __shared__ int32_t stab[kPrefillTablePages];  // block ids of the pages this chunk touches
  __shared__ int uneven;  // a tile's V dims are too unlike for one scale

  const int slot = blockIdx.x;
  const int seg_end = a.seg_off[slot + 1];
  const int rep = a.hq / a.hkv;
  const int groups = rep / HPW;
  const int kvh = blockIdx.y / groups;
  // Wave-uniform, and known to be: every value derived from it lives in scalar registers.
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int h = kvh * rep + (blockIdx.y - kvh * groups) * HPW + wave % HPW;
  const int qb = wave / HPW;
  const int lane = threadIdx.x & 63;
  const int i = lane & 31;     // MFMA row / column index of this lane
  const int half = lane >> 5;  // MFMA k-slot
  const int W = a.window;
  // Scores are kept unscaled until the exponential; a negative scale goes into q's sign, so that
  // the largest product is the largest score.
  const float sl2 = fabsf(a.scale) * kLog2e;
  const float qsign = a.scale < 0.0f ? -1.0f : 1.0f;
  const size_t rs = (size_t)a.hkv * D;
  const float *kbase = a.kv.k + (size_t)kvh * D;
  const float *vbase = a.kv.v + (size_t)kvh * D;

  Again again{a.seg_off[slot], 0};
  for (int seg = again.first; seg < seg_end; seg++) {
    // Every wave is done with the previous segment's LDS tiles and table before they are reused.
    __syncthreads();
    if (threadIdx.x == 0) uneven = 0;
    const TileItem it = a.items[seg];
    const int off = it.klen - it.qlen;  // absolute position of query 0
    // This lane's query (column i of S^T) and its visible key range.
    const int wq0 = it.q0 + qb * QW;
    const int qi = wq0 + i;
    const bool qvalid = qi < it.qlen;
    const int qic = qvalid ? qi : it.qlen - 1;
    const int aq = off + qic;
    const int vis_lo = W > 0 ? max(0, aq - W + 1) : 0;
    const int vis_hi = aq + 1;
    // The wave's 32 queries: bounds of their visible ranges.
    const bool wave_active = wq0 < it.qlen;
    const int wq1 = min(wq0 + QW - 1, it.qlen - 1);
    const int wlo_min = W > 0 ? max(0, off + wq0 - W + 1) : 0;
    const int wlo_max = W > 0 ? max(0, off + wq1 - W + 1) : 0;
    const int whi_min = off + wq0 + 1;
    const int whi_max = off + wq1 + 1;

    // The first tile's loads are issued before Q is read: a short segment waits once for both.
    TileShare<D, NW> share{a.kv, kbase, vbase, rs, stab, stage_table(a, it, stab), it.kbase, it.ks, it.ke,
                           wave, lane, -1, 0};
    f32x8 rk[UW], rv[UW];  // this wave's share of the next tile, as loaded
    auto load_tile = [&](int kt) {
      share.load_k(kt, rk);
      share.load_v(kt, rv);
    };
    load_tile(it.ks);

    // Q^T operand: lane (i, half) holds the parts of Q[query i][16 s + 8 half + 0..7] for the
    // whole key loop (queries past the sequence read its last one).
    Split8 q[KS];
    float qscale;  // takes a product of scaled q and k (of exponent 0) to log2 units
    {
      const float *qp = a.q + ((size_t)(it.qstart + qic) * a.hq + h) * D + 8 * half;
      f32x8 x[KS];
      float mx = 0.0f;
#pragma unroll
      for (int s = 0; s < KS; s++) {
        const float4 u = ld4(qp + 16 * s), v = ld4(qp + 16 * s + 4);
        x[s] = f32x8{u.x, u.y, u.z, u.w, v.x, v.y, v.z, v.w};
        mx = abs_max(mx, x[s]);
      }
      const int e = split_exp(max_halves(mx));
#pragma unroll
      for (int s = 0; s < KS; s++) q[s] = split8(x[s], qsign * split_scale(e));
      qscale = sl2 * split_unscale(e);
    }
    f32x16 o[NB];
#pragma unroll
    for (int b = 0; b < NB; b++)
#pragma unroll
      for (int r = 0; r < 16; r++) o[b][r] = 0.0f;
    float m_run = -INFINITY, m_top = -INFINITY;  // reference and largest max, log2 units
    float l_run = 0.0f, e_run = 0.0f;
    int o_exp = kMinExp;  // exponent of the V scale that o is in
    bool coarse = false;  // the split's steps show in this query's result

    // The tile in rk / rv: each wave's largest magnitudes, then (after a barrier) the exponents of
    // its scales, and its parts in LDS.
    float v_least = INFINITY;
    int v_needed = 1;
    auto share_max = [&](int b, int t) {
      const float m = max_waves(share.largest(rk), share.largest(rv));
      v_least = share.least_chunk(rv);
      v_needed = share.dims_needed(t);
      if (i == 0) smax[b][half][wave] = m;
    };
    int k_exp_in = kMinExp, v_unit = kMinExp, v_top = kMinExp;
    auto take_scales = [&](int b) {
      const TileExps sc = tile_exps<NW>(smax[b][half][lane & (NW - 1)]);
      k_exp_in = sc.a;
      v_unit = value_unit(sc.b, v_unit, v_top);
    };
    auto store_tile = [&](int b) {
      if (__popcll(__ballot(v_least < dim_limit(v_unit))) >= v_needed) uneven = 1;
      share.store_k(rk, split_scale(k_exp_in), sk[b]);
      share.store_v(rv, split_scale(v_unit), sv[b]);
    };
    auto read_split = [&](const _Float16 *p) {
      return Split8{*reinterpret_cast<const f16x8 *>(p),
                    *reinterpret_cast<const f16x8 *>(p + PART)};
    };

    // k_exp, v_exp: the exponents of the tile's scales.
    // The next tile (in rk / rv) is split and stored to buffer nb among the products of QK, and
    // the one after it loaded (next_kt; none if < 0).
    auto compute_tile = [&](int kt, const _Float16 *tk, const _Float16 *tv, int k_exp, int v_exp,
                            int nb, int next_kt) {
      if (!wave_active || kt >= whi_max || kt + KT <= wlo_min) {
        store_tile(nb);
        if (next_kt >= 0) load_tile(next_kt);
        return;
      }
      const bool full = (kt + KT <= whi_min) && (kt >= wlo_max);

      // S^T = K Q^T: register r of st holds key kt + 8 (r / 4) + 4 half + r % 4 of query i.
      f32x16 st;
#pragma unroll
      for (int r = 0; r < 16; r++) st[r] = 0.0f;
      // Operands are read kAhead steps before their products (the compiler would read each right
      // before its use and wait out the LDS latency every time).
      Split8 f[kAhead + 1];
      auto read_k = [&](int s) { return read_split(tk + k_pos<D>(i, 2 * s + half)); };
      auto read_v = [&](int u) {
        return read_split(tv + part_pos(32 * (u % NB) + i, 2 * (u / NB) + half));
      };
#pragma unroll
      for (int s = 0; s < kAhead; s++) f[s] = read_k(s);
#pragma unroll
      for (int s = 0; s < KS; s++) {
        if (s + kAhead < KS) f[(s + kAhead) % (kAhead + 1)] = read_k(s + kAhead);
        __builtin_amdgcn_sched_barrier(kKeepReads);
        st = mfma_split(f[s % (kAhead + 1)], q[s], st);
      }
#pragma unroll
      for (int u = 0; u < kAhead; u++) f[u] = read_v(u);
      __builtin_amdgcn_sched_barrier(kKeepReads);
      store_tile(nb);
      if (next_kt >= 0) load_tile(next_kt);

      if (!full) {
#pragma unroll
        for (int r = 0; r < 16; r++) {
          const int key = kt + 8 * (r >> 2) + 4 * half + (r & 3);
          st[r] = (key >= vis_lo && key < vis_hi) ? st[r] : -INFINITY;
        }
      }
      float mx = -INFINITY;
#pragma unroll
      for (int r = 0; r < 16; r++) mx = fmaxf(mx, st[r]);
      const float c = fmaxf(qscale * split_unscale(k_exp), 0x1p-126f);  // 0 * -inf is NaN
      coarse |= c > kMaxScoreUnit;
      mx = max_halves(mx) * c;
      const float mn = reference(mx, m_run, m_top);
      if (__any(mn != m_run)) {
        const float alpha = m_run == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m_run - mn);
        l_run *= alpha;
        e_run *= alpha * alpha;
#pragma unroll
        for (int b = 0; b < NB; b++) o[b] *= alpha;
        m_run = mn;
      }
      if (v_exp != o_exp) {
        const float alpha = __uint_as_float((uint32_t)max(0, 127 + o_exp - v_exp) << 23);
        e_run *= alpha * alpha;
#pragma unroll
        for (int b = 0; b < NB; b++) o[b] *= alpha;
        o_exp = v_exp;
      }
      const float ms = m_run == -INFINITY ? 0.0f : m_run;
      Split8 p[2];
      float lt[2];
#pragma unroll
      for (int s = 0; s < 2; s++) {
        f32x8 e;
#pragma unroll
        for (int j = 0; j < 8; j++) e[j] = __builtin_amdgcn_exp2f(fmaf(st[8 * s + j], c, -ms));
        lt[s] = ((e[0] + e[1]) + (e[2] + e[3])) + ((e[4] + e[5]) + (e[6] + e[7]));
        p[s] = split8(e, (float)(1 << kProbExp));
      }
      const float l_tile = lt[0] + lt[1];
      const float steps = split_steps(l_tile);
      e_run = fmaf(steps, steps, e_run);
      l_run += l_tile;  // one addition to the long sum per tile

      // O^T += V^T P^T, 16 keys a step (V chunk 2 s + half holds the lane's keys).
#pragma unroll
      for (int u = 0; u < 2 * NB; u++) {
        if (u + kAhead < 2 * NB) f[(u + kAhead) % (kAhead + 1)] = read_v(u + kAhead);
        __builtin_amdgcn_sched_barrier(kKeepReads);
        o[u % NB] = mfma_split(f[u % (kAhead + 1)], p[u / NB], o[u % NB]);
      }
    };

    // At the barrier of tile t every wave is done with tile t - 1, whose buffer takes tile
    // t + 1, tile t is in LDS, and so are the largest magnitudes of tile t + 1.
    const int ntiles = (it.ke - it.ks + KT - 1) / KT;
    share_max(0, 0);
    __syncthreads();
    take_scales(0);
    store_tile(0);
    if (ntiles > 1) load_tile(it.ks + KT);
    for (int t = 0; t < ntiles; t++) {
      const int kt = it.ks + t * KT;
      const int b = t & 1;
      const int k_exp = k_exp_in, v_exp = v_unit;
      share_max(b ^ 1, t + 1);  // the last tile stores itself once more, where nothing reads it
      __syncthreads();
      take_scales(b ^ 1);
      compute_tile(kt, sk[b], sv[b], k_exp, v_exp, b ^ 1, t + 2 < ntiles ? kt + 2 * KT : -1);
    }

    if (!wave_active) continue;
    const float l_tot = sum_halves(l_run);
    if (__any(coarse || uneven || unsound(largest_result<NB>(o, l_tot), sum_halves(e_run), v_top))) {
      again.add(seg);
      continue;
    }
    if (!qvalid) continue;
    const Dest d = destination(a, it, qi, h, D);
    const float f = result_factor(d, l_tot, m_run, m_top);
    // Register r of o[b] is dim 32 b + 8 (r / 4) + 4 half + r % 4.
#pragma unroll
    for (int b = 0; b < NB; b++)
#pragma unroll
      for (int r = 0; r < 16; r += 4)
        *reinterpret_cast<float4 *>(d.row + 32 * b + 2 * r + 4 * half) =
            result4(o[b], r, f, o_exp);
    if (d.partial && half == 0) {
      a.part_m[d.pidx] = m_top;
      a.part_l[d.pidx] = l_tot * f;
    }
  }
  for (int seg = again.next(again.first, seg_end); seg < seg_end; seg = again.next(seg + 1, seg_end)) {
    const TileItem it = a.items[seg];
    if (it.q0 + qb * QW < it.qlen) fp32_segment<D, NB>(a, it, kvh, h, it.q0 + qb * QW, 0);
  }
}

// Head dims 256 and 512: the dims of 32 queries are split over DS = D / 128 waves, which keeps a
// wave's Q, O and operand registers at those of d = 128 and eight waves (two per SIMD) on a CU.
// Each wave contracts its 128 dims of QK; the partial S^T meet in LDS and are added in a fixed
// order (S_0 + S_1, or (S_0 + S_1) + (S_2 + S_3)), so the DS waves hold the same scores, run the
// same softmax and accumulate their own 128 dims of O^T.
//
// One LDS buffer for K and one for V, each refilled while the other is in use: V of tile t is
// split and stored during QK of tile t, K of tile t + 1 during PV of tile t.  At d = 512 the
// tiles take 128 KB, so the partial scores are added pairwise in place (16 KB instead of 32),
// which costs one more barrier.
template <int D, int HPW>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2)))
prefill_split_wide_kernel(TileLaunch a) {
  constexpr int NW = 8, DW = 128, DS = D / DW;
  constexpr int KS = DW / 16, NB = DW / 32;
  constexpr int PART = KT * D;
  constexpr int UW = TileShare<D, NW>::UW;
  constexpr int SLOTS = DS == 2 ? NW : NW / 2;
  static_assert(DS == 2 || DS == 4, "two or four waves share a query group");
  __shared__ __attribute__((aligned(16))) _Float16 sk[2 * PART], sv[2 * PART];
  __shared__ __attribute__((aligned(16))) float spart[SLOTS][4][64][4];  // partial S^T
  __shared__ float smax[2][NW];  // each wave's largest |k| (of the next tile), |v|
  __shared__ int32_t stab[kPrefillTablePages];
  __shared__ int uneven;  // a tile's V dims are too unlike for one scale

  const int slot = blockIdx.x;
  const int seg_end = a.seg_off[slot + 1];
  const int rep = a.hq / a.hkv;
  const int groups = rep / HPW;
  const int kvh = blockIdx.y / groups;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ds = wave % DS, qg = wave / DS;  // dims [128 ds, 128 ds + 128) of query group qg
  const int h = kvh * rep + (blockIdx.y - kvh * groups) * HPW + qg % HPW;
  const int qb = qg / HPW;
  const int lane = threadIdx.x & 63;
  const int i = lane & 31, half = lane >> 5;
  const int W = a.window;
  // Scores are kept unscaled until the exponential; a negative scale goes into q's sign.  (Not 0:
  // 0 * -inf is NaN.)
  const float sl2 = fmaxf(fabsf(a.scale) * kLog2e, 0x1p-126f);
  const float qsign = a.scale < 0.0f ? -1.0f : 1.0f;
  const size_t rs = (size_t)a.hkv * D;

  Again again{a.seg_off[slot], 0};
  for (int seg = again.first; seg < seg_end; seg++) {
    __syncthreads();
    if (threadIdx.x == 0) uneven = 0;
    const TileItem it = a.items[seg];
    const int off = it.klen - it.qlen;
    const int wq0 = it.q0 + qb * QW;
    const int qi = wq0 + i;
    const bool qvalid = qi < it.qlen;
    const int qic = qvalid ? qi : it.qlen - 1;
    const int aq = off + qic;
    const int vis_lo = W > 0 ? max(0, aq - W + 1) : 0;
    const int vis_hi = aq + 1;
    const bool group_active = wq0 < it.qlen;
    const int wq1 = min(wq0 + QW - 1, it.qlen - 1);
    const int wlo_min = W > 0 ? max(0, off + wq0 - W + 1) : 0;
    const int wlo_max = W > 0 ? max(0, off + wq1 - W + 1) : 0;
    const int whi_min = off + wq0 + 1;
    const int whi_max = off + wq1 + 1;

    // The first tile's loads are issued before Q is read: a short segment waits once for both.
    TileShare<D, NW> share{a.kv, a.kv.k + (size_t)kvh * D, a.kv.v + (size_t)kvh * D, rs, stab,
                           stage_table(a, it, stab), it.kbase, it.ks, it.ke, wave, lane, -1, 0};
    f32x8 rk[UW], rv[UW];
    share.load_k(it.ks, rk);
    share.load_v(it.ks, rv);

    Split8 q[KS];  // lane (i, half): the parts of Q[query i][128 ds + 16 s + 8 half + 0..7]
    float qscale;
    {
      const float *qp = a.q + ((size_t)(it.qstart + qic) * a.hq + h) * D + DW * ds + 8 * half;
      f32x8 x[KS];
      float mx = 0.0f;
#pragma unroll
      for (int s = 0; s < KS; s++) {
        const float4 u = ld4(qp + 16 * s), v = ld4(qp + 16 * s + 4);
        x[s] = f32x8{u.x, u.y, u.z, u.w, v.x, v.y, v.z, v.w};
        mx = abs_max(mx, x[s]);
      }
      const int e = split_exp(max_halves(mx));
#pragma unroll
      for (int s = 0; s < KS; s++) q[s] = split8(x[s], qsign * split_scale(e));
      qscale = split_unscale(e);
    }
    f32x16 o[NB];
#pragma unroll
    for (int b = 0; b < NB; b++)
#pragma unroll
      for (int r = 0; r < 16; r++) o[b][r] = 0.0f;
    float m_run = -INFINITY, m_top = -INFINITY;  // reference and largest max, log2 units
    float l_run = 0.0f, e_run = 0.0f;
    int o_exp = kMinExp;  // exponent of the V scale that o is in
    bool coarse = false;  // the split's steps show in this query's result

    int k_exp_in = kMinExp, v_exp = kMinExp, v_top = kMinExp;
    auto share_max = [&](int t, float m) {
      const float x = max_waves(m, m);
      if (lane == 0) smax[t][wave] = x;
    };
    auto store_k = [&]() {
      const TileExps sc = tile_exps<NW>(smax[0][lane & 7]);
      k_exp_in = sc.a;
      share.store_k(rk, split_scale(sc.a), sk);
    };
    float v_least = INFINITY;
    int v_needed = 1;
    auto share_v_max = [&](int t) {
      share_max(1, share.largest(rv));
      v_least = share.least_chunk(rv);
      v_needed = share.dims_needed(t);
    };
    auto store_v = [&]() {
      const TileExps sc = tile_exps<NW>(smax[1][lane & 7]);
      v_exp = value_unit(sc.a, v_exp, v_top);
      if (__popcll(__ballot(v_least < dim_limit(v_exp))) >= v_needed) uneven = 1;
      share.store_v(rv, split_scale(v_exp), sv);
    };
    auto read_split = [&](const _Float16 *p) {
      return Split8{*reinterpret_cast<const f16x8 *>(p),
                    *reinterpret_cast<const f16x8 *>(p + PART)};
    };

    const int ntiles = (it.ke - it.ks + KT - 1) / KT;
    share_max(0, share.largest(rk));
    share_v_max(0);
    __syncthreads();
    store_k();
    if (ntiles > 1) share.load_k(it.ks + KT, rk);
    __syncthreads();
    for (int t = 0; t < ntiles; t++) {
      const int kt = it.ks + t * KT;
      const bool more = t + 1 < ntiles;
      const bool active = group_active && kt < whi_max && kt + KT > wlo_min;
      const float c = qscale * split_unscale(k_exp_in);

      // K of tile t is in LDS; V of tile t is in rv, its maxima in smax[1]; PV of tile t - 1 is
      // done everywhere.
      store_v();
      if (more) share.load_v(kt + KT, rv);
      f32x16 st;
#pragma unroll
      for (int r = 0; r < 16; r++) st[r] = 0.0f;
      if (active) {
        // k_pos<D>(i, 16 ds + 2 s + half); opaque, or the compiler keeps all of them, in scratch.
        int at = k_pos<D>(i, (DW / 8) * ds + half);
        asm volatile("" : "+v"(at));
        auto read_k = [&](int s) { return read_split(sk + (at ^ (s << 4))); };
        Split8 f[kAhead + 1];
#pragma unroll
        for (int s = 0; s < kAhead; s++) f[s] = read_k(s);
#pragma unroll
        for (int s = 0; s < KS; s++) {
          if (s + kAhead < KS) f[(s + kAhead) % (kAhead + 1)] = read_k(s + kAhead);
          __builtin_amdgcn_sched_barrier(kKeepReads);
          st = mfma_split(f[s % (kAhead + 1)], q[s], st);
        }
        coarse |= c * sl2 > kMaxScoreUnit;
        st *= c;  // a power of two: the partial score in its own units
      }
      auto put = [&](int sl) {
#pragma unroll
        for (int r = 0; r < 16; r += 4)
          *reinterpret_cast<float4 *>(spart[sl][r >> 2][lane]) =
              make_float4(st[r], st[r + 1], st[r + 2], st[r + 3]);
      };
      auto get = [&](int sl) {
        f32x16 x;
#pragma unroll
        for (int r = 0; r < 16; r += 4) {
          const float4 y = ld4(spart[sl][r >> 2][lane]);
          x[r] = y.x, x[r + 1] = y.y, x[r + 2] = y.z, x[r + 3] = y.w;
        }
        return x;
      };
      if (more) share_max(0, share.largest(rk));
      if constexpr (DS == 2) {
        if (active) put(wave);
        __syncthreads();
        if (active) {
          const f32x16 other = get(wave ^ 1);
          st = st + other;
        }
      } else {
        if (active && (ds & 1)) put(wave >> 1);
        __syncthreads();
        if (active && !(ds & 1)) {
          st = st + get(wave >> 1);
          put(wave >> 1);
        }
        __syncthreads();
        if (active) {
          const f32x16 lo = get(2 * qg), hi = get(2 * qg + 1);
          st = lo + hi;
        }
      }

      // V of tile t is in LDS; QK of tile t is done everywhere, the maxima of K of tile t + 1 are
      // in smax[0].
      if (more) {
        store_k();
        if (t + 2 < ntiles) share.load_k(kt + 2 * KT, rk);
      }
      if (active) {
        const bool full = (kt + KT <= whi_min) && (kt >= wlo_max);
        if (!full) {
#pragma unroll
          for (int r = 0; r < 16; r++) {
            const int key = kt + 8 * (r >> 2) + 4 * half + (r & 3);
            st[r] = (key >= vis_lo && key < vis_hi) ? st[r] : -INFINITY;
          }
        }
        float mx = -INFINITY;
#pragma unroll
        for (int r = 0; r < 16; r++) mx = fmaxf(mx, st[r]);
        mx = max_halves(mx) * sl2;
        const float mn = reference(mx, m_run, m_top);
        if (__any(mn != m_run)) {
          const float alpha = m_run == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m_run - mn);
          l_run *= alpha;
          e_run *= alpha * alpha;
#pragma unroll
          for (int b = 0; b < NB; b++) o[b] *= alpha;
          m_run = mn;
        }
        if (v_exp != o_exp) {
          const float alpha = __uint_as_float((uint32_t)max(0, 127 + o_exp - v_exp) << 23);
          e_run *= alpha * alpha;
#pragma unroll
          for (int b = 0; b < NB; b++) o[b] *= alpha;
          o_exp = v_exp;
        }
        const float ms = m_run == -INFINITY ? 0.0f : m_run;
        Split8 p[2];
        float lt[2];
#pragma unroll
        for (int s = 0; s < 2; s++) {
          f32x8 e;
#pragma unroll
          for (int j = 0; j < 8; j++) e[j] = __builtin_amdgcn_exp2f(fmaf(st[8 * s + j], sl2, -ms));
          lt[s] = ((e[0] + e[1]) + (e[2] + e[3])) + ((e[4] + e[5]) + (e[6] + e[7]));
          p[s] = split8(e, (float)(1 << kProbExp));
        }
        const float l_tile = lt[0] + lt[1];
        const float steps = split_steps(l_tile);
        e_run = fmaf(steps, steps, e_run);
        l_run += l_tile;  // one addition to the long sum per tile
        auto read_v = [&](int u) {
          return read_split(sv + part_pos(DW * ds + 32 * (u % NB) + i, 2 * (u / NB) + half));
        };
        Split8 f[kAhead + 1];
#pragma unroll
        for (int u = 0; u < kAhead; u++) f[u] = read_v(u);
#pragma unroll
        for (int u = 0; u < 2 * NB; u++) {
          if (u + kAhead < 2 * NB) f[(u + kAhead) % (kAhead + 1)] = read_v(u + kAhead);
          __builtin_amdgcn_sched_barrier(kKeepReads);
          o[u % NB] = mfma_split(f[u % (kAhead + 1)], p[u / NB], o[u % NB]);
        }
      }
      if (more) share_v_max(t + 1);
      __syncthreads();
    }

    const float l_tot = sum_halves(l_run);
    // The waves that share the queries decide together, over all of their dims.
    float result = coarse || uneven ? -INFINITY : largest_result<NB>(o, l_tot);
    float *results = &spart[0][0][0][0];
    if (half == 0) results[wave * QW + i] = result;
    __syncthreads();
#pragma unroll
    for (int j = 0; j < DS; j++) {
      const float x = results[(qg * DS + j) * QW + i];
      result = result < 0.0f || x < 0.0f ? -INFINITY : fmaxf(result, x);
    }
    if (__any(unsound(result, sum_halves(e_run), v_top))) {
      again.add(seg);
      continue;
    }
    if (!qvalid) continue;
    const Dest d = destination(a, it, qi, h, D);
    const float f = result_factor(d, l_tot, m_run, m_top);
#pragma unroll
    for (int b = 0; b < NB; b++)
#pragma unroll
      for (int r = 0; r < 16; r += 4)
        *reinterpret_cast<float4 *>(d.row + DW * ds + 32 * b + 2 * r + 4 * half) =
            result4(o[b], r, f, o_exp);
    if (d.partial && half == 0 && ds == 0) {
      a.part_m[d.pidx] = m_top;
      a.part_l[d.pidx] = l_tot * f;
    }
  }
  for (int seg = again.next(again.first, seg_end); seg < seg_end; seg = again.next(seg + 1, seg_end)) {
    const TileItem it = a.items[seg];
    if (it.q0 + qb * QW < it.qlen) fp32_segment<D, NB>(a, it, kvh, h, it.q0 + qb * QW, DW * ds);
  }
}

namespace {

template <int D>
constexpr int split_waves() {
  return D == 64 ? 4 : 8;
}
// Waves that share 32 queries.
constexpr int dim_waves(int head_dim) { return head_dim <= 128 ? 1 : head_dim / 128; }

// Calls f with the kernel for this head dim and number of query heads per workgroup.
template <typename F>
hipError_t with_kernel(int head_dim, int hpw, F f) {
  switch (head_dim * 8 + hpw) {
    case 64 * 8 + 1: return f(prefill_split_kernel<64, 1, split_waves<64>()>);
    case 128 * 8 + 1: return f(prefill_split_kernel<128, 1, split_waves<128>()>);
    case 128 * 8 + 2: return f(prefill_split_kernel<128, 2, split_waves<128>()>);
    case 256 * 8 + 1: return f(prefill_split_wide_kernel<256, 1>);
    case 256 * 8 + 2: return f(prefill_split_wide_kernel<256, 2>);
    case 512 * 8 + 1: return f(prefill_split_wide_kernel<512, 1>);
    default: return hipErrorInvalidValue;
  }
}

int waves(int head_dim) { return head_dim == 64 ? split_waves<64>() : split_waves<128>(); }

}  // namespace

// Most query heads one prefill workgroup carries at this head dim (it covers at least 64 queries of
// each).
int prefill_max_heads(int head_dim) { return head_dim == 64 || head_dim == 512 ? 1 : 2; }

int prefill_tile_queries(int head_dim, int heads_per_wg) {
  return QW * (waves(head_dim) / dim_waves(head_dim) / heads_per_wg);
}

bool prefill_kernel_supports(int head_dim, int heads_per_wg) {
  return (head_dim == 64 || head_dim == 128 || head_dim == 256 || head_dim == 512) &&
         (heads_per_wg == 1 || heads_per_wg == 2) && heads_per_wg <= prefill_max_heads(head_dim);
}

// Uncached: the caller (one context per device) keeps the answer.  The query reads the
// current device's properties, so the caller makes its device current first.
int prefill_blocks_per_cu(int head_dim, int heads_per_wg) {
  int b = 0;
  if (with_kernel(head_dim, heads_per_wg, [&](auto k) {
        return hipOccupancyMaxActiveBlocksPerMultiprocessor(&b, k, 64 * waves(head_dim), 0);
      }) != hipSuccess ||
      b < 1)
    b = 1;
  return b;
}

hipError_t launch_prefill_tiles(const TileLaunch &a, int hpw, hipStream_t s) {
  if (a.num_items <= 0 || a.num_slots <= 0) return hipSuccess;
  const dim3 grid(a.num_slots, a.hkv * ((a.hq / a.hkv) / hpw)), block(64 * waves(a.head_dim));
  return with_kernel(a.head_dim, hpw, [&](auto k) {
    hipLaunchKernelGGL(k, grid, block, 0, s, a);
    return hipGetLastError();
  });
}

}  // namespace nva
