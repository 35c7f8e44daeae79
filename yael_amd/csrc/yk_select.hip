// yk_select.hip -- fused FP32 distance + k-smallest selection on MFMA.
//
// Reference semantics (yael nn.c):
//   dist(q,b) = float( double(sum_j q_j*q_j) [float products, double sum]
//                    + double(float-accumulated sum_j b_j*b_j) )  - 2 * q.b
//   (nn.c:108-126), optionally times w[b] (nn.c:497-500); type 16 is the
//   plain dot product (nn.c:266-306).  k = 1: strict '<' from (-1, 1e30)
//   (nn.c:404-440).  k > 1: the k smallest non-NaN values, sorted, padded
//   with (-1, 0xffffffff) (nn.c:463-525).  Equal values are ordered by base
//   index (the reference's ascending scan gives the same for k = 1).
//
// Every selection works on 64-bit keys (order-preserving float bits << 32 |
// base index): key order is (value, index) order, so the result does not
// depend on how the base is split across lanes, waves and workgroups.
//
// Scan kernel (gfx950, wave64, v_mfma_f32_32x32x2_f32):
//   * a workgroup of W waves; each wave owns 32*NB queries (the MFMA
//     columns, held in registers when d <= 128, in the LDS-staged kernel
//     d <= 256) and takes its workgroup's base range in blocks of 32 rows (the
//     MFMA rows), streamed from global memory or staged through LDS;
//   * per 16-wide k-chunk a lane loads 8 contiguous floats (two dwordx4) of
//     its row: A and B use the same k permutation, each 64-byte row segment
//     is read once per block;
//   * the 32x32 accumulator gives each lane one query and 16 base rows, so
//     the epilogue is lane-local:
//       MODE 0  running (value, index) minimum           -> k = 1
//       MODE 1  each lane's own minimum over its rows     -> the threshold
//               sketch for k > 1
//       MODE 2  register top-R of keys (R <= 16)          -> what the filtered
//               pass leaves over for k <= 16
//       MODE 3  append every key <= the query's threshold T_q to a per-query
//               candidate list (staged in LDS, one global
//               atomic per YK_CSTAGE keys)                -> k > 1
//   * a persistent grid (resident workgroups only) walks the work items;
//     each XCD owns a contiguous run of items so workgroups that share a
//     base range share that XCD's L2;
//   * the base is split over work items when the query tiles alone cannot
//     fill 256 CUs; split results are merged by small sort kernels.
//
// k > 1 is exact in two passes: (A) MODE 1 over a 1-in-stride sample of
// base blocks with >= k splits gives, per query, >= 2k minima of disjoint
// row subsets -- distinct real keys -- whose k-th smallest bounds the true
// k-th smallest key from above: the starting bound T_q for k <= 16.  For k >
// 16 a smaller one of the minima is the estimated bound (yk_bound_rank).  (B)
// MODE 3 over the whole base collects every key <= T_q, then a per-query sort
// keeps the k smallest.  A query with fewer than k keys under an estimate is
// scanned without a bound; one whose candidates overflow the list gets a
// tighter T_q (the k-th smallest of the keys it did capture, an upper bound)
// and is scanned again, or for k <= 16 left to MODE 2.
#include <hip/hip_runtime.h>
#include <math.h>
#include <pthread.h>
#include <stdio.h>

#include <type_traits>

#include "../../include/yael_mi355x.h"
#include "yk.h"
#include "yk_dev.h"
#include "yk_wsel.h"

typedef float f32x16 __attribute__((ext_vector_type(16)));
// word 3 of a raw (untyped, stride 0) buffer descriptor on gfx9-family GPUs
#define YK_BUF_DWORD3 0x00020000

#define YK_CAND_CAP 4096  // candidate keys kept per query at most (MODE 3)
#define YK_CSTAGE 8       // MODE 3: keys staged in LDS per (lane, query tile)
#define YK_REG_R 16       // register top-R of MODE 2

struct ScanArgs {
  const float *q;
  const double *qn;
  long nq;
  const float *b;
  const float *bn;  // >= round_up(nb, 32) entries
  const float *w;   // optional, >= round_up(nb, 32) entries
  long nb;
  int ld;
  int type;
  long brange;  // base rows per split, multiple of bstep
  long bstep;   // rows between processed 32-row blocks (32 * sampling stride)
  int nsplit;
  int tiles_x;
  int total;
  int per_xcd;
  int *out_i;      // MODE 0, nsplit == 1
  float *out_d;
  uint64_t *part;  // MODE 0: [nq][nsplit]; MODE 2: [nq][nsplit][2][R]
  const uint64_t *thr;  // MODE 3: per-query threshold key (0 = inactive)
  int *cnt;             // MODE 3: per-query candidate count
  uint64_t *cand;       // MODE 3: [nq][cap]
  int cap;              // places of a query's list (yk_cand_cap)
  // batched form (item_inst != NULL): work item -> (instance, point tile);
  // q/qn/out_* are the concatenated points of all instances, b/bn the
  // instances' centroid sets (kpad rows apart), nb is unused
  const int *item_inst;
  const int *item_tile;
  const long *inst_off;  // ninst + 1 point offsets
  int kc, kpad;
  const int *done;  // instances already finished (skipped)
  const int *qidx;  // optional: point j of the concatenation is row qidx[j] of q / qn
  int *tick;        // per XCD, zero at launch: item tickets (nullptr: static order)
  const int *flag;  // MODE 2 as the fallback of the filtered search: 0 = nothing left to do
  int units;        // yk_scan_f32_lds, MODE 0: > 0 even shares of tiles x units blocks
  int inter;        // MODE 1: split s takes sampled blocks s, s + nsplit, ...
};

// The hardware hands consecutive block ids to the 8 XCDs in turn; give each
// XCD a contiguous run of work items (split-major), so the workgroups that
// share a base range also share that XCD's L2.
__device__ __forceinline__ int yk_xcd_item(int per_xcd) {
  int id = blockIdx.x;
  return (id & 7) * per_xcd + (id >> 3);
}

// sorted (ascending) register list: insert x, drop the largest
template <int R>
__device__ __forceinline__ void yk_reg_insert(uint64_t (&t)[R], uint64_t x) {
#pragma unroll
  for (int i = R - 1; i > 0; i--) {
    uint64_t lo = t[i - 1], cur = t[i];
    t[i] = x < lo ? lo : (x < cur ? x : cur);
  }
  t[0] = x < t[0] ? x : t[0];
}

// A lane's 16 row norms, in registers or (the kernels that stage them) read
// from LDS where they are used: value i's norm is entry 8 (i >> 2) + (i & 3)
// of the lane half's block norms.  dbl: the norm as a double, held as one in
// LDS (a conversion per value and block less); from a register it is converted
// where it is used (the compiler moved the 16 conversions in front of the
// branch, 17 of 117 vector instructions that every block executed).
struct YkNormRegs {
  float n[16];
  __device__ __forceinline__ float operator[](int i) const { return n[i]; }
  __device__ __forceinline__ double dbl(int i) const {
    float x = n[i];
    asm volatile("" : "+v"(x));
    return x;
  }
  __device__ __forceinline__ void all(float (&x)[16]) const {
#pragma unroll
    for (int i = 0; i < 16; i++) x[i] = n[i];
  }
};
struct YkNormLds {
  const float *p;
  const double *pd;
  __device__ __forceinline__ double dbl(int i) const { return pd[8 * (i >> 2) + (i & 3)]; }
  __device__ __forceinline__ float operator[](int i) const { return p[8 * (i >> 2) + (i & 3)]; }
  __device__ __forceinline__ float pick(int is) const { return p[8 * (is >> 2) + (is & 3)]; }
  __device__ __forceinline__ void all(float (&x)[16]) const {
#pragma unroll
    for (int g = 0; g < 4; g++) {
      const float4 v = *(const float4 *)(p + 8 * g);
      x[4 * g] = v.x, x[4 * g + 1] = v.y, x[4 * g + 2] = v.z, x[4 * g + 3] = v.w;
    }
  }
};

// The approximations of a lane's 16 values, m_i = bn - 2 acc (type 16: acc);
// fl(qn + m_i) differs from the exact expression by far less than slack =
// 2^-19 (|q|^2 + max|b|^2) (|2 q.b| <= |q|^2 + |b|^2).  Returns their minimum;
// x -> fl(qn + x) is monotone, so the query norm is added once, to it.
template <bool DOT, class Norms>
__device__ __forceinline__ float yk_approx16(const f32x16 &acc, const Norms &nn, float (&m)[16]) {
  float mm = INFINITY;
#pragma unroll
  for (int i = 0; i < 16; i++) {
    m[i] = DOT ? acc[i] : __builtin_fmaf(-2.0f, acc[i], nn[i]);
    mm = fminf(mm, m[i]);
  }
  return mm;
}

// Of the lane's values with m_i <= th: how many, and the last one's i and
// acc.  One candidate per lane is the common case of the filtered pass: the
// wave then evaluates, tests and appends one exact value, not sixteen.
__device__ __forceinline__ int yk_pick16(const f32x16 &acc, const float (&m)[16], float th,
                                         int &is, float &as) {
  int cnt = 0;
  is = 0;
  as = acc[0];
#pragma unroll
  for (int i = 0; i < 16; i++) {
    const bool c = m[i] <= th;
    cnt += c ? 1 : 0;
    is = c ? i : is;
    as = c ? acc[i] : as;
  }
  return cnt;
}

// One full block's epilogue for k = 1 and the sketch (each lane keeps the best
// of its own rows), unweighted.  With `test` the float approximations decide
// first whether any of the lane's values can improve its best; a range's
// first blocks go without: a wave runs the exact pass when any of its 64
// lanes may improve, which at block j of a range happens with probability
// about 1 - (1 - 1/(j+1))^64, so early blocks would pay for both.  The exact
// pass takes the exact FP64-normed expression for all 16 values and their
// minimum; where a lane improves, the first row of that value is looked up
// (the smallest index wins a tie).  What counts is the number of vector
// instructions: they do not overlap with the FP32 MFMAs of the SIMD's other
// waves (d = 16, k = 256: the matrix unit busy 46% and vector instructions
// issuing 58% of the cycles; the norms read as doubles and the row found after
// the minimum: 8 sub-spaces of 1e6 points, 10 iterations 16.3 -> 15.4 ms).
// Rows past the base are zeros with a norm of YK_FAR_NORM: no such value is
// below 1e30, where bv starts.
// (Picking out the lanes' one candidate by the approximations first, to
// evaluate one exact value per lane, measured slower: 26.8 against 18.2 ms
// for the 8 sub-spaces of 1e6 points, d = 16, k = 256, 10 iterations -- the
// selects cost as much as the FP64 operations they replace.)
#define YK_FAR_NORM 1e36f

template <bool DOT, class Norms>
__device__ __forceinline__ void yk_best1_block(const f32x16 &acc, const Norms &nn, double qnd,
                                               long bb, int h, bool test, float &bv, int &bi) {
  // Empty asm statements on the operands keep each pass inside its branch
  // (the compiler would otherwise hoist parts it shares with the general
  // path, executing them for every block).
  if (test) {
    const float qf = (float)qnd;
    float mm = INFINITY, nmax = 0.f, ns[16];
    nn.all(ns);  // (four 16-byte reads: between the statements below, sixteen)
#pragma unroll
    for (int i = 0; i < 16; i++) {
      float ax = acc[i], nx = ns[i];
      asm volatile("" : "+v"(ax), "+v"(nx));
      mm = fminf(mm, DOT ? ax : __builtin_fmaf(-2.0f, ax, nx));
      nmax = fmaxf(nmax, nx);
    }
    const float m = DOT ? mm : qf + mm;
    const float slack = DOT ? 0.f : 0x1p-19f * (qf + nmax);
    if (!(m - slack <= bv) && m == m) return;
  }
  double qd = qnd;
  asm volatile("" : "+v"(qd));
  // value i sits at row bb + 4 h + 8 (i >> 2) + (i & 3).  (The fused form
  // rounds as bn+qn - 2 acc does: 2 acc is exact, and where it would
  // overflow the norms' sum has too.)
  float v[16], mm = INFINITY;
#pragma unroll
  for (int i = 0; i < 16; i++) {
    v[i] = DOT ? acc[i] : __builtin_fmaf(-2.0f, acc[i], (float)(qd + nn.dbl(i)));
    mm = fminf(mm, v[i]);
  }
  if (!(mm < bv)) return;
  int bo = 0;
#pragma unroll
  for (int i = 15; i >= 0; i--) bo = v[i] == mm ? 8 * (i >> 2) + (i & 3) : bo;
  // (of a +0 and a -0, which only the dot product has, the first one's bits)
  if (DOT && mm == 0.0f) {
#pragma unroll
    for (int i = 15; i >= 0; i--) mm = v[i] == 0.0f ? v[i] : mm;
  }
  bv = mm;
  bi = (int)bb + 4 * h + bo;
}

// the largest of a lane's 16 row norms
template <class Norms>
__device__ __forceinline__ float yk_max16(const Norms &nn) {
  float nmax = 0.f;
#pragma unroll
  for (int i = 0; i < 16; i++) nmax = fmaxf(nmax, nn[i]);
  return nmax;
}

// NCH > 0: queries register-resident, exactly NCH 16-wide chunks (ld = 16
// NCH, so every chunk loop is unrolled without guards); NCH = 0: both
// operands streamed from memory.
template <int NB, int NCH, int MODE, int R>
__global__ __launch_bounds__(256) void yk_scan_f32(ScanArgs a0) {
  constexpr bool QRES = NCH > 0;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nwave = blockDim.x >> 6;
  const int r = lane & 31, h = lane >> 5;
  // Persistent grid: the hardware deals block ids to the 8 XCDs in turn;
  // XCD x owns the contiguous run of work items [x*per_xcd, (x+1)*per_xcd)
  // (split-major, so concurrently running workgroups of one XCD share a base
  // range in its L2), and its workgroups stride through that run.
  if (MODE == 2 && a0.flag && *a0.flag == 0) return;
  const int xcd = blockIdx.x & 7, local = blockIdx.x >> 3, wpx = gridDim.x >> 3;
  const int ibeg = xcd * a0.per_xcd, iend = min(a0.total, ibeg + a0.per_xcd);
  // MODE 3: candidate keys are staged in LDS, YK_CSTAGE per (query tile,
  // lane), and appended to the query's global list a region at a time (one
  // atomic per region instead of one per key; the count keeps growing past
  // YK_CAND_CAP so the select kernel sees an overflow)
  __shared__ uint64_t cstage[MODE == 3 ? 4 * NB * 64 * YK_CSTAGE : 1];
  uint64_t *const cs = cstage + (MODE == 3 ? wave * NB * 64 * YK_CSTAGE : 0);
  // a fixed first item, then tickets from the XCD's counter: the XCD's
  // workgroups keep to a window of consecutive items (one or two base ranges
  // in its L2) instead of drifting apart
  __shared__ int s_item;
  auto next_item = [&](int it) {
    if (!a0.tick) return it + wpx;
    __syncthreads();  // every wave has read the previous ticket
    if (threadIdx.x == 0) s_item = ibeg + wpx + atomicAdd(&a0.tick[xcd], 1);
    __syncthreads();
    return s_item;
  };
  for (int item = ibeg + local; item < iend; item = next_item(item)) {
  ScanArgs a = a0;
  int tile, split;
  if (a0.item_inst) {
    const int inst = a0.item_inst[item];
    // -1: an item past a level's last one (the tree descent's launch bound)
    if (inst < 0 || (a0.done && a0.done[inst])) continue;
    tile = a0.item_tile[item];
    split = 0;
    const long off = a0.inst_off[inst];
    if (a0.qidx) {
      a.qidx = a0.qidx + off;  // rows through the index table, q and qn as given
    } else {
      a.q = a0.q + off * a0.ld;
      a.qn = a0.qn + off;
    }
    a.nq = a0.inst_off[inst + 1] - off;
    a.b = a0.b + (long)inst * a0.kpad * a0.ld;
    a.bn = a0.bn + (long)inst * a0.kpad;
    a.nb = a0.kc;
    a.out_i = a0.out_i + off;
    a.out_d = a0.out_d + off;
  } else {
    tile = item % a0.tiles_x;
    split = item / a0.tiles_x;
  }
  const long qbase = ((long)tile * nwave + wave) * (32 * NB);
  // (interleaved sketch splits: neighbouring sampled blocks fall into
  // different splits, so rows near each other in the base do not all end up
  // in one subset's minimum)
  const bool inter = MODE == 1 && a.inter;
  const long bbeg = (long)split * (inter ? a.bstep : a.brange);
  const long bend = inter ? a.nb : min(a.nb, bbeg + a.brange);
  if (inter) a.bstep *= a.nsplit;
  const int nch = a.ld >> 4;
  const int ld = a.ld;
  const bool dot = (a.type == YK_DOT);

  long qrow[NB];  // the query's position (outputs)
  long qsrc[NB];  // its row of q / qn
  bool qok[NB];
  double qnd[NB];
#pragma unroll
  for (int j = 0; j < NB; j++) {
    long qi = qbase + j * 32 + r;
    qok[j] = qi < a.nq;
    qrow[j] = qok[j] ? qi : a.nq - 1;
    qsrc[j] = a.qidx ? (long)a.qidx[qrow[j]] : qrow[j];
    qnd[j] = dot ? 0.0 : a.qn[qsrc[j]];
  }

  // selection state
  float bv[NB];
  int bi[NB];
  int ncs[NB];
  auto flush = [&](int j, int n) {
    const int base = atomicAdd(&a.cnt[qrow[j]], n);
    const uint64_t *src = cs + (j * 64 + lane) * YK_CSTAGE;
    for (int s_ = 0; s_ < n; s_++)
      if (base + s_ < a.cap) a.cand[qrow[j] * a.cap + base + s_] = src[s_];
  };
  uint64_t top[NB][MODE == 2 ? R : 1];
  uint64_t T[NB];
  float Tv[NB];
#pragma unroll
  for (int j = 0; j < NB; j++) {
    bv[j] = 1e30f;
    bi[j] = -1;
    ncs[j] = 0;
#pragma unroll
    for (int s = 0; s < (MODE == 2 ? R : 1); s++) top[j][s] = YK_KEY_NONE;
    T[j] = MODE == 3 || (MODE == 2 && a.thr) ? a.thr[qrow[j]] : 0;
    Tv[j] = (T[j] == 0) ? -INFINITY
                        : (T[j] == YK_KEY_NONE ? INFINITY : yk_fkey_inv((uint32_t)(T[j] >> 32)));
  }
  if (MODE == 3 || (MODE == 2 && a.thr)) {
    bool act = false;
#pragma unroll
    for (int j = 0; j < NB; j++) act |= qok[j] && T[j] != 0;
    if (!__any(act)) continue;  // every query of this wave is already final
  }

  float4 qreg[NB][QRES ? 2 * NCH : 1];
  if (QRES) {
#pragma unroll
    for (int j = 0; j < NB; j++)
#pragma unroll
      for (int c = 0; c < NCH; c++) {
        const float *p = a.q + qsrc[j] * ld + c * 16 + h * 8;
        qreg[j][2 * c] = *(const float4 *)p;
        qreg[j][2 * c + 1] = *(const float4 *)(p + 4);
      }
  }

  // the next block's base operand is loaded while the current one is
  // multiplied (register double buffer, QRES only).  Buffer loads: a
  // descriptor based at the item's first row, the block's row offset in a
  // scalar register, the lane's (row, half) offset in a vector register
  // (rows past nb clamped to the last row, masked by the epilogue) -- no
  // 64-bit vector address arithmetic per block.  The planner keeps an
  // item's rows within 2^31 bytes.
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
      (void *)(a.b + bbeg * ld), 0, (int)min((a.nb - bbeg) * ld * 4, 0x7fffffffL), YK_BUF_DWORD3);
  // With one or two chunks a block is only 8-16 MFMAs: its base norms
  // (rows 8g + 4h .. +3) are loaded at the end of the previous block, into
  // the registers the epilogue reads, so that the epilogue does not wait for
  // them -- nor, with them, for the next block's operands issued meanwhile
  // (those are younger).  Dot-product searches read no norms.
  // Weighted searches are served by the other variants (the launcher's
  // choice), so these kernels compile without the weights' loads.
  constexpr bool NPF = QRES && NCH <= 2;
  const float *const wts = NPF ? nullptr : a.w;
  float4 anext[QRES ? 2 * NCH : 1];
  // Buffer loads based at the item's first row (bn holds round_up(nb, 32)
  // entries); for a dot-product search the descriptor has no records, so
  // the loads are unconditional and return zeros without touching memory.
  float4 nn4[NPF ? 4 : 1];
  const __amdgpu_buffer_rsrc_t rsn = __builtin_amdgcn_make_buffer_rsrc(
      (void *)(dot ? a.b : a.bn + bbeg), 0,
      dot ? 0 : (int)min((((a.nb + 31) & ~31L) - bbeg) * 4, 0x7fffffffL), YK_BUF_DWORD3);
  auto loadn = [&](long bb) {
#pragma unroll
    for (int g = 0; g < 4; g++)
      nn4[g] = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(
                                              rsn, 16 * h, (int)((bb - bbeg) * 4) + 32 * g, 0));
  };
  auto loadb = [&](long bb) {
    const int soff = (int)((bb - bbeg) * ld * 4);
    const int voff = ((int)min((long)r, a.nb - 1 - bb) * ld + h * 8) * 4;
#pragma unroll
    for (int c = 0; c < NCH; c++) {
      anext[2 * c] = __builtin_bit_cast(
          float4, __builtin_amdgcn_raw_buffer_load_b128(rs, voff, soff + c * 64, 0));
      anext[2 * c + 1] = __builtin_bit_cast(
          float4, __builtin_amdgcn_raw_buffer_load_b128(rs, voff + 16, soff + c * 64, 0));
    }
  };
  if (QRES && bbeg < bend) loadb(bbeg);
  if (NPF && bbeg < bend) loadn(bbeg);
  for (long bb = bbeg; bb < bend; bb += a.bstep) {
    const long brow = min(bb + r, a.nb - 1);
    const float *bp = a.b + brow * ld + h * 8;
    f32x16 acc[NB];
#pragma unroll
    for (int j = 0; j < NB; j++)
#pragma unroll
      for (int e = 0; e < 16; e++) acc[j][e] = 0.f;

    if (QRES) {
      float4 av[QRES ? 2 * NCH : 1];
#pragma unroll
      for (int c = 0; c < 2 * NCH; c++) av[c] = anext[c];
      {
        // unconditional (past the range it reloads the current block): a
        // conditional prefetch joins paths with different outstanding-load
        // counts, and the wait before the MFMAs would then also wait for the
        // loads just issued
        loadb(bb + a.bstep < bend ? bb + a.bstep : bb);
      }
#pragma unroll
      for (int c = 0; c < NCH; c++)
        {
#pragma unroll
          for (int j = 0; j < NB; j++) {
            float4 a0 = av[2 * c], a1 = av[2 * c + 1];
            float4 b0 = qreg[j][QRES ? 2 * c : 0], b1 = qreg[j][QRES ? 2 * c + 1 : 0];
            acc[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a0.x, b0.x, acc[j], 0, 0, 0);
            acc[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a0.y, b0.y, acc[j], 0, 0, 0);
            acc[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a0.z, b0.z, acc[j], 0, 0, 0);
            acc[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a0.w, b0.w, acc[j], 0, 0, 0);
            acc[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a1.x, b1.x, acc[j], 0, 0, 0);
            acc[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a1.y, b1.y, acc[j], 0, 0, 0);
            acc[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a1.z, b1.z, acc[j], 0, 0, 0);
            acc[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a1.w, b1.w, acc[j], 0, 0, 0);
          }
        }
    } else {
      for (int c = 0; c < nch; c++) {
        float4 a0 = *(const float4 *)(bp + c * 16);
        float4 a1 = *(const float4 *)(bp + c * 16 + 4);
#pragma unroll
        for (int j = 0; j < NB; j++) {
          const float *qp = a.q + qsrc[j] * ld + c * 16 + h * 8;
          float4 b0 = *(const float4 *)qp, b1 = *(const float4 *)(qp + 4);
          acc[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a0.x, b0.x, acc[j], 0, 0, 0);
          acc[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a0.y, b0.y, acc[j], 0, 0, 0);
          acc[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a0.z, b0.z, acc[j], 0, 0, 0);
          acc[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a0.w, b0.w, acc[j], 0, 0, 0);
          acc[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a1.x, b1.x, acc[j], 0, 0, 0);
          acc[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a1.y, b1.y, acc[j], 0, 0, 0);
          acc[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a1.z, b1.z, acc[j], 0, 0, 0);
          acc[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a1.w, b1.w, acc[j], 0, 0, 0);
        }
      }
    }

    // epilogue: lane holds query column r and base rows 8g + 4h + e
    YkNormRegs nrm;
    float (&nn)[16] = nrm.n;
    float ww[16];
#pragma unroll
    for (int g = 0; g < 4; g++) {
      const long b4 = bb + 8 * g + 4 * h;
      float4 n4 = NPF   ? nn4[NPF ? g : 0]
                  : dot ? make_float4(0.f, 0.f, 0.f, 0.f)
                        : *(const float4 *)(a.bn + b4);
      float4 w4 = wts ? *(const float4 *)(wts + b4) : make_float4(1.f, 1.f, 1.f, 1.f);
      nn[4 * g] = n4.x; nn[4 * g + 1] = n4.y; nn[4 * g + 2] = n4.z; nn[4 * g + 3] = n4.w;
      ww[4 * g] = w4.x; ww[4 * g + 1] = w4.y; ww[4 * g + 2] = w4.z; ww[4 * g + 3] = w4.w;
    }
#pragma unroll
    for (int j = 0; j < NB; j++) {
      if constexpr (MODE == 0 || MODE == 1) {
        // full blocks of unweighted searches (the last, partial block of a
        // range and weighted searches take the general path below)
        if (!wts && bb + 32 <= bend) {
          const bool test = bb - bbeg >= 48L * a.bstep;
          if (dot)
            yk_best1_block<true>(acc[j], nrm, qnd[j], bb, h, test, bv[j], bi[j]);
          else
            yk_best1_block<false>(acc[j], nrm, qnd[j], bb, h, test, bv[j], bi[j]);
          continue;
        }
      }
      // Prefilter on float approximations qn + (bn - 2 acc), which differ
      // from the exact expression by far less than 2^-19 (|q|^2 + max|b|^2)
      // (|2 q.b| <= |q|^2 + |b|^2): a min over the lane's 16 values, then a
      // per-value test; only values that may matter take the exact
      // FP64-normed expression.  Weighted searches evaluate every value.
      float nmax = 0.f;
#pragma unroll
      for (int i = 0; i < 16; i++) nmax = fmaxf(nmax, nn[i]);
      const float qf = (float)qnd[j];
      const float slack = dot ? 0.f : 0x1p-19f * (qf + nmax);
      float ap[16];
#pragma unroll
      for (int i = 0; i < 16; i++)
        ap[i] = dot ? acc[j][i] : qf + __builtin_fmaf(-2.0f, acc[j][i], nn[i]);
      const float lim = MODE == 3 ? Tv[j] : (MODE == 2 ? INFINITY : bv[j]);
      if (!wts && MODE != 2) {
        float m = ap[0];
#pragma unroll
        for (int i = 1; i < 16; i++) m = fminf(m, ap[i]);
        if (!(m - slack <= lim) && m == m) continue;
      }
#pragma unroll
      for (int i = 0; i < 16; i++) {
        if (!wts && MODE != 2 && !(ap[i] - slack <= (MODE == 3 ? Tv[j] : bv[j])) && ap[i] == ap[i])
          continue;
        const long bidx = bb + 8 * (i >> 2) + 4 * h + (i & 3);
        const bool bok = bidx < bend;
        float v = dot ? acc[j][i] : (float)(qnd[j] + (double)nn[i]) - 2.0f * acc[j][i];
        if (wts) v *= ww[i];
        if (MODE == 0 || MODE == 1) {
          if (bok && v < bv[j]) {  // strict '<' in ascending index order
            bv[j] = v;
            bi[j] = (int)bidx;
          }
        } else if (MODE == 2) {
          uint64_t key = (bok && v == v) ? yk_key(v, (int)bidx) : YK_KEY_NONE;
          if (key < top[j][R - 1]) yk_reg_insert<R>(top[j], key);
        } else if (bok && qok[j] && v == v) {
          uint64_t key = yk_key(v, (int)bidx);
          if (key <= T[j]) {
            const int n = ncs[j];
            cs[(j * 64 + lane) * YK_CSTAGE + n] = key;
            if (n + 1 == YK_CSTAGE) {
              flush(j, YK_CSTAGE);
              ncs[j] = 0;
            } else {
              ncs[j] = n + 1;
            }
          }
        }
      }
    }
    // the next block's norms (unconditional, as the operands' prefetch)
    if constexpr (NPF) loadn(bb + a.bstep < bend ? bb + a.bstep : bb);
  }

  if (MODE == 0) {
#pragma unroll
    for (int j = 0; j < NB; j++) {
      float ov = __shfl_xor(bv[j], 32);
      int oi = __shfl_xor(bi[j], 32);
      if (ov < bv[j] || (ov == bv[j] && oi < bi[j])) {
        bv[j] = ov;
        bi[j] = oi;
      }
      const long qi = qbase + j * 32 + r;
      if (h == 0 && qok[j]) {
        if (a.nsplit == 1) {
          a.out_d[qi] = bv[j];
          a.out_i[qi] = bi[j];
        } else {
          a.part[qi * a.nsplit + split] = bi[j] < 0 ? YK_KEY_NONE : yk_key(bv[j], bi[j]);
        }
      }
    }
  } else if (MODE == 1) {
    // sketch: each lane's own minimum (distinct rows per lane -> distinct keys)
#pragma unroll
    for (int j = 0; j < NB; j++) {
      const long qi = qbase + j * 32 + r;
      if (qok[j])
        a.part[(qi * a.nsplit + split) * 2 + h] = bi[j] < 0 ? YK_KEY_NONE : yk_key(bv[j], bi[j]);
    }
  } else if (MODE == 2) {
#pragma unroll
    for (int j = 0; j < NB; j++) {
      const long qi = qbase + j * 32 + r;
      if (!qok[j]) continue;
      uint64_t *dst = a.part + ((qi * a.nsplit + split) * 2 + h) * R;
#pragma unroll
      for (int s = 0; s < R; s++) dst[s] = top[j][s];
    }
  } else {
#pragma unroll
    for (int j = 0; j < NB; j++)
      if (ncs[j] > 0) flush(j, ncs[j]);
  }
  }  // work items
}

// ---------------------------------------------------------------------------
// LDS-staged scan: k = 1, the sketch and the filtered pass for more than 64
// queries and d <= 256.
//
// The streaming kernel above loads every base fragment once per wave, 16
// bytes from each of 32 rows per instruction: the vector L1 takes those rows
// one line at a time and bounded it at 55-60% of the FP32 MFMA rate (d = 128;
// n = 1e5 points to 1,024 centroids 0.290 ms, 90 TFLOP/s).  Here the
// workgroup's four waves share each block: a 32-row block is one contiguous
// piece of memory, loaded 1 KB per wave instruction straight into the other
// of two LDS buffers while a stage is multiplied (no registers hold it).  The
// four 16-byte units of a row's chunk are stored in the order unit ^ (row & 3),
// which spreads the rows' reads over four times the banks and leaves the chunk
// a constant offset of the read's address.  One barrier per stage; short vectors stage G
// blocks at once so that a stage is at least 64 MFMAs.  Two query tiles per
// wave (NB = 2) would use each fragment read from LDS twice, but at d = 128
// their 128 registers of queries leave two waves per SIMD and spills, and 256
// queries a workgroup fewer of them: 1e5 queries x 1,024 0.260 against 0.236 ms,
// 20,000 x 16,384, k = 100 2.00 and 1.84, 300 x 1e6 1.27 and 1.00 (1.17
// streamed).  Only k = 1 at d <= 16 keeps them, from 65,536 queries on (3e5 x
// 1,024 0.144 and 0.150).  Same MFMA operands, same order, same epilogue
// arithmetic as the streaming kernel: the same bits.  n = 1e5 points to 1,024
// centroids: 0.290 -> 0.222 ms (118 TFLOP/s of the 153 of a large library
// product; 1e4 queries x 1e6, k = 100: 124).  What is left is the epilogue's
// vector instructions, which do not overlap with the MFMAs, and at n = 1e5 the
// start (every workgroup's queries at once).
template <int NCH>
struct YkLdsShape {
  static constexpr int U = 4 * NCH;  // float4 units of a row
  static constexpr int G = NCH == 1 ? 8 : NCH == 2 ? 4 : NCH <= 4 ? 2 : 1;  // blocks per stage
  static constexpr int KL = G * 32 * U / 64;  // 1 KB wave loads of a stage
  static constexpr int NL = (KL + 3) / 4;     // of them per wave
  // MODE 3: keys staged per lane; fewer where two workgroups
  // would not fit a CU's LDS otherwise
  static constexpr int CST = NCH > 8 ? 4 : 8;
};

// the first of the W even shares of T units that covers unit u; shares are
// [w T / W, (w + 1) T / W)
__device__ __forceinline__ long yk_share_of(long u, long T, long W) {
  long w = u * W / T;
  while ((w + 1) * T / W <= u) w++;
  while (w * T / W > u) w--;
  return w;
}

// 16 bytes per lane from rs at voff straight to LDS at dst + 16 lane (dst
// uniform over the wave; complete when vmcnt says so)
__device__ __forceinline__ void yk_load_lds16(__amdgpu_buffer_rsrc_t rs, float4 *dst, int voff) {
#ifdef __HIP_DEVICE_COMPILE__  // (the host pass does not know the 16-byte form)
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (__attribute__((address_space(3))) void *)dst, 16,
                                           voff, 0, 0, 0);
#endif
}

template <int NB, int NCH, int MODE, bool WT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void
yk_scan_f32_lds(ScanArgs a0) {
  using S = YkLdsShape<NCH>;
  constexpr int U = S::U, G = S::G, KL = S::KL, NL = S::NL, CST = S::CST;
  constexpr int ld = 16 * NCH, TQ = 128 * NB;
  constexpr bool BEST1 = MODE != 3 && !WT;  // yk_best1_block
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 31, h = lane >> 5;
  // (the tiles first: the LDS offset of a direct load is 16 bits wide)
  struct Shared {
    float4 tile[2][G * 32 * U];
    float norm[2][G * 32];
    double normd[2][BEST1 ? G * 32 : 1];
    float wt[2][WT ? G * 32 : 1];
    uint64_t cstage[MODE == 3 ? 4 * NB * 64 * CST : 1];
    int item;
  };
  __shared__ Shared sm;
  uint64_t *const cs = sm.cstage + (MODE == 3 ? wave * NB * 64 * CST : 0);
  const bool dot = a0.type == YK_DOT;

  // Work: split items with per-XCD tickets, as above; or, MODE 0 over a base
  // that stays in the L2 (a0.units blocks), an even share of the tiles x
  // units (tile, block) pairs per workgroup: a share that covers a tile only
  // in part leaves its minima in part[(share, head or tail), query] for
  // yk_merge_share_kernel.
  const int xcd = blockIdx.x & 7, local = blockIdx.x >> 3, wpx = gridDim.x >> 3;
  const int ibeg = xcd * a0.per_xcd, iend = min(a0.total, ibeg + a0.per_xcd);
  const long T_units = (long)a0.tiles_x * a0.units;
  long cur = a0.units ? blockIdx.x * T_units / gridDim.x : 0;
  const long cend = a0.units ? (blockIdx.x + 1L) * T_units / gridDim.x : 0;
  auto next_item = [&](int it) {
    if (!a0.tick) return it + wpx;
    __syncthreads();
    if (tid == 0) sm.item = ibeg + wpx + atomicAdd(&a0.tick[xcd], 1);
    __syncthreads();
    return sm.item;
  };
  for (int item = ibeg + local; a0.units ? cur < cend : item < iend;
       item = a0.units ? 0 : next_item(item)) {
    ScanArgs a = a0;
    int tile, split = 0, slot = -1;
    long bbeg, bend, bstep = a0.bstep;
    if (a0.units) {
      tile = (int)(cur / a0.units);
      const long b0 = cur - (long)tile * a0.units;
      const long b1 = min((long)a0.units, b0 + (cend - cur));
      cur += b1 - b0;
      slot = b0 > 0 ? 0 : (b1 < a0.units ? 1 : -1);
      bbeg = 32 * b0;
      bend = min(a.nb, 32 * b1);
    } else if (MODE == 0 && NB == 1 && a0.item_inst) {
      const int inst = a0.item_inst[item];
      if (inst < 0 || (a0.done && a0.done[inst])) continue;
      tile = a0.item_tile[item];
      const long off = a0.inst_off[inst];
      if (a0.qidx) {
        a.qidx = a0.qidx + off;
      } else {
        a.q = a0.q + off * ld;
        a.qn = a0.qn + off;
      }
      a.nq = a0.inst_off[inst + 1] - off;
      a.b = a0.b + (long)inst * a0.kpad * ld;
      a.bn = a0.bn + (long)inst * a0.kpad;
      a.nb = a0.kc;
      a.out_i = a0.out_i + off;
      a.out_d = a0.out_d + off;
      bbeg = 0;
      bend = a.nb;
    } else {
      tile = item % a0.tiles_x;
      split = item / a0.tiles_x;
      if (MODE == 1 && a0.inter) {
        bbeg = (long)split * a0.bstep;
        bend = a.nb;
        bstep = a0.bstep * a0.nsplit;
      } else {
        bbeg = (long)split * a0.brange;
        bend = min(a.nb, bbeg + a0.brange);
      }
    }
    const long qbase = ((long)tile * 4 + wave) * (32 * NB);
    const bool live = qbase < a.nq;  // the wave's queries exist (uniform)

    int qrow[NB];
    long qsrc[NB];
    bool qok[NB];
    double qnd[NB];
    float bv[NB], Tv[NB];
    int bi[NB], ncs[NB];
    bool act = false;
#pragma unroll
    for (int j = 0; j < NB; j++) {
      const long qi = qbase + j * 32 + r;
      qok[j] = qi < a.nq;
      qrow[j] = (int)(qok[j] ? qi : a.nq - 1);
      qsrc[j] = MODE == 0 && NB == 1 && a.qidx ? (long)a.qidx[qrow[j]] : qrow[j];
      qnd[j] = dot ? 0.0 : a.qn[qsrc[j]];
      bv[j] = 1e30f;
      bi[j] = -1;
      ncs[j] = 0;
      // MODE 3: the bound's value (its row is looked up where a value equals
      // it); a query that is already final (T = 0), or past the last one, has
      // -inf here, which a bound's value may be too: a value equal to it
      // enters by its whole key only (no key is <= 0)
      const uint64_t T = MODE == 3 ? a.thr[qrow[j]] : 0;
      Tv[j] = T == 0 || !qok[j] ? -INFINITY
                                : (T == YK_KEY_NONE ? INFINITY : yk_fkey_inv((uint32_t)(T >> 32)));
      act |= qok[j] && T != 0;
    }
    if (MODE == 3 && !__syncthreads_or(act)) continue;  // every query of the tile is final
    float4 qreg[NB][2 * NCH];
    if (live) {
#pragma unroll
      for (int j = 0; j < NB; j++)
#pragma unroll
        for (int c = 0; c < NCH; c++) {
          const float *p = a.q + qsrc[j] * ld + c * 16 + h * 8;
          qreg[j][2 * c] = *(const float4 *)p;
          qreg[j][2 * c + 1] = *(const float4 *)(p + 4);
        }
    }
    auto flush = [&](int j, int n) {
      const int base = atomicAdd(&a.cnt[qrow[j]], n);
      const uint64_t *src = cs + (j * 64 + lane) * CST;
      for (int s_ = 0; s_ < n; s_++)
        if (base + s_ < a.cap) a.cand[(long)qrow[j] * a.cap + base + s_] = src[s_];
    };

    // wave load i of a stage: lane l stores unit 64 (4 i + wave) + l of the
    // stage's LDS image, (row, place) = (unit / U, unit % U)
    int voff[NL];
#pragma unroll
    for (int i = 0; i < NL; i++) {
      const int unit = 64 * (4 * i + wave) + lane, g = unit / (32 * U);
      const int row = unit / U % 32, u = unit % U ^ (row & 3);
      voff[i] = (int)((g * bstep * ld + row * ld + u * 4) * 4);
    }
    const int nst = (int)(((bend - bbeg + bstep - 1) / bstep + G - 1) / G);
    const long nb32 = (a.nb + 31) & ~31L;
    float ld_n = 0.f, ld_w = 0.f;
    auto load = [&](int st, int buf) {
      const long row = bbeg + (long)st * G * bstep;  // the stage's first row, below bend
      // (rows past the base read as zeros; their values are masked)
      const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
          (void *)(a.b + row * ld), 0, (int)min((a.nb - row) * ld * 4, 0x7fffffffL),
          YK_BUF_DWORD3);
#pragma unroll
      for (int i = 0; i < NL; i++)
        if (KL % 4 == 0 || 4 * i + wave < KL)
          yk_load_lds16(rs, sm.tile[buf] + 64 * (4 * i + wave), voff[i]);
      if (tid < 32 * G) {
        const long nr = row + (tid >> 5) * bstep + (tid & 31);
        if (!dot) ld_n = nr < (BEST1 ? a.nb : nb32) ? a.bn[nr] : BEST1 ? YK_FAR_NORM : 0.f;
        if (WT) ld_w = nr < nb32 ? a.w[nr] : 0.f;
      }
    };
    // the stage's norms, and the wait for its direct loads
    auto store = [&](int buf) {
      if (tid < 32 * G) {
        sm.norm[buf][tid] = ld_n;
        if (BEST1) sm.normd[buf][tid] = (double)ld_n;
        if (WT) sm.wt[buf][tid] = ld_w;
      }
      __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
    };

    auto block = [&](const float4 *tp, const float *np, const double *npd, const float *wp,
                     long bb, bool test) {
      f32x16 acc[NB];
#pragma unroll
      for (int j = 0; j < NB; j++)
#pragma unroll
        for (int e = 0; e < 16; e++) acc[j][e] = 0.f;
      // row r's units 2 h and 2 h + 1 of chunk c sit at 4 c + (unit ^ (r & 3))
      const float4 *tp0 = tp + ((2 * h) ^ (r & 3)), *tp1 = tp + ((2 * h + 1) ^ (r & 3));
      float4 av[2][2];
      av[0][0] = tp0[0];
      av[0][1] = tp1[0];
#pragma unroll
      for (int c = 0; c < NCH; c++) {
        if (c + 1 < NCH) {
          av[(c + 1) & 1][0] = tp0[4 * c + 4];
          av[(c + 1) & 1][1] = tp1[4 * c + 4];
        }
        const float4 x0 = av[c & 1][0], x1 = av[c & 1][1];
        const float xs[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
#pragma unroll
        for (int t = 0; t < 8; t++)
#pragma unroll
          for (int j = 0; j < NB; j++) {
            const float4 y = qreg[j][2 * c + (t >> 2)];
            const float ys = (t & 3) == 0 ? y.x : (t & 3) == 1 ? y.y : (t & 3) == 2 ? y.z : y.w;
            acc[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(xs[t], ys, acc[j], 0, 0, 0);
          }
        __builtin_amdgcn_sched_barrier(0);
      }
      const YkNormLds nn = {np, npd};
#pragma unroll
      for (int j = 0; j < NB; j++) {
        if constexpr (MODE != 3) {
          if (!WT && !dot) {
            yk_best1_block<false>(acc[j], nn, qnd[j], bb, h, test, bv[j], bi[j]);
            continue;
          }
          if (!WT && bb + 32 <= bend) {
            yk_best1_block<true>(acc[j], nn, qnd[j], bb, h, test, bv[j], bi[j]);
            continue;
          }
        }
        // Only a lane with a value that may enter goes on; one such value
        // is taken by itself, several by the loop over all 16.  Weighted
        // values are w times the approximations, so within |w| slack of the
        // exact ones (and 1e-36 covers products that round in the denormal
        // range).  Negated comparisons: a NaN goes on to the exact test.
        const float lim = MODE == 3 ? Tv[j] : bv[j];
        const float qf = (float)qnd[j];
        const float slack = dot ? 0.f : 0x1p-19f * (qf + yk_max16(nn));
        const long b0 = bb + 4 * h;
        auto enter = [&](float v, int i) {  // the exact value i of the lane
          const long bidx = b0 + 8 * (i >> 2) + (i & 3);
          if (MODE != 3) {
            if (bidx < bend && v < bv[j]) {  // strict '<' in ascending index order
              bv[j] = v;
              bi[j] = (int)bidx;
            }
          } else if (bidx < bend && v <= Tv[j]) {  // (drops NaN)
            const uint64_t key = yk_key(v, (int)bidx);
            if (v < Tv[j] || (qok[j] && key <= a.thr[qrow[j]])) {
              const int n = ncs[j];
              cs[(j * 64 + lane) * CST + n] = key;
              if (n + 1 == CST) {
                flush(j, CST);
                ncs[j] = 0;
              } else {
                ncs[j] = n + 1;
              }
            }
          }
        };
        auto exact = [&](float ac, float nm) {
          return dot ? ac : (float)(qnd[j] + (double)nm) - 2.0f * ac;
        };
        if constexpr (!WT) {
          float m[16];
          const float mm = dot ? yk_approx16<true>(acc[j], nn, m) : yk_approx16<false>(acc[j], nn, m);
          if (qf + mm - slack > lim || mm == INFINITY) {
            if (lim < INFINITY) continue;
          }
          // m_i <= th for every value that may enter: qf + m_i - slack <=
          // lim, with twice the slack for the roundings of this line (an
          // infinite lim: no such line, every value is tested)
          int is;
          float as;
          const int cnt = yk_pick16(acc[j], m, dot ? lim : lim - qf + 2.0f * slack, is, as);
          if (cnt == 1) {
            enter(exact(as, nn.pick(is)), is);
          } else if (cnt > 1 || !(fabsf(lim) < INFINITY)) {
#pragma unroll
            for (int i = 0; i < 16; i++) enter(exact(acc[j][i], nn[i]), i);
          }
        } else {
          // (the value's weighted approximation less its error, against the
          // bound: a lane's one such value by itself, several by the loop)
          const float limw = lim + 1e-36f;
          const YkNormLds ww = {wp, nullptr};
          int cnt = 0, is = 0;
          float as = acc[j][0];
#pragma unroll
          for (int i = 0; i < 16; i++) {
            const float ap = dot ? acc[j][i] : qf + __builtin_fmaf(-2.0f, acc[j][i], nn[i]);
            const bool c = !(ap * ww[i] - slack * fabsf(ww[i]) > limw);
            cnt += c ? 1 : 0;
            is = c ? i : is;
            as = c ? acc[j][i] : as;
          }
          if (cnt == 1) {
            enter(exact(as, nn.pick(is)) * ww.pick(is), is);
          } else if (cnt > 1) {
#pragma unroll
            for (int i = 0; i < 16; i++) enter(exact(acc[j][i], nn[i]) * ww[i], i);
          }
        }
      }
    };

    load(0, 0);
    store(0);
    __syncthreads();
    for (int st = 0; st < nst; st++) {
      const int buf = st & 1;
      if (st + 1 < nst) load(st + 1, buf ^ 1);
      if (live) {
#pragma unroll 1
        for (int g = 0; g < G; g++) {
          const long bb = bbeg + ((long)st * G + g) * bstep;
          if (bb >= bend) break;
          block(sm.tile[buf] + (g * 32 + r) * U, sm.norm[buf] + g * 32 + 4 * h,
                sm.normd[buf] + (BEST1 ? g * 32 + 4 * h : 0),
                sm.wt[buf] + (WT ? g * 32 + 4 * h : 0), bb, st * G + g >= 48);
        }
      }
      if (st + 1 < nst) store(buf ^ 1);
      __syncthreads();
    }

    if (MODE == 0) {
#pragma unroll
      for (int j = 0; j < NB; j++) {
        const float ov = __shfl_xor(bv[j], 32);
        const int oi = __shfl_xor(bi[j], 32);
        if (ov < bv[j] || (ov == bv[j] && oi < bi[j])) {
          bv[j] = ov;
          bi[j] = oi;
        }
        const long qi = qbase + j * 32 + r;
        if (h == 0 && qok[j]) {
          const uint64_t key = bi[j] < 0 ? YK_KEY_NONE : yk_key(bv[j], bi[j]);
          if (slot >= 0) {
            a.part[(blockIdx.x * 2L + slot) * TQ + wave * 32 * NB + j * 32 + r] = key;
          } else if (a.nsplit > 1) {
            a.part[qi * a.nsplit + split] = key;
          } else {
            a.out_d[qi] = bv[j];
            a.out_i[qi] = bi[j];
          }
        }
      }
    } else if (MODE == 1) {
#pragma unroll
      for (int j = 0; j < NB; j++) {
        const long qi = qbase + j * 32 + r;
        if (qok[j])
          a.part[(qi * a.nsplit + split) * 2 + h] = bi[j] < 0 ? YK_KEY_NONE : yk_key(bv[j], bi[j]);
      }
    } else {
#pragma unroll
      for (int j = 0; j < NB; j++)
        if (ncs[j] > 0) flush(j, ncs[j]);
    }
  }  // work
}

// k = 1 over even shares (yk_scan_f32_lds with units): the queries of tiles
// cut by a share's end, from the shares' minima (at most W + 1 of the tiles
// are cut; the others were written by the scan).  A thread per query, or where
// a tile has many shares (few queries) a wave, its lanes striding them: 70
// queries x 16,000 vectors, d = 16, 500 shares: the search 0.23 -> 0.024 ms.
template <bool WAVE>
__global__ __launch_bounds__(256) void yk_merge_share_kernel(const uint64_t *__restrict__ part,
                                                             long nq, int tq, long units, long T,
                                                             long W, int *out_i, float *out_d) {
  const long q = WAVE ? blockIdx.x * 4L + (threadIdx.x >> 6) : blockIdx.x * 256L + threadIdx.x;
  const int lane = WAVE ? threadIdx.x & 63 : 0;
  if (q >= nq) return;
  const long tile = q / tq, lo = tile * units, hi = lo + units;
  const long w0 = yk_share_of(lo, T, W);
  if ((w0 + 1) * T / W >= hi) return;  // one share covers the tile
  uint64_t best = YK_KEY_NONE;
  for (long w = w0 + lane; w < W; w += WAVE ? 64 : 1) {
    const long s = w * T / W;
    if (s >= hi) break;
    if ((w + 1) * T / W == s) continue;  // an empty share
    const uint64_t v = part[(w * 2 + (s > lo ? 0 : 1)) * tq + q % tq];
    best = v < best ? v : best;
  }
  if (WAVE) best = yk_wave_min64(best);
  if (lane > 0) return;
  out_i[q] = best == YK_KEY_NONE ? -1 : (int)(uint32_t)best;
  out_d[q] = best == YK_KEY_NONE ? 1e30f : yk_fkey_inv((uint32_t)(best >> 32));
}

// ---------------------------------------------------------------------------
// small per-query sorts

__device__ __forceinline__ void yk_store_key(uint64_t key, int *oi, float *od) {
  *oi = key == YK_KEY_NONE ? -1 : (int)(uint32_t)key;
  *od = key == YK_KEY_NONE ? __uint_as_float(0xffffffffu) : yk_fkey_inv((uint32_t)(key >> 32));
}

// k = 1 merge of per-split minima (nothing below 1e30 -> (-1, 1e30)): one
// wave per query, its lanes striding the splits (a thread per query walked
// them one by one)
__global__ __launch_bounds__(256) void yk_merge1_kernel(const uint64_t *__restrict__ part, long nq,
                                                        int nsplit, int *out_i, float *out_d) {
  const long q = blockIdx.x * 4L + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (q >= nq) return;
  uint64_t best = YK_KEY_NONE;
  for (int s = lane; s < nsplit; s += 64) {
    const uint64_t v = part[q * nsplit + s];
    best = v < best ? v : best;
  }
  best = yk_wave_min64(best);
  if (lane == 0) {
    out_i[q] = best == YK_KEY_NONE ? -1 : (int)(uint32_t)best;
    out_d[q] = best == YK_KEY_NONE ? 1e30f : yk_fkey_inv((uint32_t)(best >> 32));
  }
}

// ascending bitonic sort of s[0..p2) by the block (p2 a power of two)
__device__ void yk_block_bitonic(uint64_t *s, int p2) {
  for (int size = 2; size <= p2; size <<= 1) {
    for (int stride = size >> 1; stride > 0; stride >>= 1) {
      for (int t = threadIdx.x; t < p2 / 2; t += blockDim.x) {
        int lo = 2 * t - (t & (stride - 1));
        int hi = lo + stride;
        bool up = (lo & size) == 0;
        uint64_t x = s[lo], y = s[hi];
        if ((x > y) == up) {
          s[lo] = y;
          s[hi] = x;
        }
      }
      __syncthreads();
    }
  }
}

// The k smallest of each query's n keys (src + q*n), sorted: the end of the
// register top-R scan, for every query or (with flag and thr) those that the
// filtered pass left (*flag != 0, thr[q] != 0).
__global__ __launch_bounds__(256) void yk_sortsel_kernel(const uint64_t *__restrict__ src,
                                                         int n, int k, int p2, int *out_i,
                                                         float *out_d,
                                                         const uint64_t *__restrict__ thr,
                                                         const int *__restrict__ flag) {
  extern __shared__ uint64_t s[];
  if (flag && *flag == 0) return;
  const long q = blockIdx.x;
  if (thr && thr[q] == 0) return;
  const uint64_t *p = src + q * (long)n;
  for (int i = threadIdx.x; i < p2; i += blockDim.x) s[i] = i < n ? p[i] : YK_KEY_NONE;
  __syncthreads();
  yk_block_bitonic(s, p2);
  for (int i = threadIdx.x; i < k; i += blockDim.x)
    yk_store_key(i < p2 ? s[i] : YK_KEY_NONE, out_i + q * k + i, out_d + q * k + i);
}

// The filtered pass's starting bounds, one wave per query: the m-th smallest
// of the query's n <= 4096 sketch minima (YK_KEY_NONE, admit all, when fewer
// than need of them are real keys); the query's candidate count and the
// flag start at zero.
__global__ __launch_bounds__(256) void yk_thr_kernel(const uint64_t *__restrict__ src, long nq,
                                                     int n, int m, int need,
                                                     uint64_t *__restrict__ thr,
                                                     int *__restrict__ cnt, int *flag) {
  const long q = blockIdx.x * 4L + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (q == 0 && lane == 0) *flag = 0;
  if (q >= nq) return;
  const uint64_t *p = src + q * (long)n;
  uint64_t t = YK_KEY_NONE;
  auto kth = [&](auto e) {
    constexpr int E = decltype(e)::value;
    uint64_t v[E];
    yk_wave_load<E>(p, n, lane, v);
    int nreal = 0;
#pragma unroll
    for (int i = 0; i < E; i++) nreal += __popcll(__builtin_amdgcn_ballot_w64(v[i] != YK_KEY_NONE));
    if (nreal >= need) t = yk_wave_kth<E>(v, m, false);
  };
  if (n >= need) {
    if (n <= 256)
      kth(std::integral_constant<int, 4>());
    else if (n <= 512)
      kth(std::integral_constant<int, 8>());
    else if (n <= 1024)
      kth(std::integral_constant<int, 16>());
    else if (n <= 2048)
      kth(std::integral_constant<int, 32>());
    else
      kth(std::integral_constant<int, 64>());
  }
  if (lane == 0) {
    thr[q] = t;
    cnt[q] = 0;
  }
}

template <int E, int E2>
__device__ __forceinline__ void yk_cand_topk(const uint64_t *p, int m, int n, int k, int lane,
                                             uint64_t *lds, int *oi, float *od, uint64_t *thr,
                                             int *cnt, int *flag) {
  uint64_t v[E];
  yk_wave_load<E>(p, m, lane, v);
  if (n > m) {  // the list overflowed
    const uint64_t x = yk_wave_kth<E>(v, k, false);
    if (lane == 0) {
      *thr = x;
      *cnt = 0;
      atomicOr(flag, 1);
    }
    return;
  }
  uint64_t w[E2];
  yk_wave_topk_reg<E, E2>(v, k, lane, lds, w);
#pragma unroll
  for (int i = 0; i < E2; i++) {
    const int e = lane * E2 + i;
    if (e < k) yk_store_key(w[i], oi + e, od + e);
  }
  if (lane == 0) *thr = 0;
}

// After a MODE 3 pass, one wave per query (k <= 64 E2): queries whose list
// fitted get their k smallest and become inactive (thr = 0); overflowing
// queries get the k-th smallest captured key as a tighter threshold, their
// count is reset, *flag is set.  A query with fewer than k keys under a bound
// (the estimated starting bound, or with NaN distances, which no bound
// admits, any bound) gets no bound, its count reset and the flag: its next
// pass admits every value (and overflows, the overflow's bound then being a
// proven one); a query with fewer than k keys and no bound has no more to
// find.  `last`: no scan follows, so every query's outputs are written here
// (the caller knows that no list overflows, and that the bound admits k keys).
// (The keys are held in registers and the k-th found by ballot
// counts, as in the precision form: 1e4 lists of ~700 keys, k = 100, 0.049
// -> 0.012 ms against a workgroup's bitonic sort per query.)
template <int E2>
__global__ __launch_bounds__(256) void yk_select_kernel(const uint64_t *__restrict__ cand, int cap,
                                                        long nq, int *cnt, uint64_t *thr, int k,
                                                        int *out_i, float *out_d, int *flag,
                                                        int last) {
  __shared__ uint64_t lds[4][64 * E2];
  const long q = blockIdx.x * 4L + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (q >= nq || thr[q] == 0) return;
  const int n = cnt[q];
  if (!last && n < k && thr[q] != YK_KEY_NONE) {
    if (lane == 0) {
      thr[q] = YK_KEY_NONE;
      cnt[q] = 0;
      atomicOr(flag, 1);
    }
    return;
  }
  const int m = n < cap ? n : cap;
  const uint64_t *p = cand + q * (long)cap;
  int *oi = out_i + q * k;
  float *od = out_d + q * k;
  if (m <= 256)
    yk_cand_topk<4, E2>(p, m, n, k, lane, lds[wave], oi, od, thr + q, cnt + q, flag);
  else if (m <= 512)
    yk_cand_topk<8, E2>(p, m, n, k, lane, lds[wave], oi, od, thr + q, cnt + q, flag);
  else if (m <= 1024)
    yk_cand_topk<16, E2>(p, m, n, k, lane, lds[wave], oi, od, thr + q, cnt + q, flag);
  else if (m <= 2048)
    yk_cand_topk<32, E2>(p, m, n, k, lane, lds[wave], oi, od, thr + q, cnt + q, flag);
  else
    yk_cand_topk<64, E2>(p, m, n, k, lane, lds[wave], oi, od, thr + q, cnt + q, flag);
}

__global__ void yk_zero_cnt_kernel(int *cnt, long n) {
  long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
  if (i < n) cnt[i] = 0;
}

// ---------------------------------------------------------------------------
// planning and launch

// Which scan a search takes.  Up to 64 queries a pass over the base is bound
// by its bytes, and a wave streams rows straight to registers (YK_STREAM; one
// or two waves per workgroup, so that every wave has queries of its own);
// beyond that the workgroup shares the base through LDS (YK_LDS1: 32 queries
// per wave, YK_LDS2: 64, k = 1 of many short queries).  d > 256 streams both operands.
enum { YK_STREAM = 0, YK_LDS1 = 1, YK_LDS2 = 2 };
#define YK_STREAM_NQ 64

struct YkPlan {
  int kind;
  int waves;   // waves per workgroup
  int tiles;   // query tiles
  int nsplit;  // base splits
  long brange;
  long bstep;
  int inter;   // sketch: interleaved splits
  int slots;   // workgroups resident at once
  int units;   // k = 1: even shares of tiles x units blocks over `slots` workgroups
};

// Launch-plan knobs the autotuner chooses among (every choice gives the
// same bits): the number of work items the base split aims at, and a
// scale of the k > 16 sketch's sampling stride.  cfg = target index + 3 x
// stride index; 0 is the default plan.
static const long yk_item_targets[3] = {4096, 2048, 8192};
static const int yk_stride_scale[4][2] = {{1, 1}, {1, 2}, {2, 1}, {16, 3}};  // num., denom.
#define YK_NCFG 12

typedef void (*YkScanKernel)(ScanArgs);

// the streaming kernel with exactly ld/16 register-resident chunks (ld <=
// 128), else the one streaming both operands
template <int MODE, int R>
static YkScanKernel yk_stream_pick(int ld, bool weighted) {
  if (weighted && ld <= 32) return yk_scan_f32<1, 0, MODE, R>;  // no weights in NCH <= 2
  switch (ld >> 4) {
    case 1: return yk_scan_f32<1, 1, MODE, R>;
    case 2: return yk_scan_f32<1, 2, MODE, R>;
    case 3: return yk_scan_f32<1, 3, MODE, R>;
    case 4: return yk_scan_f32<1, 4, MODE, R>;
    case 5: return yk_scan_f32<1, 5, MODE, R>;
    case 6: return yk_scan_f32<1, 6, MODE, R>;
    case 7: return yk_scan_f32<1, 7, MODE, R>;
    case 8: return yk_scan_f32<1, 8, MODE, R>;
    default: return yk_scan_f32<1, 0, MODE, R>;
  }
}

template <int MODE, bool WT>
static YkScanKernel yk_lds_pick(int ld) {
  switch (ld >> 4) {
    case 1: return yk_scan_f32_lds<1, 1, MODE, WT>;
    case 2: return yk_scan_f32_lds<1, 2, MODE, WT>;
    case 3: return yk_scan_f32_lds<1, 3, MODE, WT>;
    case 4: return yk_scan_f32_lds<1, 4, MODE, WT>;
    case 5: return yk_scan_f32_lds<1, 5, MODE, WT>;
    case 6: return yk_scan_f32_lds<1, 6, MODE, WT>;
    case 7: return yk_scan_f32_lds<1, 7, MODE, WT>;
    case 8: return yk_scan_f32_lds<1, 8, MODE, WT>;
    case 9: return yk_scan_f32_lds<1, 9, MODE, WT>;
    case 10: return yk_scan_f32_lds<1, 10, MODE, WT>;
    case 11: return yk_scan_f32_lds<1, 11, MODE, WT>;
    case 12: return yk_scan_f32_lds<1, 12, MODE, WT>;
    case 13: return yk_scan_f32_lds<1, 13, MODE, WT>;
    case 14: return yk_scan_f32_lds<1, 14, MODE, WT>;
    case 15: return yk_scan_f32_lds<1, 15, MODE, WT>;
    default: return yk_scan_f32_lds<1, 16, MODE, WT>;
  }
}

static YkScanKernel yk_scan_pick(int mode, int kind, int ld, bool weighted) {
  if (kind == YK_LDS2) return yk_scan_f32_lds<2, 1, 0, false>;
  if (kind == YK_LDS1 && weighted)
    return mode == 0   ? yk_lds_pick<0, true>(ld)
           : mode == 1 ? yk_lds_pick<1, true>(ld)
                       : yk_lds_pick<3, true>(ld);
  if (kind == YK_LDS1)
    return mode == 0   ? yk_lds_pick<0, false>(ld)
           : mode == 1 ? yk_lds_pick<1, false>(ld)
                       : yk_lds_pick<3, false>(ld);
  return mode == 0   ? yk_stream_pick<0, 1>(ld, weighted)
         : mode == 1 ? yk_stream_pick<1, 1>(ld, weighted)
         : mode == 2 ? yk_stream_pick<2, YK_REG_R>(ld, weighted)
                     : yk_stream_pick<3, 1>(ld, weighted);
}

// blocks a stage of the LDS-staged kernel holds (YkLdsShape::G)
static long yk_lds_stage_blocks(int ld) { return ld <= 16 ? 8 : ld <= 32 ? 4 : ld <= 64 ? 2 : 1; }

// The plan of one scan: mode 0 (k = 1), 1 (the sketch, one block in `sample`),
// 2 (register top-R) or 3 (filtered).
static YkPlan yk_plan(int mode, long nq, long nb, int ld, bool weighted, long sample,
                      long min_splits, long max_split, long min_blocks, int cfg) {
  YkPlan p = {};
  p.bstep = 32 * sample;
  const long nblocks = (nb + p.bstep - 1) / p.bstep;  // processed blocks
  p.kind = YK_STREAM;
  p.waves = 4;
  // (a sketch or filtered scan of one or two chunks has too few MFMAs per block
  // for the stages' barriers: 5,000 queries x 16,000, d = 16, k = 10 0.166 ms
  // staged, 0.130 streamed; 300 x 1e6, k = 100 0.32 and 0.245)
  if (mode != 2 && ld <= 256 && (nq > YK_STREAM_NQ || ld > 128) && (mode == 0 || ld > 32)) {
    p.kind = mode == 0 && ld <= 16 && !weighted && nq >= 65536 ? YK_LDS2 : YK_LDS1;
  } else if (mode != 2 && nq <= YK_STREAM_NQ) {
    p.waves = nq <= 32 ? 1 : 2;
  }
  const long qt = (p.kind == YK_LDS2 ? 64 : 32) * p.waves;
  p.tiles = (int)((nq + qt - 1) / qt);
  // the filtered scan of vectors too long for registers streams its queries
  // too, from beyond the L2: three workgroups per CU (1e4 queries x 1e5, d =
  // 960, k = 100: 37.9 ms; the four that fit 40.6, two 38.8); the queries of one
  // tile, or of a tile and a wave, stay in it (65 x 1e6, d = 960, k = 60 0.92 of
  // the time with four)
  const int most = mode == 3 && ld > 256 && p.waves == 4 && nq > qt + 32 ? 3 : 0;
  const YkScanKernel kern = yk_scan_pick(mode, p.kind, ld, weighted);
  p.slots = yk_resident_wgs((const void *)kern, 64 * p.waves, most);
  if (mode == 0 && p.kind != YK_STREAM && nb * ld <= (1L << 19) && nblocks >= 8 &&
      (p.tiles * nblocks >= 4L * p.slots ||
       p.tiles >= yk_resident_wgs((const void *)kern, 64 * p.waves, 1))) {
    // k = 1 over a base of at most 2 MB, which every XCD's L2 holds (the
    // k-means assign): even shares of the (tile, block) pairs, so that no CU
    // waits for a last round of whole tiles (n = 1e5 points are 782 tiles).
    // Fewer than 8 blocks make a tile too short for the merge's launch to pay;
    // with fewer tiles than CUs, shares of fewer than 4 blocks are mostly
    // queries loaded (20,000 x 250, d = 8: 0.87 of the time in whole tiles;
    // 10,000 x 500 0.80; 100,000 x 250, 391 tiles, 1.28).
    p.units = (int)nblocks;
    p.nsplit = 1;
    p.brange = nblocks * p.bstep;
    return p;
  }
  // ~8 work items per resident workgroup keeps the tail of the persistent
  // grid short, of at least min_blocks processed blocks each
  long want = (yk_item_targets[cfg % 3] + p.tiles - 1) / p.tiles;
  long maxs = (nblocks + min_blocks - 1) / min_blocks;
  if (want > maxs) want = maxs;
  // k = 1 of long vectors, four workgroups per CU streaming both operands:
  // beyond 20 blocks each the uneven rounds cost more than they save; 100,000 x
  // 1,000, d = 750 0.70 of the time without, 10,000 x 16,000 0.91, but 50,000 x
  // 1,600 1.09 and 5,000 x 10,000 1.11.
  // A filtered scan of long vectors whose last tile has one wave of queries: the
  // workgroups of that tile end early, and with much to scan only many items in
  // turn fill their place (130 x 1e6, d = 512, k = 60 0.72 of the time).
  const bool uneven =
      mode == 3 && ld > 256 && nblocks > 8192 && nq > qt && (nq - 1) % qt < 32;
  const long few = uneven ? 0 : mode == 0 && ld > 256 ? 20 : 96;
  if (((mode == 0 && nblocks >= 8) || mode == 3) && p.tiles * nblocks < few * p.slots) {
    // few blocks per workgroup (a k = 1 tile of fewer than 8 is not split: the
    // merge takes longer; 50,000 queries x 64 rows, d = 16, 0.82 of the rate):
    // of the splits that fill r rounds of the resident workgroups, the one whose
    // rounds take least (a round is a split's blocks, and ~3 more for its
    // queries and its end)
    long best = -1;
    for (long r = 1; r <= 16; r++) {
      const long s = min(nblocks, r * p.slots / p.tiles);
      if (s < 1) continue;
      const long per = (nblocks + s - 1) / s, n = (nblocks + per - 1) / per;
      const long cost = (p.tiles * n + p.slots - 1) / p.slots * (per + 3);
      if (best < 0 || cost < best) {
        best = cost;
        want = n;
      }
    }
  }
  if (want < min_splits) want = min_splits;
  if (want > max_split) want = max_split;
  if (want > nblocks) want = nblocks;
  if (want < 1) want = 1;
  long per = (nblocks + want - 1) / want;  // processed blocks per split
  // an item's rows stay within 2^30 bytes (the streaming kernel's buffer
  // offsets are 32-bit)
  const long max_per = (1L << 30) / (32L * (ld > 128 ? ld : 128) * 4 * sample);
  if (per > max_per) per = max_per;
  p.brange = per * p.bstep;
  p.nsplit = (int)((nb + p.brange - 1) / p.brange);
  // interleaved sketch splits where the byte offsets of a split's walk (or
  // of a stage's blocks) fit 31 bits
  if (mode == 1) {
    const long span = p.kind == YK_STREAM
                          ? nb * ld * 4
                          : (yk_lds_stage_blocks(ld) - 1) * p.bstep * p.nsplit * ld * 4 + 32L * ld * 4;
    p.inter = span < 0x7fffffffL;
  }
  return p;
}

extern "C" int yk_knn_plan(long nq, long nb, int d, int k, int *nsplit, int *waves, int *nblk) {
  const YkPlan p = yk_plan(k > 1 ? 3 : 0, nq, nb, yk_ld(d), false, 1, 1, 4096, 16, 0);
  *nsplit = p.nsplit;
  *waves = p.waves;
  *nblk = p.kind == YK_LDS2 ? 2 : 1;
  return YK_OK;
}

// Device scratch of the selection pipeline.  Two sources: the grow-only
// buffers the library allocates and keeps (arena == nullptr: slot i is one
// buffer, reallocated when a call needs more), or a caller-given region
// carved front to back in 256-byte-aligned pieces (the no-allocation entry
// point's static array).  A request that does not fit the region is an
// error, never an allocation.
static void *g_scratch[4];
static size_t g_scratch_bytes[4];

struct YkArena {
  char *base;
  size_t cap, used;
};

static size_t yk_align256(size_t b) { return (b + 255) & ~(size_t)255; }

static int yk_scratch(YkArena *ar, int slot, size_t bytes, void **out) {
  if (ar) {
    const size_t at = yk_align256(ar->used);
    if (at > ar->cap || bytes > ar->cap - at)
      return yk_set_error(YK_EINVAL, "scratch request of %zu bytes exceeds the %zu-byte region",
                          bytes, ar->cap);
    *out = ar->base + at;
    ar->used = at + bytes;
    return YK_OK;
  }
  if (bytes > g_scratch_bytes[slot]) {
    if (g_scratch[slot] && hipFree(g_scratch[slot]) != hipSuccess) (void)hipGetLastError();
    g_scratch[slot] = nullptr;
    g_scratch_bytes[slot] = 0;
    hipError_t e = hipMalloc(&g_scratch[slot], bytes);
    if (e != hipSuccess) return yk_hip_fail(e, "hipMalloc(selection scratch)");
    g_scratch_bytes[slot] = bytes;
  }
  *out = g_scratch[slot];
  return YK_OK;
}

static int yk_launch_scan(int mode, const YkPlan &p, ScanArgs a) {
  a.brange = p.brange;
  a.bstep = p.bstep;
  a.nsplit = p.nsplit;
  a.inter = p.inter;
  a.units = p.units;
  a.tiles_x = p.tiles;
  a.total = p.tiles * p.nsplit;
  a.per_xcd = (a.total + 7) / 8;
  YkScanKernel kern = yk_scan_pick(mode, p.kind, a.ld, a.w != nullptr);
  const int per_xcd_res = p.slots / 8;
  dim3 grid(8 * (a.per_xcd < per_xcd_res ? a.per_xcd : per_xcd_res)), block(64 * p.waves);
  a.tick = nullptr;
  if (p.units)
    grid.x = p.slots;
  else if (a.per_xcd > per_xcd_res)  // more items than resident workgroups
    YK_TRY(yk_item_tickets(&a.tick));
  int tok = yk_prof_begin(mode == 1 ? YK_PROF_F32_SKETCH : YK_PROF_FUSED);
  hipLaunchKernelGGL(kern, grid, block, 0, yk_stream(), a);
  yk_prof_end(tok);
  YK_HIP(hipGetLastError());
  return YK_OK;
}

// the m-th smallest of the sketch's n minima per query -> thr
static int yk_thr(const uint64_t *src, long nq, int n, int m, int need, uint64_t *thr, int *cnt,
                  int *flag) {
  if (n > 4096) return yk_set_error(YK_EINVAL, "sketch of %d minima per query", n);
  int tok = yk_prof_begin(YK_PROF_MERGE);
  hipLaunchKernelGGL(yk_thr_kernel, dim3((unsigned)((nq + 3) / 4)), dim3(256), 0, yk_stream(), src,
                     nq, n, m, need, thr, cnt, flag);
  yk_prof_end(tok);
  YK_HIP(hipGetLastError());
  return YK_OK;
}

static int yk_select(const ScanArgs &a, uint64_t *thr, int k, int *assign, float *dis, int *flag,
                     int last) {
  const dim3 grid((unsigned)((a.nq + 3) / 4)), block(256);
  int tok = yk_prof_begin(YK_PROF_MERGE);
  auto kern = k <= 64    ? yk_select_kernel<1>
              : k <= 256 ? yk_select_kernel<4>
              : k <= 512 ? yk_select_kernel<8>
                         : yk_select_kernel<16>;
  hipLaunchKernelGGL(kern, grid, block, 0, yk_stream(), a.cand, a.cap, a.nq, a.cnt, thr, k, assign, dis,
                     flag, last);
  yk_prof_end(tok);
  YK_HIP(hipGetLastError());
  return YK_OK;
}

// Sketch stride of the filtered search: every lane's minimum over its rows
// of a 1-in-stride sample of base blocks, with >= k splits -> >= 2k distinct
// real keys per query.  The k-th smallest of 2k subset minima sits near
// global rank 1.4 * stride * k, the expected candidate count; ~800 keeps
// the filtered pass's append path rare and the list far from overflow.  For
// k <= 16, whose bound is always the proven k-th minimum, 1 in 16 (about
// 360 candidates at k = 16).
static long yk_sketch_stride(long nb, int k, int cfg = 0) {
  const int *sc = yk_stride_scale[(cfg / 3) % 4];
  long stride = 600L * sc[0] / sc[1] / k;
  const long cap = sc[0] == 16 || k <= YK_REG_R ? 16 : 8;  // the last scale may sample 1 in 16
  if (stride > cap) stride = cap;
  if (stride < 1) stride = 1;
  const long nblocks = (nb + 31) / 32;
  while (stride > 1 && nblocks / stride < 2L * k) stride >>= 1;
  return stride;
}

// the sketch's plan
static YkPlan yk_sketch_plan(long nq, long nb, int ld, bool weighted, int k, int cfg) {
  const long stride = yk_sketch_stride(nb, k, cfg);
  if (k <= YK_REG_R)  // more, smaller subsets: a tighter bound
    return yk_plan(1, nq, nb, ld, weighted, stride, 2 * k, 512, 4, cfg);
  return yk_plan(1, nq, nb, ld, weighted, stride, k, k > 256 ? k : 256, 16, cfg);
}

// places of a query's candidate list: no more than the base has rows (whole
// lists for bases of 100 and 1,000 rows left the no-allocation search's 64 MB
// room for 1,024 queries a pass: 16,384 queries, d = 32, 0.41 and 0.42 ms, now
// 0.089 and 0.132)
static int yk_cand_cap(long nb) { return nb < YK_CAND_CAP ? (int)((nb + 7) & ~7L) : YK_CAND_CAP; }

// queries per batch of the filtered search: candidate memory of 512 MB at
// most, the batches of one size
static long yk_filter_batch(long nq, long nb) {
  const long most = 16384L * YK_CAND_CAP / yk_cand_cap(nb), n = (nq + most - 1) / most;
  const long even = ((nq + n - 1) / n + 255) & ~255L;
  return even < nq ? even : nq;
}
// splits of the register top-R scan behind it (k <= 16)
#define YK_FALLBACK_SPLITS 16

// k > 1: sketch threshold, filtered scan, per-query select (queries in
// batches that bound the candidate memory).  k > 16 starts from an estimated
// bound and reads back a flag: queries that overflowed their list or were
// left short are scanned again.  For k <= 16 the bound is the proven k-th
// minimum, so only an overflow (thousands of rows within the bound: ties, or
// near rows concentrated between the sampled blocks) leaves a query over,
// and nothing is read back: the register top-16 scan is queued behind, each
// of its workgroups leaving at once unless the flag is set.  (That scan alone
// -- an exact FP64-normed value and a list test for every pair -- took 0.97
// of 1.34 ms for 1,003 queries x 100,003 vectors, d = 100, k = 10, with the
// sort of its lists 0.36 ms.)
static int yk_knn_filtered(ScanArgs base, int k, int *assign, float *dis, YkArena *ar, int cfg) {
  const long nq_all = base.nq, qb = yk_filter_batch(nq_all, base.nb);
  const bool small = k <= YK_REG_R, weighted = base.w != nullptr;
  // k <= 16 and a base that fits a list: no list overflows, and the proven
  // bound leaves no query short (the sketch and the filtered scan evaluate
  // the same expression), so the queued scan and its sort would find the flag
  // unset: two launches, 3.3 of the 35 - 55 us of such a search
  const bool last = small && base.nb <= YK_CAND_CAP;
  void *vthr, *vcnt, *vcand, *vpart;
  YK_TRY(yk_scratch(ar, 0, sizeof(uint64_t) * qb, &vthr));
  YK_TRY(yk_scratch(ar, 1, sizeof(int) * (qb + 64), &vcnt));
  YK_TRY(yk_scratch(ar, 2, sizeof(uint64_t) * qb * yk_cand_cap(base.nb), &vcand));
  const size_t fixed_used = ar ? ar->used : 0;
  uint64_t *thr = (uint64_t *)vthr;
  int *cnt = (int *)vcnt;
  int *flag = cnt + qb + 32;
  const long stride = yk_sketch_stride(base.nb, k, cfg);

  for (long q0 = 0; q0 < nq_all; q0 += qb) {
    const long nq = nq_all - q0 < qb ? nq_all - q0 : qb;
    ScanArgs a = base;
    a.q = base.q + q0 * base.ld;
    a.qn = base.qn ? base.qn + q0 : nullptr;
    a.nq = nq;
    // (A) sketch: per-lane minima over a strided sample
    const YkPlan pa = yk_sketch_plan(nq, a.nb, a.ld, weighted, k, cfg);
    const YkPlan pc = yk_plan(2, nq, a.nb, a.ld, weighted, 1, 1, YK_FALLBACK_SPLITS, 16, 0);
    const size_t bytes_a = sizeof(uint64_t) * nq * pa.nsplit * 2;
    const size_t bytes_c = small && !last ? sizeof(uint64_t) * nq * pc.nsplit * 2 * YK_REG_R : 0;
    if (ar) ar->used = fixed_used;  // each pass reuses the region's partial-key piece
    YK_TRY(yk_scratch(ar, 3, bytes_a > bytes_c ? bytes_a : bytes_c, &vpart));
    a.part = (uint64_t *)vpart;
    YK_TRY(yk_launch_scan(1, pa, a));
    // the starting bound: the k-th smallest minimum, or for k > 16 the m-th
    // (yk_bound_rank)
    const int m = small ? k : yk_bound_rank(k, stride);
    YK_TRY(yk_thr(a.part, nq, pa.nsplit * 2, m, m, thr, cnt, flag));
    // (B) filtered scan + per-query select
    const YkPlan pb = yk_plan(3, nq, a.nb, a.ld, weighted, 1, 1, 4096, 16, cfg);
    a.thr = thr;
    a.cnt = cnt;
    a.cand = (uint64_t *)vcand;
    a.cap = yk_cand_cap(a.nb);
    int tries = 0;
    for (;;) {
      YK_TRY(yk_launch_scan(3, pb, a));
      YK_TRY(yk_select(a, thr, k, assign + q0 * k, dis + q0 * k, flag, last));
      if (last) break;
      if (small) {  // (C) what is left, if anything
        a.flag = flag;
        YK_TRY(yk_launch_scan(2, pc, a));
        const int n = pc.nsplit * 2 * YK_REG_R;
        int p2 = 1;
        while (p2 < n) p2 <<= 1;
        hipLaunchKernelGGL(yk_sortsel_kernel, dim3((unsigned)nq), dim3(256), sizeof(uint64_t) * p2,
                           yk_stream(), a.part, n, k, p2, assign + q0 * k, dis + q0 * k, thr,
                           flag);
        YK_HIP(hipGetLastError());
        break;
      }
      int hflag = 0;
      YK_TRY(yk_read_small(&hflag, flag, sizeof(int)));
      if (!hflag) break;
      if (++tries == 6)
        return yk_set_error(YK_EINVAL,
                            "k=%d: more than %d keys tie below the k-th distance of a query", k,
                            YK_CAND_CAP);
      hipLaunchKernelGGL(yk_zero_cnt_kernel, dim3(1), dim3(64), 0, yk_stream(), flag, 1L);
    }
  }
  return YK_OK;
}

// Checks shared by the FP32 entry points; 1 when there is nothing to do.
static int yk_knn_f32_check(int *type, long nq, long nb, int k) {
  if (*type == 12) *type = YK_L2;
  if (*type != YK_L2 && *type != YK_DOT)
    return yk_set_error(YK_EINVAL, "distance type %d has no GPU path (2, 12, 16 only)", *type);
  if (k < 1 || k > nb)
    return yk_set_error(YK_EINVAL, "k=%d out of range (nb=%ld)", k, nb);
  if (nb > 0x7fffffffL || nq > 0x7fffffffL) return yk_set_error(YK_EINVAL, "sizes exceed int32");
  return nq <= 0 ? 1 : YK_OK;
}

// k <= 16 by the register top-16 scan alone, without sketch and filter.  The
// lines lie where the two routes meet, in 2,800 shapes of 1 .. 200,000 queries,
// 16 .. 1e6 rows, d = 16 .. 2,048, k = 2, 10 and 16; filter and lists in ms:
// * two blocks of rows at most: the lists' two launches against four (1 query x
//   33 rows, d = 128 0.032 / 0.029; x 80 0.033 / 0.037), and some more rows as
//   the queries grow in number (d = 128, k = 2: 12,400 x 100 0.088 / 0.078, 16,000
//   x 130 0.108 / 0.089; k = 10: 4,000 x 49 0.047 / 0.043, 12,400 x 64 0.071 /
//   0.063, 16,000 x 82 0.088 / 0.076; d = 762, k = 4: 8,000 x 82 0.120 / 0.135);
// * many queries of few rows, where a query's selections cost more than its
//   distances (50,000 queries, d = 64: x 200 0.31 / 0.19, x 600 0.37 / 0.36;
//   200,000 x 1,000 1.63 / 1.45, x 2,000 2.18 / 2.40);
// * d > 256, where both routes stream from memory: from 12,500 queries on
//   (16,384 queries, d = 512: x 100 0.145 / 0.151, x 1,000 0.68 / 0.52, x 16,000
//   4.79 / 4.82), and as the work grows, where the sketch's sixteenth of the MFMAs
//   and the filter's fewer waves cost more than the lists' insertions save (d =
//   400: 4,000 x 1e5 5.32 / 5.63, 10,000 x 4e5 60.1 / 57.8; d = 640: 1,000 x 4e5
//   8.18 / 8.17, 4,000 x 4e5 41.7 / 38.5; d = 960: 1,000 x 1e5 3.30 / 3.82,
//   4,000 x 1e5 14.95 / 14.07).  One tile is the filter's, and so are a few whose
//   last one has a single wave of queries (144 x 1e6, d = 960 6.6 / 8.2), but a
//   second tile of one wave over few blocks (yk_plan's uneven: 144 x 2e5, d = 960
//   1.98 / 1.81, d = 512 0.96 / 1.05; x 1e5 1.05 / 1.16).
// Past the lines the lists take 0.5 - 1.0 of the filter's time, before them 1.0
// - 5 times as long.
static bool yk_knn_by_lists(int k, int ld, long nq, long nb) {
  if (k < 2 || k > YK_REG_R) return false;
  if (nb <= 48 + nq / 240 || (k < 8 && nb <= 30 + nq / 160)) return true;
  if (nq >= 16384 && nb <= 100 + nq / 250) return true;
  if (ld <= 256 || nq <= 128) return false;
  const double work = (double)nq * (double)nb * ld * ld;
  if (nq <= 160) return nb <= (1L << 18) && work >= 2e13;
  if (nq <= 512 && (nq - 1) % 128 < 32) return false;
  return nq > 12500 || work >= 1.3e14;
}
static YkPlan yk_lists_plan(long nq, long nb, int ld, bool weighted, int cfg) {
  return yk_plan(2, nq, nb, ld, weighted, 1, 1, 256, 16, cfg);
}
static int yk_knn_lists(ScanArgs a, int k, int *assign, float *dis, YkArena *ar, int cfg) {
  const YkPlan p = yk_lists_plan(a.nq, a.nb, a.ld, a.w != nullptr, cfg);
  const int n = p.nsplit * 2 * YK_REG_R;
  void *buf;
  YK_TRY(yk_scratch(ar, 3, sizeof(uint64_t) * a.nq * n, &buf));
  a.part = (uint64_t *)buf;
  YK_TRY(yk_launch_scan(2, p, a));
  int p2 = 1;
  while (p2 < n) p2 <<= 1;
  int tok = yk_prof_begin(YK_PROF_MERGE);
  hipLaunchKernelGGL(yk_sortsel_kernel, dim3((unsigned)a.nq), dim3(256), sizeof(uint64_t) * p2,
                     yk_stream(), a.part, n, k, p2, assign, dis, nullptr, nullptr);
  yk_prof_end(tok);
  YK_HIP(hipGetLastError());
  return YK_OK;
}

// The FP32 search of nq queries, scratch from ar (nullptr: the grow-only
// buffers); lists: yk_knn_by_lists
static int yk_knn_f32_run(int type, long nq, long nb, int d, int k, const float *q,
                          const double *qn, const float *b, const float *bn, const float *w,
                          int *assign, float *dis, bool lists, YkArena *ar, int cfg = 0) {
  if (k > YK_KMAX) {  // beyond the on-chip selection: distance rows + radix select
    if (ar) return yk_set_error(YK_EINVAL, "k=%d > %d needs allocated scratch", k, YK_KMAX);
    return yk_knn_bigk(type, nq, nb, d, k, q, qn, b, bn, w, assign, dis);
  }
  ScanArgs a = {};
  a.q = q;
  a.qn = qn;
  a.nq = nq;
  a.b = b;
  a.bn = bn;
  a.w = w;
  a.nb = nb;
  a.ld = yk_ld(d);
  a.type = type;
  a.out_i = assign;
  a.out_d = dis;
  if (lists) return yk_knn_lists(a, k, assign, dis, ar, cfg);
  if (k > 1) return yk_knn_filtered(a, k, assign, dis, ar, cfg);
  const YkPlan p = yk_plan(0, nq, nb, a.ld, w != nullptr, 1, 1, 4096, 16, cfg);
  const long tq = p.kind == YK_LDS2 ? 256 : 128;
  if (p.nsplit > 1 || p.units) {
    void *buf;
    YK_TRY(yk_scratch(ar, 3, sizeof(uint64_t) * (p.units ? 2 * tq * p.slots : nq * p.nsplit), &buf));
    a.part = (uint64_t *)buf;
  }
  YK_TRY(yk_launch_scan(0, p, a));
  if (p.units) {
    int tok = yk_prof_begin(YK_PROF_MERGE);
    const bool wave = p.slots > 8L * p.tiles;  // shares per tile
    const auto merge = wave ? yk_merge_share_kernel<true> : yk_merge_share_kernel<false>;
    hipLaunchKernelGGL(merge, dim3((unsigned)(wave ? (nq + 3) / 4 : (nq + 255) / 256)), dim3(256),
                       0, yk_stream(), a.part, nq, (int)tq, (long)p.units,
                       (long)p.tiles * p.units, (long)p.slots, assign, dis);
    yk_prof_end(tok);
    YK_HIP(hipGetLastError());
  } else if (p.nsplit > 1) {
    int tok = yk_prof_begin(YK_PROF_MERGE);
    hipLaunchKernelGGL(yk_merge1_kernel, dim3((unsigned)((nq + 3) / 4)), dim3(256), 0, yk_stream(),
                       a.part, nq, p.nsplit, assign, dis);
    yk_prof_end(tok);
    YK_HIP(hipGetLastError());
  }
  return YK_OK;
}

// a search through yk_time_ms
struct YkF32Call {
  int type;
  long nq, nb;
  int d, k;
  const float *q;
  const double *qn;
  const float *b, *bn, *w;
  int *assign;
  float *dis;
  int cfg;
};
static int yk_f32_call(void *p) {
  const YkF32Call &c = *(const YkF32Call *)p;
  return yk_knn_f32_run(c.type, c.nq, c.nb, c.d, c.k, c.q, c.qn, c.b, c.bn, c.w, c.assign, c.dis,
                        yk_knn_by_lists(c.k, yk_ld(c.d), c.nq, c.nb), nullptr, c.cfg);
}

// log2 bucket of a size (shape classes of the tuning cache)
static int yk_lg(long x) {
  int l = 0;
  while (x > 1) {
    x >>= 1;
    l++;
  }
  return l;
}

// The plan: the tuning cache's choice for the shape class; on a miss (and
// a search of at least 2^30 flop, where one timing is meaningful), every
// candidate plan is timed once after an untimed run of the default, the
// fastest recorded.  The outputs then hold the last candidate's results --
// the same bits as any other plan's.  *ran = 1 when the outputs are already
// written.
static int yk_f32_plan(const YkF32Call &call, int *cfg, int *ran) {
  *cfg = 0;
  *ran = 0;
  if (call.k > YK_KMAX || !yk_tune_enabled()) return YK_OK;
  if ((double)call.nq * call.nb * call.d < (double)(1 << 29)) return YK_OK;
  const int kc = call.k == 1 ? 1 : call.k <= YK_REG_R ? 16 : 1 << yk_lg(call.k);
  char key[128];
  // (a plan of one route, or of the weighted kernels, says nothing of the
  // other's: both may meet within a bucket of sizes)
  snprintf(key, sizeof key, "f32:v2:t%d:k%d:ld%d:q%d:b%d%s%s", call.type, kc, yk_ld(call.d),
           yk_lg(call.nq), yk_lg(call.nb),
           yk_knn_by_lists(call.k, yk_ld(call.d), call.nq, call.nb) ? ":lists" : "",
           call.w ? ":w" : "");
  if (yk_tune_get(key, cfg)) {
    if (*cfg < 0 || *cfg >= YK_NCFG) *cfg = 0;
    return YK_OK;
  }
  const int ncand = call.k > YK_REG_R ? YK_NCFG : 3;  // the stride matters for k > 16 only
  // candidates whose plans come out the same as an earlier one's are not
  // timed again (e.g. queries enough to fill the chip without any split)
  long sig[YK_NCFG][3];
  int distinct = 0;
  bool dup[YK_NCFG] = {};
  const int ld = yk_ld(call.d);
  const bool weighted = call.w != nullptr;
  for (int i = 0; i < ncand; i++) {
    const long nqb = yk_filter_batch(call.nq, call.nb);
    if (call.k == 1 || yk_knn_by_lists(call.k, ld, call.nq, call.nb)) {
      const YkPlan p = call.k > 1
                           ? yk_lists_plan(call.nq, call.nb, ld, weighted, i)
                           : yk_plan(0, call.nq, call.nb, ld, weighted, 1, 1, 4096, 16, i);
      sig[i][0] = p.nsplit, sig[i][1] = p.brange, sig[i][2] = 0;
    } else {
      const YkPlan pa = yk_sketch_plan(nqb, call.nb, ld, weighted, call.k, i);
      const YkPlan pb = yk_plan(3, nqb, call.nb, ld, weighted, 1, 1, 4096, 16, i);
      sig[i][0] = pa.bstep, sig[i][1] = pa.nsplit, sig[i][2] = pb.nsplit;
    }
    for (int j = 0; j < i && !dup[i]; j++)
      dup[i] = !dup[j] && sig[j][0] == sig[i][0] && sig[j][1] == sig[i][1] &&
               sig[j][2] == sig[i][2];
    distinct += !dup[i];
  }
  if (distinct < 2) return YK_OK;  // one plan: nothing to choose
  YkF32Call c = call;
  c.cfg = 0;
  YK_TRY(yk_f32_call(&c));  // warm-up
  float best = 1e30f;
  for (int i = 0; i < ncand; i++) {
    if (dup[i]) continue;
    c.cfg = i;
    float ms = 0;
    YK_TRY(yk_time_ms(yk_f32_call, &c, &ms));
    if (ms < best) {
      best = ms;
      *cfg = i;
    }
  }
  yk_tune_put(key, *cfg);
  *ran = 1;
  return YK_OK;
}

extern "C" int yk_knn_f32(int type, long nq, long nb, int d, int k, const float *q,
                          const double *qn, const float *b, const float *bn, const float *w,
                          int *assign, float *dis) {
  YK_TRY(yk_init());
  YkGuard guard;
  const int c = yk_knn_f32_check(&type, nq, nb, k);
  if (c != YK_OK) return c > 0 ? YK_OK : c;
  const YkF32Call call = {type, nq, nb, d, k, q, qn, b, bn, w, assign, dis, 0};
  int cfg = 0, ran = 0;
  YK_TRY(yk_f32_plan(call, &cfg, &ran));
  if (ran) return YK_OK;
  return yk_knn_f32_run(type, nq, nb, d, k, q, qn, b, bn, w, assign, dis,
                        yk_knn_by_lists(k, yk_ld(d), nq, nb), nullptr, cfg);
}

// ---------------------------------------------------------------------------
// the FP32 search without allocation: scratch in a static device array

// Every GPU the library runs on holds one copy of this array for the life
// of the process.  Host code never passes its name to a kernel (on the host
// it is only a stand-in for the symbol): the device address of each GPU's
// copy comes from hipGetSymbolAddress, taken once per device.
static __device__ __align__(256) unsigned char scratch[YK_NOALLOC_SCRATCH_BYTES];

#define YK_NOALLOC_MAX_DEV 64
static void *g_noalloc_ptr[YK_NOALLOC_MAX_DEV];
static pthread_mutex_t g_noalloc_mu = PTHREAD_MUTEX_INITIALIZER;

// the current device's copy of the array (set-up on the first call there)
static int yk_noalloc_region(char **out) {
  int dev = -1;
  YK_HIP(hipGetDevice(&dev));
  if (dev < 0 || dev >= YK_NOALLOC_MAX_DEV)
    return yk_set_error(YK_EINVAL, "device %d beyond the %d the scratch table covers", dev,
                        YK_NOALLOC_MAX_DEV);
  pthread_mutex_lock(&g_noalloc_mu);
  int rc = YK_OK;
  if (!g_noalloc_ptr[dev]) {
    void *ptr = nullptr;
    const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess)
      rc = yk_hip_fail(e, "hipGetSymbolAddress(scratch)");
    else if (!ptr)
      rc = yk_set_error(YK_EHIP, "hipGetSymbolAddress(scratch) gave a null address");
    else
      g_noalloc_ptr[dev] = ptr;
  }
  *out = (char *)g_noalloc_ptr[dev];
  pthread_mutex_unlock(&g_noalloc_mu);
  return rc;
}

// Scratch bytes one yk_knn_f32_run over nq queries takes from a region (the
// same plans and pieces as the run itself, each rounded up to 256 bytes).
static size_t yk_knn_f32_need(long nq, long nb, int ld, bool weighted, int k, bool lists) {
  if (lists)
    return yk_align256(sizeof(uint64_t) * nq * 2 * YK_REG_R *
                       yk_lists_plan(nq, nb, ld, weighted, 0).nsplit);
  if (k == 1) {
    const YkPlan p = yk_plan(0, nq, nb, ld, weighted, 1, 1, 4096, 16, 0);
    if (p.units) return yk_align256(sizeof(uint64_t) * 2 * (p.kind == YK_LDS2 ? 256 : 128) * p.slots);
    return p.nsplit > 1 ? yk_align256(sizeof(uint64_t) * nq * p.nsplit) : 0;
  }
  const long qb = yk_filter_batch(nq, nb);
  const YkPlan pa = yk_sketch_plan(qb, nb, ld, weighted, k, 0);
  const YkPlan pc = yk_plan(2, qb, nb, ld, weighted, 1, 1, YK_FALLBACK_SPLITS, 16, 0);
  const size_t bytes_a = sizeof(uint64_t) * qb * pa.nsplit * 2;
  const size_t bytes_c =
      k <= YK_REG_R && nb > YK_CAND_CAP ? sizeof(uint64_t) * qb * pc.nsplit * 2 * YK_REG_R : 0;
  return yk_align256(sizeof(uint64_t) * qb) + yk_align256(sizeof(int) * (qb + 64)) +
         yk_align256(sizeof(uint64_t) * qb * yk_cand_cap(nb)) +
         yk_align256(bytes_a > bytes_c ? bytes_a : bytes_c);
}

extern "C" int yk_knn_f32_noalloc(int type, long nq, long nb, int d, int k, const float *q,
                                  const double *qn, const float *b, const float *bn,
                                  const float *w, int *assign, float *dis) {
  YK_TRY(yk_init());
  YkGuard guard;
  const int c = yk_knn_f32_check(&type, nq, nb, k);
  if (c != YK_OK) return c > 0 ? YK_OK : c;
  char *region = nullptr;
  YK_TRY(yk_noalloc_region(&region));
  // Queries go in passes small enough for the region: of 16384 queries or
  // fewer, halved until the scratch of a pass and of what the last one leaves
  // over fits, then a quarter more at a time while that still fits.  Each
  // query's result depends only on that query, so the passes give the single
  // call's results.  (The route is the first pass's for them all.)
  const int ld = yk_ld(d);
  bool lists = false;
  auto need_of = [&](long pass) {
    const long n = pass < nq ? pass : nq, left = nq % n;
    lists = yk_knn_by_lists(k, ld, n, nb);
    const size_t a = yk_knn_f32_need(n, nb, ld, w != nullptr, k, lists);
    const size_t b = left ? yk_knn_f32_need(left, nb, ld, w != nullptr, k, lists) : 0;
    return a > b ? a : b;
  };
  long pass = 16384;
  size_t need = need_of(pass);
  while (need > YK_NOALLOC_SCRATCH_BYTES && pass > 32) need = need_of(pass >>= 1);
  if (pass >= 128 && pass < 16384 && pass < nq) {
    long more = 7;  // quarters of the pass that fits
    while (more > 4 && need_of(pass / 4 * more) > YK_NOALLOC_SCRATCH_BYTES) more--;
    pass = pass / 4 * more;
    need = need_of(pass);
  }
  if (need > YK_NOALLOC_SCRATCH_BYTES)
    return yk_set_error(YK_EINVAL,
                        "k=%d, nb=%ld needs %zu scratch bytes even for %ld queries at a time; "
                        "the no-allocation search holds %zu",
                        k, nb, need, pass, (size_t)YK_NOALLOC_SCRATCH_BYTES);
  for (long q0 = 0; q0 < nq; q0 += pass) {
    const long n = nq - q0 < pass ? nq - q0 : pass;
    YkArena ar = {region, (size_t)YK_NOALLOC_SCRATCH_BYTES, 0};
    YK_TRY(yk_knn_f32_run(type, n, nb, d, k, q + q0 * ld, qn ? qn + q0 : nullptr, b, bn, w,
                          assign + q0 * k, dis + q0 * k, lists, &ar));
  }
  return YK_OK;
}

// ---------------------------------------------------------------------------
// batched form: the assign step of many k-means instances in one launch

// Small centroid sets (NBLK 32-row blocks, d <= 16 NCH): a work item is one
// of the nsub pieces (`sub` consecutive points) of an update chunk (up to
// `chunk` consecutive points of one instance); its workgroup stages the
// instance's centroid fragments in LDS and streams the chunk's points
// through in 32-point blocks, wave w taking blocks w, w + W, ...; a block's
// fragments are reloaded chunk by chunk right after the centroid blocks'
// MFMAs have read them, so every load has the next block's MFMAs to
// arrive in.  (The general scan holds the points and streams the
// centroids, which for k <= 64 leaves each 32-point tile two centroid blocks
// of work against the full latency of loading its points.)  Same MFMA
// operands, same order and the same epilogue arithmetic as the general
// scan's MODE 0: the outputs are its bits.
struct BassignArgs {
  const float *v;
  const double *vn;
  const float *cent, *cn;
  int ld, kc, kpad, chunk, sub, nsub;
  const long *inst_off;
  const int *uitem_inst, *uitem_first;
  int nitems, per_xcd;
  const int *done;
  int *assign;
  float *dis;
  int *tick;
};

template <int NCH, int NBLK>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void
yk_bassign_res_kernel(BassignArgs a) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nwave = blockDim.x >> 6;
  const int r = lane & 31, h = lane >> 5;
  const int xcd = blockIdx.x & 7, local = blockIdx.x >> 3, wpx = gridDim.x >> 3;
  const int ibeg = xcd * a.per_xcd, iend = min(a.nitems, ibeg + a.per_xcd);
  const int ld = a.ld;
  __shared__ float4 cfs[NBLK * 2 * NCH * 64];
  __shared__ double nns[NBLK * 32];
  __shared__ int s_item;
  auto next_item = [&](int it) {
    __syncthreads();  // also: every wave is done with the staged centroids
    if (threadIdx.x == 0) s_item = ibeg + wpx + atomicAdd(&a.tick[xcd], 1);
    __syncthreads();
    return s_item;
  };
  for (int it = ibeg + local; it < iend; it = next_item(it)) {
    const int u = it / a.nsub, inst = a.uitem_inst[u];
    if (a.done[inst]) continue;
    const long off = a.inst_off[inst], n = a.inst_off[inst + 1] - off;
    const long pc = (long)(u - a.uitem_first[inst]) * a.chunk;
    const long pe = pc + a.chunk < n ? pc + a.chunk : n;
    const long p0 = pc + (long)(it % a.nsub) * a.sub;
    const long p1 = p0 + a.sub < pe ? p0 + a.sub : pe;
    if (p0 >= p1) continue;
    const float *cb0 = a.cent + (long)inst * a.kpad * ld;
    const float *cnb = a.cn + (long)inst * a.kpad;
    // centroid fragments and norms, staged in LDS once for the workgroup
    // in the lanes' order: fragment entry (cb, half-chunk q, lane) holds row
    // 32 cb + r, dimensions 16 (q / 2) + 8 h + 4 (q % 2) .. + 3 (rows past kc
    // are zeros of norm YK_FAR_NORM)
    for (int i = threadIdx.x; i < NBLK * 2 * NCH * 64; i += blockDim.x) {
      const int ln = i & 63, q = (i >> 6) % (2 * NCH), cb = (i >> 6) / (2 * NCH);
      const int cr = 32 * cb + (ln & 31);
      const float *row = cb0 + (long)cr * ld + (ln >> 5) * 8;
      cfs[i] = cr < a.kc ? *(const float4 *)(row + 16 * (q >> 1) + 4 * (q & 1))
                         : make_float4(0.f, 0.f, 0.f, 0.f);
    }
    for (int i = threadIdx.x; i < NBLK * 32; i += blockDim.x)
      nns[i] = (double)(i < a.kc ? cnb[i] : YK_FAR_NORM);
    __syncthreads();
    const long step = 32L * nwave;
    long pb = p0 + 32L * wave;
    if (pb >= p1) continue;
    // the block's point fragments and norm (rows past the chunk clamped to
    // its last point, not written)
    float4 bq[2 * NCH];
    auto loadq = [&](long blk, int c) {
      const float *pr = a.v + (off + min(blk + r, p1 - 1)) * ld + h * 8 + 16 * c;
      bq[2 * c] = *(const float4 *)pr;
      bq[2 * c + 1] = *(const float4 *)(pr + 4);
    };
#pragma unroll
    for (int c = 0; c < NCH; c++) loadq(pb, c);
    double qd = a.vn[off + min(pb + r, p1 - 1)];
    for (; pb < p1; pb += step) {
      const long pn = pb + step < p1 ? pb + step : pb;  // past the chunk: reload this block
      const double qdn = a.vn[off + min(pn + r, p1 - 1)];
      // the centroid blocks' MFMA chains interleaved chunk by chunk (two
      // independent accumulators); chunk c of the next point block loads
      // once every chain has read it, a whole block of MFMAs ahead of use
      f32x16 acc[NBLK];
#pragma unroll
      for (int cb = 0; cb < NBLK; cb++)
#pragma unroll
        for (int e = 0; e < 16; e++) acc[cb][e] = 0.f;
      // the centroid operand of chunk c + 1 is read from LDS while chunk
      // c's MFMAs run
      float4 av[2][NBLK][2];
#pragma unroll
      for (int cb = 0; cb < NBLK; cb++) {
        av[0][cb][0] = cfs[(cb * 2 * NCH) * 64 + lane];
        av[0][cb][1] = cfs[(cb * 2 * NCH + 1) * 64 + lane];
      }
#pragma unroll
      for (int c = 0; c < NCH; c++) {
        const float4 b0 = bq[2 * c], b1 = bq[2 * c + 1];
        if (c + 1 < NCH) {
#pragma unroll
          for (int cb = 0; cb < NBLK; cb++) {
            av[(c + 1) & 1][cb][0] = cfs[(cb * 2 * NCH + 2 * c + 2) * 64 + lane];
            av[(c + 1) & 1][cb][1] = cfs[(cb * 2 * NCH + 2 * c + 3) * 64 + lane];
          }
        }
#pragma unroll
        for (int cb = 0; cb < NBLK; cb++) {
          const float4 a0 = av[c & 1][cb][0], a1 = av[c & 1][cb][1];
          acc[cb] = __builtin_amdgcn_mfma_f32_32x32x2f32(a0.x, b0.x, acc[cb], 0, 0, 0);
          acc[cb] = __builtin_amdgcn_mfma_f32_32x32x2f32(a0.y, b0.y, acc[cb], 0, 0, 0);
          acc[cb] = __builtin_amdgcn_mfma_f32_32x32x2f32(a0.z, b0.z, acc[cb], 0, 0, 0);
          acc[cb] = __builtin_amdgcn_mfma_f32_32x32x2f32(a0.w, b0.w, acc[cb], 0, 0, 0);
          acc[cb] = __builtin_amdgcn_mfma_f32_32x32x2f32(a1.x, b1.x, acc[cb], 0, 0, 0);
          acc[cb] = __builtin_amdgcn_mfma_f32_32x32x2f32(a1.y, b1.y, acc[cb], 0, 0, 0);
          acc[cb] = __builtin_amdgcn_mfma_f32_32x32x2f32(a1.z, b1.z, acc[cb], 0, 0, 0);
          acc[cb] = __builtin_amdgcn_mfma_f32_32x32x2f32(a1.w, b1.w, acc[cb], 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
        loadq(pn, c);
        __builtin_amdgcn_sched_barrier(0);
      }
      float bv = 1e30f;
      int bi = -1;
#pragma unroll
      for (int cb = 0; cb < NBLK; cb++) {
        const YkNormLds nn = {nullptr, nns + 32 * cb + 4 * h};
        yk_best1_block<false>(acc[cb], nn, qd, 32L * cb, h, false, bv, bi);
      }
      const float ov = __shfl_xor(bv, 32);
      const int oi = __shfl_xor(bi, 32);
      if (ov < bv || (ov == bv && oi < bi)) {
        bv = ov;
        bi = oi;
      }
      if (h == 0 && pb + r < p1) {
        a.dis[off + pb + r] = bv;
        a.assign[off + pb + r] = bi;
      }
      qd = qdn;
    }
  }
}

template <int NCH, int NBLK>
static void (*yk_bassign_pick2())(BassignArgs) {
  return yk_bassign_res_kernel<NCH, NBLK>;
}

// The kernel for (nch, nblk), or null when the centroid set does not fit
// (centroid fragments of nblk x nch x 2 KB of LDS, at most 32 KB).
static void (*yk_bassign_pick(int nch, int nblk))(BassignArgs) {
  if (nblk == 1) {
    switch (nch) {
      case 1: return yk_bassign_pick2<1, 1>();
      case 2: return yk_bassign_pick2<2, 1>();
      case 3: return yk_bassign_pick2<3, 1>();
      case 4: return yk_bassign_pick2<4, 1>();
      case 5: return yk_bassign_pick2<5, 1>();
      case 6: return yk_bassign_pick2<6, 1>();
      case 7: return yk_bassign_pick2<7, 1>();
      case 8: return yk_bassign_pick2<8, 1>();
    }
  } else if (nblk == 2) {
    switch (nch) {
      case 1: return yk_bassign_pick2<1, 2>();
      case 2: return yk_bassign_pick2<2, 2>();
      case 3: return yk_bassign_pick2<3, 2>();
      case 4: return yk_bassign_pick2<4, 2>();
      case 5: return yk_bassign_pick2<5, 2>();
      case 6: return yk_bassign_pick2<6, 2>();
      case 7: return yk_bassign_pick2<7, 2>();
      case 8: return yk_bassign_pick2<8, 2>();
    }
  } else if (nblk <= 4 && nch <= 4) {
    switch (nch * 8 + nblk) {
      case 1 * 8 + 3: return yk_bassign_pick2<1, 3>();
      case 2 * 8 + 3: return yk_bassign_pick2<2, 3>();
      case 3 * 8 + 3: return yk_bassign_pick2<3, 3>();
      case 4 * 8 + 3: return yk_bassign_pick2<4, 3>();
      case 1 * 8 + 4: return yk_bassign_pick2<1, 4>();
      case 2 * 8 + 4: return yk_bassign_pick2<2, 4>();
      case 3 * 8 + 4: return yk_bassign_pick2<3, 4>();
      case 4 * 8 + 4: return yk_bassign_pick2<4, 4>();
    }
  }
  return nullptr;
}

// The batched assign over the update chunks with the centroids
// register-resident; returns 1 when the shape has no such kernel (the
// caller then uses yk_batch_assign).
int yk_batch_assign_res(int ninst, int d, int kc, int kpad, int chunk, const float *v,
                        const double *vn, const float *cent, const float *cn,
                        const long *inst_off, long nuitems, const int *uitem_inst,
                        const int *uitem_first, const int *done, int *assign, float *dis) {
  YK_TRY(yk_init());
  (void)ninst;
  const int ld = yk_ld(d);
  auto kern = yk_bassign_pick(ld >> 4, (kc + 31) / 32);
  if (!kern || nuitems <= 0 || nuitems > 0x7fffffffL) return 1;
  BassignArgs a = {};
  a.v = v;
  a.vn = vn;
  a.cent = cent;
  a.cn = cn;
  a.ld = ld;
  a.kc = kc;
  a.kpad = kpad;
  a.chunk = chunk;
  a.inst_off = inst_off;
  a.uitem_inst = uitem_inst;
  a.uitem_first = uitem_first;
  a.done = done;
  a.assign = assign;
  a.dis = dis;
  YK_TRY(yk_item_tickets(&a.tick));
  // (two workgroups per CU: a third, where the registers allow it, made an
  // iteration's assign 0.387 instead of 0.380 ms)
  const int per_res = yk_resident_wgs((const void *)kern, 256, 2) / 8;
  // The update's chunk is chosen for the update; whole chunks as work items
  // left the last of ~1.4 rounds half empty (2e6 points, 1,094 chunks for 768
  // workgroups: 0.412 ms, now 0.380; two workgroups per CU with whole chunks, as
  // many registers once made it, were as good: 0.37 - 0.39).  At least six items a workgroup, of
  // 256 points or more (the centroids are staged once per item).
  long nsub = (48L * per_res + nuitems - 1) / nuitems;
  if (nsub > chunk / 256) nsub = chunk / 256;
  if (nsub < 1) nsub = 1;
  a.sub = (int)(((chunk + nsub - 1) / nsub + 127) / 128 * 128);
  a.nsub = (chunk + a.sub - 1) / a.sub;
  if (nuitems * a.nsub > 0x7fffffffL) a.sub = chunk, a.nsub = 1;
  a.nitems = (int)(nuitems * a.nsub);
  a.per_xcd = (a.nitems + 7) / 8;
  const dim3 grid(8 * (a.per_xcd < per_res ? a.per_xcd : per_res)), block(256);
  hipLaunchKernelGGL(kern, grid, block, 0, yk_stream(), a);
  YK_HIP(hipGetLastError());
  return YK_OK;
}

extern "C" int yk_batch_assign(long nitems, const int *item_inst, const int *item_tile,
                               const long *inst_off, int d, int kc, int kpad, const float *v,
                               const double *vn, const float *cent, const float *cn,
                               const int *done, int *assign, float *dis) {
  return yk_batch_assign_idx(nitems, item_inst, item_tile, inst_off, d, kc, kpad, v, vn, nullptr,
                             cent, cn, done, assign, dis);
}

int yk_batch_assign_idx(long nitems, const int *item_inst, const int *item_tile,
                        const long *inst_off, int d, int kc, int kpad, const float *v,
                        const double *vn, const int *qidx, const float *cent, const float *cn,
                        const int *done, int *assign, float *dis) {
  YK_TRY(yk_init());
  if (nitems <= 0) return YK_OK;
  ScanArgs a = {};
  a.q = v;
  a.qn = vn;
  a.b = cent;
  a.bn = cn;
  a.ld = yk_ld(d);
  a.type = YK_L2;
  a.brange = kpad;
  a.bstep = 32;
  a.nsplit = 1;
  a.tiles_x = 1;
  a.out_i = assign;
  a.out_d = dis;
  a.item_inst = item_inst;
  a.item_tile = item_tile;
  a.inst_off = inst_off;
  a.kc = kc;
  a.kpad = kpad;
  a.done = done;
  a.qidx = qidx;
  a.total = (int)nitems;
  a.per_xcd = (a.total + 7) / 8;
  // (the points are the kernel's queries: 128 per item, four waves)
  auto kern = yk_scan_pick(0, a.ld <= 256 ? YK_LDS1 : YK_STREAM, a.ld, false);
  YK_TRY(yk_item_tickets(&a.tick));
  const int per_res = yk_resident_wgs((const void *)kern, 256) / 8;
  dim3 grid(8 * (a.per_xcd < per_res ? a.per_xcd : per_res)), block(256);
  hipLaunchKernelGGL(kern, grid, block, 0, yk_stream(), a);
  YK_HIP(hipGetLastError());
  return YK_OK;
}
