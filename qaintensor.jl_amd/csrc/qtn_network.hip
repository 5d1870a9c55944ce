// Whole-network contraction with every intermediate resident on the device:
// the work of TensorOperations.ncon(tensors, labels; order) behind
// contract(net) (src/contract.jl:242-264; ncon at :257 and :263).
//
// Labels follow ncon: a positive label names a contracted leg pair (it
// appears twice in the network, in one tensor for a trace), a negative one
// an open leg; the result's legs are ordered -1, -2, ... .  The contraction
// sequence is the caller's (the reference's planner, or increasing labels):
// the first label not yet contracted names the next pair of tensors, which
// are contracted over every label they share.  Tensors left unconnected at
// the end are joined by outer products in their order.
//
// The steps form a tree; all steps of one depth are independent and run in
// one launch (net_level), each as the block kind its sizes call for:
//   elem    one thread per product entry (short inner dimension)
//   tile    complex FP64 GEMM tiles on MFMA whose operand staging gathers
//           through the tensors' own strides (the permutes of a permute +
//           GEMM scheme folded into the global -> LDS loads)
//   long    few entries over a long inner dimension (the closing product of
//           two wide tensors): threads over the inner index
//   reduce  the sum of the partial products of a split inner dimension
// The free legs of A index the rows, the shared legs the inner dimension,
// the free legs of B the columns, and the product is written contiguous
// with legs (free A, free B).  Intermediates live in one device arena whose
// layout (first fit, freed operands reused) is planned on the host before
// anything runs; the inputs and the step descriptors arrive in one staging
// copy, the result leaves in one.
#include <algorithm>
#include <cstring>
#include <functional>
#include <map>
#include <numeric>
#include <vector>

#include "qtn_internal.hpp"

namespace qtn {
namespace {

constexpr int kMaxLegs = 24;
constexpr int kSlotArena = 220;

// One leg of an index group (first leg fastest): its size, log2 of it (-1
// when not a power of two) and the element offsets its values add in the
// group's one or two tensors (the inner legs step through A and B).
struct NetLeg {
  uint32_t dim;
  int32_t sh;
  int64_t s0, s1;
};

enum NetKind { kElem = 0, kTile, kLong, kReduce, kIdent, kGather };

// One step of a level as its blocks read it.  Offsets are in elements of
// the arena; legs lie in the pool from `legs` on: n_am rows legs, then n_k
// inner legs, then n_bn column legs.
struct NetStep {
  int64_t a, b, c, M, N, K;
  int64_t kchunk;       // inner indices per block (tile and long kinds)
  uint32_t first;       // first block of the step in its level
  uint32_t nx, ny;      // tiles along M and N (tile kind)
  int32_t kind, tile;   // tile: rows and columns of a tile, 32 or 64
  int32_t legs, n_am, n_k, n_bn;
  int32_t a_kfast, b_nfast;
  int32_t nsplit;       // partial products (reduce: how many to add)
};

__device__ __forceinline__ int64_t net_off(const NetLeg* l, int n,
                                           uint64_t idx) {
  int64_t off = 0;
  if (idx <= 0xffffffffu) {
    // 32-bit divisions where the index allows (64-bit ones are long
    // instruction sequences), shifts where the leg allows
    uint32_t u = (uint32_t)idx;
    for (int i = 0; i < n; ++i) {
      const uint32_t d = l[i].dim;
      const uint32_t q = l[i].sh >= 0 ? u >> l[i].sh : u / d;
      off += (int64_t)(u - q * d) * l[i].s0;
      u = q;
    }
    return off;
  }
  for (int i = 0; i < n; ++i) {
    const uint64_t d = l[i].dim;
    const uint64_t q = idx / d;
    off += (int64_t)(idx - q * d) * l[i].s0;
    idx = q;
  }
  return off;
}

// Offsets of an inner index in A and B.
__device__ __forceinline__ void net_off2(const NetLeg* l, int n, uint64_t idx,
                                         int64_t& oa, int64_t& ob) {
  oa = 0;
  ob = 0;
  if (idx <= 0xffffffffu) {
    uint32_t u = (uint32_t)idx;
    for (int i = 0; i < n; ++i) {
      const uint32_t d = l[i].dim;
      const uint32_t q = l[i].sh >= 0 ? u >> l[i].sh : u / d;
      const int64_t r = u - q * d;
      oa += r * l[i].s0;
      ob += r * l[i].s1;
      u = q;
    }
    return;
  }
  for (int i = 0; i < n; ++i) {
    const uint64_t d = l[i].dim;
    const uint64_t q = idx / d;
    const int64_t r = (int64_t)(idx - q * d);
    oa += r * l[i].s0;
    ob += r * l[i].s1;
    idx = q;
  }
}

typedef double d4_t __attribute__((ext_vector_type(4)));

constexpr int kElemK = 64;       // longest inner dimension of the elem kind
constexpr int kLongOut = 16;     // most entries of the long kind
constexpr int kTileK = 16;       // inner indices of a staged slice

// Shared memory of a block (the kinds use different parts of it).
struct NetShared {
  NetLeg leg[3 * kMaxLegs];
  union {
    struct {
      double a_re[kTileK][65], a_im[kTileK][65];
      double b_re[kTileK][65], b_im[kTileK][65];
      int64_t am[64], bn[64], ak[kTileK], bk[kTileK];
    } t;
    struct {
      int64_t ak[kElemK], bk[kElemK];
    } e;
    struct {
      int64_t am[kLongOut], bn[kLongOut];
      double2 part[4][kLongOut];
    } l;
  };
};

// kElem: C[m + n M] = sum_k A[am(m) + ak(k)] B[bk(k) + bn(n)], one thread
// per entry.
__device__ __forceinline__ void net_elem(const double2* __restrict__ dev,
                                         double2* __restrict__ C,
                                         const NetStep& st, uint32_t blk,
                                         NetShared& sh) {
  const int tid = threadIdx.x;
  const NetLeg* lk = sh.leg + st.n_am;
  const int K = (int)st.K;
  if (tid < K) {
    int64_t oa, ob;
    net_off2(lk, st.n_k, tid, oa, ob);
    sh.e.ak[tid] = oa;
    sh.e.bk[tid] = ob;
  }
  __syncthreads();
  const uint32_t o = blk * 256u + tid;
  const uint32_t M = (uint32_t)st.M;
  if (o >= (uint32_t)(st.M * st.N)) return;
  const uint32_t n = o / M, m = o - n * M;
  const double2* A = dev + st.a + net_off(sh.leg, st.n_am, m);
  const double2* B = dev + st.b + net_off(lk + st.n_k, st.n_bn, n);
  double re = 0.0, im = 0.0;
#pragma unroll 4
  for (int k = 0; k < K; ++k) {
    const double2 x = A[sh.e.ak[k]], y = B[sh.e.bk[k]];
    re = fma(x.x, y.x, re);
    re = fma(-x.y, y.y, re);
    im = fma(x.x, y.y, im);
    im = fma(x.y, y.x, im);
  }
  C[st.c + o] = make_double2(re, im);
}

// kTile: a (32 T) x (32 T) tile over kchunk inner indices, slices of 16,
// four waves of (16 T) x (16 T) on v_mfma_f64_16x16x4f64 (four real products
// per complex one).  The tile's row and column offsets and each slice's
// offsets are computed once into LDS; a_kfast / b_nfast pick the staging
// order that reads the operand's unit-stride leg along consecutive threads.
template <int T>
__device__ __forceinline__ void net_tile(const double2* __restrict__ dev,
                                         double2* __restrict__ Cb,
                                         const NetStep& st, uint32_t blk,
                                         NetShared& sh) {
  constexpr int BM = 32 * T, BK = kTileK;
  const double2* __restrict__ A = dev + st.a;
  const double2* __restrict__ B = dev + st.b;
  const NetLeg* lk = sh.leg + st.n_am;
  const NetLeg* ln = lk + st.n_k;
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const uint32_t tx = blk % st.nx, rest = blk / st.nx;
  const uint32_t ty = rest % st.ny, split = rest / st.ny;
  const int64_t M = st.M, N = st.N;
  const int64_t m0 = (int64_t)tx * BM, n0 = (int64_t)ty * BM;
  const int64_t kb = (int64_t)split * st.kchunk;
  const int64_t ke = min(st.K, kb + st.kchunk);
  double2* __restrict__ C = Cb + st.c + (int64_t)split * M * N;
  for (int i = tid; i < BM; i += 256) {
    sh.t.am[i] = m0 + i < M ? net_off(sh.leg, st.n_am, m0 + i) : 0;
    sh.t.bn[i] = n0 + i < N ? net_off(ln, st.n_bn, n0 + i) : 0;
  }
  const int wm = (wave & 1) * T * 16, wn = (wave >> 1) * T * 16;
  d4_t acc_re[T][T], acc_im[T][T];
#pragma unroll
  for (int i = 0; i < T; ++i)
#pragma unroll
    for (int j = 0; j < T; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        acc_re[i][j][e] = 0.0;
        acc_im[i][j][e] = 0.0;
      }
  for (int64_t k0 = kb; k0 < ke; k0 += BK) {
    __syncthreads();  // the previous slice's MFMA reads are done
    if (tid < BK) {
      int64_t oa = 0, ob = 0;
      if (k0 + tid < ke) net_off2(lk, st.n_k, k0 + tid, oa, ob);
      sh.t.ak[tid] = oa;
      sh.t.bk[tid] = ob;
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < BM * BK / 256; ++u) {
      const int idx = tid + 256 * u;
      const int i = st.a_kfast ? idx / BK : idx % BM;
      const int kk = st.a_kfast ? idx % BK : idx / BM;
      double2 v = make_double2(0.0, 0.0);
      if (m0 + i < M && k0 + kk < ke) v = A[sh.t.am[i] + sh.t.ak[kk]];
      sh.t.a_re[kk][i] = v.x;
      sh.t.a_im[kk][i] = v.y;
    }
#pragma unroll
    for (int u = 0; u < BM * BK / 256; ++u) {
      const int idx = tid + 256 * u;
      const int j = st.b_nfast ? idx % BM : idx / BK;
      const int kk = st.b_nfast ? idx / BM : idx % BK;
      double2 v = make_double2(0.0, 0.0);
      if (n0 + j < N && k0 + kk < ke) v = B[sh.t.bk[kk] + sh.t.bn[j]];
      sh.t.b_re[kk][j] = v.x;
      sh.t.b_im[kk][j] = v.y;
    }
    __syncthreads();
#pragma unroll
    for (int ks = 0; ks < BK; ks += 4) {
      const int kr = ks + (lane >> 4);
      double a_re[T], a_im[T], b_re[T], b_im[T];
#pragma unroll
      for (int i = 0; i < T; ++i) {
        a_re[i] = sh.t.a_re[kr][wm + i * 16 + (lane & 15)];
        a_im[i] = sh.t.a_im[kr][wm + i * 16 + (lane & 15)];
        b_re[i] = sh.t.b_re[kr][wn + i * 16 + (lane & 15)];
        b_im[i] = sh.t.b_im[kr][wn + i * 16 + (lane & 15)];
      }
#pragma unroll
      for (int i = 0; i < T; ++i)
#pragma unroll
        for (int j = 0; j < T; ++j) {
          acc_re[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(
              a_re[i], b_re[j], acc_re[i][j], 0, 0, 0);
          acc_re[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(
              -a_im[i], b_im[j], acc_re[i][j], 0, 0, 0);
          acc_im[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(
              a_re[i], b_im[j], acc_im[i][j], 0, 0, 0);
          acc_im[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(
              a_im[i], b_re[j], acc_im[i][j], 0, 0, 0);
        }
    }
  }
  // result element e of lane l: row 4 e + l / 16, column l % 16
#pragma unroll
  for (int i = 0; i < T; ++i)
#pragma unroll
    for (int j = 0; j < T; ++j) {
      const int64_t col = n0 + wn + j * 16 + (lane & 15);
      if (col >= N) continue;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int64_t row = m0 + wm + i * 16 + 4 * e + (lane >> 4);
        if (row < M)
          C[row + col * M] = make_double2(acc_re[i][j][e], acc_im[i][j][e]);
      }
    }
}

// kLong: the block's kchunk inner indices of all M N <= kLongOut entries,
// threads over the inner index, partial sums at C[blk M N + entry].
__device__ __forceinline__ void net_long(const double2* __restrict__ dev,
                                         double2* __restrict__ C,
                                         const NetStep& st, uint32_t blk,
                                         NetShared& sh) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const NetLeg* lk = sh.leg + st.n_am;
  const int M = (int)st.M, MN = (int)(st.M * st.N);
  if (tid < MN) {
    sh.l.am[tid] = net_off(sh.leg, st.n_am, tid % M);
    sh.l.bn[tid] = net_off(lk + st.n_k, st.n_bn, tid / M);
  }
  __syncthreads();
  double re[kLongOut], im[kLongOut];
#pragma unroll
  for (int o = 0; o < kLongOut; ++o) re[o] = im[o] = 0.0;
  const int64_t kb = (int64_t)blk * st.kchunk;
  const int64_t ke = min(st.K, kb + st.kchunk);
  for (int64_t k = kb + tid; k < ke; k += 256) {
    int64_t oa, ob;
    net_off2(lk, st.n_k, k, oa, ob);
    const double2* A = dev + st.a + oa;
    const double2* B = dev + st.b + ob;
#pragma unroll
    for (int o = 0; o < kLongOut; ++o) {
      if (o < MN) {
        const double2 x = A[sh.l.am[o]], y = B[sh.l.bn[o]];
        re[o] = fma(x.x, y.x, re[o]);
        re[o] = fma(-x.y, y.y, re[o]);
        im[o] = fma(x.x, y.y, im[o]);
        im[o] = fma(x.y, y.x, im[o]);
      }
    }
  }
#pragma unroll
  for (int o = 0; o < kLongOut; ++o) {
    if (o < MN) {
      for (int w = 32; w > 0; w >>= 1) {
        re[o] += __shfl_xor(re[o], w, 64);
        im[o] += __shfl_xor(im[o], w, 64);
      }
      if (lane == 0) sh.l.part[wave][o] = make_double2(re[o], im[o]);
    }
  }
  __syncthreads();
  if (tid < MN) {
    double2 v = sh.l.part[0][tid];
    for (int w = 1; w < 4; ++w) {
      v.x += sh.l.part[w][tid].x;
      v.y += sh.l.part[w][tid].y;
    }
    C[st.c + (int64_t)blk * MN + tid] = v;
  }
}

// kReduce: C[o] = sum_s P[s M N + o].  Up to kLongOut entries: a block per
// entry, threads over the partials; more: a thread per entry.
__device__ __forceinline__ void net_reduce(const double2* __restrict__ dev,
                                           double2* __restrict__ C,
                                           const NetStep& st, uint32_t blk,
                                           NetShared& sh) {
  const int tid = threadIdx.x;
  const int64_t MN = st.M * st.N;
  double2 v = make_double2(0.0, 0.0);
  if (MN > kLongOut) {
    const int64_t o = (int64_t)blk * 256 + tid;
    if (o >= MN) return;
    for (int s = 0; s < st.nsplit; ++s) {
      const double2 x = dev[st.a + s * MN + o];
      v.x += x.x;
      v.y += x.y;
    }
    C[st.c + o] = v;
    return;
  }
  for (int s = tid; s < st.nsplit; s += 256) {
    const double2 x = dev[st.a + s * MN + blk];
    v.x += x.x;
    v.y += x.y;
  }
  for (int w = 32; w > 0; w >>= 1) {
    v.x += __shfl_xor(v.x, w, 64);
    v.y += __shfl_xor(v.y, w, 64);
  }
  if ((tid & 63) == 0) sh.l.part[tid >> 6][0] = v;
  __syncthreads();
  if (tid == 0) {
    for (int w = 1; w < 4; ++w) {
      v.x += sh.l.part[w][0].x;
      v.y += sh.l.part[w][0].y;
    }
    C[st.c + blk] = v;
  }
}

// All steps of one level.  A small network is bound by its chain of
// dependent launches, so independent steps share one (the 20-qubit QFT
// network in its treewidth order, 249 steps in 26 levels: 7.26 ms -> 1.99 ms
// per contract(); the 17-qubit one in the default order, a chain of 170
// steps closed by a 1 x 1 x 131072 product: 40.4 ms -> 2.01 ms).  dev is the
// arena (the operands of a level and its results are disjoint), steps its
// nsteps descriptors with ascending first blocks, pool the legs; this launch
// takes the level's blocks from base on.  kHeavy: the level holds tile or
// long steps, whose accumulators allow two waves per SIMD; the levels without
// them take the lighter instance.
template <bool kHeavy>
__global__ __launch_bounds__(256) void net_level(
    const double2* __restrict__ dev, double2* __restrict__ out,
    const NetStep* __restrict__ steps, int nsteps,
    const NetLeg* __restrict__ pool, uint32_t base) {
  __shared__ NetShared sh;
  __shared__ int s_at;
  const int tid = threadIdx.x;
  const uint32_t bid = base + blockIdx.x;
  int at = 0;
  if (nsteps > 1) {
    // the last step whose first block is not after this one
    if (tid == 0) s_at = 0;
    __syncthreads();
    for (int i = tid; i < nsteps; i += 256)
      if (steps[i].first <= bid &&
          (i + 1 == nsteps || steps[i + 1].first > bid))
        s_at = i;
    __syncthreads();
    at = __builtin_amdgcn_readfirstlane(s_at);
  }
  const NetStep st = steps[at];
  const uint32_t blk = bid - st.first;
  const int nl = st.n_am + st.n_k + st.n_bn;
  if (tid < nl) sh.leg[tid] = pool[st.legs + tid];
  __syncthreads();
  switch (st.kind) {
    case kElem:
      net_elem(dev, out, st, blk, sh);
      break;
    case kTile:
      if constexpr (kHeavy) {
        if (st.tile == 64)
          net_tile<2>(dev, out, st, blk, sh);
        else
          net_tile<1>(dev, out, st, blk, sh);
      }
      break;
    case kLong:
      if constexpr (kHeavy) net_long(dev, out, st, blk, sh);
      break;
    case kReduce:
      net_reduce(dev, out, st, blk, sh);
      break;
    case kIdent: {
      // d x d identity (a trace is a contraction with it), d = M
      const int64_t i = (int64_t)blk * 256 + tid;
      if (i < st.M * st.M)
        out[st.c + i] =
            make_double2((i % st.M) == (i / st.M) ? 1.0 : 0.0, 0.0);
      break;
    }
    default: {  // kGather: out[o] = in[am(o)] (the final leg order)
      const int64_t o = (int64_t)blk * 256 + tid;
      if (o < st.M) out[st.c + o] = dev[st.a + net_off(sh.leg, st.n_am, o)];
    }
  }
}

struct Item {
  std::vector<int64_t> labels, dims;
  int64_t off = 0, size = 1;  // in elements
  int level = 0;              // level after which it exists (inputs: 0)
};

std::vector<int64_t> col_strides(const std::vector<int64_t>& dims) {
  std::vector<int64_t> s(dims.size());
  int64_t acc = 1;
  for (size_t i = 0; i < dims.size(); ++i) {
    s[i] = acc;
    acc *= dims[i];
  }
  return s;
}

int32_t log2_or(int64_t d) {
  return (d & (d - 1)) ? -1 : (int32_t)__builtin_ctzll((uint64_t)d);
}

// Legs (dims, strides in one tensor or two) -> the pool, merging neighbours
// that are contiguous in memory (in both).  False when more than kMaxLegs
// groups remain or a group is too long.
bool add_legs(const std::vector<int64_t>& dims, const std::vector<int64_t>& sa,
              const std::vector<int64_t>& sb, std::vector<NetLeg>* pool,
              int32_t* n) {
  std::vector<int64_t> d, ta, tb;
  for (size_t i = 0; i < dims.size(); ++i) {
    if (dims[i] == 1) continue;
    if (!d.empty() && ta.back() * d.back() == sa[i] &&
        tb.back() * d.back() == sb[i]) {
      d.back() *= dims[i];
    } else {
      d.push_back(dims[i]);
      ta.push_back(sa[i]);
      tb.push_back(sb[i]);
    }
  }
  if ((int)d.size() > kMaxLegs) return false;
  for (size_t i = 0; i < d.size(); ++i) {
    if (d[i] > INT32_MAX) return false;
    pool->push_back({(uint32_t)d[i], log2_or(d[i]), ta[i], tb[i]});
  }
  *n = (int32_t)d.size();
  return true;
}

// First-fit placement in an arena of elements (offsets 16-aligned).
struct Arena {
  std::map<int64_t, int64_t> used;  // offset -> size
  int64_t peak = 0;
  int64_t alloc(int64_t size) {
    const int64_t sz = std::max<int64_t>(16, (size + 15) / 16 * 16);
    int64_t at = 0;
    for (const auto& u : used) {
      if (u.first - at >= sz) break;
      at = std::max(at, u.first + (u.second + 15) / 16 * 16);
    }
    used[at] = sz;
    peak = std::max(peak, at + sz);
    return at;
  }
  void release(int64_t off) { used.erase(off); }
};

// One step of the planned execution (offsets filled once the arena is
// placed): `item` operands and result, its place in the tree.
struct Step {
  NetStep d;
  int a = -1, b = -1, out = -1, level = 0;
};

int64_t prod(const std::vector<int64_t>& v) {
  int64_t p = 1;
  for (int64_t x : v) p *= x;
  return p;
}

// Block kind and launch shape of a pairwise step.
//   long: at most 16 entries over 512 or more inner indices.  One tile
//     would walk them in slices of 16, 0.42 us each (the closing 1 x 1 x
//     131072 product of the 17-qubit default-order network took 34 ms).
//   elem: short inner dimensions, where the product is bound by its
//     operands and result (K < 8, or thin with K < 16) or too small to
//     fill the chip with tiles (M N K <= 2^22 and K <= 64).
//   tile: everything else; 64 x 64 tiles once they give 256 workgroups,
//     else 32 x 32.  From K = 512 on, a step of fewer than 512 tiles splits
//     its inner dimension (128 indices or more per block, at most 64 MiB of
//     partial products).
void choose_kind(NetStep& d) {
  const int64_t M = d.M, N = d.N, K = d.K, thin = std::min(M, N);
  d.nsplit = 1;
  d.kchunk = K;
  d.nx = d.ny = 1;
  d.tile = 0;
  const bool idx32 = M <= INT32_MAX && N <= INT32_MAX && M * N <= INT32_MAX;
  if (idx32 && M * N <= kLongOut && K >= 512) {
    d.kind = kLong;
    // 1024 inner indices per block, at most 1024 blocks
    d.kchunk = std::max<int64_t>(1024, ((K + 1023) / 1024 + 255) / 256 * 256);
    d.nsplit = (int32_t)((K + d.kchunk - 1) / d.kchunk);
    return;
  }
  if (idx32 && K <= kElemK &&
      (K < 8 || (thin < 32 && K < 16) || M * N * K <= (1 << 22))) {
    d.kind = kElem;
    return;
  }
  d.kind = kTile;
  const int64_t big = ((M + 63) / 64) * ((N + 63) / 64);
  d.tile = big >= 256 ? 64 : 32;
  d.nx = (uint32_t)((M + d.tile - 1) / d.tile);
  d.ny = (uint32_t)((N + d.tile - 1) / d.tile);
  const int64_t tiles = (int64_t)d.nx * d.ny;
  if (K >= 512 && tiles < 512) {
    const int64_t ns = std::min<int64_t>(
        {512 / tiles, K / 128, (int64_t)(1 << 22) / (M * N), 64});
    if (ns >= 2) {
      d.kchunk = ((K + ns - 1) / ns + kTileK - 1) / kTileK * kTileK;
      d.nsplit = (int32_t)((K + d.kchunk - 1) / d.kchunk);
    }
  }
}

// Blocks of a step.
int64_t step_blocks(const NetStep& d) {
  switch (d.kind) {
    case kElem:
      return (d.M * d.N + 255) / 256;
    case kTile:
      return (int64_t)d.nx * d.ny * d.nsplit;
    case kLong:
      return d.nsplit;
    case kReduce:
      return d.M * d.N > kLongOut ? (d.M * d.N + 255) / 256 : d.M * d.N;
    case kIdent:
      return (d.M * d.M + 255) / 256;
    default:
      return (d.M + 255) / 256;
  }
}

// Places the results of every step level by level: a level's results are
// placed before its operands are released.  by_level[l] lists the steps of
// level l + 1.  Returns the arena's peak.
int64_t place(Arena arena, const std::vector<std::vector<int>>& by_level,
              const std::vector<Step>& steps, std::vector<Item>* items) {
  for (const auto& lev : by_level) {
    for (int i : lev)
      (*items)[steps[i].out].off = arena.alloc((*items)[steps[i].out].size);
    for (int i : lev) {
      if (steps[i].a >= 0) arena.release((*items)[steps[i].a].off);
      if (steps[i].b >= 0) arena.release((*items)[steps[i].b].off);
    }
  }
  return arena.peak;
}

}  // namespace
}  // namespace qtn

using namespace qtn;

extern "C" {

int32_t qtn_contract_network(qtn_ctx* ctx, int32_t ntensors,
                             const int32_t* ndims, const int64_t* dims,
                             const int32_t* labels,
                             const double* const* tensors, int32_t norder,
                             const int32_t* order, double* out,
                             int64_t out_len) try {
  clear_error();
  QTN_ARG(ctx && ntensors >= 1 && ndims && tensors && out,
          "qtn_contract_network: NULL argument or no tensors");
  QTN_ARG(norder >= 0 && (norder == 0 || order),
          "qtn_contract_network: bad contraction order");
  // ---- read the network
  std::vector<Item> items(ntensors);
  std::map<int64_t, int> count;
  std::map<int64_t, int64_t> ldim;
  int64_t pos = 0;
  for (int t = 0; t < ntensors; ++t) {
    QTN_ARG(ndims[t] >= 0, "qtn_contract_network: negative rank");
    QTN_ARG(tensors[t], "qtn_contract_network: NULL tensor");
    for (int l = 0; l < ndims[t]; ++l, ++pos) {
      const int64_t lab = labels[pos], d = dims[pos];
      QTN_ARG(lab != 0, "qtn_contract_network: label 0 is not allowed");
      QTN_ARG(d >= 1, "qtn_contract_network: leg dimensions must be >= 1");
      items[t].labels.push_back(lab);
      items[t].dims.push_back(d);
      count[lab] += 1;
      if (ldim.count(lab))
        QTN_ARG(ldim[lab] == d,
                "Dimensions of contraction legs do not match");
      ldim[lab] = d;
    }
    items[t].size = prod(items[t].dims);
  }
  std::vector<int64_t> open;
  for (const auto& kv : count) {
    if (kv.first > 0)
      QTN_ARG(kv.second == 2, "qtn_contract_network: a positive label must "
                              "appear exactly twice");
    else {
      QTN_ARG(kv.second == 1, "qtn_contract_network: a negative label must "
                              "appear once");
      open.push_back(kv.first);
    }
  }
  {
    std::vector<int64_t> o(order, order + norder), p;
    for (const auto& kv : count)
      if (kv.first > 0) p.push_back(kv.first);
    std::sort(o.begin(), o.end());
    QTN_ARG(o == p, "qtn_contract_network: the order must list every "
                    "positive label once");
  }
  // ncon's output order: -1, -2, ...
  std::sort(open.begin(), open.end(), std::greater<int64_t>());
  int64_t out_size = 1;
  for (int64_t lab : open) out_size *= ldim[lab];
  QTN_ARG(out_len == out_size,
          "qtn_contract_network: out_len differs from the result's size");

  // ---- plan: steps, their levels and arena placement (host only)
  Arena arena;
  std::vector<int> alive;
  int64_t in_total = 0;
  for (int t = 0; t < ntensors; ++t) {
    items[t].off = arena.alloc(items[t].size);
    in_total = std::max(in_total, items[t].off + items[t].size);
    alive.push_back(t);
  }
  std::vector<Step> steps;
  std::vector<NetLeg> pool;
  int64_t next_label = 1;
  for (const auto& kv : count) next_label = std::max(next_label, kv.first + 1);
  auto pair_step = [&](int ia, int ib) -> int32_t {
    Item &A = items[ia], &B = items[ib];
    std::vector<int64_t> shared;
    for (int64_t x : A.labels)
      if (x > 0 &&
          std::find(B.labels.begin(), B.labels.end(), x) != B.labels.end())
        shared.push_back(x);
    const std::vector<int64_t> sA = col_strides(A.dims),
                               sB = col_strides(B.dims);
    // inner legs follow the larger operand's leg order
    if (B.size > A.size) {
      std::vector<int64_t> sh;
      for (int64_t x : B.labels)
        if (std::find(shared.begin(), shared.end(), x) != shared.end())
          sh.push_back(x);
      shared = sh;
    }
    Item C;
    std::vector<int64_t> dm, sm, dn, sn, dk, ska, skb;
    for (size_t i = 0; i < A.labels.size(); ++i)
      if (std::find(shared.begin(), shared.end(), A.labels[i]) ==
          shared.end()) {
        C.labels.push_back(A.labels[i]);
        C.dims.push_back(A.dims[i]);
        dm.push_back(A.dims[i]);
        sm.push_back(sA[i]);
      }
    for (size_t i = 0; i < B.labels.size(); ++i)
      if (std::find(shared.begin(), shared.end(), B.labels[i]) ==
          shared.end()) {
        C.labels.push_back(B.labels[i]);
        C.dims.push_back(B.dims[i]);
        dn.push_back(B.dims[i]);
        sn.push_back(sB[i]);
      }
    for (int64_t x : shared) {
      const size_t ia_ = std::find(A.labels.begin(), A.labels.end(), x) -
                         A.labels.begin();
      const size_t ib_ = std::find(B.labels.begin(), B.labels.end(), x) -
                         B.labels.begin();
      dk.push_back(A.dims[ia_]);
      ska.push_back(sA[ia_]);
      skb.push_back(sB[ib_]);
    }
    Step st;
    std::memset(&st.d, 0, sizeof(st.d));
    st.a = ia;
    st.b = ib;
    NetStep& d = st.d;
    d.M = prod(dm);
    d.N = prod(dn);
    d.K = prod(dk);
    d.legs = (int32_t)pool.size();
    if (!add_legs(dm, sm, sm, &pool, &d.n_am) ||
        !add_legs(dk, ska, skb, &pool, &d.n_k) ||
        !add_legs(dn, sn, sn, &pool, &d.n_bn)) {
      set_error("qtn_contract_network: a step has more than 24 leg groups");
      return QTN_ERR_ARG;
    }
    QTN_ARG((d.N + 63) / 64 <= 65535 && (d.M + 63) / 64 <= INT32_MAX,
            "qtn_contract_network: a step is too large for the launch grid");
    // stage along the operand's unit-stride leg where it is in the group
    d.a_kfast = (d.n_k > 0 && pool[d.legs + d.n_am].s0 == 1) ? 1 : 0;
    d.b_nfast =
        (d.n_bn > 0 && pool[d.legs + d.n_am + d.n_k].s0 == 1) ? 1 : 0;
    choose_kind(d);
    st.level = std::max(A.level, B.level) + 1;
    C.size = d.M * d.N;
    C.level = st.level;
    if (d.nsplit > 1) {
      // partial products, then their sum one level on
      Item P;
      P.size = C.size * d.nsplit;
      P.level = st.level;
      items.push_back(P);
      st.out = (int)items.size() - 1;
      steps.push_back(st);
      Step rd;
      rd.d = d;
      rd.d.kind = kReduce;
      rd.d.n_am = rd.d.n_k = rd.d.n_bn = 0;
      rd.a = st.out;
      rd.level = st.level + 1;
      C.level = rd.level;
      items.push_back(C);
      rd.out = (int)items.size() - 1;
      steps.push_back(rd);
    } else {
      items.push_back(C);
      st.out = (int)items.size() - 1;
      steps.push_back(st);
    }
    alive.erase(std::find(alive.begin(), alive.end(), ia));
    alive.erase(std::find(alive.begin(), alive.end(), ib));
    alive.push_back((int)items.size() - 1);
    return QTN_OK;
  };
  std::map<int64_t, bool> done;
  for (int q = 0; q < norder; ++q) {
    const int64_t lab = order[q];
    if (done[lab]) continue;
    std::vector<int> holders;
    for (int t : alive)
      if (std::find(items[t].labels.begin(), items[t].labels.end(), lab) !=
          items[t].labels.end())
        holders.push_back(t);
    if (holders.size() == 1) {
      // a trace: the second leg takes a fresh label and the tensor meets
      // the identity on both
      Item& A = items[holders[0]];
      auto it = std::find(A.labels.begin(), A.labels.end(), lab);
      it = std::find(it + 1, A.labels.end(), lab);
      const int64_t fresh = next_label++;
      *it = fresh;
      Item I;
      I.labels = {lab, fresh};
      I.dims = {ldim[lab], ldim[lab]};
      I.size = ldim[lab] * ldim[lab];
      I.level = 1;
      items.push_back(I);
      Step f;
      std::memset(&f.d, 0, sizeof(f.d));
      f.d.kind = kIdent;
      f.d.M = ldim[lab];
      f.level = 1;
      f.out = (int)items.size() - 1;
      steps.push_back(f);
      alive.push_back(f.out);
      holders.push_back(f.out);
      done[fresh] = true;
    }
    QTN_ARG(holders.size() == 2, "qtn_contract_network: inconsistent labels");
    for (int64_t x : items[holders[0]].labels)
      if (x > 0 && std::find(items[holders[1]].labels.begin(),
                             items[holders[1]].labels.end(),
                             x) != items[holders[1]].labels.end())
        done[x] = true;
    QTN_TRY(pair_step(holders[0], holders[1]));
  }
  while (alive.size() > 1) QTN_TRY(pair_step(alive[0], alive[1]));
  // final gather into ncon's leg order
  {
    const Item& R = items[alive[0]];
    const std::vector<int64_t> sR = col_strides(R.dims);
    std::vector<int64_t> d, st;
    for (int64_t lab : open) {
      const size_t i =
          std::find(R.labels.begin(), R.labels.end(), lab) - R.labels.begin();
      d.push_back(R.dims[i]);
      st.push_back(sR[i]);
    }
    Step g;
    std::memset(&g.d, 0, sizeof(g.d));
    g.d.kind = kGather;
    g.d.M = out_size;
    g.d.legs = (int32_t)pool.size();
    QTN_ARG(add_legs(d, st, st, &pool, &g.d.n_am),
            "qtn_contract_network: the result has more than 24 leg groups");
    g.a = alive[0];
    g.level = R.level + 1;
    Item O;
    O.size = out_size;
    O.level = g.level;
    items.push_back(O);
    g.out = (int)items.size() - 1;
    steps.push_back(g);
  }
  // the descriptors and legs travel behind the inputs in the same copy and
  // stay for the whole run
  const int64_t step_el =
      (int64_t)((steps.size() * sizeof(NetStep) + 15) / 16);
  const int64_t leg_el = (int64_t)((pool.size() * sizeof(NetLeg) + 15) / 16);
  const int64_t desc_off = arena.alloc(step_el + leg_el);
  in_total = std::max(in_total, desc_off + step_el + leg_el);
  // Steps of one depth run together (the 20-qubit QFT network in its
  // treewidth order: 26 launches instead of 249) unless keeping all their
  // results at once would take more than the caller's order does and more
  // than 64 MiB; then one step runs after the other in that order.
  std::vector<std::vector<int>> seq, lev;
  for (size_t i = 0; i < steps.size(); ++i) {
    seq.push_back({(int)i});
    if ((size_t)steps[i].level > lev.size()) lev.resize(steps[i].level);
    lev[steps[i].level - 1].push_back((int)i);
  }
  std::vector<Item> placed = items;
  const int64_t seq_peak = place(arena, seq, steps, &placed);
  int64_t peak = place(arena, lev, steps, &items);
  if (peak > std::max<int64_t>(seq_peak, 1 << 22)) {
    peak = seq_peak;
    items = placed;
    lev = seq;
  }

  // ---- run
  QTN_CHECK_HIP(hipSetDevice(ctx->device));
  hipStream_t s = ctx->stream;
  void* base;
  QTN_TRY(ctx->buffer(kSlotArena, (size_t)peak * sizeof(double2), &base));
  double2* dev = (double2*)base;
  // inputs and descriptors through one pinned staging copy
  void* pin = nullptr;
  QTN_TRY(ctx->pinned_buffer((size_t)in_total * sizeof(double2), &pin));
  for (int t = 0; t < ntensors; ++t)
    std::memcpy((double2*)pin + items[t].off, tensors[t],
                (size_t)items[t].size * sizeof(double2));
  NetStep* hs = (NetStep*)((double2*)pin + desc_off);
  std::vector<uint32_t> blocks;
  for (const auto& l : lev) {
    int64_t nb = 0;
    for (int i : l) {
      NetStep d = steps[i].d;
      d.a = steps[i].a >= 0 ? items[steps[i].a].off : 0;
      d.b = steps[i].b >= 0 ? items[steps[i].b].off : 0;
      d.c = items[steps[i].out].off;
      d.first = (uint32_t)nb;
      *hs++ = d;
      nb += step_blocks(d);
      QTN_ARG(nb <= INT32_MAX, "qtn_contract_network: a step is too large "
                               "for the launch grid");
    }
    blocks.push_back((uint32_t)nb);
  }
  if (!pool.empty())
    std::memcpy((double2*)pin + desc_off + step_el, pool.data(),
                pool.size() * sizeof(NetLeg));
  QTN_CHECK_HIP(hipMemcpyAsync(dev, pin, (size_t)in_total * sizeof(double2),
                               hipMemcpyHostToDevice, s));
  const NetStep* ds = (const NetStep*)(dev + desc_off);
  const NetLeg* dl = (const NetLeg*)(dev + desc_off + step_el);
  for (size_t l = 0; l < lev.size(); ++l) {
    const int ns = (int)lev[l].size();
    bool heavy = false;
    for (int i : lev[l])
      heavy = heavy || steps[i].d.kind == kTile || steps[i].d.kind == kLong;
    // a grid holds fewer than 2^32 threads
    constexpr uint32_t kMost = 1u << 23;
    for (uint32_t at = 0; at < blocks[l]; at += kMost)
      hipLaunchKernelGGL(heavy ? net_level<true> : net_level<false>,
                         dim3(std::min(blocks[l] - at, kMost)), dim3(256), 0,
                         s, (const double2*)dev, dev, ds, ns, dl, at);
    ds += ns;
  }
  QTN_CHECK_HIP(hipGetLastError());
  QTN_CHECK_HIP(hipMemcpyAsync(out, dev + items[steps.back().out].off,
                               (size_t)out_size * sizeof(double2),
                               hipMemcpyDeviceToHost, s));
  QTN_CHECK_HIP(hipStreamSynchronize(s));
  return QTN_OK;
} catch (...) {
  return qtn::abi_exception();
}

}  // extern "C"
