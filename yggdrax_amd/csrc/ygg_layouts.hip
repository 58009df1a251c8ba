// Downstream layouts of the far-field lists, the formats M2L kernels consume:
//  * dense level-major buffers (yggdrax/dense_interactions.py:35-140): for
//    slot (level, j) the target node nodes_by_level[level_offsets[level] + j],
//    its far sources padded to the longest list, the validity mask, the count
//    and the target-minus-source centre displacements;
//  * displacement classes (yggdrax/grouped_interactions.py:74-207): far pairs
//    keyed by (target level, source level, rint(delta / cell) per axis),
//    ordered lexicographically by key and, inside a class, by input position,
//    with CSR class offsets and the class of every input pair.
#include "ygg_common.h"

namespace ygg {
namespace {

// A CSR row reaching outside the num_far sources, or a source outside
// [0, num_nodes), is written as padding and raises *err (checked by the
// caller after the launch).
// Elements of the [num_levels][max_nodes][K] buffers, four consecutive ones
// per thread and 1024 per workgroup and step: a workgroup divides once, its
// threads step on from there, and with aligned buffers (VEC) whole spans go
// out as 16-byte stores over contiguous runs, past the caches (nothing here
// reads them again). Bound by the writes, 21 bytes per element: 2.16 GB (2^18
// Plummer points, leaf 32) in 360 us, 6.0 TB/s where a plain fill reaches
// 6.9; 491 us with one element per thread (two 64-bit divisions each), 469 us
// with four per thread and stores of a thread's own, 565 us through LDS with
// cached stores.
constexpr int kDensePer = 4, kDenseThreads = 256, kDenseSpan = kDensePer * kDenseThreads;

template <typename IdxT, bool VEC>
__global__ __launch_bounds__(kDenseThreads) void k_dense_m2l(
    const IdxT* __restrict__ offsets, const IdxT* __restrict__ counts,
    const IdxT* __restrict__ sources, int64_t num_nodes, int64_t num_far,
    const int32_t* __restrict__ nbl, const int32_t* __restrict__ loff, int num_levels,
    int64_t max_nodes, int64_t K, const float* __restrict__ center, IdxT* __restrict__ out_src,
    float* __restrict__ out_disp, uint8_t* __restrict__ out_mask, IdxT* __restrict__ out_counts,
    int32_t* __restrict__ err) {
  __shared__ __align__(16) IdxT s_src[VEC ? kDenseSpan : 1];
  __shared__ __align__(16) float s_disp[VEC ? 3 * kDenseSpan : 1];
  const int64_t total = (int64_t)num_levels * max_nodes * K;
  for (int64_t base = (int64_t)blockIdx.x * kDenseSpan; base < total;
       base += (int64_t)gridDim.x * kDenseSpan) {
    // uniform: the span's first slot, its level and place in it
    const int64_t slot0 = base / K;
    const int64_t l0 = slot0 / max_nodes;
    const int64_t e0 = base + (int64_t)threadIdx.x * kDensePer;
    if (e0 >= total) continue;
    int64_t j = base - slot0 * K + (int64_t)threadIdx.x * kDensePer;
    int64_t slot = slot0;
    if (K >= kDenseSpan) {
      if (j >= K) {  // at most one slot ends inside the span
        j -= K;
        ++slot;
      }
    } else {
      const uint32_t q = (uint32_t)j / (uint32_t)K;
      slot += q;
      j -= (int64_t)q * K;
    }
    int64_t s = slot - l0 * max_nodes;
    int l = (int)l0;
    int64_t node = -1, cnt = 0, off = 0;
    float tc[3] = {0.0f, 0.0f, 0.0f};
    bool bad = false;
    auto enter_slot = [&]() {
      while (s >= max_nodes) {
        s -= max_nodes;
        ++l;
      }
      const int64_t lc = (int64_t)loff[l + 1] - loff[l];
      node = s < lc ? (int64_t)nbl[loff[l] + s] : -1;
      cnt = node >= 0 ? (int64_t)counts[node] : 0;
      if (cnt < 0) {
        bad = true;
        cnt = 0;
      }
      if (j < cnt) {
        off = (int64_t)offsets[node];
#pragma unroll
        for (int d = 0; d < 3; ++d) tc[d] = center[3 * node + d];
      }
    };
    enter_slot();
    IdxT src[kDensePer];
    float disp[3 * kDensePer];
    uint32_t mask = 0;
    const int64_t left = total - e0;
#pragma unroll
    for (int k = 0; k < kDensePer; ++k) {
      src[k] = (IdxT)-1;
      disp[3 * k] = disp[3 * k + 1] = disp[3 * k + 2] = 0.0f;
      if (k < left) {
        if (j == K) {
          j = 0;
          ++slot;
          ++s;
          enter_slot();
        }
        if (j < cnt) {
          const int64_t at = off + j;
          int64_t v = -1;
          if (at >= 0 && at < num_far) v = (int64_t)sources[at];
          if (v < 0 || v >= num_nodes) {
            bad = true;
          } else {
            src[k] = (IdxT)v;
            mask |= 1u << (8 * k);
#pragma unroll
            for (int d = 0; d < 3; ++d) disp[3 * k + d] = tc[d] - center[3 * v + d];
          }
        }
        if (j == 0) out_counts[slot] = (IdxT)cnt;
        ++j;
      }
    }
    if (bad) *err = 1;
    if (VEC && base + kDenseSpan <= total) {
      // uniform: a whole span; sources and displacements change hands in LDS
      // so that each wide store of a wavefront covers one run of memory
      *(uint32_t*)(out_mask + e0) = mask;
      const bool any = __syncthreads_or((int)mask);
      if (any) {
#pragma unroll
        for (int k = 0; k < kDensePer; ++k) {
          s_src[threadIdx.x * kDensePer + k] = src[k];
#pragma unroll
          for (int d = 0; d < 3; ++d)
            s_disp[(threadIdx.x * kDensePer + k) * 3 + d] = disp[3 * k + d];
        }
        __syncthreads();
      }
      constexpr int kSrcWords = kDenseSpan * (int)sizeof(IdxT) / 16, kDispWords = kDenseSpan * 12 / 16;
      typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
      const u32x4 ones = {~0u, ~0u, ~0u, ~0u}, zeros = {0u, 0u, 0u, 0u};
#pragma unroll
      for (int k = 0; k < kSrcWords / kDenseThreads; ++k) {
        const int i = k * kDenseThreads + (int)threadIdx.x;
        __builtin_nontemporal_store(any ? ((const u32x4*)s_src)[i] : ones,
                                    &((u32x4*)(out_src + base))[i]);
      }
#pragma unroll
      for (int k = 0; k < kDispWords / kDenseThreads; ++k) {
        const int i = k * kDenseThreads + (int)threadIdx.x;
        __builtin_nontemporal_store(any ? ((const u32x4*)s_disp)[i] : zeros,
                                    &((u32x4*)(out_disp + 3 * base))[i]);
      }
      if (any) __syncthreads();  // before the next span's values
    } else {
#pragma unroll
      for (int k = 0; k < kDensePer; ++k) {
        if (k >= left) break;
        out_src[e0 + k] = src[k];
        out_mask[e0 + k] = (uint8_t)(mask >> (8 * k));
#pragma unroll
        for (int d = 0; d < 3; ++d) out_disp[3 * (e0 + k) + d] = disp[3 * k + d];
      }
    }
  }
}

// numpy's float64 -> int32 cast on x86-64 (cvttsd2si): values outside the
// int32 range, and NaN, become INT32_MIN. The argument is already integral.
__device__ __forceinline__ int32_t to_i32_like_numpy(double r) {
  return (r >= -2147483648.0 && r <= 2147483647.0) ? (int32_t)r : INT32_MIN;
}

// Per-axis cell size of a level: max(extent / max(2^level, 1), 1e-12)
// (grouped_interactions.py:34-38); the division by 2^level is exact where the
// quotient is not below 1e-12, so it is a change of exponent.
__device__ __forceinline__ double cell_size(double extent, int level) {
  return fmax(ldexp(extent, -max(level, 0)), 1e-12);
}

struct GroupGeom {
  int64_t num_nodes;     // T
  const int32_t* level;  // node_level [T]
  const float* center;   // [T, 3]
  const float* bmin;     // [3]
  const float* bmax;     // [3]
  const float4* node;    // [T] centre and level, or null
};

// Key fields of pair i: target level, source level and the rounded
// displacement in target-level cells (grouped_interactions.py:139-165).
// Arithmetic is float64 as in the reference's NumPy code: the centre
// difference, the IEEE division and the round-half-even are all exact
// restatements, so the key is bit-identical.
struct GroupNode {
  float c[3];
  int32_t level;
};

__device__ __forceinline__ GroupNode group_node(const GroupGeom& g, int64_t v) {
  if (g.node) {
    const float4 r = g.node[v];
    return GroupNode{{r.x, r.y, r.z}, __float_as_int(r.w)};
  }
  return GroupNode{{g.center[3 * v], g.center[3 * v + 1], g.center[3 * v + 2]}, g.level[v]};
}

__device__ __forceinline__ void group_fields(const GroupNode& t, const GroupNode& s,
                                             const GroupGeom& g, int32_t f[5]) {
  f[0] = t.level;
  f[1] = s.level;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const double ext = (double)g.bmax[a] - (double)g.bmin[a];
    const double delta = (double)t.c[a] - (double)s.c[a];
    f[2 + a] = to_i32_like_numpy(rint(delta / cell_size(ext, t.level)));
  }
}

// Centre and level side by side: a pair's nodes come in two cache lines instead
// of four, which is what bounds the two kernels over the pairs. 2.1e7 pairs: 211 and 258 us, 256 and 310 us
// without.
__global__ void k_group_nodes(GroupGeom g, float4* __restrict__ out) {
  for (int64_t v = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; v < g.num_nodes;
       v += (int64_t)gridDim.x * blockDim.x)
    out[v] = make_float4(g.center[3 * v], g.center[3 * v + 1], g.center[3 * v + 2],
                         __int_as_float(g.level[v]));
}

// Pairs per thread and step of the two kernels over the pairs: all their node
// ids, then all their nodes are on the way before the first is used.
constexpr int kGroupPer = 4;

// Field-wise min (partials[b][0..4]) and max ([5..9]) of block b's pairs:
// wavefront shuffles, then one LDS row per wavefront. No atomics, so the
// reduction costs no cross-XCD traffic. The nodes' gathers bound it (2.1e7
// pairs: 211 us for 0.33 GB of node ids).
constexpr int kMinmaxBlocks = 2048;

// Pairs naming a node outside [0, T) are skipped and raise *err; the
// classify call then fails before any kernel reads through them.
template <typename IdxT>
__global__ void __launch_bounds__(256)
k_group_minmax(const IdxT* __restrict__ src, const IdxT* __restrict__ tgt, int64_t n,
               GroupGeom g, int32_t* __restrict__ partials, int32_t* __restrict__ err) {
  __shared__ int32_t red[256 / YGG_WAVE][10];
  int32_t lo[5], hi[5];
#pragma unroll
  for (int k = 0; k < 5; ++k) {
    lo[k] = INT32_MAX;
    hi[k] = INT32_MIN;
  }
  const int64_t step = (int64_t)gridDim.x * blockDim.x * kGroupPer;
  for (int64_t b = blockIdx.x * (int64_t)blockDim.x * kGroupPer + threadIdx.x; b < n; b += step) {
    int64_t t[kGroupPer], s[kGroupPer];
    bool ok[kGroupPer];
#pragma unroll
    for (int q = 0; q < kGroupPer; ++q) {
      const int64_t i = b + (int64_t)q * blockDim.x;
      ok[q] = i < n;
      t[q] = ok[q] ? (int64_t)tgt[i] : 0;
      s[q] = ok[q] ? (int64_t)src[i] : 0;
    }
    GroupNode tn[kGroupPer], sn[kGroupPer];
#pragma unroll
    for (int q = 0; q < kGroupPer; ++q) {
      if (t[q] < 0 || t[q] >= g.num_nodes || s[q] < 0 || s[q] >= g.num_nodes) {
        *err = 1;
        ok[q] = false;
        t[q] = s[q] = 0;
      }
      tn[q] = group_node(g, t[q]);
      sn[q] = group_node(g, s[q]);
    }
#pragma unroll
    for (int q = 0; q < kGroupPer; ++q) {
      int32_t f[5];
      group_fields(tn[q], sn[q], g, f);
      if (!ok[q]) continue;
#pragma unroll
      for (int k = 0; k < 5; ++k) {
        lo[k] = min(lo[k], f[k]);
        hi[k] = max(hi[k], f[k]);
      }
    }
  }
#pragma unroll
  for (int k = 0; k < 5; ++k) {
    for (int o = YGG_WAVE / 2; o > 0; o >>= 1) {
      lo[k] = min(lo[k], __shfl_xor(lo[k], o));
      hi[k] = max(hi[k], __shfl_xor(hi[k], o));
    }
  }
  const int wave = threadIdx.x / YGG_WAVE;
  if ((threadIdx.x & (YGG_WAVE - 1)) == 0) {
#pragma unroll
    for (int k = 0; k < 5; ++k) {
      red[wave][k] = lo[k];
      red[wave][5 + k] = hi[k];
    }
  }
  __syncthreads();
  if (threadIdx.x < 10) {
    const int k = threadIdx.x;
    int32_t v = red[0][k];
    for (int w = 1; w < 256 / YGG_WAVE; ++w) v = k < 5 ? min(v, red[w][k]) : max(v, red[w][k]);
    partials[10 * blockIdx.x + k] = v;
  }
}

// Field offsets and widths of the packed key; the fields are concatenated
// most significant first (target level, source level, dx, dy, dz), each
// minus its minimum, so unsigned order of the packed value is the
// lexicographic order of the signed fields. total = sum of widths. The sort
// key is the top `head` bits of it: all of them, or 63 of a longer key (seven
// 9-bit passes; 64 where more than 64 would be left).
struct Pack {
  int32_t min[5];
  int32_t width[5];
  int32_t total;
  int32_t bad;  // a pair named a node outside [0, T)
  int32_t head;
  int32_t repeats;  // sort keys met again in a sample of kGroupSample pairs
};

// The bits of a pair's key below its sort key, and the pair: what the sorted
// order gathers.
struct __attribute__((aligned(16))) KeyedPair {
  uint64_t rest;
  uint64_t pair;  // target << 32 | source
};

__global__ void __launch_bounds__(256)
k_group_pack_params(const int32_t* __restrict__ partials, int nblocks,
                    const int32_t* __restrict__ err, Pack* __restrict__ pk) {
  __shared__ int32_t red[256 / YGG_WAVE][10];
  int32_t v[10];
#pragma unroll
  for (int k = 0; k < 5; ++k) {
    v[k] = INT32_MAX;
    v[5 + k] = INT32_MIN;
  }
  for (int b = threadIdx.x; b < nblocks; b += blockDim.x) {
#pragma unroll
    for (int k = 0; k < 5; ++k) {
      v[k] = min(v[k], partials[10 * b + k]);
      v[5 + k] = max(v[5 + k], partials[10 * b + 5 + k]);
    }
  }
#pragma unroll
  for (int k = 0; k < 5; ++k) {
    for (int o = YGG_WAVE / 2; o > 0; o >>= 1) {
      v[k] = min(v[k], __shfl_xor(v[k], o));
      v[5 + k] = max(v[5 + k], __shfl_xor(v[5 + k], o));
    }
  }
  if ((threadIdx.x & (YGG_WAVE - 1)) == 0) {
#pragma unroll
    for (int k = 0; k < 10; ++k) red[threadIdx.x / YGG_WAVE][k] = v[k];
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    int total = 0;
    for (int k = 0; k < 5; ++k) {
      int32_t lo = red[0][k], hi = red[0][5 + k];
      for (int w = 1; w < 256 / YGG_WAVE; ++w) {
        lo = min(lo, red[w][k]);
        hi = max(hi, red[w][5 + k]);
      }
      const uint32_t span = (uint32_t)((int64_t)hi - (int64_t)lo);
      const int width = span == 0 ? 0 : 32 - __clz((int)span);
      pk->min[k] = lo;
      pk->width[k] = width;
      total += width;
    }
    pk->total = total;
    pk->bad = *err;
    pk->repeats = 0;
    pk->head = total <= 63 ? total : (total > 127 ? 64 : 63);
  }
}

// The sort key and the bits below it of a pair with fields f.
__device__ __forceinline__ void pack_key(const int32_t f[5], const Pack& pk, uint64_t& key,
                                         uint64_t& rest) {
  uint64_t lo = 0, hi = 0;
#pragma unroll
  for (int k = 0; k < 5; ++k) {
    const int w = pk.width[k];  // 0..32
    if (w == 0) continue;
    const uint64_t u = (uint64_t)((int64_t)f[k] - (int64_t)pk.min[k]);
    hi = (hi << w) | (lo >> (64 - w));
    lo = (lo << w) | u;
  }
  const int cut = pk.total - pk.head;  // 0..64
  key = lo;
  rest = 0;
  if (cut == 64) {
    rest = lo;
    key = hi;
  } else if (cut > 0) {
    rest = lo & ((1ull << cut) - 1ull);
    key = (lo >> cut) | (hi << (64 - cut));
  }
}

// How often the sort keys of kGroupSample pairs, evenly spaced, repeat: one
// workgroup, a table of twice as many slots in LDS. Pairs with bad node ids are
// left out (the call fails for them).
constexpr int kGroupSample = 4096;

template <typename IdxT>
__global__ void __launch_bounds__(1024)
k_group_sample(const IdxT* __restrict__ src, const IdxT* __restrict__ tgt, int64_t n, GroupGeom g,
               Pack* __restrict__ pkp) {
  constexpr unsigned kSlots = 2 * kGroupSample;
  constexpr unsigned long long kEmpty = ~0ull;
  __shared__ unsigned long long s_key[kSlots];
  __shared__ int s_again;
  const Pack pk = *pkp;
  if (threadIdx.x == 0) s_again = 0;
  for (unsigned k = threadIdx.x; k < kSlots; k += 1024) s_key[k] = kEmpty;
  __syncthreads();
  const int64_t taken = n < kGroupSample ? n : kGroupSample;
  for (int64_t q = threadIdx.x; q < taken; q += 1024) {
    const int64_t i = q * n / taken;
    const int64_t t = (int64_t)tgt[i], v = (int64_t)src[i];
    if (t < 0 || t >= g.num_nodes || v < 0 || v >= g.num_nodes) continue;
    int32_t f[5];
    group_fields(group_node(g, t), group_node(g, v), g, f);
    uint64_t key, rest;
    pack_key(f, pk, key, rest);
    unsigned slot = (unsigned)((key * 0x9E3779B97F4A7C15ull) >> 51);  // 13 bits
    for (unsigned probe = 0; probe < kSlots; ++probe, slot = (slot + 1) % kSlots) {
      const unsigned long long was = atomicCAS(&s_key[slot], kEmpty, (unsigned long long)key);
      if (was == (unsigned long long)key) atomicAdd(&s_again, 1);
      if (was == (unsigned long long)key || was == kEmpty) break;
    }
  }
  __syncthreads();
  if (threadIdx.x == 0) pkp->repeats = s_again;
}

template <typename IdxT>
__global__ void __launch_bounds__(256)
k_group_pack(const IdxT* __restrict__ src, const IdxT* __restrict__ tgt,
                int64_t n, GroupGeom g, Pack pk, uint64_t* __restrict__ key_out,
                             KeyedPair* __restrict__ recs) {
  const int64_t step = (int64_t)gridDim.x * blockDim.x * kGroupPer;
  for (int64_t b = blockIdx.x * (int64_t)blockDim.x * kGroupPer + threadIdx.x; b < n; b += step) {
    int64_t t[kGroupPer], s[kGroupPer];
#pragma unroll
    for (int q = 0; q < kGroupPer; ++q) {
      const int64_t i = b + (int64_t)q * blockDim.x;
      t[q] = i < n ? (int64_t)tgt[i] : 0;
      s[q] = i < n ? (int64_t)src[i] : 0;
    }
    GroupNode tn[kGroupPer], sn[kGroupPer];
#pragma unroll
    for (int q = 0; q < kGroupPer; ++q) {
      tn[q] = group_node(g, t[q]);
      sn[q] = group_node(g, s[q]);
    }
#pragma unroll
    for (int q = 0; q < kGroupPer; ++q) {
      const int64_t i = b + (int64_t)q * blockDim.x;
      if (i >= n) break;
      int32_t f[5];
      group_fields(tn[q], sn[q], g, f);
      uint64_t lo, rest;
      pack_key(f, pk, lo, rest);
      // node ids are below 2^31
      recs[i] = KeyedPair{rest, ((uint64_t)(uint32_t)t[q] << 32) | (uint64_t)(uint32_t)s[q]};
      key_out[i] = lo;
    }
  }
}

__global__ void k_gather_keys(const uint64_t* __restrict__ v, const uint32_t* __restrict__ idx,
                              int64_t n, uint64_t* __restrict__ out) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    out[i] = v[idx[i]];
}

__global__ void k_iota_u32(uint32_t* __restrict__ out, int64_t n) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    out[i] = (uint32_t)i;
}

__global__ void k_rest_keys(const KeyedPair* __restrict__ recs, int64_t n,
                            uint64_t* __restrict__ out) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    out[i] = recs[i].rest;
}

// The pairs and the rests of their keys (if any) in sorted order: one gather of
// 16-byte records.
__global__ void __launch_bounds__(256)
k_group_gather(const KeyedPair* __restrict__ recs, const uint32_t* __restrict__ order, int64_t n,
               uint64_t* __restrict__ pairs_s, uint64_t* __restrict__ rest_s) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    const KeyedPair r = recs[order[i]];
    pairs_s[i] = r.pair;
    if (rest_s) rest_s[i] = r.rest;
  }
}

// 1 where sorted position i starts a class: its key (key_s, rest_s if any)
// differs from position i - 1's.
__global__ void k_group_flags(const uint64_t* __restrict__ key_s,
                              const uint64_t* __restrict__ rest_s, int64_t n,
                              int32_t* __restrict__ flags) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    flags[i] = i == 0 || key_s[i] != key_s[i - 1] || (rest_s && rest_s[i] != rest_s[i - 1]);
}

// Finishes a stable sort by the top 63 bits of longer keys: the positions of
// one sort key are put in the order of their rests (equal ones stay in theirs),
// and the classes' first positions are marked. Keys of far pairs hardly ever
// share 63 bits, so nearly all this does is read the sort keys once, where
// sorting the rests too takes a third of the whole build: 2.1e7 pairs with
// 100-bit keys, seven passes and 220 us here against twelve passes and a gather
// of the second word, 3.3 ms in all against 4.5.
// A wavefront takes the runs that start among its 64 positions, one after the
// other, through LDS; a run belongs to one wavefront. A run longer than
// kTieRun raises *too_long (the order is then not valid): ranking it costs its
// square, and 20 KB of LDS per workgroup let eight of them share a CU (with runs
// of up to 512, 320 us).
constexpr int kTieThreads = 256;
constexpr int kTieRun = 256;

__global__ void __launch_bounds__(kTieThreads)
k_group_ties(const uint64_t* __restrict__ key_s, int64_t n, uint32_t* __restrict__ order,
             uint64_t* __restrict__ pairs_s, uint64_t* __restrict__ rest_s,
             int32_t* __restrict__ flags, int32_t* __restrict__ too_long) {
  __shared__ uint64_t s_rest[kTieThreads / YGG_WAVE][kTieRun];
  __shared__ uint64_t s_pair[kTieThreads / YGG_WAVE][kTieRun];
  __shared__ uint32_t s_ord[kTieThreads / YGG_WAVE][kTieRun];
  const int w = (int)threadIdx.x / YGG_WAVE, lane = (int)lane_id();
  const int64_t waves = (int64_t)gridDim.x * (kTieThreads / YGG_WAVE);
  for (int64_t b = ((int64_t)blockIdx.x * (kTieThreads / YGG_WAVE) + w) * YGG_WAVE; b < n;
       b += waves * YGG_WAVE) {
    const int64_t i = b + lane;
    const bool ok = i < n;
    const uint64_t k = ok ? key_s[i] : 0;
    const bool head = ok && (i == 0 || key_s[i - 1] != k);
    const bool tied = ok && i + 1 < n && key_s[i + 1] == k;
    if (head && !tied) flags[i] = 1;
    uint64_t runs = __ballot(head && tied);
    while (runs) {
      const int first = __ffsll((unsigned long long)runs) - 1;
      runs &= runs - 1;
      const int64_t h = b + first;
      const uint64_t key = (uint64_t)__shfl((unsigned long long)k, first, YGG_WAVE);
      int len = 0;
      while (len <= kTieRun) {
        const int64_t j = h + len + lane;
        const uint64_t same = __ballot(j < n && key_s[j] == key);
        if (~same == 0ull) {
          len += YGG_WAVE;
          continue;
        }
        len += __ffsll((unsigned long long)~same) - 1;
        break;
      }
      if (len > kTieRun) {
        if (lane == 0) *too_long = 1;
        continue;
      }
      for (int e = lane; e < len; e += YGG_WAVE) {
        s_rest[w][e] = rest_s[h + e];
        s_pair[w][e] = pairs_s[h + e];
        s_ord[w][e] = order[h + e];
      }
      // the wavefront's own LDS: written before it is read, read before the
      // next run writes it
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
      for (int e = lane; e < len; e += YGG_WAVE) {
        const uint64_t mine = s_rest[w][e];
        int rank = 0;
        bool starts = true;
        for (int j = 0; j < len; ++j) {
          const uint64_t o = s_rest[w][j];
          rank += o < mine || (o == mine && j < e);
          starts = starts && !(o == mine && j < e);
        }
        order[h + rank] = s_ord[w][e];
        pairs_s[h + rank] = s_pair[w][e];
        rest_s[h + rank] = mine;
        flags[h + rank] = starts;
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
    }
  }
}

// class_scan[i] = classes started before sorted position i, so position i
// belongs to class class_scan[i + 1] - 1 and starts it iff the two differ.
// A class head decodes its key fields from its packed key.
// Bound by its writes: 2.1e7 pairs of as many classes, 64 contiguous bytes and
// one scattered class id each, 590 us (930 us when the heads' keys were gathered
// and each thread wrote its own class row).
constexpr int kEmitThreads = 256;

template <typename IdxT>
__global__ void __launch_bounds__(kEmitThreads)
k_group_emit(const uint64_t* __restrict__ pairs_s, int64_t n,
                             const float* __restrict__ bmin,
                             const float* __restrict__ bmax, const Pack* __restrict__ pkp,
                             const uint64_t* __restrict__ key_s,
                             const uint64_t* __restrict__ rest_s,
                             const uint32_t* __restrict__ order, const int64_t* __restrict__ scan,
                             IdxT* __restrict__ csrc, IdxT* __restrict__ ctgt,
                             IdxT* __restrict__ cids, IdxT* __restrict__ coff,
                             int32_t* __restrict__ ckeys, float* __restrict__ cdisp) {
  // the rows of a workgroup's classes are contiguous: they leave through LDS
  __shared__ int32_t s_key[5 * kEmitThreads];
  __shared__ float s_disp[3 * kEmitThreads];
  const Pack pk = *pkp;
  const int cut = pk.total - pk.head;  // 0..64
  const int tid = (int)threadIdx.x;
  for (int64_t b = blockIdx.x * (int64_t)kEmitThreads; b < n;
       b += (int64_t)gridDim.x * kEmitThreads) {
    const int64_t i = b + tid, end = min(b + kEmitThreads, n);
    const int64_t c0 = scan[b];  // classes that start before this workgroup's
    const int rows = (int)(scan[end] - c0);
    if (i < n) {
      const int64_t p = order[i];
      const int64_t c = scan[i + 1] - 1;
      const uint64_t tp = pairs_s[i];
      csrc[i] = (IdxT)(uint32_t)tp;
      ctgt[i] = (IdxT)(uint32_t)(tp >> 32);
      cids[p] = (IdxT)c;
      if (scan[i + 1] != scan[i]) {
        coff[c] = (IdxT)i;
        const int r = (int)(c - c0);
        uint64_t lo = key_s[i], hi = 0;
        if (cut == 64) {
          hi = lo;
          lo = rest_s[i];
        } else if (cut > 0) {
          hi = lo >> (64 - cut);
          lo = (lo << cut) | rest_s[i];
        }
        int32_t f[5];
#pragma unroll
        for (int k = 4; k >= 0; --k) {
          const int w = pk.width[k];
          uint64_t bits = 0;
          if (w > 0) {
            bits = lo & ((1ull << w) - 1ull);
            lo = (lo >> w) | (hi << (64 - w));
            hi >>= w;
          }
          f[k] = (int32_t)((int64_t)pk.min[k] + (int64_t)bits);
        }
#pragma unroll
        for (int k = 0; k < 5; ++k) s_key[5 * r + k] = f[k];
        // class displacement = index * target-level cell, rounded to float32
#pragma unroll
        for (int a = 0; a < 3; ++a) {
          const double ext = (double)bmax[a] - (double)bmin[a];
          s_disp[3 * r + a] = (float)((double)f[2 + a] * cell_size(ext, f[0]));
        }
      }
      if (i == n - 1) coff[scan[n]] = (IdxT)n;
    }
    __syncthreads();
    for (int k = tid; k < 5 * rows; k += kEmitThreads) ckeys[5 * c0 + k] = s_key[k];
    for (int k = tid; k < 3 * rows; k += kEmitThreads) cdisp[3 * c0 + k] = s_disp[k];
    __syncthreads();
  }
}

// The radix sort ranks at most 2^30 - 1 elements per call.
constexpr int64_t kMaxGroupedPairs = (1ll << 30) - 1;

// Workspace shared by the classify and emit calls. After classify, pairs_s
// holds the pairs, key_s the sort keys and rest_s the bits below them, all in
// sorted order, and pack the packing parameters.
struct GroupWs {
  int32_t* partials;
  int32_t* err;  // [2]: a bad node id, a run of equal sort keys too long
  Pack* pack;
  uint64_t* key;
  uint64_t* key_s;
  uint64_t* alt;
  uint64_t* rest_s;
  uint64_t* pairs_s;
  KeyedPair* recs;
  uint32_t* order1;
  int32_t* flags;
  void* sort_ws;
  size_t sort_bytes;
  void* scan_ws;
  size_t scan_bytes;
};

static bool group_ws_layout(int64_t n, void* ws, size_t ws_bytes, GroupWs* w, size_t* bytes) {
  Arena a(ws, ws_bytes);
  w->partials = a.take<int32_t>(10 * kMinmaxBlocks);
  w->err = a.take<int32_t>(2);
  w->pack = a.take<Pack>(1);
  w->key = a.take<uint64_t>((size_t)n);
  w->key_s = a.take<uint64_t>((size_t)n);
  w->alt = a.take<uint64_t>((size_t)n);
  w->rest_s = a.take<uint64_t>((size_t)n);
  w->pairs_s = w->alt;  // written once the keys are sorted
  w->recs = a.take<KeyedPair>((size_t)n);
  w->order1 = a.take<uint32_t>((size_t)n);
  w->flags = a.take<int32_t>((size_t)n);
  w->sort_bytes = std::max(sort_workspace_bytes(n, 8, 64, 8), sort_workspace_bytes(n, 8, 64, 9));
  w->sort_ws = a.take<char>(w->sort_bytes);
  w->scan_bytes = scan_workspace_bytes(n);
  w->scan_ws = a.take<char>(w->scan_bytes);
  if (bytes) *bytes = a.off;
  return w->partials && w->err && w->pack && w->key && w->key_s && w->alt && w->rest_s &&
         w->recs && w->order1 && w->flags && w->sort_ws && w->scan_ws;
}

// Digit width of a class-key sort over `bits` bits: 9 unless 8 takes fewer
// passes (a pass over 2e7 pairs takes 160 us with 9 bits, 176 us with 8).
static int group_digit_bits(int bits) { return (bits + 8) / 9 <= (bits + 7) / 8 ? 9 : 8; }

// Class starts counted from w.flags: *total classes, and *too_long if a run of
// equal sort keys was too long for k_group_ties.
static int group_count(const GroupWs& w, int64_t n, int64_t* scan, int64_t* total,
                       int32_t* too_long, hipStream_t st) {
  if (int rc = exclusive_scan_i32_to_i64(w.flags, nullptr, scan, n, w.scan_ws, w.scan_bytes, st))
    return rc;
  YGG_CHECK(hipMemcpyAsync(total, scan + n, sizeof(*total), hipMemcpyDeviceToHost, st));
  if (too_long)
    YGG_CHECK(hipMemcpyAsync(too_long, w.err + 1, sizeof(*too_long), hipMemcpyDeviceToHost, st));
  YGG_CHECK(hipStreamSynchronize(st));
  return YGG_OK;
}

// Keys of one word: sorted whole (identity order for the single class of a key
// without bits).
static int group_order_one_word(const GroupWs& w, int64_t n, int bits, uint32_t* order,
                                hipStream_t st) {
  const int grid = grid_for(n, 256);
  int rc;
  if (bits == 0) {
    hipLaunchKernelGGL(k_iota_u32, dim3(grid), dim3(256), 0, st, order, n);
    YGG_LAUNCH_CHECK();
    rc = copy_u32((uint32_t*)w.key_s, (const uint32_t*)w.key, 2 * n, st);
  } else {
    rc = sort_pairs_u64(w.key, nullptr, w.key_s, order, n, 0, bits, w.sort_ws, w.sort_bytes, st,
                        nullptr, group_digit_bits(bits));
  }
  if (rc) return rc;
  hipLaunchKernelGGL(k_group_gather, dim3(grid), dim3(256), 0, st, w.recs, order, n, w.pairs_s,
                     nullptr);
  hipLaunchKernelGGL(k_group_flags, dim3(grid), dim3(256), 0, st, w.key_s, nullptr, n, w.flags);
  YGG_LAUNCH_CHECK();
  return YGG_OK;
}

// Longer keys that hardly ever share their sort key: sorted by it, and the runs
// that do put in order in place.
static int group_order_ties(const GroupWs& w, int64_t n, const Pack& pk, uint32_t* order,
                            hipStream_t st) {
  if (int rc = sort_pairs_u64(w.key, nullptr, w.key_s, order, n, 0, pk.head, w.sort_ws,
                              w.sort_bytes, st, nullptr, group_digit_bits(pk.head)))
    return rc;
  hipLaunchKernelGGL(k_group_gather, dim3(grid_for(n, 256)), dim3(256), 0, st, w.recs, order, n,
                     w.pairs_s, w.rest_s);
  hipLaunchKernelGGL(k_group_ties, dim3(grid_for(n, kTieThreads, 4096)), dim3(kTieThreads), 0, st,
                     w.key_s, n, order, w.pairs_s, w.rest_s, w.flags, w.err + 1);
  YGG_LAUNCH_CHECK();
  return YGG_OK;
}

// Longer keys of which many share their sort key: a stable LSD sort over both
// words, the rests first, then the sort keys carrying that order.
static int group_order_two_words(const GroupWs& w, int64_t n, const Pack& pk, uint32_t* order,
                                 hipStream_t st) {
  const int grid = grid_for(n, 256), cut = pk.total - pk.head;
  hipLaunchKernelGGL(k_rest_keys, dim3(grid), dim3(256), 0, st, w.recs, n, w.alt);
  YGG_LAUNCH_CHECK();
  int rc = sort_pairs_u64(w.alt, nullptr, w.rest_s, w.order1, n, 0, cut, w.sort_ws, w.sort_bytes,
                          st, nullptr, group_digit_bits(cut));
  if (rc) return rc;
  hipLaunchKernelGGL(k_gather_keys, dim3(grid), dim3(256), 0, st, w.key, w.order1, n, w.alt);
  YGG_LAUNCH_CHECK();
  rc = sort_pairs_u64(w.alt, w.order1, w.key_s, order, n, 0, pk.head, w.sort_ws, w.sort_bytes, st,
                      nullptr, group_digit_bits(pk.head));
  if (rc) return rc;
  hipLaunchKernelGGL(k_group_gather, dim3(grid), dim3(256), 0, st, w.recs, order, n, w.pairs_s,
                     w.rest_s);
  hipLaunchKernelGGL(k_group_flags, dim3(grid), dim3(256), 0, st, w.key_s, w.rest_s, n, w.flags);
  YGG_LAUNCH_CHECK();
  return YGG_OK;
}

template <typename IdxT>
int grouped_classify(const IdxT* src, const IdxT* tgt, int64_t n, GroupGeom g,
                     uint32_t* order, int64_t* scan, int64_t* num_classes, void* ws,
                     size_t ws_bytes, hipStream_t st) {
  GroupWs w;
  if (!group_ws_layout(n, ws, ws_bytes, &w, nullptr)) return YGG_ERR_WORKSPACE;
  const int mgrid = grid_for(n, 256 * kGroupPer, kMinmaxBlocks);
  int rc;
  if ((rc = fill_u32((uint32_t*)w.err, 0u, 2, st))) return rc;
  // the table lies where the sort will work, if it fits: not for a tree of more
  // nodes than pairs
  if (sizeof(float4) * (size_t)g.num_nodes <= w.sort_bytes) {
    float4* table = (float4*)w.sort_ws;
    hipLaunchKernelGGL(k_group_nodes, dim3(grid_for(g.num_nodes, 256)), dim3(256), 0, st, g,
                       table);
    g.node = table;
  }
  hipLaunchKernelGGL(k_group_minmax<IdxT>, dim3(mgrid), dim3(256), 0, st, src, tgt, n, g,
                     w.partials, w.err);
  YGG_LAUNCH_CHECK();
  hipLaunchKernelGGL(k_group_pack_params, dim3(1), dim3(256), 0, st, w.partials, mgrid, w.err,
                     w.pack);
  YGG_LAUNCH_CHECK();
  hipLaunchKernelGGL(k_group_sample<IdxT>, dim3(1), dim3(1024), 0, st, src, tgt, n, g, w.pack);
  YGG_LAUNCH_CHECK();
  Pack pk;
  YGG_CHECK(hipMemcpyAsync(&pk, w.pack, sizeof(Pack), hipMemcpyDeviceToHost, st));
  YGG_CHECK(hipStreamSynchronize(st));
  if (pk.bad) return YGG_ERR_ARG;
  const int W = pk.total;
  if (W > 128) return YGG_ERR_UNSUPPORTED;
  const int cut = W - pk.head;  // bits below the sort key
  // r pairs to a sort key show as r sample^2 / 2 n repeats. From about 100 on
  // ranking the ties, or finding a run too long, costs more than sorting the
  // rests: with 200 (400) pairs to each of 16384 keys of 83 bits, 0.99 (1.59) ms
  // sorting both words at once, 1.13 (2.26) ms the other way. The sample costs 40
  // us at 2.1e7 pairs, 3.2 ms in all.
  const double sample = (double)std::min<int64_t>(n, kGroupSample);
  const bool both = cut > 0 && 2.0 * (double)pk.repeats * (double)n > 100.0 * sample * sample;
  hipLaunchKernelGGL(k_group_pack<IdxT>, dim3(grid_for(n, 256 * kGroupPer)), dim3(256), 0, st, src,
                     tgt, n, g, pk, w.key, w.recs);
  YGG_LAUNCH_CHECK();
  int64_t total = 0;
  int32_t too_long = 0;
  if (cut == 0) {
    if ((rc = group_order_one_word(w, n, W, order, st))) return rc;
    if ((rc = group_count(w, n, scan, &total, nullptr, st))) return rc;
  } else if (!both) {
    if ((rc = group_order_ties(w, n, pk, order, st))) return rc;
    if ((rc = group_count(w, n, scan, &total, &too_long, st))) return rc;
  }
  if (both || too_long) {
    if ((rc = group_order_two_words(w, n, pk, order, st))) return rc;
    if ((rc = group_count(w, n, scan, &total, nullptr, st))) return rc;
  }
  *num_classes = total;
  return YGG_OK;
}

}  // namespace
}  // namespace ygg

using namespace ygg;

extern "C" {

int ygg_dense_interactions(const void* offsets, const void* counts, const void* sources,
                           int idx_i64, int64_t num_nodes, int64_t num_far,
                           const int32_t* nodes_by_level, const int32_t* level_offsets,
                           int32_t num_levels, int64_t max_nodes, int64_t max_interactions,
                           const float* center, void* out_sources, float* out_displacements,
                           uint8_t* out_mask, void* out_counts, int32_t* error_flag,
                           void* stream) {
  if (num_levels < 1 || max_nodes < 1 || max_interactions < 1 || num_nodes < 1 ||
      num_far < 0 || !offsets || !counts || !sources || !nodes_by_level || !level_offsets ||
      !center || !out_sources || !out_displacements || !out_mask || !out_counts || !error_flag)
    return YGG_ERR_ARG;
  if ((int64_t)num_levels * max_nodes > (1ll << 40) / max_interactions) return YGG_ERR_ARG;
  hipStream_t st = (hipStream_t)stream;
  int rc;
  if ((rc = fill_u32((uint32_t*)error_flag, 0u, 1, st))) return rc;
  const int64_t total = (int64_t)num_levels * max_nodes * max_interactions;
  const dim3 g(grid_for(total, kDenseSpan));
  // wide stores need 16-byte aligned sources and displacements, a 4-byte
  // aligned mask
  const bool vec = (((uintptr_t)out_sources | (uintptr_t)out_displacements) & 15) == 0 &&
                   ((uintptr_t)out_mask & 3) == 0;
  auto launch = [&](auto kernel, auto idx) {
    using IdxT = decltype(idx);
    hipLaunchKernelGGL(kernel, g, dim3(kDenseThreads), 0, st, (const IdxT*)offsets,
                       (const IdxT*)counts, (const IdxT*)sources, num_nodes, num_far,
                       nodes_by_level, level_offsets, num_levels, max_nodes, max_interactions,
                       center, (IdxT*)out_sources, out_displacements, out_mask,
                       (IdxT*)out_counts, error_flag);
  };
  if (idx_i64)
    vec ? launch(k_dense_m2l<int64_t, true>, int64_t()) : launch(k_dense_m2l<int64_t, false>, int64_t());
  else
    vec ? launch(k_dense_m2l<int32_t, true>, int32_t()) : launch(k_dense_m2l<int32_t, false>, int32_t());
  YGG_LAUNCH_CHECK();
  return YGG_OK;
}

size_t ygg_grouped_workspace_bytes(int64_t num_pairs) {
  if (num_pairs < 1) return 0;
  GroupWs w;
  size_t bytes = 0;
  group_ws_layout(num_pairs, nullptr, 0, &w, &bytes);
  return bytes;
}

int ygg_grouped_classify(const void* sources, const void* targets, int64_t num_pairs,
                         int idx_i64, int64_t num_nodes, const int32_t* node_level,
                         const float* center,
                         const float* bounds_min, const float* bounds_max, uint32_t* order,
                         int64_t* class_scan, int64_t* num_classes, void* ws, size_t ws_bytes,
                         void* stream) {
  if (num_pairs < 1 || !sources || !targets || !node_level || !center || !bounds_min ||
      !bounds_max || !order || !class_scan || !num_classes)
    return YGG_ERR_ARG;
  if (num_pairs > kMaxGroupedPairs) return YGG_ERR_UNSUPPORTED;
  if (num_nodes < 1) return YGG_ERR_ARG;
  GroupGeom g{num_nodes, node_level, center, bounds_min, bounds_max, nullptr};
  hipStream_t st = (hipStream_t)stream;
  if (idx_i64)
    return grouped_classify((const int64_t*)sources, (const int64_t*)targets, num_pairs, g,
                            order, class_scan, num_classes, ws, ws_bytes, st);
  return grouped_classify((const int32_t*)sources, (const int32_t*)targets, num_pairs, g, order,
                          class_scan, num_classes, ws, ws_bytes, st);
}

int ygg_grouped_emit(int64_t num_pairs, int idx_i64, const float* bounds_min,
                     const float* bounds_max, const uint32_t* order, const int64_t* class_scan,
                     void* class_sources, void* class_targets, void* class_ids,
                     void* class_offsets, int32_t* class_keys, float* class_displacements,
                     void* ws, size_t ws_bytes, void* stream) {
  if (num_pairs < 1 || !bounds_min || !bounds_max || !order ||
      !class_scan || !class_sources || !class_targets || !class_ids || !class_offsets ||
      !class_keys || !class_displacements)
    return YGG_ERR_ARG;
  if (num_pairs > kMaxGroupedPairs) return YGG_ERR_UNSUPPORTED;
  GroupWs w;
  if (!group_ws_layout(num_pairs, ws, ws_bytes, &w, nullptr)) return YGG_ERR_WORKSPACE;
  hipStream_t st = (hipStream_t)stream;
  dim3 grid(grid_for(num_pairs, kEmitThreads));
  if (idx_i64)
    hipLaunchKernelGGL(k_group_emit<int64_t>, grid, dim3(256), 0, st, w.pairs_s, num_pairs,
                       bounds_min, bounds_max, w.pack, w.key_s, w.rest_s, order, class_scan,
                       (int64_t*)class_sources,
                       (int64_t*)class_targets, (int64_t*)class_ids, (int64_t*)class_offsets,
                       class_keys, class_displacements);
  else
    hipLaunchKernelGGL(k_group_emit<int32_t>, grid, dim3(256), 0, st, w.pairs_s, num_pairs,
                       bounds_min, bounds_max, w.pack, w.key_s, w.rest_s, order, class_scan,
                       (int32_t*)class_sources,
                       (int32_t*)class_targets, (int32_t*)class_ids, (int32_t*)class_offsets,
                       class_keys, class_displacements);
  YGG_LAUNCH_CHECK();
  return YGG_OK;
}

}  // extern "C"
