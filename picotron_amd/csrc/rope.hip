// Rotary position embedding (forward and its inverse, the backward) for gfx950.
//
// Reference semantics (AndyMLAndAI/picotron):
//   tables   src/picotron/nn/rope.py:13-32    angle[s, i] = s * theta^(-2i/D); cos/sin
//   rotation src/picotron/nn/rope.py:35-51    interleaved pairs (2i, 2i+1):
//            (a, b) -> (a*c - b*s, a*s + b*c)
//   Triton   src/picotron/nn/triton_kernels/rope.py:25-49 (same pairs, forward only)
// The rotate-half layout pairs (i, i + D/2) with the same angle table.  The inverse
// rotation (a, b) -> (a*c + b*s, -a*s + b*c) is the exact transpose of the forward, so it
// is the backward of the forward.
//
// Work item = one 16-byte vector of a row (interleaved: V/2 pairs) or one vector from each
// half of a row (rotate-half: V pairs), for up to kHeads heads of one position: the heads share
// the item's cos and sin, which are twice the bytes of one head's vectors where those are 16-bit,
// and the decode of its indices.  Rows are the (batch, head, seq) positions of a
// strided view whose head_dim is contiguous; the host orders the three row dimensions by
// decreasing stride so consecutive work items walk memory in address order (item c of a
// position's `chunks` takes heads c, c + chunks, ...).  Query and key
// are handled by one launch (blocks [0, nb0) and [nb0, nb0 + nb1)).
#include "pt_common.hpp"

namespace pt {
namespace {

// Work items per row: interleaved rows split into V-element vectors (V/2 pairs each, or one
// pair on the element path); rotate-half rows into P-pair groups taken from both halves.
template <typename T, int LAYOUT, bool ALIGNED>
__host__ __device__ constexpr int items_per_row(int head_dim) {
  return LAYOUT == 0 ? head_dim / (ALIGNED ? Elem<T>::VEC : 2)
                     : (head_dim / 2) / (ALIGNED ? Elem<T>::VEC : 1);
}

struct RopeTensor {
  const void* x;
  void* y;
  int64_t n[3];    // row dimensions, outer to inner (iteration order); the heads' in chunks
  int64_t xs[3];   // x strides of those dimensions (elements)
  int64_t ys[3];   // y strides
  int seq_dim;     // which of the three is the sequence dimension
  int head_dim;    // and which the heads
  int64_t heads;
  int64_t chunks;  // items that share a position's heads
  int64_t xstep;   // elements from one of an item's heads to the next
  int64_t ystep;
  int64_t rows;    // batch * heads * seq
  int64_t items;   // n[0] * n[1] * n[2] * items_per_row
  int64_t blocks;  // blocks assigned to this tensor
  int64_t ybytes;  // bytes from y to the end of its last row
};

// What the kernel reads of a RopeTensor.  A small call is bound by the chain of scalar loads that fetches
// these arguments: as the host's struct, behind the tables' pointers, they cost it 0.1 us of 2.1.
struct RopeArgs {
  const void* x;
  void* y;
  int64_t xs[3];
  int64_t ys[3];
  int64_t xstep;
  int64_t ystep;
  uint32_t n1, n2;  // n[1], n[2]
  uint32_t heads;
  uint32_t chunks;
  uint32_t items;
  uint32_t blocks;
  int seq_dim;
  int head_dim;
  int ybytes;  // write-through stores only
};

// One work item in two phases, so that a thread has every head's loads in flight before it
// computes and stores any of them (the output may alias the input, so the
// compiler would not move a later head's loads above an earlier head's stores).  The pair
// members are held as a[p] (first) and b[p] (second): interleaved rows pair elements
// (2i, 2i+1) of one vector, rotate-half rows pair element i of the first half with element
// i of the second.  Item, row and the three row indices fit in 32 bits (pt_rope bounds
// items by 2^32), so they are decoded with 32-bit divisions; only memory offsets are 64-bit.
// WT (aligned rows only): stores through a buffer resource over y with the write-through
// policy instead of nontemporal global stores.
// Heads per item (U): two for interleaved rows, whose item is one vector of 16 bytes per head beside 32
// bytes of cos and sin; one for rotate-half rows (two vectors beside 64 bytes).  Measured per launch
// on q [8, 2048, 32, 128] + k [8, 2048, 8, 128] bf16 (the bytes at copy speed: 51.5 us): interleaved one
// head 55.7, two 53.9, four 54.9, and at [1, 2048] 10.1, 8.9, 8.6; rotate-half 54.7, 55.2, 57.2 and
// 8.6, 8.3, 8.8.  Calls of fewer than 65536 vectors (a decode step) are one wave's chain of loads, which the
// second head only lengthens: interleaved, mean over the sizes up to 16384 vectors two heads 2.16 us
// and one 2.06, up to 65536 2.24 and 2.14; up to 262144 3.15 and 3.18, up to 1048576 5.84 and 6.15.
constexpr int64_t kTwoHeadVectors = 65536;

template <typename T, int LAYOUT, bool ALIGNED, bool NT, bool WT, int U>
struct RopeWork {
  static constexpr int V = ALIGNED ? Elem<T>::VEC : 2;
  static constexpr int P = LAYOUT == 0 ? V / 2 : (ALIGNED ? Elem<T>::VEC : 1);  // pairs
  // Raw storage until store(): converting in load() would wait for the data there.
  Vec16<T> va[U], vb[U];  // aligned: interleaved vector (va) or the two half vectors (va, vb)
  T ea[2], eb[2];   // element path: interleaved (ea[0], ea[1]) or rotate-half (ea[0], eb[0])
  float c[P], s[P];
  T* ya;            // the first head's first members (interleaved: the whole vector)
  int64_t ystep;    // from head to head
  int count;        // heads

  __device__ __forceinline__ void load(const RopeArgs& t, uint32_t item, int head_dim,
                                       const float* __restrict__ cos_t,
                                       const float* __restrict__ sin_t) {
    const int half = head_dim / 2;
    const uint32_t per_row = static_cast<uint32_t>(items_per_row<T, LAYOUT, ALIGNED>(head_dim));
    const uint32_t row = item / per_row;
    const int j = static_cast<int>(item - row * per_row);
    int64_t idx[3];
    const uint32_t r1 = row / t.n2;
    idx[2] = row - r1 * t.n2;
    idx[0] = r1 / t.n1;
    idx[1] = r1 - static_cast<uint32_t>(idx[0]) * t.n1;
    const int64_t xo = idx[0] * t.xs[0] + idx[1] * t.xs[1] + idx[2] * t.xs[2];
    const int64_t yo = idx[0] * t.ys[0] + idx[1] * t.ys[1] + idx[2] * t.ys[2];
    // selects, not an indexed array (which would live in scratch memory)
    const int64_t pos = t.seq_dim == 0 ? idx[0] : (t.seq_dim == 1 ? idx[1] : idx[2]);
    const T* xr = static_cast<const T*>(t.x) + xo;
    const int i0 = j * P;  // first pair of the item
    ya = static_cast<T*>(t.y) + yo + (LAYOUT == 0 ? 2 * i0 : i0);
    ystep = U > 1 ? t.ystep : 0;
    count = 1;
    if constexpr (ALIGNED) {
      const int64_t xstep = U > 1 ? t.xstep : 0;
      if constexpr (U > 1) {
        static_assert(U == 2 && ALIGNED, "an item's heads are first and first + chunks");
        // below 2^31: pt_rope bounds the pairs by 2^32, and these rows have at least two vectors
        const uint32_t first =
            static_cast<uint32_t>(t.head_dim == 0 ? idx[0] : (t.head_dim == 1 ? idx[1] : idx[2]));
        count = first + t.chunks < t.heads ? 2 : 1;
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (u == 0 || u < count) {
          const T* p = xr + u * xstep;
          if constexpr (LAYOUT == 0) {
            va[u].raw = load16<NT>(p + j * V);
          } else {
            va[u].raw = load16<NT>(p + i0);
            vb[u].raw = load16<NT>(p + half + i0);
          }
        }
      }
    } else if constexpr (LAYOUT == 0) {
      ea[0] = xr[2 * j];
      ea[1] = xr[2 * j + 1];
    } else {
      ea[0] = xr[j];
      eb[0] = xr[half + j];
    }
    const float* cr = cos_t + pos * half + i0;
    const float* sr = sin_t + pos * half + i0;
#pragma unroll
    for (int p = 0; p < P; ++p) {
      c[p] = cr[p];
      s[p] = sr[p];
    }
  }

  template <int N>
  __device__ __forceinline__ static void put(__amdgpu_buffer_rsrc_t buf, const T* ybase, T* p,
                                             const float (&o)[N]) {
    if constexpr (WT) {
      Vec16<T> v;
#pragma unroll
      for (int i = 0; i < N; ++i) v.e[i] = Elem<T>::from_f32(o[i]);
      const uint32_t off = static_cast<uint32_t>(reinterpret_cast<const char*>(p) -
                                                 reinterpret_cast<const char*>(ybase));
      __builtin_amdgcn_raw_buffer_store_b128(v.raw, buf, off, 0, kWriteThrough);
    } else {
      store_f32<T, true, NT>(p, o, N);
    }
  }

  __device__ __forceinline__ void store(float sign, int head_dim, __amdgpu_buffer_rsrc_t buf,
                                        const T* ybase) const {
    const int half = head_dim / 2;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (u > 0 && u >= count) continue;
      float a[P], b[P];
#pragma unroll
      for (int p = 0; p < P; ++p) {
        if constexpr (LAYOUT == 0) {
          a[p] = Elem<T>::to_f32(ALIGNED ? va[u].e[2 * p] : ea[2 * p]);
          b[p] = Elem<T>::to_f32(ALIGNED ? va[u].e[2 * p + 1] : ea[2 * p + 1]);
        } else {
          a[p] = Elem<T>::to_f32(ALIGNED ? va[u].e[p] : ea[p]);
          b[p] = Elem<T>::to_f32(ALIGNED ? vb[u].e[p] : eb[p]);
        }
      }
      float oa[P], ob[P];
#pragma unroll
      for (int p = 0; p < P; ++p) {
        // Written out, since the compiler's own choice of the product that it rounds differs from
        // instance to instance: the same bits from every number of heads per item.  (For fp16 it may
        // still fuse the last operation with the conversion, one rounding in place of two.)
        const float sn = sign * s[p];
        oa[p] = __builtin_fmaf(a[p], c[p], -(b[p] * sn));
        ob[p] = LAYOUT == 0 && ALIGNED ? __builtin_fmaf(a[p], sn, b[p] * c[p])
                                       : __builtin_fmaf(b[p], c[p], a[p] * sn);
      }
      T* y = ya + u * ystep;
      if constexpr (LAYOUT == 0) {
        float o[V];
#pragma unroll
        for (int p = 0; p < P; ++p) {
          o[2 * p] = oa[p];
          o[2 * p + 1] = ob[p];
        }
        if constexpr (ALIGNED) {
          put(buf, ybase, y, o);
        } else {
          y[0] = Elem<T>::from_f32(o[0]);
          y[1] = Elem<T>::from_f32(o[1]);
        }
      } else if constexpr (ALIGNED) {
        put(buf, ybase, y, oa);
        put(buf, ybase, y + half, ob);
      } else {
        y[0] = Elem<T>::from_f32(oa[0]);
        y[half] = Elem<T>::from_f32(ob[0]);
      }
    }
  }
};

// Thread t of block b takes item b * 256 + t of its tensor.
template <typename T, int LAYOUT, bool ALIGNED, bool NT, bool WT, int U>
__global__ __launch_bounds__(256) void rope_kernel(const float* __restrict__ cos_t,
                                                   const float* __restrict__ sin_t, int head_dim,
                                                   float sign, RopeArgs t0, RopeArgs t1) {
  uint32_t b = blockIdx.x;
  const RopeArgs* t = &t0;
  if (b >= t0.blocks) {
    b -= t0.blocks;
    t = &t1;
  }
  const uint32_t item = b * 256u + threadIdx.x;
  // y's span fits a buffer resource whenever WT is set (checked on the host); unused otherwise
  const auto ybuf = uniform_buffer(t->y, WT ? t->ybytes : 0);
  if (item >= t->items) return;
  // Fetches the table pointers with the other arguments (left alone, the compiler loads them only after
  // the states' loads, and the tables' loads wait for one more round trip).
  asm volatile("" : : "s"(cos_t), "s"(sin_t));
  RopeWork<T, LAYOUT, ALIGNED, NT, WT, U> w;
  w.load(*t, item, head_dim, cos_t, sin_t);
  w.store(sign, head_dim, ybuf, static_cast<const T*>(t->y));
}

bool parse(const void* x, void* y, const int64_t* d, int64_t head_dim, int64_t table_rows,
           int esize, int layout, RopeTensor* t, bool* aligned, std::string* err) {
  const int64_t sz[3] = {d[0], d[1], d[2]};  // batch, heads, seq
  const int64_t xs[3] = {d[3], d[4], d[5]};
  const int64_t ys[3] = {d[6], d[7], d[8]};
  for (int i = 0; i < 3; ++i) {
    if (sz[i] < 0) {
      *err = "negative dimension";
      return false;
    }
  }
  if (sz[2] > table_rows) {
    *err = "sequence length exceeds the cos/sin table rows";
    return false;
  }
  // iteration order: dimensions by decreasing x stride (stable), so the innermost
  // iterated dimension has the smallest stride.
  int ord[3] = {0, 1, 2};
  for (int a = 0; a < 3; ++a)
    for (int b = a + 1; b < 3; ++b)
      if (xs[ord[b]] > xs[ord[a]]) {
        const int tmp = ord[a];
        ord[a] = ord[b];
        ord[b] = tmp;
      }
  t->x = x;
  t->y = y;
  for (int i = 0; i < 3; ++i) {
    t->n[i] = sz[ord[i]];
    t->xs[i] = xs[ord[i]];
    t->ys[i] = ys[ord[i]];
    if (ord[i] == 2) t->seq_dim = i;
    if (ord[i] == 1) t->head_dim = i;
  }
  t->heads = sz[1];
  t->rows = sz[0] * sz[1] * sz[2];
  // y's extent in bytes (-1 when a stride is negative): the write-through stores address y
  // through a buffer resource, so they need it to fit 31 bits
  int64_t last = head_dim;
  for (int i = 0; i < 3; ++i) {
    if (sz[i] > 1 && ys[i] < 0) last = -1;
    if (last >= 0 && sz[i] > 1) last += (sz[i] - 1) * ys[i];
  }
  t->ybytes = last < 0 ? -1 : last * esize;
  // 16-byte vectors need aligned bases, strides that keep every row aligned, and
  // (rotate-half) a half that is a whole number of vectors.
  const int vec = 16 / esize;
  bool al = aligned16(x) && aligned16(y) && head_dim % (2 * vec) == 0;
  for (int i = 0; i < 3; ++i) {
    if (sz[i] > 1 && ((xs[i] * esize) % 16 != 0 || (ys[i] * esize) % 16 != 0)) al = false;
  }
  if (layout == 0 && head_dim % vec != 0) al = false;
  *aligned = al;
  return true;
}

constexpr int64_t kNontemporalBytes = int64_t{64} << 20;

// Resident workgroups per CU (0: no limit); PT_ROPE_OCCUPANCY overrides it.  One item
// per thread keeps little in flight, so the limit stays high: rotate-half rows at 6 measured
// 54.3-54.5 us per launch on the 4-layer q + k benchmark against 54.7 with the full 8, and 60.5-66.1
// at 4 and 3; interleaved rows, with half as much in flight per head, lose at 6 (one head per item 62.6
// against 55.7 without a limit, two 54.1 against 53.9).
int rope_occupancy(int layout) {
  static const int v = static_cast<int>(env_int("PT_ROPE_OCCUPANCY", -1));
  return v >= 0 ? v : (layout == 0 ? 0 : 6);
}

template <typename K>
void launch_limited(K kernel, int layout, unsigned grid, hipStream_t st, const RopeArgs& t0,
                    const RopeArgs& t1, int head_dim, const float* c, const float* s,
                    float sign) {
  size_t lds = occupancy_lds(rope_occupancy(layout), 0);
  if (allow_dynamic_lds(reinterpret_cast<const void*>(kernel), lds) != PT_OK) lds = 0;
  hipLaunchKernelGGL(kernel, dim3(grid), dim3(256), lds, st, c, s, head_dim, sign, t0, t1);
}

template <typename T, int LAYOUT, bool ALIGNED, int U>
void launch(RopeTensor& t0, RopeTensor& t1, int head_dim, const float* c, const float* s,
            float sign, hipStream_t st) {
  const int per_row = items_per_row<T, LAYOUT, ALIGNED>(head_dim);
  for (RopeTensor* t : {&t0, &t1}) {
    t->chunks = (t->heads + U - 1) / U;
    t->xstep = t->xs[t->head_dim] * t->chunks;
    t->ystep = t->ys[t->head_dim] * t->chunks;
    t->items = 0;
    if (t->rows > 0) {
      t->n[t->head_dim] = t->chunks;
      t->items = t->rows / t->heads * t->chunks * per_row;
    }
    t->blocks = (t->items + 255) / 256;
  }
  const int64_t blocks = t0.blocks + t1.blocks;
  if (blocks == 0) return;
  // pt_rope has checked that (rows0 + rows1) * head_dim / 2 + 512 < 2^32, which bounds
  // blocks * 256 for every layout.  Streams larger than the caches are touched once:
  // nontemporal loads and stores.
  // Aligned streams whose outputs fit a buffer resource store through it with the
  // write-through policy: the q + k benchmark (4 layers, rotate-half bf16) measured 419.7
  // against 424.6 us per step with nontemporal global stores, the same bits.
  const int64_t bytes = (t0.rows + t1.rows) * head_dim * static_cast<int64_t>(sizeof(T));
  const auto fits = [](const RopeTensor& t) {
    return t.rows == 0 || (t.ybytes > 0 && t.ybytes <= 0x7fffffff);
  };
  const auto args = [](const RopeTensor& t) {
    RopeArgs a{t.x, t.y, {t.xs[0], t.xs[1], t.xs[2]}, {t.ys[0], t.ys[1], t.ys[2]}, t.xstep, t.ystep};
    a.n1 = static_cast<uint32_t>(t.n[1]);
    a.n2 = static_cast<uint32_t>(t.n[2]);
    a.heads = static_cast<uint32_t>(t.heads);
    a.chunks = static_cast<uint32_t>(t.chunks);
    a.items = static_cast<uint32_t>(t.items);
    a.blocks = static_cast<uint32_t>(t.blocks);
    a.seq_dim = t.seq_dim;
    a.head_dim = t.head_dim;
    a.ybytes = static_cast<int>(t.ybytes);
    return a;
  };
  const auto go = [&](auto kernel) {
    launch_limited(kernel, LAYOUT, static_cast<unsigned>(blocks), st, args(t0), args(t1), head_dim, c, s,
                   sign);
  };
  if (bytes <= kNontemporalBytes) {
    go(rope_kernel<T, LAYOUT, ALIGNED, false, false, U>);
  } else if (ALIGNED && fits(t0) && fits(t1)) {
    go(rope_kernel<T, LAYOUT, ALIGNED, true, ALIGNED, U>);
  } else {
    go(rope_kernel<T, LAYOUT, ALIGNED, true, false, U>);
  }
}

template <typename T>
void launch_t(int layout, bool aligned, RopeTensor& t0, RopeTensor& t1, int head_dim,
              const float* c, const float* s, float sign, hipStream_t st) {
  if (layout == 0) {
    if (!aligned) {
      launch<T, 0, false, 1>(t0, t1, head_dim, c, s, sign, st);
    } else if ((t0.rows + t1.rows) * head_dim / Elem<T>::VEC < kTwoHeadVectors) {
      launch<T, 0, true, 1>(t0, t1, head_dim, c, s, sign, st);
    } else {
      launch<T, 0, true, 2>(t0, t1, head_dim, c, s, sign, st);
    }
  } else {
    if (aligned) {
      launch<T, 1, true, 1>(t0, t1, head_dim, c, s, sign, st);
    } else {
      launch<T, 1, false, 1>(t0, t1, head_dim, c, s, sign, st);
    }
  }
}

}  // namespace
}  // namespace pt

using namespace pt;

extern "C" {

int pt_rope(const void* x0, void* y0, const int64_t* desc0, const void* x1, void* y1,
            const int64_t* desc1, int64_t head_dim, const float* cos_table,
            const float* sin_table, int64_t table_rows, int layout, int inverse, int dtype,
            void* stream) {
  if (!valid_dtype(dtype)) return fail(PT_EINVAL, "pt_rope: unknown dtype code");
  if (layout != 0 && layout != 1) return fail(PT_EINVAL, "pt_rope: layout must be 0 or 1");
  if (head_dim <= 0 || head_dim % 2 != 0 || head_dim > (1 << 20))
    return fail(PT_EINVAL, "pt_rope: head_dim must be a positive even number");
  if (!cos_table || !sin_table) return fail(PT_EINVAL, "pt_rope: null cos/sin table");
  if (!desc0) return fail(PT_EINVAL, "pt_rope: null first tensor descriptor");
  if ((x1 == nullptr) != (y1 == nullptr) || (x1 != nullptr && desc1 == nullptr))
    return fail(PT_EINVAL, "pt_rope: second tensor needs x, y and desc");
  const int esize = dtype_size(dtype);
  RopeTensor t0{}, t1{};
  bool al0 = true, al1 = true;
  std::string err;
  if (!parse(x0, y0, desc0, head_dim, table_rows, esize, layout, &t0, &al0, &err))
    return fail(PT_EINVAL, "pt_rope: first tensor: " + err);
  if (x1 != nullptr) {
    if (!parse(x1, y1, desc1, head_dim, table_rows, esize, layout, &t1, &al1, &err))
      return fail(PT_EINVAL, "pt_rope: second tensor: " + err);
  } else {
    t1.n[0] = t1.n[1] = t1.n[2] = 1;
    t1.rows = 0;
    t1.heads = 1;
  }
  // Empty tensors may carry null data pointers; non-empty ones may not.
  if (t0.rows > 0 && (!x0 || !y0)) return fail(PT_EINVAL, "pt_rope: null first tensor");
  const bool aligned = al0 && al1;
  if ((t0.rows + t1.rows) * (head_dim / 2) + 512 > 0xffffffffLL)
    return fail(PT_EUNSUPPORTED, "pt_rope: too many rows for one launch");
  const float sign = inverse ? -1.0f : 1.0f;
  hipStream_t st = as_stream(stream);
  const int hd = static_cast<int>(head_dim);
  if (dtype == PT_FLOAT32) {
    launch_t<float>(layout, aligned, t0, t1, hd, cos_table, sin_table, sign, st);
  } else if (dtype == PT_FLOAT16) {
    launch_t<_Float16>(layout, aligned, t0, t1, hd, cos_table, sin_table, sign, st);
  } else {
    launch_t<__bf16>(layout, aligned, t0, t1, hd, cos_table, sin_table, sign, st);
  }
  return check_launch("pt_rope");
}

}  // extern "C"
