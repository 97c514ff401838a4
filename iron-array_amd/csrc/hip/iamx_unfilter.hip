// iamx_unfilter.hip -- the second launch of a block decode: un-shuffle or
// bit-un-shuffle of every block's streams into its tile of a dense row-major
// destination (or of its transposed image).
//
// A block's streams are the decoded LZ4 scratch, the compressed chunk arena
// (raw streams, read in place) or a constant byte.  Three ways through a block:
//   groups   byte-shuffled and unfiltered 4- and 8-byte elements, untransposed:
//            4 elements a thread, one dword from each byte plane and 4x4 byte
//            transposes (or the elements as they are), stored together; four
//            such groups in flight per thread.
//   staged   bit-shuffled elements, and the others with a transposed
//            destination: some rows of the block at a time (16 KB) are put
//            together in LDS, 32 (bits) or 4 elements a thread, and written out
//            along the destination's rows.
//   general  any other layout, element by element.
// All three are bound by memory, the first two by having enough loads in
// flight: a block is shared by up to 16 workgroups when blocks are few.
#include "iamx_internal.h"

namespace {

using iamx::tr4;
using iamx::transpose8;
using iamx::transpose8_32;
using iamx::u32_any;
using iamx::u32x4_any;

constexpr int kThreads = 128;
// Bytes of a staged piece (9 workgroups then fit a CU's LDS), with an element
// of padding after every 32: a thread's 32 elements start in another bank than
// its neighbour's.
constexpr int kPieceBytes = 16128;
__device__ __forceinline__ int32_t pad(int32_t k) { return k + (k >> 5); }
constexpr int kBufBytes = kPieceBytes + kPieceBytes / 32 + 8;

// A block's streams; a null pointer is a constant one.
struct Streams {
  const IAMX_GLOBAL uint8_t *ptr[IAMX_MAX_STREAMS];
  uint8_t fill[IAMX_MAX_STREAMS];
};

template <typename T>
__device__ __forceinline__ void put_elem(uint8_t *dst, int64_t idx, uint64_t v) {
  reinterpret_cast<T *>(dst)[idx] = (T)v;
}

__device__ __forceinline__ void store_elem(uint8_t *dst, int ts, int64_t idx, uint64_t v) {
  switch (ts) {
    case 8: put_elem<uint64_t>(dst, idx, v); break;
    case 4: put_elem<uint32_t>(dst, idx, v); break;
    case 2: put_elem<uint16_t>(dst, idx, v); break;
    default: put_elem<uint8_t>(dst, idx, v); break;
  }
}

template <int TS>
struct Elem;
template <>
struct Elem<4> {
  typedef uint32_t T;
  static __device__ __forceinline__ T of(uint32_t lo, uint32_t) { return lo; }
};
template <>
struct Elem<8> {
  typedef uint64_t T;
  static __device__ __forceinline__ T of(uint32_t lo, uint32_t hi) { return ((uint64_t)hi << 32) | lo; }
};

// Division of x < 2^31 by a fixed d >= 1: m = floor(2^32 / d) + 1 gives the
// quotient or one more.
struct Div {
  uint32_t d, m;
  __device__ __forceinline__ explicit Div(int32_t v) : d((uint32_t)v), m((uint32_t)(0xffffffffu / (uint32_t)v) + 1u) {}
  __device__ __forceinline__ int32_t operator()(int32_t x) const {
    if (d == 1) return x;
    const uint32_t q = __umulhi((uint32_t)x, m);
    return (int32_t)(q * d > (uint32_t)x ? q - 1 : q);
  }
};

// Byte q of the block's concatenated streams of `ne` bytes each.
__device__ __forceinline__ uint32_t block_byte(const Streams &S, int32_t ne, const Div &by_ne, int32_t q) {
  const int s = by_ne(q);
  return S.ptr[s] ? S.ptr[s][q - s * ne] : S.fill[s];
}

// Where a block's elements are.  load takes four of them from e0 on (those below
// n) as TS words, and join puts them together.
//
// Shuffled: byte j of all n >= 4 elements in stream j of S.  A plane's last
// bytes come from its last dword, shifted (a branch for them a load cost 10% on
// float64 blocks).
template <int TS>
struct Shuffled {
  const Streams &S;
  int32_t n;
  __device__ __forceinline__ void load(int32_t e0, uint32_t *w) const {
    const int32_t at = min(e0, n - 4);
#pragma unroll
    for (int j = 0; j < TS; j++) {
      const IAMX_GLOBAL uint8_t *p = S.ptr[j];
      w[j] = 0x01010101u * S.fill[j];
      if (p) w[j] = *(const IAMX_GLOBAL u32_any *)(p + at);
    }
  }
  __device__ __forceinline__ void join(int32_t e0, uint32_t *w, typename Elem<TS>::T *v) const {
    const int32_t sh = 8 * (e0 - min(e0, n - 4));
#pragma unroll
    for (int j = 0; j < TS; j++) w[j] >>= sh;
    uint32_t lo[4], hi[4] = {0, 0, 0, 0};
    tr4(w[0], w[1], w[2], w[3], lo);
    if (TS == 8) tr4(w[4 % TS], w[5 % TS], w[6 % TS], w[7 % TS], hi);
#pragma unroll
    for (int i = 0; i < 4; i++) v[i] = Elem<TS>::of(lo[i], hi[i]);
  }
};

// Unfiltered: one after the other in streams of `ne` bytes.  Read byte by byte on
// the general path, with this kernel's 16 wavefronts a CU, a 4096x4096 float64
// matrix in blocks of 128^2 took 235 us and its transposed image 342; 55 and 73
// as groups of four.
template <int TS>
struct Plain {
  const Streams &S;
  int32_t n, ne;
  Div by_ne;
  __device__ __forceinline__ void load(int32_t e0, uint32_t *w) const {
    const int32_t q = e0 * TS, s = by_ne(q), o = q - s * ne;
    const IAMX_GLOBAL uint8_t *p = S.ptr[s];
    if (o + 4 * TS <= ne) {
      if (p) {
#pragma unroll
        for (int h = 0; h < TS / 4; h++) {
          const u32x4_any x = *(const IAMX_GLOBAL u32x4_any *)(p + o + 16 * h);
#pragma unroll
          for (int t = 0; t < 4; t++) w[4 * h + t] = x[t];
        }
      } else {
#pragma unroll
        for (int t = 0; t < TS; t++) w[t] = 0x01010101u * S.fill[s];
      }
    } else {  // past a stream's end, or the block's
#pragma unroll
      for (int t = 0; t < TS; t++) w[t] = 0;
#pragma unroll 1
      for (int b = 0; b < 4 * TS && q + b < n * TS; b++) {
        const uint32_t v = block_byte(S, ne, by_ne, q + b) << (8 * (b & 3));
#pragma unroll
        for (int t = 0; t < TS; t++) w[t] |= t == b >> 2 ? v : 0;
      }
    }
  }
  __device__ __forceinline__ void join(int32_t, const uint32_t *w, typename Elem<TS>::T *v) const {
#pragma unroll
    for (int i = 0; i < 4; i++) v[i] = Elem<TS>::of(w[i * (TS / 4)], w[i * (TS / 4) + TS / 4 - 1]);
  }
};

// groups: the block's rows [0, vrows), this workgroup's share.  A 256x256
// float32 block is 16384 groups; with one group in flight the pass moved 2.4
// TB/s on an 8192x8192 matrix (214 us), with four 4.9 TB/s (104 us).
template <int TS, typename SRC>
__device__ __forceinline__ void unfilter_groups(const SRC &src, const iamx_block_job_t &J, uint8_t *__restrict__ dst) {
  typedef typename Elem<TS>::T T;
  constexpr int U = 4;
  const int32_t cols = J.cols, vrows = J.vrows, vcols = J.vcols;
  const int64_t ld = J.dst_ld;
  T *out = reinterpret_cast<T *>(dst) + J.dst_off;
  const Div by_cols(cols);
  const int32_t ng = (int32_t)(((int64_t)vrows * cols + 3) >> 2);
  const int32_t step = kThreads * gridDim.y;
  for (int32_t q0 = blockIdx.y * kThreads + threadIdx.x; q0 < ng; q0 += U * step) {
    uint32_t w[U][TS];
#pragma unroll
    for (int u = 0; u < U; u++)
      if (q0 + u * step < ng) src.load(4 * (q0 + u * step), w[u]);
#pragma unroll
    for (int u = 0; u < U; u++) {
      if (q0 + u * step >= ng) continue;
      const int32_t e0 = 4 * (q0 + u * step);
      T v[4];
      src.join(e0, w[u], v);
      int32_t r = by_cols(e0), c = e0 - r * cols;
      if (c + 4 <= vcols) {  // one row (r < vrows)
        T *o = out + (int64_t)r * ld + c;
        if (TS == 4) {
          *(IAMX_GLOBAL u32x4_any *)iamx::gptr<uint8_t>((uint64_t)o) =
              u32x4_any{(uint32_t)v[0], (uint32_t)v[1], (uint32_t)v[2], (uint32_t)v[3]};
        } else {
          IAMX_GLOBAL u32x4_any *g = (IAMX_GLOBAL u32x4_any *)iamx::gptr<uint8_t>((uint64_t)o);
          g[0] = u32x4_any{(uint32_t)v[0], (uint32_t)((uint64_t)v[0] >> 32), (uint32_t)v[1],
                           (uint32_t)((uint64_t)v[1] >> 32)};
          g[1] = u32x4_any{(uint32_t)v[2], (uint32_t)((uint64_t)v[2] >> 32), (uint32_t)v[3],
                           (uint32_t)((uint64_t)v[3] >> 32)};
        }
      } else {
#pragma unroll
        for (int i = 0; i < 4; i++) {
          if (r < vrows && c < vcols) out[(int64_t)r * ld + c] = v[i];
          if (++c == cols) {
            c = 0;
            ++r;
          }
        }
      }
    }
  }
}

// Where a bit-shuffled block's planes are: 8j .. 8j + 7 one after the other at
// of(j), or bytes fill(j) where that is null.  Back to back in one stream (by a
// table in LDS like the others these took 15 to 30% longer), or one stream for
// each j: 4096x4096 float32 in blocks of 128^2 105 us on the general path, 46 so.
struct OneStream {
  const IAMX_GLOBAL uint8_t *base;
  int32_t n8;
  __device__ __forceinline__ const IAMX_GLOBAL uint8_t *of(int j) const { return base + (int64_t)j * n8; }
  __device__ __forceinline__ uint32_t fill(int) const { return 0; }
  static constexpr bool kAny = false;  // none is null
};
struct ByByte {
  const Streams &S;
  __device__ __forceinline__ const IAMX_GLOBAL uint8_t *of(int j) const { return S.ptr[j]; }
  __device__ __forceinline__ uint32_t fill(int j) const { return S.fill[j]; }
  static constexpr bool kAny = true;
};

// Elements [32 u, 32 u + 32) of a bit-shuffled block, all of them below n8, the
// ones in [ea, eb) into buf, 4 bytes of them at a time (32 planes: twice the
// registers for 64 planes together spilled).
template <int TS, typename BITS>
__device__ __forceinline__ void stage_bits(const BITS &bits, int32_t rowlen, int32_t u, int32_t ea, int32_t eb,
                                           typename Elem<TS>::T *buf) {
  const int32_t e0 = 32 * u;
  uint32_t *out = reinterpret_cast<uint32_t *>(buf);
#pragma unroll 1
  for (int half = 0; half < TS / 4; half++) {
    uint32_t d[32];
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const IAMX_GLOBAL uint8_t *base = bits.of(4 * half + j);
      if (BITS::kAny && !base) {
#pragma unroll
        for (int k = 0; k < 8; k++) d[8 * j + k] = 0x01010101u * bits.fill(4 * half + j);
      } else {
#pragma unroll
        for (int k = 0; k < 8; k++) d[8 * j + k] = *(const IAMX_GLOBAL u32_any *)(base + (int64_t)k * rowlen + 4 * u);
      }
    }
#pragma unroll
    for (int g = 0; g < 4; g++) {
      // Y[j] = bit transpose of byte g of planes 8j..8j+7: byte i is byte j of element 8g+i
      uint32_t ylo[4], yhi[4];
      const uint32_t sel = (uint32_t)g | ((uint32_t)(g + 4) << 8);
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const uint32_t a0 = __builtin_amdgcn_perm(d[8 * j + 1], d[8 * j + 0], sel);
        const uint32_t a1 = __builtin_amdgcn_perm(d[8 * j + 3], d[8 * j + 2], sel);
        const uint32_t a2 = __builtin_amdgcn_perm(d[8 * j + 5], d[8 * j + 4], sel);
        const uint32_t a3 = __builtin_amdgcn_perm(d[8 * j + 7], d[8 * j + 6], sel);
        uint32_t lo = __builtin_amdgcn_perm(a1, a0, 0x05040100u);
        uint32_t hi = __builtin_amdgcn_perm(a3, a2, 0x05040100u);
        transpose8_32(lo, hi);
        ylo[j] = lo;
        yhi[j] = hi;
      }
      uint32_t v[8];
      tr4(ylo[0], ylo[1], ylo[2], ylo[3], v);
      tr4(yhi[0], yhi[1], yhi[2], yhi[3], v + 4);
#pragma unroll
      for (int i = 0; i < 8; i++) {
        const int32_t e = e0 + 8 * g + i;
        if (e >= ea && e < eb) out[pad(e - ea) * (TS / 4) + half] = v[i];
      }
    }
  }
}

// One element of a bit-shuffled block of n elements; elements [n8, n) follow
// the planes of a single stream unshuffled.
template <int TS, typename BITS>
__device__ __forceinline__ typename Elem<TS>::T one_of_bits(const BITS &bits, int32_t n8, int32_t e) {
  uint64_t v = 0;
  if (e < n8) {
#pragma unroll 8
    for (int p = 0; p < 8 * TS; p++) {
      const IAMX_GLOBAL uint8_t *base = bits.of(p >> 3);
      const uint32_t b = !BITS::kAny || base ? base[(int64_t)(p & 7) * (n8 / 8) + (e >> 3)] : bits.fill(p >> 3);
      v |= (uint64_t)((b >> (e & 7)) & 1u) << p;
    }
  } else {
    const IAMX_GLOBAL uint8_t *q = bits.of(0);
#pragma unroll
    for (int b = 0; b < TS; b++)
      v |= (uint64_t)(!BITS::kAny || q ? q[(int64_t)e * TS + b] : bits.fill(0)) << (8 * b);
  }
  return (typename Elem<TS>::T)v;
}

// staged: elements put together from bit planes (src null), or four at a time
// from src.  The general path's byte gathers and scattered 8-byte stores took 199 us
// on a 3001x4507 bit-shuffled float64 matrix (70 here) and 340 on the transposed
// image of a 4001x6007 byte-shuffled one (104 here).
template <int TS, typename BITS, typename SRC>
__device__ __forceinline__ void unfilter_staged(const BITS &bits, const SRC *src, int32_t n8,
                                                const iamx_block_job_t &J, bool tr, typename Elem<TS>::T *buf,
                                                uint8_t *__restrict__ dst) {
  typedef typename Elem<TS>::T T;
  constexpr int32_t kPiece = kPieceBytes / TS;
  const int tid = threadIdx.x;
  const int32_t cols = J.cols, vrows = J.vrows, vcols = J.vcols;
  const int64_t ld = J.dst_ld;
  T *out = reinterpret_cast<T *>(dst) + J.dst_off;
  // pieces of whole rows, or of one row's kPiece columns
  const bool whole = cols <= kPiece;
  const int32_t prows = whole ? kPiece / cols : 1;
  const int32_t segs = whole ? 1 : (vcols + kPiece - 1) / kPiece;
  const int32_t npieces = whole ? (vrows + prows - 1) / prows : vrows * segs;
  for (int32_t k = blockIdx.y; k < npieces; k += gridDim.y) {
    int32_t r0, c0, nr, nc;  // rows and columns of the piece (whole rows keep their padding columns in LDS)
    if (whole) {
      r0 = k * prows;
      nr = min(prows, vrows - r0);
      c0 = 0;
      nc = cols;
    } else {
      r0 = k / segs;
      nr = 1;
      c0 = (k - r0 * segs) * kPiece;
      nc = min(kPiece, vcols - c0);
    }
    const int32_t ea = r0 * cols + c0, eb = ea + (nr - 1) * cols + nc;
    if (!src) {
      const int32_t eq = min(eb, n8 & ~31);  // whole groups of 32 end here
      for (int32_t u = ea / 32 + tid; 32 * u < eq; u += kThreads) stage_bits<TS>(bits, n8 / 8, u, ea, eb, buf);
      for (int32_t e = max(ea, n8 & ~31) + tid; e < eb; e += kThreads) buf[pad(e - ea)] = one_of_bits<TS>(bits, n8, e);
    } else {
      constexpr int U = 4;
      for (int32_t e0 = ea + 4 * tid; e0 < eb; e0 += 4 * U * kThreads) {
        uint32_t w[U][TS];
#pragma unroll
        for (int u = 0; u < U; u++)
          if (e0 + 4 * u * kThreads < eb) src->load(e0 + 4 * u * kThreads, w[u]);
#pragma unroll
        for (int u = 0; u < U; u++) {
          T v[4];
          src->join(e0 + 4 * u * kThreads, w[u], v);
#pragma unroll
          for (int i = 0; i < 4; i++) {
            const int32_t e = e0 + 4 * u * kThreads + i;
            if (e < eb) buf[pad(e - ea)] = v[i];
          }
        }
      }
    }
    __syncthreads();
    const int32_t wc = min(nc, vcols - c0);  // columns written
    if (tr) {
      const Div by_rows(nr);
      for (int32_t i = tid; i < nr * wc; i += kThreads) {
        const int32_t c = by_rows(i), r = i - c * nr;
        out[(int64_t)(c0 + c) * ld + r0 + r] = buf[pad(r * nc + c)];
      }
    } else {
      const Div by_wc(wc);
      for (int32_t i = tid; i < nr * wc; i += kThreads) {
        const int32_t r = by_wc(i), c = i - r * wc;
        out[(int64_t)(r0 + r) * ld + c0 + c] = buf[pad(r * nc + c)];
      }
    }
    __syncthreads();
  }
}

template <int TS, typename SRC>
__device__ __forceinline__ void unfilter_elements(const SRC &src, const iamx_block_job_t &J, bool tr, uint64_t *buf,
                                                  uint8_t *__restrict__ dst) {
  if (tr)
    unfilter_staged<TS>(OneStream{}, &src, 0, J, true, reinterpret_cast<typename Elem<TS>::T *>(buf), dst);
  else
    unfilter_groups<TS>(src, J, dst);
}

__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(4, 8))) void k_unfilter(
    const iamx_block_job_t *__restrict__ jobs, int njobs, const uint8_t *__restrict__ scratch,
    uint8_t *__restrict__ dst) {
  __shared__ iamx_block_job_t J;
  __shared__ Streams S, planes;  // as the job has them; and by byte of the elements
  __shared__ uint64_t buf[kBufBytes / 8];
  const int bj = blockIdx.x;
  if (bj >= njobs) return;
  // the job, a dword a thread, beside its streams, one a thread: many small
  // blocks are bound by the wait for it
  if (threadIdx.x < sizeof(J) / 4)
    reinterpret_cast<uint32_t *>(&J)[threadIdx.x] = reinterpret_cast<const uint32_t *>(jobs + bj)[threadIdx.x];
  if (threadIdx.x < IAMX_MAX_STREAMS) {
    const iamx_block_job_t &G = jobs[bj];
    const int s = threadIdx.x;
    auto at = [&](int k) -> const IAMX_GLOBAL uint8_t * {
      return k >= G.nstreams                 ? nullptr
             : G.kind[k] == IAMX_SRC_ADDR    ? iamx::gptr<const uint8_t>(G.src[k])
             : G.kind[k] == IAMX_SRC_SCRATCH ? iamx::gptr<const uint8_t>((uint64_t)(scratch + G.src[k]))
                                             : nullptr;
    };
    S.ptr[s] = at(s);
    S.fill[s] = s < G.nstreams ? G.fill[s] : 0;
    // one stream holds all planes back to back
    const bool one = G.nstreams == 1;
    const IAMX_GLOBAL uint8_t *p = at(one ? 0 : s);
    planes.ptr[s] = p && one ? p + (int64_t)s * (G.bsize / G.typesize) : p;
    planes.fill[s] = G.fill[one ? 0 : s];
  }
  __syncthreads();
  const int ts = J.typesize, nstreams = J.nstreams;
  const int32_t n = J.bsize / ts;  // elements in the block
  const int32_t cols = J.cols, ne = J.neblock;
  const int64_t ld = J.dst_ld;
  const int64_t base = J.dst_off;
  // a transposed destination takes tile element (r, c) at base + c * ld + r
  const bool tr = (J.filter & IAMX_JOB_TRANSPOSE) != 0;
  const int filter = J.filter & ~IAMX_JOB_TRANSPOSE;
  const bool bits = filter == IAMX_FILTER_BITSHUFFLE || filter == IAMX_FILTER_BITSHUFFLE_V2;
  const bool shuffled = filter == IAMX_FILTER_SHUFFLE && ts > 1;
  const int32_t n8 = filter == IAMX_FILTER_BITSHUFFLE ? n - n % 8 : n;
  if (cols < 1 || J.vrows < 1 || J.vcols < 1) return;
  const bool wide = (int64_t)J.vrows * cols <= n && J.vcols <= cols && (ts == 4 || ts == 8);
  if (wide && shuffled && n >= 4 && (nstreams == ts || nstreams == 1)) {
    if (ts == 4) unfilter_elements<4>(Shuffled<4>{planes, n}, J, tr, buf, dst);
    else unfilter_elements<8>(Shuffled<8>{planes, n}, J, tr, buf, dst);
    return;
  }
  if (wide && bits && nstreams == 1 && S.ptr[0]) {
    const OneStream one = {S.ptr[0], n8};
    if (ts == 4)
      unfilter_staged<4>(one, (const Plain<4> *)nullptr, n8, J, tr, reinterpret_cast<uint32_t *>(buf), dst);
    else
      unfilter_staged<8>(one, (const Plain<8> *)nullptr, n8, J, tr, buf, dst);
    return;
  }
  if (wide && bits && ((nstreams == 1 && !S.ptr[0]) || (nstreams == ts && n % 8 == 0 && ne == n))) {
    if (ts == 4)
      unfilter_staged<4>(ByByte{planes}, (const Plain<4> *)nullptr, n8, J, tr, reinterpret_cast<uint32_t *>(buf), dst);
    else
      unfilter_staged<8>(ByByte{planes}, (const Plain<8> *)nullptr, n8, J, tr, buf, dst);
    return;
  }
  if (wide && !shuffled && !bits && ne >= 1 && (int64_t)ne * nstreams >= J.bsize) {
    if (ts == 4) unfilter_elements<4>(Plain<4>{S, n, ne, Div(ne)}, J, tr, buf, dst);
    else unfilter_elements<8>(Plain<8>{S, n, ne, Div(ne)}, J, tr, buf, dst);
    return;
  }
  // general
  const int64_t sr = tr ? 1 : ld, sc = tr ? ld : 1;
  const Div by_ne(ne), by_cols(cols);
  auto byte_at = [&](int32_t q) -> uint32_t { return block_byte(S, ne, by_ne, q); };
  if (bits) {
    const int32_t rowlen = n8 / 8;
    const int32_t ngroups = rowlen + (n - n8);  // 8-element groups, then tail elements one by one
    for (int32_t g = blockIdx.y * kThreads + threadIdx.x; g < ngroups; g += kThreads * gridDim.y) {
      uint64_t elems[8];
      int cnt;
      int32_t e0;
      if (g < rowlen) {
        for (int i = 0; i < 8; i++) elems[i] = 0;
        for (int j = 0; j < ts; j++) {
          uint64_t x = 0;
#pragma unroll
          for (int k = 0; k < 8; k++) x |= (uint64_t)byte_at((8 * j + k) * rowlen + g) << (8 * k);
          const uint64_t y = transpose8(x);
          for (int i = 0; i < 8; i++) elems[i] |= ((y >> (8 * i)) & 0xffull) << (8 * j);
        }
        cnt = 8;
        e0 = 8 * g;
      } else {
        const int32_t e = n8 + (g - rowlen);
        uint64_t v = 0;
        for (int j = 0; j < ts; j++) v |= (uint64_t)byte_at(e * ts + j) << (8 * j);
        elems[0] = v;
        cnt = 1;
        e0 = e;
      }
      int32_t r = by_cols(e0), c = e0 - r * cols;
      for (int i = 0; i < cnt; i++) {
        if (r < J.vrows && c < J.vcols) store_elem(dst, ts, base + (int64_t)r * sr + (int64_t)c * sc, elems[i]);
        if (++c == cols) { c = 0; ++r; }
      }
    }
    return;
  }
  // byte shuffle (planes) or no filter
  auto plane_byte = [&](int j, int32_t e) -> uint64_t {
    if (nstreams == ts) return S.ptr[j] ? S.ptr[j][e] : S.fill[j];
    return S.ptr[0] ? S.ptr[0][(int64_t)j * n + e] : S.fill[0];
  };
  // (a tile may name more than the block's n elements: those there are)
  const int32_t wcols = shuffled ? min(J.vcols, cols) : J.vcols;
  for (int32_t r = blockIdx.y * (kThreads / 64) + threadIdx.x / 64; r < J.vrows; r += kThreads / 64 * gridDim.y) {
    for (int32_t c = threadIdx.x % 64; c < wcols; c += 64) {
      if ((int64_t)r * cols + c >= n) break;
      const int32_t e = r * cols + c;
      uint64_t v = 0;
      if (shuffled) {
        for (int j = 0; j < ts; j++) v |= plane_byte(j, e) << (8 * j);
      } else {
        for (int j = 0; j < ts; j++) v |= (uint64_t)byte_at(e * ts + j) << (8 * j);
      }
      store_elem(dst, ts, base + (int64_t)r * sr + (int64_t)c * sc, v);
    }
  }
}

}  // namespace

int iamx::launch_unfilter(const iamx_block_job_t *d_blocks, int n_blocks, const void *d_scratch, void *d_dst) {
  // enough workgroups for 16 a CU, up to 16 to a block
  const int want = 16 * g_num_cus;
  const int share = n_blocks >= want ? 1 : (want + n_blocks - 1) / n_blocks;
  IAMX_LAUNCH("unfilter", k_unfilter, dim3((unsigned)n_blocks, (unsigned)(share < 16 ? share : 16)), dim3(kThreads), 0,
              d_blocks, n_blocks, (const uint8_t *)d_scratch, (uint8_t *)d_dst);
  return IAMX_OK;
}
