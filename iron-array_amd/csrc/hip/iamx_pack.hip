// iamx_pack.hip -- the blocks of a dense product, filtered, as the encoder
// reads them: the other direction of the un-filter pass.
#include "iamx_internal.h"

using iamx::tr4;
using iamx::transpose8;
using iamx::transpose8_32;
using iamx::u32_any;
using iamx::u32x4_any;

namespace {

__device__ __forceinline__ uint64_t load_elem(const uint8_t *src, int ts, int64_t idx) {
  switch (ts) {
    case 8: return reinterpret_cast<const uint64_t *>(src)[idx];
    case 4: return reinterpret_cast<const uint32_t *>(src)[idx];
    case 2: return reinterpret_cast<const uint16_t *>(src)[idx];
    default: return src[idx];
  }
}

// A block's tile of the dense array: `rows` x `cols` elements from src, of
// which the first vr rows and vc columns exist (the rest is zero).
struct Tile {
  const uint8_t *src;
  int64_t ld;
  int32_t n, cols;
  int64_t vr, vc;
};

__device__ __forceinline__ Tile tile_of(const iamx_tiling_t &t, const uint8_t *src, int64_t ld, int64_t id) {
  const int64_t nbpc = t.nblocks[0] * t.nblocks[1];
  const int64_t nc = id / nbpc, nb = id % nbpc;
  const int64_t r_in = nb / t.nblocks[1] * t.block[0], c_in = nb % t.nblocks[1] * t.block[1];
  const int64_t gr0 = nc / t.nchunks[1] * t.chunk[0] + r_in, gc0 = nc % t.nchunks[1] * t.chunk[1] + c_in;
  Tile b;
  b.src = src + (gr0 * ld + gc0) * t.typesize;
  b.ld = ld;
  b.n = (int32_t)(t.block[0] * t.block[1]);
  b.cols = (int32_t)t.block[1];
  b.vr = min(t.chunk[0] - r_in, t.shape[0] - gr0);
  b.vc = min(t.chunk[1] - c_in, t.shape[1] - gc0);
  return b;
}

__device__ __forceinline__ uint64_t tile_elem(const Tile &b, int ts, int32_t e) {
  const int32_t r = (int32_t)((uint32_t)e / (uint32_t)b.cols), c = e - r * b.cols;
  return r < b.vr && c < b.vc ? load_elem(b.src, ts, r * b.ld + c) : 0;
}

// the low and high words of elements e0 .. e0 + 3 (zero from e0 + ne on): read
// together, at whatever address, where they share a row and all exist
template <int TS>
__device__ __forceinline__ void load_quad(const Tile &b, int32_t e0, int32_t ne, uint32_t lo[4], uint32_t hi[4]) {
  int32_t r = (int32_t)((uint32_t)e0 / (uint32_t)b.cols), c = e0 - r * b.cols;
  if (ne == 4 && c + 4 <= b.cols && c + 4 <= b.vc && r < b.vr) {
    const IAMX_GLOBAL u32x4_any *s = iamx::gptr<const u32x4_any>((uint64_t)(b.src + (r * b.ld + c) * TS));
    const u32x4_any x = s[0];
    if (TS == 4) {
      lo[0] = x.x; lo[1] = x.y; lo[2] = x.z; lo[3] = x.w;
    } else {
      const u32x4_any y = s[1];
      lo[0] = x.x; hi[0] = x.y; lo[1] = x.z; hi[1] = x.w;
      lo[2] = y.x; hi[2] = y.y; lo[3] = y.z; hi[3] = y.w;
    }
    return;
  }
#pragma unroll
  for (int i = 0; i < 4; i++) {
    uint64_t v = 0;
    if (i < ne && r < b.vr && c < b.vc) v = load_elem(b.src, TS, r * b.ld + c);
    lo[i] = (uint32_t)v;
    if (TS == 8) hi[i] = (uint32_t)(v >> 32);
    if (++c == b.cols) {
      c = 0;
      r++;
    }
  }
}

// 4 bytes (or the first n of them) at any address
__device__ __forceinline__ void store4(uint8_t *d, uint32_t w, int32_t n) {
  if (n == 4) {
    *iamx::gptr<u32_any>((uint64_t)d) = w;
  } else {
    for (int i = 0; i < n; i++) d[i] = (uint8_t)(w >> (8 * i));
  }
}

// Byte planes (or the elements as they are): four consecutive elements per
// thread, two of these sets in flight; bytes j of a set are 4 bytes of plane j.
template <int TS>
__device__ __forceinline__ void pack_bytes(const Tile &b, bool planes, uint8_t *o, int32_t first, int32_t step) {
  auto put = [&](int32_t e0, const uint32_t lo[4], const uint32_t hi[4]) {
    const int32_t ne = min(4, b.n - e0);
    if (!planes) {
      uint8_t *d = o + (int64_t)e0 * TS;
      IAMX_GLOBAL u32x4_any *d4 = iamx::gptr<u32x4_any>((uint64_t)d);
      if (ne == 4 && TS == 4) {
        d4[0] = u32x4_any{lo[0], lo[1], lo[2], lo[3]};
      } else if (ne == 4) {
        d4[0] = u32x4_any{lo[0], hi[0], lo[1], hi[1]};
        d4[1] = u32x4_any{lo[2], hi[2], lo[3], hi[3]};
      } else {
#pragma unroll
        for (int i = 0; i < 3; i++) {
          if (i >= ne) continue;
          store4(d + i * TS, lo[i], 4);
          if (TS == 8) store4(d + i * TS + 4, hi[i], 4);
        }
      }
      return;
    }
    uint32_t w[8];
    tr4(lo[0], lo[1], lo[2], lo[3], w);
    if (TS == 8) tr4(hi[0], hi[1], hi[2], hi[3], w + 4);
#pragma unroll
    for (int j = 0; j < TS; j++) store4(o + (int64_t)j * b.n + e0, w[j], ne);
  };
  const int32_t nq = (int32_t)(((int64_t)b.n + 3) / 4);
  for (int64_t q = first; q < nq; q += 2 * step) {
    uint32_t la[4], ha[4], lb[4], hb[4];
    const int32_t e0 = (int32_t)(4 * q);
    load_quad<TS>(b, e0, min(4, b.n - e0), la, ha);
    const bool two = q + step < nq;
    const int32_t e1 = (int32_t)(4 * (q + step));
    if (two) load_quad<TS>(b, e1, min(4, b.n - e1), lb, hb);
    put(e0, la, ha);
    if (two) put(e1, lb, hb);
  }
}

// Bit planes of elements 8 g .. 8 g + 7: their bytes j are an 8x8 bit matrix
// whose columns are byte g of the planes 8 j .. 8 j + 7; a wavefront stores 64
// bytes of a plane at a time.
template <int TS>
__device__ __forceinline__ void pack_bits(const Tile &b, uint8_t *o, int32_t rowlen, int32_t g) {
  uint32_t la[4], ha[4], lb[4], hb[4], x[8], y[8];
  load_quad<TS>(b, 8 * g, 4, la, ha);
  load_quad<TS>(b, 8 * g + 4, 4, lb, hb);
  tr4(la[0], la[1], la[2], la[3], x);
  tr4(lb[0], lb[1], lb[2], lb[3], y);
  if (TS == 8) {
    tr4(ha[0], ha[1], ha[2], ha[3], x + 4);
    tr4(hb[0], hb[1], hb[2], hb[3], y + 4);
  }
#pragma unroll
  for (int j = 0; j < TS; j++) {
    transpose8_32(x[j], y[j]);
    uint8_t *d = o + (int64_t)(8 * j) * rowlen + g;
#pragma unroll
    for (int k = 0; k < 4; k++) {
      d[(int64_t)k * rowlen] = (uint8_t)(x[j] >> (8 * k));
      d[(int64_t)(4 + k) * rowlen] = (uint8_t)(y[j] >> (8 * k));
    }
  }
}

// Part `part` of `parts` of one block: gather the tile, apply the filter,
// write the bytes at o.
//
// Bound by HBM: every element is read and written once.  With one workgroup a
// block, a 2000^2 float64 product in 256 blocks of 125^2 left the chip a
// wavefront a SIMD, each waiting for its own loads, and odd rows and block
// lengths took divisions, element loads and byte stores: 48 us for 64 MB.
// Several workgroups share a block, so that a thread has eight elements, and
// loads and the stores of byte planes are wide at any address: 16 us (bit
// planes 41 to 19).  A 3001 x 2503 float32 product in blocks of 128^2 45 to 16
// us, 4096^2 in blocks of 256^2 58 to 24, 300 x 170 float64 18.6 to 6.7; two
// groups of 48 ragged products 56 to 14 us each.
//
// WIDE: elements of 4 and 8 bytes.  Other sizes, element by element, are bound by
// the wavefronts there are: in one kernel with the wide paths they took up to 38%
// longer (4096^2 2-byte elements, unfiltered, in blocks of 50^2 64 us, 46 alone).
template <bool WIDE>
__device__ __forceinline__ void pack_part(const iamx_tiling_t &t, const uint8_t *src, int64_t ld, uint8_t *o,
                                          int64_t id, int part, int parts) {
  const Tile b = tile_of(t, src, ld, id);
  const int ts = t.typesize;
  const int32_t first = part * 256 + (int32_t)threadIdx.x, step = parts * 256;
  if (t.filter == IAMX_FILTER_BITSHUFFLE) {
    const int32_t n8 = b.n - b.n % 8, rowlen = n8 / 8;
    for (int64_t g = first; g < rowlen; g += step) {
      if (WIDE && ts == 4) {
        pack_bits<4>(b, o, rowlen, (int32_t)g);
      } else if (WIDE) {
        pack_bits<8>(b, o, rowlen, (int32_t)g);
      } else {
        uint64_t v[8];
        for (int i = 0; i < 8; i++) v[i] = tile_elem(b, ts, (int32_t)(8 * g + i));
        for (int j = 0; j < ts; j++) {
          uint64_t x = 0;
          for (int i = 0; i < 8; i++) x |= ((v[i] >> (8 * j)) & 0xffull) << (8 * i);
          const uint64_t y = transpose8(x);
          for (int k = 0; k < 8; k++) o[(int64_t)(8 * j + k) * rowlen + g] = (uint8_t)(y >> (8 * k));
        }
      }
    }
    for (int64_t e = n8 + first; e < b.n; e += step) {
      const uint64_t v = tile_elem(b, ts, (int32_t)e);
      for (int j = 0; j < ts; j++) o[e * ts + j] = (uint8_t)(v >> (8 * j));
    }
    return;
  }
  const bool shuffled = t.filter == IAMX_FILTER_SHUFFLE && ts > 1;
  if (WIDE && ts == 4) {
    pack_bytes<4>(b, shuffled, o, first, step);
  } else if (WIDE) {
    pack_bytes<8>(b, shuffled, o, first, step);
  } else {
    for (int64_t e = first; e < b.n; e += step) {
      const uint64_t v = tile_elem(b, ts, (int32_t)e);
      for (int j = 0; j < ts; j++) o[shuffled ? (int64_t)j * b.n + e : e * ts + j] = (uint8_t)(v >> (8 * j));
    }
  }
}

// Workgroups (x, y): block id0 + x of C, part y; block `id`'s bytes go to
// out + id * bsize.
template <bool WIDE>
__global__ __launch_bounds__(256) void k_pack(iamx_tiling_t t, const uint8_t *__restrict__ src, int64_t ld,
                                              uint8_t *__restrict__ out, int64_t id0) {
  const int64_t id = id0 + blockIdx.x;
  pack_part<WIDE>(t, src, ld, out + id * (t.block[0] * t.block[1] * t.typesize), id, blockIdx.y, gridDim.y);
}

// The C blocks of any product: blk[2*i] = product, blk[2*i+1] = block index
// inside that product (chunk-major, block-major).
__global__ __launch_bounds__(256) void k_pack_batch(const iamx_batch_pack_t *__restrict__ packs,
                                                    const int32_t *__restrict__ blk, const uint8_t *__restrict__ base_c,
                                                    uint8_t *__restrict__ out) {
  const iamx_batch_pack_t Q = packs[blk[2 * blockIdx.x]];
  const int64_t id = blk[2 * blockIdx.x + 1];
  const iamx_tiling_t &t = Q.tiling;
  uint8_t *o = out + Q.out_off + id * (t.block[0] * t.block[1] * t.typesize);
  if (t.typesize == 4 || t.typesize == 8)
    pack_part<true>(t, base_c + Q.c_off_bytes, t.shape[1], o, id, blockIdx.y, gridDim.y);
  else
    pack_part<false>(t, base_c + Q.c_off_bytes, t.shape[1], o, id, blockIdx.y, gridDim.y);
}

}  // namespace

extern "C" {

IAMX_API int iamx_pack_blocks_range(const iamx_tiling_t *t, const void *d_src, int64_t src_ld, void *d_out,
                                    int64_t chunk_begin, int64_t chunk_end) {
  int rc = iamx::ensure_init();
  if (rc) return rc;
  if (!t || t->typesize < 1 || t->typesize > 8 || t->block[0] <= 0 || t->block[1] <= 0)
    return iamx::set_error(IAMX_EINVAL, "iamx_pack_blocks: bad tiling");
  const int64_t nchunks = t->nchunks[0] * t->nchunks[1], nbpc = t->nblocks[0] * t->nblocks[1];
  if (chunk_begin < 0 || chunk_end > nchunks || chunk_begin > chunk_end)
    return iamx::set_error(IAMX_EINVAL, "iamx_pack_blocks: chunk range [%lld, %lld) outside [0, %lld)",
                           (long long)chunk_begin, (long long)chunk_end, (long long)nchunks);
  const int64_t nblk = (chunk_end - chunk_begin) * nbpc;
  if (nblk == 0) return IAMX_OK;
  if (nblk < 0 || nblk > INT32_MAX) return iamx::set_error(IAMX_EINVAL, "iamx_pack_blocks: bad block count");
  const int64_t parts = (t->block[0] * t->block[1] + 8 * 256 - 1) / (8 * 256);  // eight elements a thread
  const dim3 grid((unsigned)nblk, (unsigned)(parts < 1024 ? parts : 1024));
  if (t->typesize == 4 || t->typesize == 8)
    IAMX_LAUNCH("pack_blocks", k_pack<true>, grid, dim3(256), 0, *t, (const uint8_t *)d_src, src_ld, (uint8_t *)d_out,
                chunk_begin * nbpc);
  else
    IAMX_LAUNCH("pack_blocks", k_pack<false>, grid, dim3(256), 0, *t, (const uint8_t *)d_src, src_ld, (uint8_t *)d_out,
                chunk_begin * nbpc);
  return IAMX_OK;
}

IAMX_API int iamx_pack_blocks(const iamx_tiling_t *t, const void *d_src, int64_t src_ld, void *d_out) {
  if (!t) return iamx::set_error(IAMX_EINVAL, "iamx_pack_blocks: bad tiling");
  return iamx_pack_blocks_range(t, d_src, src_ld, d_out, 0, t->nchunks[0] * t->nchunks[1]);
}

IAMX_API int iamx_pack_batch(const iamx_batch_pack_t *d_packs, const int32_t *d_blocks, int nblocks,
                             const void *base_c, void *d_out) {
  int rc = iamx::ensure_init();
  if (rc) return rc;
  if (nblocks <= 0) return IAMX_OK;
  // the tilings are on the device: as many parts as a 128^2 block has eight elements a thread
  IAMX_LAUNCH("pack_batch", k_pack_batch, dim3(nblocks, 8), dim3(256), 0, d_packs, d_blocks, (const uint8_t *)base_c,
              (uint8_t *)d_out);
  return IAMX_OK;
}

}  // extern "C"
