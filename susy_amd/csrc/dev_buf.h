// Matrices of plane-layout fields read through buffer descriptors: one lane
// offset per operand, the element's plane in the scalar offset.
#ifndef SUSY_DEV_BUF_H
#define SUSY_DEV_BUF_H
#include "susy_internal.h"

template <typename C, typename R>
__device__ __forceinline__ void cfma(C &acc, R ar, R ai, C b) {
  acc.x = fma(ar, b.x, acc.x);
  acc.x = fma(-ai, b.y, acc.x);
  acc.y = fma(ar, b.y, acc.y);
  acc.y = fma(ai, b.x, acc.y);
}

typedef __amdgpu_buffer_rsrc_t Rsrc;

__device__ __forceinline__ Rsrc make_rsrc(const void *p, uint32_t bytes) {
  // dword3 0x00020000: raw (untyped) access on the gfx9 family
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), (short)0, (int)bytes,
                                           0x00020000);
}
template <typename C> __device__ __forceinline__ C bload(Rsrc r, uint32_t voff, uint32_t soff);
template <>
__device__ __forceinline__ double2 bload<double2>(Rsrc r, uint32_t voff, uint32_t soff) {
  return __builtin_bit_cast(double2, __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0));
}
template <>
__device__ __forceinline__ float2 bload<float2>(Rsrc r, uint32_t voff, uint32_t soff) {
  return __builtin_bit_cast(float2, __builtin_amdgcn_raw_buffer_load_b64(r, voff, soff, 0));
}
__device__ __forceinline__ int bload_i32(Rsrc r, uint32_t voff, uint32_t soff) {
  return (int)__builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, 0);
}
// A matrix operand: field descriptor, lane byte offset of the site, uniform
// byte offset of element (0,0); element (i,j) is (i*NCOL+j) planes further.
struct Opnd {
  Rsrc r;
  uint32_t v, s;
};

// acc += s * op(A) * op(B).  TA/TB select the dagger.  B is streamed one row
// at a time (row j of op(B) meets column j of op(A)), so every operand
// element is loaded once and only the accumulator plus one row stay live.
template <typename R, bool TA, bool TB>
__device__ __forceinline__ void mmacc(typename CT<R>::t (&acc)[NCOL][NCOL], R s, Opnd A,
                                      Opnd B, uint32_t plane) {
  typedef typename CT<R>::t C;
#pragma unroll
  for (int j = 0; j < NCOL; j++) {
    C brow[NCOL];
#pragma unroll
    for (int k = 0; k < NCOL; k++) {
      C v = bload<C>(B.r, B.v, B.s + (uint32_t)(TB ? k * NCOL + j : j * NCOL + k) * plane);
      if (TB) v.y = -v.y;
      brow[k] = v;
    }
#pragma unroll
    for (int i = 0; i < NCOL; i++) {
      C a = bload<C>(A.r, A.v, A.s + (uint32_t)(TA ? j * NCOL + i : i * NCOL + j) * plane);
      R ar = s * a.x, ai = TA ? -s * a.y : s * a.y;
#pragma unroll
      for (int k = 0; k < NCOL; k++) cfma(acc[i][k], ar, ai, brow[k]);
    }
  }
}

// Site of a lane in the block order `ord` with chunks of `sites` sites: qq is
// the chunk's position in the queue of XCD x.  False: no such site (*s is then
// out of range).
__device__ __forceinline__ bool ord_site(const DsOrder &ord, int sites, int x, int qq, int lane,
                                         int V, int *s) {
  if (ord.paired) {
    // even chunk k, odd chunk k, even chunk k+1, ... of this XCD's slab
    const int par = qq & 1, pos = qq >> 1;
    const int chunk = x * ord.slab + (ord.paired == 2 ? (pos % ord.T) * ord.P + pos / ord.T : pos);
    const int i = chunk * sites + lane;
    *s = par ? ord.half + i : i;
    return i < (par ? V - ord.half : ord.half);
  }
  *s = (x * ord.slab + qq) * sites + lane;
  return *s < V;
}
// The same for chunks of 64 sites, with site 0 given to a lane that has none.
__device__ __forceinline__ bool ord_site64(const DsOrder &ord, int x, int qq, int lane, int V,
                                           int *s) {
  const bool live = ord_site(ord, 64, x, qq, lane, V, s);
  if (!live) *s = 0;
  return live;
}

#endif  // SUSY_DEV_BUF_H
