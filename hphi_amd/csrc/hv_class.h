// Device side of the class layout shared by its kernels (hv_class.hip, serve.hip).
#pragma once
#include <hip/hip_runtime.h>

#include "engine_internal.h"

#define CL_NONE 0xffffffffu  // the term does not act in this block

typedef const uint32_t __attribute__((address_space(4))) *CU32;
typedef const ClsTerm __attribute__((address_space(4))) *CClsTerm;

__device__ __forceinline__ double2 cl_at(const double2 *base, uint32_t off) {
  return *(const double2 *)((const char *)base + off);
}

__device__ __forceinline__ ClsTerm cl_term(CClsTerm p) {
  ClsTerm t;
  t.cre = p->cre;
  t.cim = p->cim;
  t.flip = p->flip;
  t.tmask = p->tmask;
  t.tval = p->tval;
  t.sgn = p->sgn;
  t.lo = p->lo;
  t.tlo = p->tlo;
  t.parity = t.src = 0;
  return t;
}
