// mf_params.hpp -- the operator of a matrix-free kernel: its forms and their coefficients.
#pragma once

#include "hgdt_internal.hpp"

namespace hgdt {

constexpr int MF_MAXF = 8;
enum { MFK_CG_QUAD = 0, MFK_CG_HEX = 1, MFK_DG_QUAD = 2 };

// the parameters of an appended form, in one record (a kernel's few forms then span few lines of its argument
// block, which the kernel reads before anything else)
struct MfElementForm {
  const double* coef;
  double value, scale;
  int kind;
};
struct MfFaceForm {
  const double* kappa;
  const double* omega;
  double kv, ov, param, scale;
  int kind;
};

struct MfParams {
  int ninst;
  // per row block: first DoF and first element of the instance, cells n0 n1 n2, instance, first and last
  // row of the block relative to the instance's first DoF
  const int64_t* blk;
  int64_t ref_stride; // doubles per instance of the reference data: h0 h1 1/h1 1/h0, element, face, boundary matrices
  int64_t eoff; // offset of the element matrices inside an instance's block (continuous spaces)
  int dirichlet;
  int nef, ncf, nbf;
  int nb; // row blocks (the solver's operator partition): one row or element per lane
  const double* single; // the one coefficient field of every form (kernels that prefetch it), or NULL
  MfVectors v;
  // the forms last: a kernel reads the first nef / ncf / nbf records of each array
  MfElementForm ef[MF_MAXF];
  MfFaceForm ff[2][MF_MAXF]; // [0] inner, [1] boundary forms
};

// the forms of a matrix-free operator (no vectors, blocks of the whole operator)
MfParams mf_params(const Operator& op);

namespace {

// coefficient of a form at element e: the field's value, or the constant
__device__ __forceinline__ double cf(const double* __restrict__ f, double value, int64_t e)
{
  return f ? f[e] : value;
}

} // namespace
} // namespace hgdt
