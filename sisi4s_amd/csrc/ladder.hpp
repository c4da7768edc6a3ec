// Particle-particle ladder of a CCSD run on kept pair integrals.
//
// With T_abij = T_baji, X = T2 + T1 T1 and the pair combinations
//   X+-[cd,ij] = (X[c,d,i,j] +- X[d,c,i,j]) / 2      (c <= d, i <= j)
//   V+-[pq,cd] = V[p,q,c,d] +- V[p,q,d,c]            (V+ halved at c = d)
// the undressed ladder Q[p,q,i,j] = sum_cd (pc|qd) X[c,d,i,j] is
//   Q[p,q,i,j] = Q+ + Q-,  Q[p,q,j,i] = Q+ - Q-,  Q+-[pq,ij] = sum_cd V+- X+-,
// a quarter of the multiplications of the four-index form.  V+- does not
// depend on the amplitudes: it is built once per run, for the particle pairs
// (a <= b), the hole-particle pairs (k, b) and the hole pairs (k <= l), and
// the T1 dressing of the vertex (CcsdEnergyFromCoulombIntegrals.cxx:397-400)
// is applied to Q:
//   L[a,b,i,j] = Q[ab] - T_ak Q[kb] - T_bl Q[al] + T_ak T_bl Q[kl].
#pragma once

#include "engine.hpp"

namespace sisi {

// A slice width below the default (No) asks for a ladder in less memory than
// the doubles amplitudes take, (width x width x Nv x Nv): no pair integrals
// are kept then.
inline bool slices_bound_memory(int slice_size, int No) {
  return slice_size > 0 && slice_size < No;
}

// Whether T2 (device) equals its transpose T_baji bit by bit.
bool doubles_symmetric(Engine &e, const double *T2);

// Build the pair integrals (in the pool's block) if the engine has none; false
// when they do not fit (more than kLadderShare of the memory that is free or
// cached in the pool, less than the rest of the run needs left over, or an
// allocation fails).  Between begin_use() and
// end_use() of the pool.
bool kept_ladder_build(Engine &e);
// Device memory of an engine's pair integrals.
double kept_ladder_bytes(int64_t No, int64_t Nv);

// Q of X: Qp (kept_ladder_rows x pairs, + and - parts), its hole-particle
// rows expanded to Qh[k,b,i,j] and its hole rows to W[k,l,i,j].
size_t kept_ladder_q_size(const Engine &e);
void kept_ladder_apply(Engine &e, const double *X, double *Q, double *Qh, double *W,
                       int precision);
// R2 += V + the particle rows of Q (undressed part of the ladder).
void kept_ladder_add(Engine &e, const double *Q, const double *V, double *R2);

}  // namespace sisi
