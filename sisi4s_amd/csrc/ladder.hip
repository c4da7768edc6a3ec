// Kept pair integrals of the particle-particle ladder (see ladder.hpp).
#include "ladder.hpp"

#include <algorithm>

#include "contract.hpp"
#include "tape.hpp"
#include "tensor_ops.hpp"

namespace sisi {

namespace {

// Largest share of the free (or pool-cached) device memory the pair
// integrals may take: 124 GB of about 260 free at No = 40, Nv = 400.
constexpr double kLadderShare = 0.55;

// Device memory that the rest of a run will allocate, at most: the mixer's
// slots not yet filled, the residual's intermediates and permuted copies
// (about 14 doubles tensors and three vertex-sized ones), with a captured
// residual a second set of these.
double run_needs(const Engine &e) {
  const double n2 = 8.0 * double(e.n1() + e.n2()), g = 8.0 * double(e.NG) * e.Nv * e.Nv;
  const sisi_ccsd_opts &o = e.opts;
  double slots = 2.0;
  if (o.mixer == SISI_MIXER_DIIS) {
    int filled = 0;
    for (const DiisSlot &s : e.diis) filled += s.d2.get() != nullptr;
    slots = std::max(0, std::min(o.max_residua, o.max_iterations - e.iteration + filled) - filled);
  }
  return 2.0 * n2 * slots + (o.graphs ? 2.0 : 1.0) * (14.0 * n2 + 3.0 * g);
}

constexpr int64_t kSlab = 4096;  // pairs per FP32 product of the ladder

// Rows of a pair tensor: particle pairs a <= b at b(b+1)/2 + a, then (k, b) at
// k + No b, then hole pairs k <= l at l(l+1)/2 + k.
struct Rows {
  int64_t v, o;
  __host__ __device__ int64_t pairs() const { return v * (v + 1) / 2; }
  __host__ __device__ int64_t opairs() const { return o * (o + 1) / 2; }
  __host__ __device__ int64_t hp() const { return pairs(); }
  __host__ __device__ int64_t hh() const { return pairs() + o * v; }
  __host__ __device__ int64_t count() const { return hh() + opairs(); }
};

enum PackMode { kParticleRows, kHoleRows, kAmplitudes };

struct PackArgs {
  const double *src;  // matrices [c + v d]
  double *out;        // plus parts; minus parts at out + plane
  int64_t plane;
  int v, o, mode, np, b0;  // matrix p + np (b - b0) of kParticleRows, p + o q of the others
  double scale, diag;      // out+- = scale (x +- y), the plus part times diag at c = d
};

// One matrix x[c, d] of v x v into a row of pairs c <= d, its plus and minus
// combinations with the transposed matrix.  HBM bound: each matrix is read
// once, tile by tile, with its mirror tile staged in LDS (both reads run along
// c), and the packed rows are written along c.
__device__ __forceinline__ void pack_pairs_body(const PackArgs &g, int ct, int dt, int z) {
  const int v = g.v;
  if (ct > dt) return;
  const int p = z % g.np, q = z / g.np;
  const Rows rows{v, g.o};
  int64_t row;
  if (g.mode == kParticleRows) {
    const int b = g.b0 + q;
    if (p < g.o) row = rows.hp() + p + int64_t(g.o) * b;
    else if (p - g.o <= b) row = int64_t(b) * (b + 1) / 2 + (p - g.o);
    else return;
  } else {
    if (p > q) return;
    row = int64_t(q) * (q + 1) / 2 + p + (g.mode == kHoleRows ? rows.hh() : 0);
  }
  const double *m = g.src + int64_t(z) * v * v;
  __shared__ double s0[32][33], s1[32][33];  // [d][c] of the tile, and of its mirror
  const int x = int(threadIdx.x) & 31, y0 = int(threadIdx.x) >> 5;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int y = y0 + 8 * r;
    const int c = 32 * ct + x, d = 32 * dt + y, c1 = 32 * dt + x, d1 = 32 * ct + y;
    s0[y][x] = (c < v && d < v) ? m[c + int64_t(v) * d] : 0.0;
    s1[y][x] = (c1 < v && d1 < v) ? m[c1 + int64_t(v) * d1] : 0.0;
  }
  __syncthreads();
  double *out = g.out + row * rows.pairs();
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int y = y0 + 8 * r;
    const int c = 32 * ct + x, d = 32 * dt + y;
    if (d >= v || c > d) continue;
    const double a = s0[y][x], b = s1[x][y];  // m[c,d], m[d,c]
    const int64_t k = int64_t(d) * (d + 1) / 2 + c;
    out[k] = g.scale * (a + b) * (c == d ? g.diag : 1.0);
    out[g.plane + k] = g.scale * (a - b);
  }
}

__global__ __launch_bounds__(256) void pack_pairs_kernel(PackArgs g) {
  pack_pairs_body(g, int(blockIdx.x), int(blockIdx.y), int(blockIdx.z));
}

// The amplitudes' pack: matrices X[:, :, i, j] into rows i <= j.
__host__ __device__ inline PackArgs amplitude_pack(const double *X, double *out, int64_t plane,
                                                   int v, int o) {
  PackArgs a{};
  a.src = X;
  a.out = out;
  a.plane = plane;
  a.v = v;
  a.o = o;
  a.mode = kAmplitudes;
  a.np = o;
  a.scale = 0.5;
  a.diag = 1.0;
  return a;
}

void pack_pairs(Engine &e, const PackArgs &g, int64_t matrices) {
  const unsigned t = unsigned((g.v + 31) / 32);
  PackArgs a = g;
  // the grid's z extent is limited: whole columns of np matrices per launch
  const int64_t step = std::max<int64_t>(1, 65535 / g.np) * g.np;
  SISI_REQUIRE(g.np <= 65535, SISI_ERR_INVALID, "pack_pairs: too many matrices");
  Timed tm(*e.timers, Kind::Bandwidth, 16.0 * double(matrices) * g.v * g.v);
  for (int64_t m = 0; m < matrices; m += step) {
    SISI_REQUIRE(m == 0 || g.mode == kParticleRows, SISI_ERR_INVALID, "pack_pairs: grid");
    const int64_t n = std::min(step, matrices - m);
    a.src = g.src + m * g.v * g.v;
    a.b0 = g.b0 + int(m / g.np);
    hipLaunchKernelGGL(pack_pairs_kernel, dim3(t, t, unsigned(n)), dim3(256), 0, e.stream, a);
  }
  SISI_HIP(hipGetLastError());
}

// Hole-particle rows to Qh[k,b,i,j] and hole rows to W[k,l,i,j].
__device__ __forceinline__ void unpack_holes_body(const double *Qp, int64_t plane, int v, int o,
                                                  double *Qh, double *W, unsigned bx,
                                                  unsigned gx) {
  const Rows rows{v, o};
  const int64_t M = rows.count(), nij = rows.opairs();
  const int64_t hp = int64_t(o) * v, per = hp + rows.opairs();
  const int64_t total = per * nij;
  for (int64_t t = int64_t(bx) * blockDim.x + threadIdx.x; t < total;
       t += int64_t(gx) * blockDim.x) {
    const int64_t r = t % per, n = t / per;
    int j = int((sqrt(8.0 * double(n) + 1.0) - 1.0) * 0.5);
    while (int64_t(j + 1) * (j + 2) / 2 <= n) ++j;
    while (int64_t(j) * (j + 1) / 2 > n) --j;
    const int i = int(n - int64_t(j) * (j + 1) / 2);
    const double plus = Qp[rows.hp() + r + M * n], minus = Qp[plane + rows.hp() + r + M * n];
    const double ij = plus + minus, ji = plus - minus;
    if (r < hp) {
      Qh[r + hp * (i + int64_t(o) * j)] = ij;
      Qh[r + hp * (j + int64_t(o) * i)] = ji;
    } else {
      const int64_t kl = r - hp, oo = int64_t(o) * o;
      int l = int((sqrt(8.0 * double(kl) + 1.0) - 1.0) * 0.5);
      while (int64_t(l + 1) * (l + 2) / 2 <= kl) ++l;
      while (int64_t(l) * (l + 1) / 2 > kl) --l;
      const int k = int(kl - int64_t(l) * (l + 1) / 2);
      W[k + int64_t(o) * l + oo * (i + int64_t(o) * j)] = ij;
      W[l + int64_t(o) * k + oo * (j + int64_t(o) * i)] = ij;
      W[k + int64_t(o) * l + oo * (j + int64_t(o) * i)] = ji;
      W[l + int64_t(o) * k + oo * (i + int64_t(o) * j)] = ji;
    }
  }
}

__global__ __launch_bounds__(256) void unpack_holes_kernel(const double *Qp, int64_t plane, int v,
                                                           int o, double *Qh, double *W) {
  unpack_holes_body(Qp, plane, v, o, Qh, W, blockIdx.x, gridDim.x);
}

// R2 += V + particle rows: a tile of pairs (a in ta, b in tb, ta <= tb) of one
// i <= j is read along a, and its values go to the four places (ab,ij),
// (ba,ji), (ab,ji), (ba,ij); the two mirrored ones through LDS, so that every
// write runs along the first index.  HBM bound: R2 and V once, Q once.
__device__ __forceinline__ void add_pairs_body(const double *Qp, int64_t plane, const double *V,
                                               double *R, int v, int o, int ta, int tb, int ij0,
                                               int nij) {
  if (ta > tb) return;
  const Rows rows{v, o};
  const int64_t M = rows.count(), nv2 = int64_t(v) * v;
  __shared__ double s0[32][33], s1[32][33];
  const int x = int(threadIdx.x) & 31, y0 = int(threadIdx.x) >> 5;
  for (int ij = ij0; ij < o * o; ij += nij) {
    const int i = ij % o, j = ij / o;
    if (i > j) continue;
    const int64_t n = int64_t(j) * (j + 1) / 2 + i;
    const int64_t oij = nv2 * (i + int64_t(o) * j), oji = nv2 * (j + int64_t(o) * i);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int y = y0 + 8 * r;
      const int a = 32 * ta + x, b = 32 * tb + y;
      double p = 0.0, m = 0.0;
      if (b < v && a <= b) {
        const int64_t q = int64_t(b) * (b + 1) / 2 + a + M * n;
        p = Qp[q];
        m = Qp[plane + q];
      }
      const double vij = p + m, vji = p - m;
      s0[y][x] = vij;
      s1[y][x] = vji;
      if (b < v && a <= b) {
        const int64_t k = a + int64_t(v) * b;
        R[oij + k] += V[oij + k] + vij;
        if (i != j) R[oji + k] += V[oji + k] + vji;
      }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int y = y0 + 8 * r;
      const int b = 32 * tb + x, a = 32 * ta + y;  // element (b, a), a < b
      if (b < v && a < b) {
        const int64_t k = b + int64_t(v) * a;
        R[oji + k] += V[oji + k] + s0[x][y];
        if (i != j) R[oij + k] += V[oij + k] + s1[x][y];
      }
    }
    __syncthreads();
  }
}

__global__ __launch_bounds__(256) void add_pairs_kernel(const double *Qp, int64_t plane,
                                                        const double *V, double *R, int v, int o) {
  add_pairs_body(Qp, plane, V, R, v, o, int(blockIdx.x), int(blockIdx.y), int(blockIdx.z),
                 int(gridDim.z));
}

// Grouped forms (batched solver), arguments in ElemArgs: i0 = v, i1 = o,
// n = plane; Pack x0 -> y; Unpack x0 -> y, and W at x1; Add x0, V = x1 -> y.
template <int KIND>
__global__ __launch_bounds__(256) void pairs_grouped(const ElemArgs *const *args,
                                                     const unsigned *__restrict__ start, int n) {
  int lo = 0, hi = n - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (start[mid] <= blockIdx.x) lo = mid;
    else hi = mid - 1;
  }
  const ElemArgs a = *args[lo];
  const unsigned bx = blockIdx.x - start[lo], gx = start[lo + 1] - start[lo];
  const int t = (a.i0 + 31) / 32, x = int(bx) % t, y = int(bx) / t % t, z = int(bx) / (t * t);
  if constexpr (KIND == int(OpKind::PackPairs))
    pack_pairs_body(amplitude_pack(a.x0, a.y, a.n, a.i0, a.i1), x, y, z);
  else if constexpr (KIND == int(OpKind::UnpackHoles))
    unpack_holes_body(a.x0, a.n, a.i0, a.i1, a.y, const_cast<double *>(a.x1), bx, gx);
  else
    add_pairs_body(a.x0, a.n, a.x1, a.y, a.i0, a.i1, x, y, z, a.i1 * a.i1);
}

// Record of one of them on the engine's tape.
bool tape_pairs(Engine &e, OpKind kind, const double *x0, const double *x1, double *y,
                int64_t plane, int64_t blocks) {
  if (!e.tape) return false;
  SISI_REQUIRE(blocks < (int64_t(1) << 31), SISI_ERR_INVALID, "pairs: grid too large");
  TapeOp op;
  op.kind = kind;
  op.gx = unsigned(blocks);
  op.e.x0 = x0;
  op.e.x1 = x1;
  op.e.y = y;
  op.e.n = plane;
  op.e.i0 = e.Nv;
  op.e.i1 = e.No;
  e.tape->ops.push_back(op);
  return true;
}

__global__ __launch_bounds__(256) void asymmetry_kernel(const double *T, int v, int o,
                                                        double *flag) {
  const int64_t nv2 = int64_t(v) * v, total = nv2 * o * o;
  bool bad = false;
  for (int64_t t = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; t < total;
       t += int64_t(gridDim.x) * blockDim.x) {
    const int64_t ab = t % nv2, ij = t / nv2;
    const int64_t u = ab / v + v * (ab % v) + nv2 * (ij / o + o * (ij % o));
    bad = bad || !(T[t] == T[u]);
  }
  if (bad) *flag = 1.0;  // any thread: the same value
}

}  // namespace

bool doubles_symmetric(Engine &e, const double *T2) {
  DBuf flag(&e.pool, 1);
  zero(e, flag.get(), 1);
  const int64_t n = int64_t(e.n2e());
  const int blocks = int(std::min<int64_t>((n + 255) / 256, 4096));
  hipLaunchKernelGGL(asymmetry_kernel, dim3(blocks), dim3(256), 0, e.stream, T2, e.Nv, e.No,
                     flag.get());
  SISI_HIP(hipGetLastError());
  double f = 1.0;
  e.download(&f, flag, 1);
  return f == 0.0;
}

double kept_ladder_bytes(int64_t No, int64_t Nv) {
  const Rows rows{Nv, No};
  return 16.0 * double(rows.count()) * double(rows.pairs());
}

bool kept_ladder_build(Engine &e) {
  if (e.ladder) return true;
  const int64_t o = e.No, v = e.Nv, G = e.NG, P = o + v;
  const Rows rows{v, o};
  const int64_t K = rows.pairs(), M = rows.count();
  const double bytes = kept_ladder_bytes(o, v);
  if (o * o > 65535 || P > 65535) return false;  // grids of pack_pairs
  // an earlier run's block may hold the operands that (T) caches; it builds
  // them again in a fraction of an iteration
  if (e.pool.block_carved()) e.drop_triples_operands();
  // a slice of b: a temporary of v^2 (o + v) doubles per b, at most an eighth
  // of the result and 2 GB (it stays in the engine's pool)
  const int64_t most = std::min<int64_t>(int64_t(1) << 28, M * K / 4);
  const int64_t nb = std::min<int64_t>(v, std::max<int64_t>(1, most / (v * v * P)));
  size_t free_b = 0, total_b = 0;
  if (hipMemGetInfo(&free_b, &total_b) != hipSuccess) return false;
  const double room = e.ladder_share * (double(free_b) + double(e.pool.cached_bytes()));
  const double temporaries = 8.0 * double(v * v * P * nb + G * v * P);
  // (a block kept from an earlier run has its share already)
  const bool kept = double(e.pool.idle_block()) >= bytes;
  if ((!kept && bytes + temporaries > kLadderShare * room) ||
      bytes + temporaries + (e.run_active ? run_needs(e) : 0.0) > room ||
      M >= (int64_t(1) << 31))
    return false;
  double *out = static_cast<double *>(e.pool.take_block(16 * size_t(M) * size_t(K)));
  if (!out) return false;
  e.ladder = out;
  try {
    // Gt[G, c, p]: Gamma_pc with c next to G, p over the holes, then the particles
    DBuf Gt(&e.pool, size_t(G * v * P)), tmp(&e.pool, size_t(v * v * P * nb));
    copy(e, dense(Gt.get(), {G, v, o}), dense(e.Gai.get(), {G, v, o}));
    sum(e, 1.0, dense(e.Gab.get(), {G, v, v}), "Gac", 0.0,
        dense(Gt.get() + G * v * o, {G, v, v}), "Gca");
    PackArgs a{};
    a.out = out;
    a.plane = M * K;
    a.v = int(v);
    a.o = int(o);
    a.scale = 1.0;
    a.diag = 0.5;
    for (int64_t b0 = 0; b0 < v; b0 += nb) {
      const int64_t b1 = std::min(v, b0 + nb), np = o + b1;
      // (pc|bd) at [c, d, p, b], p up to the slice's last particle
      GemmArgs g;
      g.A = Gt.get();
      g.B = Gt.get() + G * v * (o + b0);
      g.sam = g.sbn = G;
      g.sak = g.sbk = 1;
      g.M = int(v * np);
      g.N = int(v * (b1 - b0));
      g.K = int(G);
      g.C = tmp.get();
      g.dm0 = g.dn0 = int(v);
      g.dm1 = int(np);
      g.dn1 = int(b1 - b0);
      g.cm0 = 1;
      g.cm1 = v * v;
      g.cn0 = v;
      g.cn1 = v * v * np;
      gemm(e, SISI_FP64, g);
      a.src = tmp.get();
      a.mode = kParticleRows;
      a.np = int(np);
      a.b0 = int(b0);
      pack_pairs(e, a, np * (b1 - b0));
    }
    a.src = e.Vabij.get();  // (kc|ld) = V_cdkl
    a.mode = kHoleRows;
    a.np = int(o);
    a.b0 = 0;
    pack_pairs(e, a, o * o);
  } catch (const Error &err) {
    e.drop_ladder();
    if (err.code != SISI_ERR_ALLOC) throw;
    return false;
  }
  return true;
}

size_t kept_ladder_q_size(const Engine &e) {
  const Rows rows{e.Nv, e.No};
  return size_t(2 * rows.count() * rows.opairs());
}

void kept_ladder_apply(Engine &e, const double *X, double *Q, double *Qh, double *W,
                       int precision) {
  const int64_t o = e.No, v = e.Nv;
  const Rows rows{v, o};
  const int64_t K = rows.pairs(), M = rows.count(), N = rows.opairs();
  SISI_REQUIRE(e.ladder, SISI_ERR_STATE, "ladder: pair integrals not built");
  DBuf Xp(&e.pool, size_t(2 * N * K));
  const int64_t t32 = (v + 31) / 32;
  if (!tape_pairs(e, OpKind::PackPairs, X, nullptr, Xp.get(), N * K, t32 * t32 * o * o))
    pack_pairs(e, amplitude_pack(X, Xp.get(), N * K, int(v), int(o)), o * o);
  GemmArgs g;  // both combinations as one batch
  g.A = e.ladder;
  g.B = Xp.get();
  g.C = Q;
  g.sam = g.sbn = K;
  g.sak = g.sbk = 1;
  g.M = int(M);
  g.N = int(N);
  g.K = int(K);
  g.batch = 2;
  g.bsa = M * K;
  g.bsb = N * K;
  g.bsc = M * N;
  g.cm0 = 1;
  g.cn0 = M;
  g.dm0 = g.M;
  g.dn0 = g.N;
  // FP32: sums over the pairs in slabs of about kSlab, added in FP64, as the
  // 128 tile sums a launch in one FP32 chain and the sliced ladder's chains
  // are no longer than a slab.  (Recorded products run on the 64 tile, whose
  // sums have two levels.)
  const int64_t slabs = e.tape || precision == SISI_FP64
                            ? 1
                            : std::max<int64_t>(1, (K + kSlab / 2) / kSlab);
  const int64_t step = ((K + slabs - 1) / slabs + 15) / 16 * 16;
  for (int64_t k = 0; k < K; k += step) {
    g.A = e.ladder + k;
    g.B = Xp.get() + k;
    g.K = int(std::min(step, K - k));
    g.beta = k == 0 ? 0.0 : 1.0;
    gemm(e, precision, g);
  }
  const int64_t total = (o * v + N) * N;
  if (tape_pairs(e, OpKind::UnpackHoles, Q, W, Qh, M * N,
                 std::min<int64_t>((total + 255) / 256, 256)))
    return;
  Timed t(*e.timers, Kind::Bandwidth, 32.0 * double(total));
  hipLaunchKernelGGL(unpack_holes_kernel, dim3(unsigned(std::min<int64_t>((total + 255) / 256, 65536))),
                     dim3(256), 0, e.stream, Q, M * N, int(v), int(o), Qh, W);
  SISI_HIP(hipGetLastError());
}

void kept_ladder_add(Engine &e, const double *Q, const double *V, double *R2) {
  const Rows rows{e.Nv, e.No};
  const unsigned t = unsigned((e.Nv + 31) / 32);
  const unsigned gz = unsigned(std::min<int64_t>(int64_t(e.No) * e.No, 65535));
  if (tape_pairs(e, OpKind::AddPairs, Q, V, R2, rows.count() * rows.opairs(),
                 int64_t(t) * t * e.No * e.No))
    return;
  Timed tm(*e.timers, Kind::Bandwidth, 28.0 * double(e.n2e()));
  hipLaunchKernelGGL(add_pairs_kernel, dim3(t, t, gz), dim3(256), 0, e.stream, Q,
                     rows.count() * rows.opairs(), V, R2, e.Nv, e.No);
  SISI_HIP(hipGetLastError());
}

void launch_pairs_grouped(OpKind kind, const ElemArgs *const *args, const unsigned *start, int n,
                          unsigned total, hipStream_t s) {
  switch (kind) {
#define SISI_PAIRS_CASE(K)                                                                      \
  case OpKind::K:                                                                               \
    hipLaunchKernelGGL(pairs_grouped<int(OpKind::K)>, dim3(total), dim3(256), 0, s, args, start, \
                       n);                                                                      \
    break;
    SISI_PAIRS_CASE(PackPairs)
    SISI_PAIRS_CASE(UnpackHoles)
    SISI_PAIRS_CASE(AddPairs)
#undef SISI_PAIRS_CASE
    default: throw Error(SISI_ERR_INVALID, "grouped launch: unknown kind");
  }
  SISI_HIP(hipGetLastError());
}

}  // namespace sisi
