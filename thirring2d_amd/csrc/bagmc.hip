// bagmc.hip -- many fermion-bag configurations advanced by Metropolis
// proposals in lockstep on the device (the update loop of fermionbag.c:
// 284-379 with the determinant ratios and accept hooks of
// fluctuation_determinant.c:305-871, for a batch of matrices).
//
// Every matrix b keeps B_b = (D_FF)^-1 over the free sites of its
// configuration (V_b x V_b, identity rows and columns at occupied sites),
// its field and log|det D_FF| with its sign, all on the device.  One step
// proposes one change per matrix and applies it if accepted:
//   a Philox draw picks a site and a move (monomer on/off: rank 1; link
//   on/off, monomer hop to a neighbour: rank 2), the ratio follows from a few
//   entries of B (freeing R: det(D_RR - D_RF B D_FR); occupying O: det of the
//   updated B on O), and a second draw makes the Metropolis decision;
//   freeing: B += (B D_FR - e_R) S^-1 (D_RF B - e_R), the unit diagonal of R
//   out first; occupying: B -= B_FO (B_OO)^-1 B_OF, then unit rows and
//   columns.  A hop frees first, then occupies.
// The matrices do not depend on each other, and rewriting all of B for a
// change of rank 2 is bound by HBM (16 V^2 bytes), so the changes of up to
// kmax / 2 steps are kept as B + U W with V x kmax factors: k_bmc_steps runs
// these steps, one workgroup per matrix, reading B and the factors where an
// entry, a row or a column is needed; k_bmc_flush then adds U W to B on the
// matrix cores, once.  64 matrices of order 256..2304, 50 steps: B was
// rewritten up to 100 times (11.9 of 13.4 ms), now 2 times.
#include "th2d_internal.h"

#include <algorithm>
#include <cmath>
#include <vector>

#include "../../include/th2d_bag.h"
#include "bag_geo.h"

namespace {

constexpr int BMC_KMAX = 64;  // columns of U (rows of W) at most
constexpr int BMC_NT = 512;   // threads of a matrix's workgroup
constexpr int BMC_S = 10;     // sites whose entries of B a ratio needs: 2 x 4 neighbours, 2 occupied

struct BMove {
  int no, nr;
  int occ[2], fr[2], vals[2];
  int acc;
  int ns, site[BMC_S];         // the sites: the freed sites' free neighbours, then occ
  int nbn[2], nb0[2];          // neighbours of freed site a: site[nb0[a]] ..
  double din[2][4], dout[2][4];
  double Sinv[4];  // (D_RR - D_RF B D_FR)^-1, nr x nr
  double Cocc[4];  // -(B1_OO)^-1, no x no
  double ratio;
};

struct BView {
  int count;
  int kmax;          // columns of U and rows of W a matrix has room for
  const BagGeo *G;
  const int *V;
  const long *boff;  // start of B_b (elements)
  const long *foff;  // start of field_b; U_b, W_b start at kmax foff
  double *B;
  int *field;
  double *U, *W;     // [kmax][V_b] each
  int *K;            // factors in use after k_bmc_steps
  double *logabs;
  int *sign;
  long *nacc;
};

__device__ inline double det_small(const double *a, int n)
{
  return n == 1 ? a[0] : a[0] * a[3] - a[1] * a[2];
}

__device__ inline void inv_small(const double *a, int n, double *o)
{
  if (n == 1) {
    o[0] = 1.0 / a[0];
  } else {
    const double d = a[0] * a[3] - a[1] * a[2];
    o[0] = a[3] / d;
    o[1] = -a[1] / d;
    o[2] = -a[2] / d;
    o[3] = a[0] / d;
  }
}

// The move of one step: draws, kind, and the sites whose entries of B it
// needs, with D[nb][R] and D[R][nb] of the freed sites' free neighbours.
__device__ void bmc_move(const BagGeo &G, int V, const int *f, int b, unsigned long long seed,
                         uint32_t ctr, BMove &m, double &u_acc)
{
  m.no = m.nr = m.ns = 0;
  m.acc = 0;
  m.ratio = 0.0;
  m.nbn[0] = m.nbn[1] = m.nb0[0] = m.nb0[1] = 0;
  const uint2 key = make_uint2((uint32_t)seed, (uint32_t)(seed >> 32));
  const uint4 r0 = philox10(make_uint4((uint32_t)b, ctr, 0x42414731u, 0x7468u), key);
  const uint4 r1 = philox10(make_uint4((uint32_t)b, ctr, 0x42414732u, 0x7468u), key);
  const double u_site = u01(r0.x, r0.y), u_kind = u01(r0.z, r0.w), u_dir = u01(r1.x, r1.y);
  u_acc = u01(r1.z, r1.w);
  const int s = min((int)(u_site * V), V - 1);
  const int t = s / G.nx, x = s - t * G.nx;
  if (u_kind < 0.3) {  // a monomer on or off: rank 1
    if (f[s] == 0) {
      m.no = 1;
      m.occ[0] = s;
      m.vals[0] = 1;
    } else if (f[s] == 1) {
      m.nr = 1;
      m.fr[0] = s;
    }
  } else {  // a link on or off, or a monomer hop onto s: rank 2
    const int d = u_dir < 0.5 ? 0 : 1;
    int t2, x2;
    bag_nb(G, t, x, d, t2, x2);
    if (x2 >= 0) {
      const int s2 = t2 * G.nx + x2;
      if (f[s] == 0 && f[s2] == 0) {
        m.no = 2;
        m.occ[0] = s;
        m.occ[1] = s2;
        m.vals[0] = 2 + d;
        m.vals[1] = 4 + d;
      } else if (f[s] == 2 + d && f[s2] == 4 + d) {
        m.nr = 2;
        m.fr[0] = s;
        m.fr[1] = s2;
      } else if (f[s] == 0 && f[s2] == 1) {
        m.no = 1;
        m.occ[0] = s;
        m.vals[0] = 1;
        m.nr = 1;
        m.fr[0] = s2;
      }
    }
  }
  for (int a = 0; a < m.nr; a++) {
    const int ra = m.fr[a], ta = ra / G.nx, xa = ra - ta * G.nx;
    m.nb0[a] = m.ns;
    int n = 0;
    for (int dir = 0; dir < 4; dir++) {
      int t2, x2;
      bag_nb(G, ta, xa, dir, t2, x2);
      if (x2 < 0) continue;
      const int s2 = t2 * G.nx + x2;
      if (f[s2] != 0) continue;
      bool dup = false;
      for (int q = 0; q < n; q++) dup |= m.site[m.nb0[a] + q] == s2;
      if (dup) continue;
      m.site[m.nb0[a] + n] = s2;
      m.din[a][n] = bag_elem(G, s2, ra);
      m.dout[a][n] = bag_elem(G, ra, s2);
      n++;
    }
    m.nbn[a] = n;
    m.ns += n;
  }
  for (int a = 0; a < m.no; a++) m.site[m.ns++] = m.occ[a];
}

// The ratio and the decision from Bs, B on the move's sites (ns x ns).
__device__ void bmc_decide(const BagGeo &G, const double *Bs, double u_acc, BMove &m)
{
  double r_free = 1.0, r_occ = 1.0;
  const int n = m.ns, o0 = n - m.no;  // the occupied sites come last
  bool ok = m.no + m.nr > 0;
  if (ok && m.nr) {
    double S[4];
    for (int a = 0; a < m.nr; a++)
      for (int c = 0; c < m.nr; c++) {
        double val = bag_elem(G, m.fr[a], m.fr[c]);
        for (int p = 0; p < m.nbn[a]; p++)
          for (int q = 0; q < m.nbn[c]; q++)
            val -= m.dout[a][p] * Bs[(m.nb0[a] + p) * BMC_S + m.nb0[c] + q] * m.din[c][q];
        S[a * m.nr + c] = val;
      }
    r_free = det_small(S, m.nr);
    if (r_free == 0.0) ok = false;
    else inv_small(S, m.nr, m.Sinv);
  }
  if (ok && m.no) {
    // B after freeing R, on the sites O (all free now)
    double Boo[4];
    for (int a = 0; a < m.no; a++)
      for (int c = 0; c < m.no; c++) {
        double val = Bs[(o0 + a) * BMC_S + o0 + c];
        for (int p = 0; p < m.nr; p++) {
          double u = 0.0;
          for (int q = 0; q < m.nbn[p]; q++) u += Bs[(o0 + a) * BMC_S + m.nb0[p] + q] * m.din[p][q];
          for (int q = 0; q < m.nr; q++) {
            double w = 0.0;
            for (int r = 0; r < m.nbn[q]; r++) w += m.dout[q][r] * Bs[(m.nb0[q] + r) * BMC_S + o0 + c];
            val += u * m.Sinv[p * m.nr + q] * w;
          }
        }
        Boo[a * m.no + c] = val;
      }
    r_occ = det_small(Boo, m.no);
    if (r_occ == 0.0) ok = false;
    else {
      inv_small(Boo, m.no, m.Cocc);
      for (int k = 0; k < m.no * m.no; k++) m.Cocc[k] = -m.Cocc[k];
    }
  }
  if (ok) {
    m.ratio = r_free * r_occ;
    m.acc = u_acc < fabs(m.ratio) ? 1 : 0;
  }
}

// `nsteps` (at most kmax / 2) proposals of one matrix per workgroup, from
// B with no factors (K = 0).  In B and in the factors the rows and columns of
// occupied sites are 0 apart from B's unit diagonal, so that B + U W holds
// without a mask: occupying a site clears its entries in all of them.
// Bound by the latency of a step (draws, the entries of the ratio, the
// decision: about 5 us) and, when it is accepted, by the columns of B, one
// line per element, that one CU reads.
__global__ void __launch_bounds__(BMC_NT) k_bmc_steps(BView v, unsigned long long seed,
                                                      unsigned long long ctr0, int nsteps,
                                                      th2d_bag_move *trace)
{
  __shared__ BMove m;
  __shared__ double u_acc;
  __shared__ double us[BMC_S][BMC_KMAX], ws[BMC_S][BMC_KMAX];  // U_k, W_k on the sites
  __shared__ double Bs[BMC_S * BMC_S];
  __shared__ double cu[2][BMC_KMAX], cw[2][BMC_KMAX];
  const int b = blockIdx.x, tid = threadIdx.x;
  const BagGeo G = v.G[b];
  const int V = v.V[b];
  int *f = v.field + v.foff[b];
  double *B = v.B + v.boff[b];
  double *U = v.U + v.kmax * v.foff[b], *W = v.W + v.kmax * v.foff[b];
  int K = 0;  // uniform
  for (int step = 0; step < nsteps; step++) {
    if (tid == 0) bmc_move(G, V, f, b, seed, (uint32_t)(ctr0 + (unsigned long long)step), m, u_acc);
    __syncthreads();
    const int ns = m.ns;
    for (int e = tid; e < ns * K; e += BMC_NT) {
      const int q = e / K, k = e - q * K;
      us[q][k] = U[(long)k * V + m.site[q]];
      ws[q][k] = W[(long)k * V + m.site[q]];
    }
    double b0 = 0.0;
    const int p = tid / BMC_S, q = tid % BMC_S;
    const bool mine = p < ns && q < ns;
    if (mine) b0 = B[(long)m.site[p] * V + m.site[q]];
    __syncthreads();
    if (mine) {
      double acc = 0.0;
      for (int k = 0; k < K; k++) acc += us[p][k] * ws[q][k];
      Bs[p * BMC_S + q] = b0 + acc;
    }
    __syncthreads();
    if (tid == 0) {
      bmc_decide(G, Bs, u_acc, m);
      if (trace) {
        th2d_bag_move &o = trace[(long)step * v.count + b];
        o.no = m.no;
        o.nr = m.nr;
        for (int a = 0; a < 2; a++) {
          o.occ[a] = a < m.no ? m.occ[a] : -1;
          o.fr[a] = a < m.nr ? m.fr[a] : -1;
          o.vals[a] = a < m.no ? m.vals[a] : 0;
        }
        o.accepted = m.acc;
        o.pad = 0;
        o.ratio = m.ratio;
      }
    }
    __syncthreads();
    if (m.acc) {  // (uniform)
      const int nr = m.nr, no = m.no;
      if (nr) {
        // U: B D_FR less the unit vectors of R; W: S^-1 (D_RF B less them)
        for (int e = tid; e < nr * K; e += BMC_NT) {
          const int a = e / K, k = e - a * K;
          double x = 0.0, y = 0.0;
          for (int j = 0; j < m.nbn[a]; j++) {
            x += ws[m.nb0[a] + j][k] * m.din[a][j];
            y += m.dout[a][j] * us[m.nb0[a] + j][k];
          }
          cu[a][k] = x;
          cw[a][k] = y;
        }
        __syncthreads();
        for (int i = tid; i < V; i += BMC_NT) {
          double u[2] = {0.0, 0.0}, w[2] = {0.0, 0.0};
          for (int a = 0; a < nr; a++) {
            for (int j = 0; j < m.nbn[a]; j++) {
              const long nb = m.site[m.nb0[a] + j];
              u[a] += B[(long)i * V + nb] * m.din[a][j];
              w[a] += m.dout[a][j] * B[nb * V + i];
            }
          }
#pragma unroll 8
          for (int k = 0; k < K; k++) {
            const double uk = U[(long)k * V + i], wk = W[(long)k * V + i];
            u[0] += uk * cu[0][k];
            w[0] += cw[0][k] * wk;
            if (nr == 2) {
              u[1] += uk * cu[1][k];
              w[1] += cw[1][k] * wk;
            }
          }
          for (int a = 0; a < nr; a++)
            if (i == m.fr[a]) {
              u[a] -= 1.0;
              w[a] -= 1.0;
            }
          for (int a = 0; a < nr; a++) {
            U[(long)(K + a) * V + i] = u[a];
            W[(long)(K + a) * V + i] =
                nr == 2 ? m.Sinv[2 * a] * w[0] + m.Sinv[2 * a + 1] * w[1] : m.Sinv[0] * w[0];
          }
        }
        K += nr;
        __syncthreads();
        if (tid < nr) B[(long)m.fr[tid] * V + m.fr[tid]] = 0.0;  // no longer a unit row
      }
      if (no) {
        // U: the columns O of B; W: -(B_OO)^-1 times the rows O
        for (int e = tid; e < no * K; e += BMC_NT) {
          const int a = e / K, k = e - a * K;
          cu[a][k] = W[(long)k * V + m.occ[a]];
          cw[a][k] = U[(long)k * V + m.occ[a]];
        }
        __syncthreads();
        for (int i = tid; i < V; i += BMC_NT) {
          double u[2] = {0.0, 0.0}, w[2] = {0.0, 0.0};
          for (int a = 0; a < no; a++) {
            u[a] = B[(long)i * V + m.occ[a]];
            w[a] = B[(long)m.occ[a] * V + i];
          }
#pragma unroll 8
          for (int k = 0; k < K; k++) {
            const double uk = U[(long)k * V + i], wk = W[(long)k * V + i];
            u[0] += uk * cu[0][k];
            w[0] += cw[0][k] * wk;
            if (no == 2) {
              u[1] += uk * cu[1][k];
              w[1] += cw[1][k] * wk;
            }
          }
          for (int a = 0; a < no; a++) {
            U[(long)(K + a) * V + i] = u[a];
            W[(long)(K + a) * V + i] =
                no == 2 ? m.Cocc[2 * a] * w[0] + m.Cocc[2 * a + 1] * w[1] : m.Cocc[0] * w[0];
          }
        }
        K += no;
        __syncthreads();
        // the rows and columns O: unit vectors in B, 0 in the factors
        for (int a = 0; a < no; a++) {
          const long o = m.occ[a];
          for (int i = tid; i < V; i += BMC_NT) {
            const double e = i == o ? 1.0 : 0.0;
            B[o * V + i] = e;
            B[(long)i * V + o] = e;
          }
          for (int k = tid; k < K; k += BMC_NT) U[(long)k * V + o] = W[(long)k * V + o] = 0.0;
        }
      }
      if (tid == 0) {
        for (int a = 0; a < nr; a++) f[m.fr[a]] = 0;
        for (int a = 0; a < no; a++) f[m.occ[a]] = m.vals[a];
        v.logabs[b] += log(fabs(m.ratio));
        if (m.ratio < 0) v.sign[b] = -v.sign[b];
        v.nacc[b] += 1;
      }
    }
    __syncthreads();  // the step's stores, before the next step's reads
  }
  if (tid == 0) v.K[b] = K;
}

// B += U W, one 128 x 64 tile per workgroup: wave w holds rows 32 w .. of it
// as 2 x 4 blocks of 16 x 16 of the FP64 matrix instruction, B itself as the
// accumulator.  Bound by HBM (B read and written once); the factors come
// from L2.  (Result register r of lane l: row 4 r + l / 16, column l % 16.)
typedef double bmc_v4d __attribute__((ext_vector_type(4)));
__global__ void __launch_bounds__(256) k_bmc_flush(BView v)
{
  const int b = blockIdx.z;
  const int K = v.K[b], V = v.V[b];
  const int lane = threadIdx.x & 63, l15 = lane & 15, l4 = lane >> 4;
  const int i0 = blockIdx.y * 128 + (threadIdx.x >> 6) * 32, j0 = blockIdx.x * 64;
  if (K == 0 || i0 >= V || j0 >= V) return;
  double *B = v.B + v.boff[b];
  const double *U = v.U + v.kmax * v.foff[b], *W = v.W + v.kmax * v.foff[b];
  bmc_v4d acc[2][4];
#pragma unroll
  for (int a = 0; a < 2; a++)
#pragma unroll
    for (int c = 0; c < 4; c++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int i = i0 + a * 16 + 4 * r + l4, j = j0 + c * 16 + l15;
        acc[a][c][r] = i < V && j < V ? B[(long)i * V + j] : 0.0;
      }
  int iu[2], jw[4];
#pragma unroll
  for (int a = 0; a < 2; a++) iu[a] = min(i0 + a * 16 + l15, V - 1);
#pragma unroll
  for (int c = 0; c < 4; c++) jw[c] = min(j0 + c * 16 + l15, V - 1);
  for (int k0 = 0; k0 < K; k0 += 4) {
    const int k = min(k0 + l4, K - 1);
    const bool in = k0 + l4 < K;
    double av[2], wv[4];
#pragma unroll
    for (int a = 0; a < 2; a++) {
      const double x = U[(long)k * V + iu[a]];
      av[a] = in ? x : 0.0;
    }
#pragma unroll
    for (int c = 0; c < 4; c++) {
      const double x = W[(long)k * V + jw[c]];
      wv[c] = in ? x : 0.0;
    }
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
      for (int c = 0; c < 4; c++)
        acc[a][c] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[a], wv[c], acc[a][c], 0, 0, 0);
  }
#pragma unroll
  for (int a = 0; a < 2; a++)
#pragma unroll
    for (int c = 0; c < 4; c++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int i = i0 + a * 16 + 4 * r + l4, j = j0 + c * 16 + l15;
        if (i < V && j < V) B[(long)i * V + j] = acc[a][c][r];
      }
}

}  // namespace

struct th2d_bag_batch {
  th2d_ctx *ctx = nullptr;
  int count = 0, maxV = 0;
  int kmax = 0;  // factors kept between two additions to B
  std::vector<int> hV;
  std::vector<long> hboff, hfoff;
  long nB = 0, nF = 0;
  th2d_bag_geom *dgeom = nullptr;
  BagGeo *dG = nullptr;
  int *dV = nullptr;
  long *dboff = nullptr, *dfoff = nullptr;
  double *B = nullptr, *work = nullptr, *U = nullptr, *W = nullptr;
  int *field = nullptr, *piv = nullptr, *info = nullptr;
  int *K = nullptr;
  double *logabs = nullptr;
  int *sign = nullptr;
  long *nacc = nullptr;

  BView view() const
  {
    return BView{count, kmax, dG, dV, dboff, dfoff, B, field, U, W, K, logabs, sign, nacc};
  }
};

namespace {

template <typename T>
int dalloc(T **p, size_t n)
{
  return hipMalloc((void **)p, sizeof(T) * std::max<size_t>(n, 1)) == hipSuccess ? TH2D_OK
                                                                                 : TH2D_ENOMEM;
}

// B_b = (D_FF)^-1 of every configuration from scratch, with log|det D_FF|
// and its sign (update_background, fluctuation_determinant.c:126-301).
int bmc_refresh(th2d_bag_batch *s)
{
  th2d_ctx *c = s->ctx;
  th2d_batch bt{s->count, s->maxV, s->dboff, s->dV, s->dfoff};
  TH2D_TRY(th2d_bag_build_masked(c, s->dgeom, s->field, s->dfoff, &bt, s->work, TH2D_PREC_F64));
  TH2D_TRY(th2d_lu_batched(c, &bt, s->work, TH2D_PREC_F64, s->piv, s->info));
  TH2D_TRY(th2d_lu_logdet(c, &bt, s->work, TH2D_PREC_F64, s->piv, s->info, s->logabs, s->sign));
  std::vector<int> info(s->count);
  TH2D_HIP(hipMemcpyAsync(info.data(), s->info, sizeof(int) * s->count, hipMemcpyDeviceToHost,
                          c->stream));
  TH2D_HIP(hipStreamSynchronize(c->stream));
  for (int v : info)
    if (v) return TH2D_ESINGULAR;
  return th2d_lu_inverse(c, &bt, s->work, TH2D_PREC_F64, s->piv, s->B);
}

}  // namespace

extern "C" int th2d_bag_batch_destroy(th2d_bag_batch *s)
{
  if (!s) return TH2D_OK;
  if (s->ctx) (void)hipStreamSynchronize(s->ctx->stream);
  for (void *p : {(void *)s->dgeom, (void *)s->dG, (void *)s->dV, (void *)s->dboff,
                  (void *)s->dfoff, (void *)s->B, (void *)s->work, (void *)s->U, (void *)s->W,
                  (void *)s->field, (void *)s->piv, (void *)s->info, (void *)s->K,
                  (void *)s->logabs, (void *)s->sign, (void *)s->nacc})
    if (p) (void)hipFree(p);
  delete s;
  return TH2D_OK;
}

extern "C" int th2d_bag_batch_create(th2d_ctx *c, int count, const th2d_bag_geom *geoms,
                                     const int *fields, th2d_bag_batch **out)
{
  // count is a grid dimension of every batch launch
  if (!c || count < 1 || count > 65535 || !geoms || !fields || !out) return TH2D_EARG;
  for (int b = 0; b < count; b++) TH2D_TRY(check_bag_geom(&geoms[b]));
  th2d_bag_batch *s = new th2d_bag_batch();
  s->ctx = c;
  s->count = count;
  std::vector<BagGeo> hG(count);
  for (int b = 0; b < count; b++) {
    const int V = geoms[b].nt * geoms[b].nx;
    s->hV.push_back(V);
    s->hboff.push_back(s->nB);
    s->hfoff.push_back(s->nF);
    s->nB += (long)V * V;
    s->nF += V;
    s->maxV = std::max(s->maxV, V);
    hG[b] = bag_geo(&geoms[b]);
  }
  int rc = TH2D_OK;
  auto A = [&](int r) {
    if (rc == TH2D_OK) rc = r;
  };
  A(dalloc(&s->dgeom, count));
  A(dalloc(&s->dG, count));
  A(dalloc(&s->dV, count));
  A(dalloc(&s->dboff, count));
  A(dalloc(&s->dfoff, count));
  A(dalloc(&s->B, s->nB));
  A(dalloc(&s->work, s->nB));
  // few factors for small matrices: adding them to B is cheap there, and
  // they stay a small part of the batch's memory
  s->kmax = s->maxV >= 512 ? BMC_KMAX : (s->maxV >= 128 ? 32 : 8);
  A(dalloc(&s->U, (size_t)s->kmax * s->nF));
  A(dalloc(&s->W, (size_t)s->kmax * s->nF));
  A(dalloc(&s->field, s->nF));
  A(dalloc(&s->piv, s->nF));
  A(dalloc(&s->info, count));
  A(dalloc(&s->K, count));
  A(dalloc(&s->logabs, count));
  A(dalloc(&s->sign, count));
  A(dalloc(&s->nacc, count));
  if (rc != TH2D_OK) {
    th2d_bag_batch_destroy(s);
    return rc;
  }
  hipStream_t st = c->stream;
  rc = hipMemcpyAsync(s->dgeom, geoms, sizeof(th2d_bag_geom) * count, hipMemcpyHostToDevice, st) ||
               hipMemcpyAsync(s->dG, hG.data(), sizeof(BagGeo) * count, hipMemcpyHostToDevice, st) ||
               hipMemcpyAsync(s->dV, s->hV.data(), sizeof(int) * count, hipMemcpyHostToDevice, st) ||
               hipMemcpyAsync(s->dboff, s->hboff.data(), sizeof(long) * count,
                              hipMemcpyHostToDevice, st) ||
               hipMemcpyAsync(s->dfoff, s->hfoff.data(), sizeof(long) * count,
                              hipMemcpyHostToDevice, st) ||
               hipMemcpyAsync(s->field, fields, sizeof(int) * s->nF, hipMemcpyHostToDevice, st) ||
               hipMemsetAsync(s->nacc, 0, sizeof(long) * count, st)
           ? TH2D_EHIP
           : TH2D_OK;
  if (rc == TH2D_OK) rc = bmc_refresh(s);
  if (rc != TH2D_OK) {
    th2d_bag_batch_destroy(s);
    return rc;
  }
  *out = s;
  return TH2D_OK;
}

extern "C" int th2d_bag_batch_refresh(th2d_bag_batch *s)
{
  if (!s) return TH2D_EARG;
  return bmc_refresh(s);
}

extern "C" int th2d_bag_batch_sweep(th2d_bag_batch *s, int nsteps, unsigned long long seed,
                                    unsigned long long counter, th2d_bag_move *trace)
{
  if (!s || nsteps < 0) return TH2D_EARG;
  th2d_ctx *c = s->ctx;
  const BView v = s->view();
  const dim3 gf((unsigned)((s->maxV + 63) / 64), (unsigned)((s->maxV + 127) / 128),
                (unsigned)s->count);
  // runs of steps that the factors have room for (a step adds at most two),
  // each followed by the addition to B: between calls B is whole
  for (long k = 0; k < nsteps; k += s->kmax / 2) {
    hipLaunchKernelGGL(k_bmc_steps, dim3((unsigned)s->count), dim3(BMC_NT), 0, c->stream, v, seed,
                       counter + (unsigned long long)k, (int)std::min<long>(s->kmax / 2, nsteps - k),
                       trace ? trace + (size_t)k * s->count : nullptr);
    hipLaunchKernelGGL(k_bmc_flush, gf, dim3(256), 0, c->stream, v);
  }
  TH2D_HIP(hipGetLastError());
  return TH2D_OK;
}

extern "C" int th2d_bag_batch_state(th2d_bag_batch *s, double *logabs, int *sign, int *fields,
                                    long *accepted)
{
  if (!s) return TH2D_EARG;
  hipStream_t st = s->ctx->stream;
  if (logabs)
    TH2D_HIP(hipMemcpyAsync(logabs, s->logabs, sizeof(double) * s->count, hipMemcpyDeviceToHost, st));
  if (sign) TH2D_HIP(hipMemcpyAsync(sign, s->sign, sizeof(int) * s->count, hipMemcpyDeviceToHost, st));
  if (fields)
    TH2D_HIP(hipMemcpyAsync(fields, s->field, sizeof(int) * s->nF, hipMemcpyDeviceToHost, st));
  if (accepted)
    TH2D_HIP(hipMemcpyAsync(accepted, s->nacc, sizeof(long) * s->count, hipMemcpyDeviceToHost, st));
  TH2D_HIP(hipStreamSynchronize(st));
  return TH2D_OK;
}
