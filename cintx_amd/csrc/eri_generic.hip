// Runtime-class fallback kernel: any (li, lj, lk, ll) with l <= 4 (+1 for
// nabla_i), used for the classes that have no compile-time instantiation
// (high angular momentum: (ff|..), (gg|gg), the s..g basis workload).  One
// shell tuple per 256-lane workgroup, or per several when there are few (see
// gen_split).  The g tensors live in LDS when one fits in 150 KB, else in a
// per-workgroup global scratch slice; the Cartesian accumulators live in
// registers (larger blocks in chunks of rows); the chunk results are in
// scratch.  Arithmetic is the same as eri_class_kernel (libcint
// g2e.c:272-690, 4425-4620).
#include <algorithm>

#include "eri_device.h"

namespace cx {

struct GenShape {
  int l[4];
  int lic;  // l[0] + deriv
  int deriv, nr;
  int nrs;  // stride of a root's neighbours in g: nr made odd (LDS banks)
  int di, dj, dk, dl, g4;
  int nf, ncomp;
  int ibase, kbase;
  // work split (gen_split)
  int P;       // primitive tuples per step
  int nslice;  // workgroups that share a tuple's primitive tuples
  int nchunk;  // row chunks of a block
  bool split;  // slices and chunks are workgroups; a second kernel finishes
  int level;   // rows per lane (gen_rows_per_lane)
  bool glds;
  int lds;     // doubles of dynamic LDS
  int slabs;   // slabs that a workgroup finishes at a time (not split)
  int64_t per;  // scratch doubles per workgroup, or per tuple when split
};

// The recurrences of one primitive tuple in three lane-parallel phases.
// generic_vrr, one (axis, root) per lane: the VRR columns m <= MMAX, column m
// staged in slot m of the first NMAX + 1 (i, j) blocks (entry n in block n;
// (A+1)(B+1) >= A+B+1 blocks exist).  generic_bra, one (axis, root, m) per
// lane: reads its staged column, then the bra transfer into g(i, j, slot m).
// generic_ket, one (axis, root, (i, j) block) per lane: the ket transfer of
// that block from the slots m to (k, l).  The work arrays are indexed with
// compile-time positions only (loops unrolled to the largest size, guarded by
// the runtime bounds) so they stay in registers.
constexpr int kChainMax = 10;  // NMAX, MMAX <= 9 (nabla_i on (gg|..))
__device__ void generic_vrr(double* __restrict__ g, const GenShape& S, int axis, int r, double sr,
                            double qr, double wz, double inv_sum, double hij, double hkl,
                            double aij, double akl, double dx, double prb, double qrk) {
  const int NR = S.nrs;
  const int NMAX = S.lic + S.l[1], MMAX = S.l[2] + S.l[3];
  const int BLK = S.dk * S.dl;
  const double sa = sr * inv_sum, oms = qr;
  const double b00 = 0.5 * sa, b10 = 0.5 * sa + oms * hij, b01 = 0.5 * sa + oms * hkl;
  const double c00 = prb - sa * akl * dx;
  const double c0p = qrk + sa * aij * dx;
  double* ga = g + (size_t)axis * S.g4 * NR + r;
  double cm1[kChainMax], c0[kChainMax];
#pragma unroll
  for (int n = 0; n < kChainMax; ++n) {
    cm1[n] = 0.0;
    c0[n] = 0.0;
  }
  c0[0] = (axis == 2) ? wz : 1.0;
#pragma unroll
  for (int n = 0; n + 1 < kChainMax; ++n)
    if (n < NMAX) c0[n + 1] = c00 * c0[n] + (n > 0 ? n * b10 * c0[n - 1] : 0.0);
  for (int m = 0; m <= MMAX; ++m) {
    if (m > 0) {
      // descending n: c0[n - 1] is still the previous column when read
#pragma unroll
      for (int n = kChainMax - 1; n >= 0; --n) {
        double v = c0p * c0[n] + (m - 1) * b01 * cm1[n];
        if (n > 0) v += n * b00 * c0[n - 1];
        cm1[n] = c0[n];
        c0[n] = v;
      }
    }
#pragma unroll
    for (int n = 0; n < kChainMax; ++n)
      if (n <= NMAX) ga[((size_t)n * BLK + m) * NR] = c0[n];
  }
}

__device__ void generic_bra(double* __restrict__ g, const GenShape& S, int axis, int r, int m,
                            double drb, bool ibase) {
  const int NR = S.nrs;
  const int NMAX = S.lic + S.l[1];
  const int A = ibase ? S.lic : S.l[1], B = ibase ? S.l[1] : S.lic;
  const int DJ = S.dj, BLK = S.dk * S.dl;
  double* ga = g + (size_t)axis * S.g4 * NR + r + (size_t)m * NR;
  double t[kChainMax];
#pragma unroll
  for (int a = 0; a < kChainMax; ++a) t[a] = a <= NMAX ? ga[(size_t)a * BLK * NR] : 0.0;
#pragma unroll
  for (int b = 0; b < kChainMax; ++b) {
    if (b > B) break;
    if (b > 0) {
#pragma unroll
      for (int a = 0; a + 1 < kChainMax; ++a)
        if (a <= A + B - b) t[a] = t[a + 1] + drb * t[a];
    }
#pragma unroll
    for (int a = 0; a < kChainMax; ++a) {
      if (a > A) break;
      const int i = ibase ? a : b, j = ibase ? b : a;
      ga[(size_t)(i * DJ + j) * BLK * NR] = t[a];
    }
  }
}

__device__ void generic_ket(double* __restrict__ g, const GenShape& S, int axis, int r, int ij,
                            double drk, bool kbase) {
  const int NR = S.nrs;
  const int MMAX = S.l[2] + S.l[3];
  const int C = kbase ? S.l[2] : S.l[3], D = kbase ? S.l[3] : S.l[2];
  const int DL = S.dl, BLK = S.dk * S.dl;
  double* blk = g + (size_t)axis * S.g4 * NR + r + (size_t)ij * BLK * NR;
  double t[kChainMax];
#pragma unroll
  for (int c = 0; c < kChainMax; ++c) t[c] = c <= MMAX ? blk[c * NR] : 0.0;
#pragma unroll
  for (int d = 0; d < kChainMax; ++d) {
    if (d > D) break;
    if (d > 0) {
#pragma unroll
      for (int c = 0; c + 1 < kChainMax; ++c)
        if (c <= C + D - d) t[c] = t[c + 1] + drk * t[c];
    }
#pragma unroll
    for (int c = 0; c < kChainMax; ++c) {
      if (c > C) break;
      const int k = kbase ? c : d, l = kbase ? d : c;
      blk[(k * DL + l) * NR] = t[c];
    }
  }
}

// Row-blocked gout: a lane owns RPL rows of the block, a row being the
// ncart(LI) elements that share their j, k, l components (LI, the canonical
// i shell's l, is a template parameter so that the row's elements index
// registers).  Per root the lane loads the LI + 1 (nabla_i: LI + 2) g values
// of each axis once and forms every element of the row from them: about one
// LDS read per element instead of three.  The accumulators stay in
// registers; a block with more rows than one chunk (256 RPL rows) is done
// chunk by chunk, each chunk a full pass over the primitive tuples with the
// roots and chains recomputed.  RPL: one for blocks of at most 256 rows, else
// about 16 accumulators per lane (nabla_i: 45), and for blocks of more rows
// than one such chunk about 60 (nabla_i: 90) at one workgroup per CU (the
// register budget of one wave per SIMD), so a (g f|g p) block takes 3 chunks
// instead of 9.  (RPL is a template parameter: a run-time bound on an
// unrolled loop of rows spilled up to 19 KB per lane.)
// GLDS: the g tensors in (dynamic) LDS instead of a global slice.
//
// A step takes P primitive tuples through the phases together (as many g
// tensors as fit in LDS), and a chunk of fewer than 256 rows is worked on by
// several groups of lanes, each on its share of the P: one primitive tuple
// alone keeps 3 NR of the 256 lanes busy in the VRR and as many as the block
// has rows in the last phase, and pays five barriers ((p s|g d) nabla_i: 8 us
// per primitive tuple, whatever its size).
constexpr size_t kGenLdsBytes = 150 * 1024;  // dynamic LDS (gfx950: 160 KB per CU)
constexpr int kGenScalars = 16;              // doubles per primitive tuple beside its roots

// rows per lane of the three levels (an s shell i: as many as do not spill)
__host__ __device__ constexpr int gen_rows_per_lane(int li, bool deriv, int level) {
  if (level == 0) return 1;
  if (li == 0) return deriv ? 15 : (level == 1 ? 12 : 40);
  return cmax(1, (deriv ? (level == 1 ? 15 : 30) : (level == 1 ? 16 : 60)) / ncart(li));
}
// workgroups per CU that the registers are to allow
__host__ __device__ constexpr int gen_waves(bool deriv, int level) {
  return level == 2 || (deriv && level == 1) ? 1 : 2;
}

// The elements of a lane's K rows (g offsets ox, oy, oz) from one g tensor:
// roots outer, rows inner, so that a row's g values of one root are loaded
// once (the loads of the lane's rows are independent and overlap) and every
// element of the row is formed from them.
template <int LI, bool DERIV, int K>
__device__ __forceinline__ void gout_rows(const double* gp, const int* ox, const int* oy,
                                          const int* oz, double* racc, int NR, int up,
                                          double ai2) {
  constexpr int NCI = ncart(LI), NLD = LI + 1 + (DERIV ? 1 : 0), ACC = K * NCI;
  for (int r = 0; r < NR; ++r) {
#pragma unroll
    for (int k = 0; k < K; ++k) {
      double xv[NLD], yv[NLD], zv[NLD];
#pragma unroll
      for (int i = 0; i < NLD; ++i) {
        xv[i] = gp[ox[k] + i * up + r];
        yv[i] = gp[oy[k] + i * up + r];
        zv[i] = gp[oz[k] + i * up + r];
      }
#pragma unroll
      for (int fi = 0; fi < NCI; ++fi) {
        int ix, iy, iz;
        cart_decode(LI, fi, ix, iy, iz);
        if constexpr (!DERIV) {
          racc[k * NCI + fi] += xv[ix] * yv[iy] * zv[iz];
        } else {
          double fx = ai2 * xv[ix + 1];
          double fy = ai2 * yv[iy + 1];
          double fz = ai2 * zv[iz + 1];
          if (ix > 0) fx += (double)ix * xv[ix - 1];
          if (iy > 0) fy += (double)iy * yv[iy - 1];
          if (iz > 0) fz += (double)iz * zv[iz - 1];
          racc[k * NCI + fi] += fx * yv[iy] * zv[iz];
          racc[ACC + k * NCI + fi] += xv[ix] * fy * zv[iz];
          racc[2 * ACC + k * NCI + fi] += xv[ix] * yv[iy] * fz;
        }
      }
    }
  }
}

// The finish of a block, by slabs (the elements of one Cartesian component fl
// of shell l): a slab always fits in LDS, and slabs can go to different
// workgroups.  part: [nslice][ncomp][nf] partial blocks.
//
// generic_slabs: for the nfl slabs from fl on, the sum of the slices' slabs,
// the i, j and k axes turned into spherical harmonics in `lds` (twice nfl
// slabs), left in the slabs' places in slice 0.  A workgroup that finishes a
// whole block takes as many at a time as its LDS holds: each pass is a chain
// of global reads, up to four barriers and writes (5,000 nabla_i (s s|g g)
// tuples of one primitive tuple, 15 slabs each: 0.89 ms one by one, 0.27 ms
// all at once).  generic_last: the elements [e0, e1) of one component of the spherical
// block: the l axis, as a weighted sum over the slabs, and the strided write.
__device__ __forceinline__ double* generic_out(const EriArgs& a, int64_t q, int comp) {
  return a.out + a.out_base + (a.place ? a.place[q] : q) * a.block + comp * a.st_comp;
}

__device__ __forceinline__ int generic_slab_size(const GenShape& S) {
  return ncart(S.l[0]) * ncart(S.l[1]) * ncart(S.l[2]);
}

__device__ void generic_slabs(const EriArgs& a, const GenShape& S, double* part, int comp, int fl,
                              int nfl, double* lds) {
  const int t = threadIdx.x, T = blockDim.x;
  const int n = generic_slab_size(S);
  double* at = part + (size_t)comp * S.nf + (size_t)fl * n;
  for (int e = t; e < nfl * n; e += T) {
    double v = at[e];
    for (int s = 1; s < S.nslice; ++s) v += at[(size_t)s * S.ncomp * S.nf + e];
    lds[e] = v;
  }
  __syncthreads();
  int dims[4] = {ncart(S.l[0]), ncart(S.l[1]), ncart(S.l[2]), nfl};
  double* src = lds;
  double* dst = lds + nfl * n;
  for (int ax = 0; ax < 3; ++ax) {
    if (S.l[ax] < 2 || a.cart) continue;
    c2s_pass_mfma(dst, src, dims, ax, S.l[ax], a.c2s, t, T);
    dims[ax] = nsph(S.l[ax]);
    double* tmp = src;
    src = dst;
    dst = tmp;
    __syncthreads();
  }
  const int ns = dims[0] * dims[1] * dims[2];
  for (int e = t; e < nfl * ns; e += T) at[(e / ns) * n + e % ns] = src[e];
  __syncthreads();
}

__device__ void generic_last(const EriArgs& a, const GenShape& S, int64_t q, const double* part,
                             int comp, int e0, int e1) {
  const int n = generic_slab_size(S);
  const int n0 = a.cart ? ncart(S.l[0]) : nsph(S.l[0]);
  const int n1 = a.cart ? ncart(S.l[1]) : nsph(S.l[1]);
  const int n2 = a.cart ? ncart(S.l[2]) : nsph(S.l[2]);
  const int nfl = ncart(S.l[3]), ns = n0 * n1 * n2;
  const bool same = a.cart || S.l[3] < 2;  // s and p: identity
  const double* row = a.c2s + (size_t)S.l[3] * kC2sM * kC2sC;
  double* o = generic_out(a, q, comp);
  part += (size_t)comp * S.nf;
  for (int e = e0 + (int)threadIdx.x; e < e1; e += blockDim.x) {
    const int ml = e / ns, r = e - ml * ns;
    double v = 0;
    if (same) {
      v = part[(size_t)ml * n + r];
    } else {
      for (int fl = 0; fl < nfl; ++fl) v += row[ml * kC2sC + fl] * part[(size_t)fl * n + r];
    }
    const int mi = r % n0, r1 = r / n0;
    const int mj = r1 % n1, mk = r1 / n1;
    o[mi * a.st[0] + mj * a.st[1] + mk * a.st[2] + ml * a.st[3]] = v;
  }
}

__device__ __forceinline__ int generic_out_size(const EriArgs& a, const GenShape& S) {
  int n = 1;
  for (int c = 0; c < 4; ++c) n *= a.cart ? ncart(S.l[c]) : nsph(S.l[c]);
  return n;
}

// Split launches: a workgroup per slab of every tuple, then one per kGenLast
// elements of the blocks.
constexpr int kGenLast = 1024;
__global__ void __launch_bounds__(256) eri_generic_slab_kernel(EriArgs a, GenShape S) {
  extern __shared__ double gl[];
  const int nfl = ncart(S.l[3]);
  const int64_t b = blockIdx.x / nfl;
  const int fl = (int)(blockIdx.x - b * nfl);
  const int64_t q = b / S.ncomp;
  generic_slabs(a, S, a.scratch + (size_t)q * S.per, (int)(b - q * S.ncomp), fl, 1, gl);
}
__global__ void __launch_bounds__(256) eri_generic_last_kernel(EriArgs a, GenShape S, int pieces) {
  const int64_t b = blockIdx.x / pieces;
  const int e0 = (int)(blockIdx.x - b * pieces) * kGenLast;
  const int64_t q = b / S.ncomp;
  generic_last(a, S, q, a.scratch + (size_t)q * S.per, (int)(b - q * S.ncomp), e0,
               min(e0 + kGenLast, generic_out_size(a, S)));
}

template <bool GLDS, bool DERIV, int LI, int LEVEL>
__global__ void __launch_bounds__(256, gen_waves(DERIV, LEVEL))
    eri_generic_kernel(EriArgs a, GenShape S) {
  constexpr int NC = DERIV ? 3 : 1;
  constexpr int NCI = ncart(LI);                           // elements per row
  constexpr int RPL = gen_rows_per_lane(LI, DERIV, LEVEL);  // rows per lane
  constexpr int ACC = RPL * NCI;                      // elements per lane
  constexpr int CHUNK = 256 * RPL;                    // rows per chunk
  extern __shared__ double gl[];
  __shared__ int list[256];  // surviving primitive tuples, ket primitive << 12 | bra primitive
  __shared__ int wave_count[4];
  const int t = threadIdx.x;
  constexpr int T = 256;
  const int NR = S.nr, NRS = S.nrs;
  const int GSZ = 3 * S.g4 * NRS;  // doubles of one g tensor
  // LDS: [P][GSZ] (GLDS), [P][3 NR] roots, weights and 1 - roots, [P] scalars
  double* const uw = gl + (GLDS ? (size_t)S.P * GSZ : 0);
  double* const sc = uw + (size_t)S.P * 3 * NR;
  const int nfj = ncart(S.l[1]), nfk = ncart(S.l[2]), nfl = ncart(S.l[3]);
  const int SI = S.dj * S.dk * S.dl;
  const int IJ = S.di * S.dj;
  const int ket_tasks = (S.l[2] > 0 && S.l[3] > 0) ? 3 * IJ * NR : 0;
  const int NM = S.l[2] + S.l[3] + 1;  // VRR columns
  const int bra_tasks = 3 * NM * NR;
  const int nrow = nfj * nfk * nfl;
  const int per_tuple = S.split ? S.nchunk * S.nslice : 1;
  // this lane's rows: offsets (in doubles) of their x, y, z g entries with
  // i power 0
  int ox[RPL], oy[RPL], oz[RPL];
  double racc[NC * ACC];
  const int64_t nitem = a.nq * per_tuple;
  for (int64_t item = blockIdx.x; item < nitem; item += gridDim.x) {
    const int64_t it = nitem - 1 - item;  // the longest tuples first
    const int64_t q = it / per_tuple;
    const int sub = (int)(it - q * per_tuple);
    const int sl = sub / S.nchunk, ch0 = sub - sl * S.nchunk;  // (0, 0) when not split
    const int2 pq = a.quartets[q];
    const int boff = a.pair_off[pq.x], koff = a.pair_off[pq.y];
    const double* gb = a.pair_geo + 8 * (size_t)pq.x;
    const double* gk = a.pair_geo + 8 * (size_t)pq.y;
    // coordinate differences (positions are formed from these and the
    // primitive weights, never from an absolute product centre)
    double rji[3], rlk[3], rik[3];
    for (int d = 0; d < 3; ++d) {
      rji[d] = gb[3 + d] - gb[d];
      rlk[d] = gk[3 + d] - gk[d];
      rik[d] = gb[d] - gk[d];
    }
    const double logd_ij = gb[6], logd_kl = gk[6];
    const int np_ij = a.pair_np[pq.x], np_kl = a.pair_np[pq.y];
    const int npq = np_ij * np_kl;
    // scratch of the tuple, or of the workgroup: [nslice][ncomp][nf] partial
    // blocks and (without GLDS) a g tensor for each slice and chunk
    double* const own = a.scratch + (size_t)(S.split ? q : blockIdx.x) * S.per;
    double* const part = own + (size_t)sl * S.ncomp * S.nf;
    double* const g = GLDS ? gl : own + (size_t)S.nslice * S.ncomp * S.nf + (size_t)sub * GSZ;
    const int ch1 = S.split ? ch0 + 1 : S.nchunk;
    for (int ch = ch0; ch < ch1; ++ch) {
      const int r0 = ch * CHUNK;
      const int nrc = min(nrow - r0, CHUNK);     // rows of this chunk
      const int rpl = (nrc + T - 1) / T;         // rows of a lane that are in use
      const int G = rpl > 1 ? 1 : min(T / nrc, S.P);  // groups of lanes
      const int grp = G > 1 ? t / nrc : 0;
      const int lr = t - grp * nrc;              // first row of the lane in the chunk
#pragma unroll
      for (int k = 0; k < RPL; ++k) {
        const int row = r0 + lr + k * T;
        int px = 0, py = 0, pz = 0;
        if (grp < G && row < r0 + nrc) {  // others read entry 0 and are not stored
          const int fj = row % nfj, e2 = row / nfj;
          const int fk = e2 % nfk, fl = e2 / nfk;
          int jx, jy, jz, kx, ky, kz, lx_, ly_, lz_;
          cart_decode(S.l[1], fj, jx, jy, jz);
          cart_decode(S.l[2], fk, kx, ky, kz);
          cart_decode(S.l[3], fl, lx_, ly_, lz_);
          px = (jx * S.dk + kx) * S.dl + lx_;
          py = (jy * S.dk + ky) * S.dl + ly_;
          pz = (jz * S.dk + kz) * S.dl + lz_;
        }
        ox[k] = px * NRS;
        oy[k] = (S.g4 + py) * NRS;
        oz[k] = (2 * S.g4 + pz) * NRS;
      }
#pragma unroll
      for (int k = 0; k < NC * ACC; ++k) racc[k] = 0.0;
      int before = 0;  // survivors among the candidates of earlier rounds
      for (int c0 = 0; c0 < npq; c0 += T) {
        // one candidate primitive tuple per lane; of the survivors, in
        // order, this slice lists every nslice-th
        const int cand = c0 + t;
        const int kp = cand / np_ij, ip = cand - kp * np_ij;
        bool ok = cand < npq;
        if (ok) {
          const double ccekl =
              a.three_center ? 0.0 : a.prim[8 * (size_t)(koff + kp) + 6] - a.lkl_ceil * logd_kl;
          const double cceij = a.prim[8 * (size_t)(boff + ip) + 6] - a.lij_ceil * logd_ij;
          // (libcint zeroes the prefactor of a bra pair with cce >= expcutoff)
          ok = ccekl <= a.expcutoff && cceij <= a.expcutoff - ccekl && cceij < a.expcutoff;
        }
        const unsigned long long mask = __ballot(ok);
        if ((t & 63) == 0) wave_count[t >> 6] = __popcll(mask);
        __syncthreads();
        int rank = before + __popcll(mask & ((1ull << (t & 63)) - 1)), total = before;
        for (int w = 0; w < T / 64; ++w) {
          if (w < t >> 6) rank += wave_count[w];
          total += wave_count[w];
        }
        auto taken = [&](int n) { return n > sl ? (n - sl - 1) / S.nslice + 1 : 0; };
        const int first = taken(before), nlist = taken(total) - first;
        if (ok && rank % S.nslice == sl) list[rank / S.nslice - first] = kp << 12 | ip;
        before = total;
        __syncthreads();
        if (a.counters && t == 0 && ch == 0 && nlist > 0)
          atomicAdd(a.counters, (unsigned long long)nlist);
        for (int b = 0; b < nlist; b += S.P) {
          const int np = min(S.P, nlist - b);  // primitive tuples of this step
          for (int u = t; u < np * NR; u += T) {
            const int pp = u / NR, r = u - pp * NR;
            const int ki = list[b + pp];
            const double* pk = a.prim + 8 * (size_t)(koff + (ki >> 12));
            const double* pi = a.prim + 8 * (size_t)(boff + (ki & 4095));
            const double aij = pi[0], akl = pk[0];
            // transfer base of each side: libcint's (lk > ll) unless both
            // shells carry angular momentum, then the centre of the larger
            // exponent (Q lies near it, so the VRR terms stay small and the
            // transfer adds instead of cancelling; FP64 results of
            // (f|g)-type quartets with distant centres otherwise lose up to
            // 7 digits)
            const bool kb = (S.l[2] > 0 && S.l[3] > 0) ? (pk[7] >= akl - pk[7]) : (S.kbase != 0);
            const bool ib = (S.lic > 0 && S.l[1] > 0) ? (pi[7] >= aij - pi[7]) : (S.ibase != 0);
            double dx[3], prb[3], qrk[3], rr = 0;
            for (int d = 0; d < 3; ++d) {
              const double pr = pi[2] * rji[d], qk = pk[2] * rlk[d];  // P - R_i, Q - R_k
              dx[d] = (rik[d] + pr) - qk;
              rr += dx[d] * dx[d];
              prb[d] = ib ? pr : -pi[1] * rji[d];
              qrk[d] = kb ? qk : -pk[1] * rlk[d];
            }
            double root_inv, inv_sum;
            rsqrt_rcp(aij + akl, root_inv, inv_sum);
            const double hij = pi[5], hkl = pk[5];
            const double fac = a.common * pi[4] * pk[4];
            const double fac1 = 4.0 * hij * hkl * root_inv * fac;
            const double a0 = aij * akl * inv_sum;
            const double x = a0 * rr;
            double sr, qr, w;
            rys_eval(a.rys, NR, r, x, sr, qr, w);
            double* up = uw + (size_t)pp * 3 * NR;
            up[r] = sr;
            up[NR + r] = w * fac1;
            up[2 * NR + r] = qr;
            if (r == 0) {
              double* s = sc + pp * kGenScalars;
              s[0] = inv_sum;
              s[1] = hij;
              s[2] = hkl;
              s[3] = aij;
              s[4] = akl;
              for (int d = 0; d < 3; ++d) {
                s[5 + d] = dx[d];
                s[8 + d] = prb[d];
                s[11 + d] = qrk[d];
              }
              s[14] = pi[7];
              s[15] = (ib ? 1.0 : 0.0) + (kb ? 2.0 : 0.0);
            }
          }
          __syncthreads();
          for (int u = t; u < np * 3 * NR; u += T) {
            const int pp = u / (3 * NR), c = u - pp * 3 * NR;
            const int axis = c / NR, r = c - axis * NR;
            const double* s = sc + pp * kGenScalars;
            const double* up = uw + (size_t)pp * 3 * NR;
            generic_vrr(g + (size_t)pp * GSZ, S, axis, r, up[r], up[2 * NR + r], up[NR + r], s[0],
                        s[1], s[2], s[3], s[4], s[5 + axis], s[8 + axis], s[11 + axis]);
          }
          __syncthreads();
          for (int u = t; u < np * bra_tasks; u += T) {
            const int pp = u / bra_tasks, c = u - pp * bra_tasks;
            const int r = c % NR, rest = c / NR;
            const int m = rest % NM, axis = rest / NM;
            const bool ib = ((int)sc[pp * kGenScalars + 15] & 1) != 0;
            const double d = axis == 0 ? rji[0] : (axis == 1 ? rji[1] : rji[2]);
            generic_bra(g + (size_t)pp * GSZ, S, axis, r, m, ib ? -d : d, ib);
          }
          __syncthreads();
          if (ket_tasks) {  // (with min(lk, ll) = 0 the slots are already (k, l))
            for (int u = t; u < np * ket_tasks; u += T) {
              const int pp = u / ket_tasks, c = u - pp * ket_tasks;
              const int r = c % NR, rest = c / NR;
              const int ij = rest % IJ, axis = rest / IJ;
              const bool kb = ((int)sc[pp * kGenScalars + 15] & 2) != 0;
              const double d = axis == 0 ? rlk[0] : (axis == 1 ? rlk[1] : rlk[2]);
              generic_ket(g + (size_t)pp * GSZ, S, axis, r, ij, kb ? -d : d, kb);
            }
            __syncthreads();
          }
          const int up = SI * NRS;  // stride of the i power
          for (int pp = grp; pp < (grp < G ? np : 0); pp += G) {
            const double* gp = g + (size_t)pp * GSZ;
            const double ai2 = DERIV ? -2.0 * sc[pp * kGenScalars + 14] : 0.0;
            gout_rows<LI, DERIV, RPL>(gp, ox, oy, oz, racc, NR, up, ai2);
          }
          __syncthreads();
        }
      }
      if (a.counters && t == 0 && ch == 0 && sl == 0 && before > 0) atomicAdd(a.counters + 1, 1ull);
      // the chunk's results to the partial block (element fi of row `row` is
      // fi + NCI row: i fastest), the groups adding theirs in turn
      for (int gg = 0; gg < G; ++gg) {
        if (grp == gg) {
#pragma unroll
          for (int k = 0; k < RPL; ++k) {
            const int row = r0 + lr + k * T;
            if (row < r0 + nrc) {
#pragma unroll
              for (int comp = 0; comp < NC; ++comp)
#pragma unroll
                for (int fi = 0; fi < NCI; ++fi) {
                  double* d = part + (size_t)comp * S.nf + (size_t)row * NCI + fi;
                  const double v = racc[comp * ACC + k * NCI + fi];
                  *d = gg == 0 ? v : *d + v;
                }
            }
          }
        }
        __syncthreads();
      }
    }
    if (!S.split) {
      for (int comp = 0; comp < S.ncomp; ++comp) {
        for (int fl = 0; fl < nfl; fl += S.slabs)
          generic_slabs(a, S, part, comp, fl, min(S.slabs, nfl - fl), gl);
        generic_last(a, S, q, part, comp, 0, generic_out_size(a, S));
      }
      __syncthreads();
    }
  }
}

// How a launch of nq tuples of one class is cut up, `most` primitive tuples
// in the longest of them.  A large launch runs a workgroup per tuple, chunks
// in turn, and finishes blocks itself; one of few tuples makes workgroups of
// the chunks and of slices of the primitive tuples, at least 2 P of them each,
// until they fill the chip once and as long as the partial blocks stay under
// 256 MB, and finishes them in two more kernels.  (Four times as many slices:
// int2e_sph on an s..g basis, 60,000 tuples in 120 classes on parallel
// chains, 13.7 ms instead of 9.9 ms; half as many: 13.2 ms.)
static GenShape gen_split(const int* l, int deriv, int64_t nq, int64_t most) {
  GenShape S;
  for (int c = 0; c < 4; ++c) S.l[c] = l[c];
  S.deriv = deriv;
  S.lic = l[0] + deriv;
  S.nr = (S.lic + l[1] + l[2] + l[3]) / 2 + 1;
  S.nrs = S.nr | 1;
  S.di = S.lic + 1;
  S.dj = l[1] + 1;
  S.dk = l[2] + 1;
  S.dl = l[3] + 1;
  S.g4 = S.di * S.dj * S.dk * S.dl;
  S.nf = ncart(l[0]) * ncart(l[1]) * ncart(l[2]) * ncart(l[3]);
  S.ncomp = deriv ? 3 : 1;
  S.ibase = S.lic > l[1];
  S.kbase = l[2] > l[3];
  const int nrow = ncart(l[1]) * ncart(l[2]) * ncart(l[3]);
  S.level = 0;
  while (S.level < 2 && nrow > 256 * gen_rows_per_lane(l[0], deriv != 0, S.level)) ++S.level;
  const int rows = 256 * gen_rows_per_lane(l[0], deriv != 0, S.level);
  S.nchunk = (nrow + rows - 1) / rows;
  const int gsz = 3 * S.g4 * S.nrs, per_prim = 3 * S.nr + kGenScalars;
  const int cap = (int)kGenLdsBytes / 8;
  S.glds = gsz + per_prim <= cap;
  // two workgroups per CU where the registers allow it and one g tensor fits
  const int two = 9600;  // doubles: 75 KB
  const int room = gen_waves(deriv != 0, S.level) == 2 && gsz + per_prim <= two ? two : cap;
  S.P = S.glds ? std::min(16, room / (gsz + per_prim)) : 1;
  S.P = (int)std::max<int64_t>(1, std::min<int64_t>(S.P, most));
  S.nslice = 1;
  S.split = false;
  if (nq < kGenFew) {
    const int64_t want = (kGenFill + nq * S.nchunk - 1) / (nq * S.nchunk);
    S.nslice = (int)std::max<int64_t>(1, std::min(want, most / (2 * S.P)));
    const auto bytes = [&] {
      return nq * 8 * ((int64_t)S.nslice * S.ncomp * S.nf +
                       (S.glds ? 0 : (int64_t)S.nslice * S.nchunk * gsz));
    };
    while (S.nslice > 1 && bytes() > ((int64_t)256 << 20)) S.nslice /= 2;
    S.split = S.nslice * S.nchunk > 1 && bytes() <= ((int64_t)256 << 20);
    if (!S.split) S.nslice = 1;
  }
  S.lds = (S.glds ? S.P * gsz : 0) + S.P * per_prim;
  S.slabs = 1;
  if (!S.split) {  // room for more slabs, short of what costs a workgroup per CU
    const int slab = 2 * ncart(l[0]) * ncart(l[1]) * ncart(l[2]);
    const int free_lds = gen_waves(deriv != 0, S.level) == 2 ? two / 2 : cap;
    S.lds = std::max({S.lds, slab, std::min(ncart(l[3]) * slab, free_lds)});
    S.slabs = std::min(ncart(l[3]), S.lds / slab);
  }
  S.per = (int64_t)S.nslice * S.ncomp * S.nf +
          (S.glds ? 0 : (S.split ? (int64_t)S.nslice * S.nchunk : 1) * gsz);
  S.per = (S.per + 31) / 32 * 32;
  return S;
}

// doubles of scratch that a launch needs
int64_t generic_scratch(const int* l, int deriv, int64_t nq, int64_t most) {
  const GenShape S = gen_split(l, deriv, nq, most);
  return S.per * (S.split ? nq : std::min<int64_t>(nq, kGenericGrid));
}

int generic_prims_per_step(const int* l, int deriv, int64_t nq, int64_t most) {
  return gen_split(l, deriv, nq, most).P;
}

hipError_t launch_generic(const EriArgs& a, const int* l, int deriv, int64_t most,
                          hipStream_t s) {
  const GenShape S = gen_split(l, deriv, a.nq, most);
  const size_t dyn = (size_t)S.lds * 8;
  const int64_t items = S.split ? a.nq * S.nchunk * S.nslice
                                : std::min<int64_t>(a.nq, kGenericGrid);
  const dim3 grid((unsigned)items);
#define CX_GEN(GLDS, DERIV, LI, LEVEL)                                                       \
  hipLaunchKernelGGL((eri_generic_kernel<GLDS, DERIV, LI, LEVEL>), grid, dim3(256), dyn, s, a, S)
#define CX_GEN_LEVEL(DERIV, LI)                       \
  do {                                                \
    if (S.level == 0) CX_GEN(true, DERIV, LI, 0);     \
    else if (S.level == 1) CX_GEN(true, DERIV, LI, 1); \
    else CX_GEN(true, DERIV, LI, 2);                  \
  } while (0)
  if (!S.glds) {  // nabla_i on (g g|g g) alone is beyond the LDS
    if (!deriv || l[0] != 4 || S.level != 2) return hipErrorInvalidValue;
    CX_GEN(false, true, 4, 2);
  } else {
    switch (l[0] * 2 + (deriv ? 1 : 0)) {
      case 0: CX_GEN_LEVEL(false, 0); break;
      case 1: CX_GEN_LEVEL(true, 0); break;
      case 2: CX_GEN_LEVEL(false, 1); break;
      case 3: CX_GEN_LEVEL(true, 1); break;
      case 4: CX_GEN_LEVEL(false, 2); break;
      case 5: CX_GEN_LEVEL(true, 2); break;
      case 6: CX_GEN_LEVEL(false, 3); break;
      case 7: CX_GEN_LEVEL(true, 3); break;
      case 8: CX_GEN_LEVEL(false, 4); break;
      case 9: CX_GEN_LEVEL(true, 4); break;
      default: return hipErrorInvalidValue;
    }
  }
#undef CX_GEN_LEVEL
#undef CX_GEN
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || !S.split) return e;
  const int nc = S.ncomp, nfl = ncart(l[3]);
  hipLaunchKernelGGL(eri_generic_slab_kernel, dim3((unsigned)(a.nq * nc * nfl)), dim3(256),
                     (size_t)2 * (S.nf / nfl) * 8, s, a, S);
  const int64_t pieces = (a.block / nc + kGenLast - 1) / kGenLast;
  hipLaunchKernelGGL(eri_generic_last_kernel, dim3((unsigned)(a.nq * nc * pieces)), dim3(256), 0,
                     s, a, S, (int)pieces);
  return hipGetLastError();
}

}  // namespace cx
