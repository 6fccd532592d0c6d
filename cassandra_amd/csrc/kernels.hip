// kernels.hip -- device code of libcassgpu for gfx950 (CDNA4, wave64).
//
// The energy path is a gather- and ALU-bound sum, not a contraction, so no
// MFMA is used: every kernel is VALU work with FP64 accumulation, wave64
// shuffle reductions and deterministic (fixed-order) cross-block sums.
#include "kernels.h"

namespace cass {

// ------------------------------------------------------------ reductions
__device__ inline double wave_sum(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
  return v;
}

__device__ inline int wave_or(int v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v |= __shfl_down(v, o, 64);
  return v;
}

// Block sum of NV doubles and an OR flag; result valid in thread 0.
template <int NV>
__device__ inline void block_reduce(double (&v)[NV], int &flag) {
  __shared__ double sh[NV][kMaxBlock / 64];
  __shared__ int shf[kMaxBlock / 64];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = (blockDim.x + 63) >> 6;
#pragma unroll
  for (int k = 0; k < NV; ++k) v[k] = wave_sum(v[k]);
  flag = wave_or(flag);
  if (lane == 0) {
#pragma unroll
    for (int k = 0; k < NV; ++k) sh[k][wid] = v[k];
    shf[wid] = flag;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      double s = 0.0;
      for (int w = 0; w < nw; ++w) s += sh[k][w];
      v[k] = s;
    }
    int f = 0;
    for (int w = 0; w < nw; ++w) f |= shf[w];
    flag = f;
  }
  __syncthreads();
}

// ------------------------------------------------------ trial energies
// grid (nblk, ntrial): trial t against the box's molecules
// [blockIdx.x*blockDim.x, +blockDim.x).  Partials per (trial, block):
// part[(t*nblk + bx)*2 + {0,1}] = {E_vdw, E_qq}, part_ov[t*nblk + bx].
template <typename P>
__global__ void __launch_bounds__(kMaxBlock) k_trials(BoxDev b, TopoDev tp, PairConst<double> cd,
                                                      PairConst<float> cf, int species, int ni,
                                                      const double *__restrict__ txyz, int exclude,
                                                      int cbmc, double *part, int *part_ov) {
  __shared__ double px[kMaxSites], py[kMaxSites], pz[kMaxSites];
  __shared__ int pspa[kMaxSites];
  __shared__ double4 pcom;
  const int t = blockIdx.y;
  const int oi = tp.sp_atom_off[species];
  if (threadIdx.x < ni) {
    const size_t o = ((size_t)t * ni + threadIdx.x) * 3;
    px[threadIdx.x] = txyz[o];
    py[threadIdx.x] = txyz[o + 1];
    pz[threadIdx.x] = txyz[o + 2];
    pspa[threadIdx.x] = oi + threadIdx.x;
  }
  __syncthreads();
  if (threadIdx.x == 0) pcom = molecule_com(tp, oi, ni, px, py, pz);
  __syncthreads();
  const bool coul_cbmc = tp.sp_coul_cbmc[species] != 0;
  double v[2] = {0.0, 0.0};
  int ov = 0;
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j < b.nmols && j != exclude && b.live[j]) {
    if (molpair_in_range(b, cbmc, pcom, b.comd[j]))
      ov = molpair_energy<P>(b, tp, cd, cf, cbmc, coul_cbmc, ni, px, py, pz, pspa, j, v[0], v[1], nullptr);
  }
  block_reduce<2>(v, ov);
  if (threadIdx.x == 0) {
    const size_t o = (size_t)t * gridDim.x + blockIdx.x;
    part[2 * o] = v[0];
    part[2 * o + 1] = v[1];
    part_ov[o] = ov;
  }
}

// Fixed-order sum of per-block partials: one thread per trial.
__global__ void k_finalize_trials(const double *part, const int *part_ov, int nblk, int ntrial,
                                  double *out, int *out_ov) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= ntrial) return;
  double a = 0.0, c = 0.0;
  int o = 0;
  for (int k = 0; k < nblk; ++k) {
    const size_t i = (size_t)t * nblk + k;
    a += part[2 * i];
    c += part[2 * i + 1];
    o |= part_ov[i];
  }
  out[2 * t] = a;
  out[2 * t + 1] = c;
  out_ov[t] = o;
}

// Fixed-order sum of n doubles by one block.
__global__ void k_sum(const double *in, size_t n, int stride, int comp, double *out) {
  double v[1] = {0.0};
  int f = 0;
  for (size_t i = threadIdx.x; i < n; i += blockDim.x) v[0] += in[i * stride + comp];
  block_reduce<1>(v, f);
  if (threadIdx.x == 0) *out = v[0];
}

// ---------------------------------------------------- total pair energy
// Compute_System_Total_Energy inter part (energy_routines.f90:2775-2917): one
// wave per molecule i and the pairs (i, j) with j > i.  The sites of the
// molecules in range are compacted in LDS and scored 64 at a time against
// every site of i.  A workgroup of one j per lane left five lanes in six idle
// (j <= i, or out of range) and dominated the sum: 24 boxes of 512 waters took
// 0.60 ms, 0.27 here.  part[i], part_ov[i]: i's sums.
template <typename P>
__device__ inline void total_pairs_wave(const BoxDev &b, const TopoDev &tp, const PairConst<double> &cd,
                                        const PairConst<float> &cf, int i, double *part, int *part_ov) {
  using TV = typename P::V;
  using TQ = typename P::Q;
  const PairConst<TV> &cv = pconst<TV>(cd, cf);
  const PairConst<TQ> &cq = pconst<TQ>(cd, cf);
  __shared__ int2 ring[kPairMols][128];  // (site, species atom) of partners in range
  const int lane = threadIdx.x & 63;
  int2 *ent = ring[threadIdx.x >> 6];
  const int si = b.species[i], fi = b.first[i];
  const int ni = tp.sp_natoms[si], oi = tp.sp_atom_off[si];
  const double4 ci = b.comd[i];
  double ev = 0.0, eq = 0.0;
  bool ov = false;
  int head = 0, cnt = 0;
  auto sync = [] {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };
  int base = b.live[i] ? i + 1 : b.nmols, ja = 0, nj = 0, fj = 0, oj = 0;
  bool take = false;
  for (;;) {
    // the ja-th sites of 64 molecules, then the next 64
    if (__any(take && ja < nj)) {
      const bool push = take && ja < nj;
      const uint64_t bal = __ballot(push);
      const int before =
          __builtin_amdgcn_mbcnt_hi((uint32_t)(bal >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)bal, 0));
      if (push) ent[(head + cnt + before) & 127] = make_int2(fj + ja, oj + ja);
      cnt += __popcll(bal);
      ++ja;
      sync();
    } else if (base < b.nmols) {
      const int j = base + lane;
      base += 64;
      take = j < b.nmols && b.live[j] && molpair_in_range(b, false, ci, b.comd[j]);
      if (take) {
        const int sj = b.species[j];
        fj = b.first[j];
        oj = tp.sp_atom_off[sj];
        nj = tp.sp_natoms[sj];
      }
      ja = 0;
      continue;
    } else if (cnt == 0) {
      break;
    }
    const bool last = base >= b.nmols && !__any(take && ja < nj);
    if (cnt >= 64 || last) {
      const int n = cnt < 64 ? cnt : 64;
      if (lane < n) {
        const int2 e = ent[(head + lane) & 127];
        const double x = b.x[e.x], y = b.y[e.x], z = b.z[e.x], qj = tp.atom_charge[e.y];
        const int tj = tp.atom_type[e.y];
        for (int ia = 0; ia < ni; ++ia) {
          double dx = b.x[fi + ia] - x, dy = b.y[fi + ia] - y, dz = b.z[fi + ia] - z;
          min_image(b, dx, dy, dz);
          const double r2 = dx * dx + dy * dy + dz * dz;
          if (r2 < cd.rc_low2) {
            ov = true;
            continue;
          }
          bool gv, gq;
          pair_cutoff(cd, false, r2, gv, gq);
          const int ti = tp.atom_type[oi + ia];
          if (gv && ti >= 0 && tj >= 0) {
            const int k = ti * tp.ntypes + tj;
            ev += (double)vdw_inter<TV, typename P::M>(cv, (TV)r2, (TV)tp.eps[k], (TV)tp.sig[k], (TV)tp.mn[k],
                                                       (TV)tp.mm[k]);
          }
          const double qi = tp.atom_charge[oi + ia];
          if (gq && cd.q_style != CASS_Q_NONE && qi != 0.0 && qj != 0.0)
            eq += (double)qq_inter<TQ, typename P::M>(cq, (TQ)r2, (TQ)(qi * qj));
        }
      }
      head += n;
      cnt -= n;
      sync();
    }
  }
  ev = wave_total(ev);
  eq = wave_total(eq);
  const int any = __any(ov);
  if (lane == 0) {
    part[2 * (size_t)i] = ev;
    part[2 * (size_t)i + 1] = eq;
    part_ov[i] = any;
  }
}

// grid ceil(nmols / kPairMols)
template <typename P>
__global__ void __launch_bounds__(64 * kPairMols) k_total_pairs(BoxDev b, TopoDev tp, PairConst<double> cd,
                                                                PairConst<float> cf, double *part, int *part_ov) {
  const int i = blockIdx.x * kPairMols + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (i < b.nmols) total_pairs_wave<P>(b, tp, cd, cf, i, part, part_ov);
}

// The same over many boxes: one workgroup per item (box, first molecule); the
// box's partials start at part_off in part / part_ov.
template <typename P>
__global__ void __launch_bounds__(64 * kPairMols)
    k_total_pairs_multi(const RecomputeBox *__restrict__ boxes, TopoDev tp, const int2 *__restrict__ items,
                        double *part, int *part_ov) {
  const int2 it = items[blockIdx.x];
  const RecomputeBox &r = boxes[it.x];
  const int i = it.y + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (i < r.b.nmols) total_pairs_wave<P>(r.b, tp, r.cd, r.cf, i, part + 2 * r.part_off, part_ov + r.part_off);
}

// ----------------------------------------------------------------- Ewald
// Compute_System_Ewald_Reciprocal_Energy (energy_routines.f90:4111-4231),
// stage 1: the sums of one molecule over the k vectors, `parts` workgroups
// sharing them.  The powers of the sites' unit phases stand in LDS (2 pi as the
// reference truncates it), each from its own angle in two words: powers by
// products share the rounding of the first, which moves the site and left twice
// the error of a sine and cosine per vector (8.6e-16 rms of the energy; 3.7e-16
// here, as there).  A lane takes a segment of consecutive n_x, and each wave
// passes its segments' sums through LDS to store them in k order: 24 boxes of
// 512 waters took 0.32 ms with a sine and cosine per site and vector, 0.13 here,
// for 0.46 GB of stores.
__device__ inline void ewald_mol_block(const BoxDev &b, const TopoDev &tp, const EwaldDev &ew, int m, int part,
                                       int parts) {
  __shared__ cplx tab[kEwTab];
  __shared__ double2 ph[3 * kMaxSites];
  __shared__ double out[kMaxBlock / 64][64 * kKSeg];
  const int tid = threadIdx.x, lane = tid & 63;
  const int sp = b.species[m], f = b.first[m];
  const int n = tp.sp_natoms[sp], o = tp.sp_atom_off[sp], nt = ew.tx + ew.ty + ew.tz;
  if (ewald_direct(ew, b.nmols, n)) return;  // ewald_direct_block takes it
  double *cm = ew.cmol + (size_t)m * ew.nvecs, *sm = ew.smol + (size_t)m * ew.nvecs;
  if (!b.live[m]) {
    for (int k = part * blockDim.x + tid; k < ew.nvecs; k += parts * blockDim.x) cm[k] = sm[k] = 0.0;
    return;
  }
  for (int t = tid; t < 3 * n; t += blockDim.x) {
    const int a = t / 3, d = t - 3 * a;
    const double x = b.x[f + a], y = b.y[f + a], z = b.z[f + a];
    const double sh = fma(b.Li[d], x, fma(b.Li[3 + d], y, b.Li[6 + d] * z));
    const double sl = fma(b.Li[6 + d], z, fma(b.Li[3 + d], y, fma(b.Li[d], x, -sh)));
    const double hi = kTwoPi * sh;
    ph[t] = make_double2(hi, fma(kTwoPi, sl, fma(kTwoPi, sh, -hi)));
  }
  __syncthreads();
  for (int t = tid; t < n * nt; t += blockDim.x) {
    const int a = t / nt, r = t - a * nt;
    const int d = r < ew.tx ? 0 : r < ew.tx + ew.ty ? 1 : 2;
    const double k = r - (d == 0 ? 0 : d == 1 ? ew.tx : ew.tx + ew.ty);
    const double2 p = ph[3 * a + d];
    const double hi = k * p.x, lo = fma(k, p.y, fma(k, p.x, -hi));
    double sv, cv;
    sincos(hi, &sv, &cv);
    tab[t] = cplx{fma(-sv, lo, cv), fma(cv, lo, sv)};
  }
  __syncthreads();
  double *buf = out[tid >> 6];
  for (int s0 = part * blockDim.x + tid - lane; s0 < ew.nsegs; s0 += parts * blockDim.x) {  // wave-uniform
    const int4 sg = ew.segs[min(s0 + lane, ew.nsegs - 1)];
    const int k0 = sg.x & 0xfffff, len = sg.x >> 20;
    const int ny = sg.z < 0 ? -sg.z : sg.z, nz = sg.w < 0 ? -sg.w : sg.w;
    double c[kKSeg], s[kKSeg];
#pragma unroll
    for (int t = 0; t < kKSeg; ++t) c[t] = s[t] = 0.0;
    for (int a = 0; a < n; ++a) {
      const cplx *ta = tab + a * nt;
      const cplx X = ta[sg.y], E = ta[1];
      cplx Y = ta[ew.tx + ny], Z = ta[ew.tx + ew.ty + nz];
      Y.im = sg.z < 0 ? -Y.im : Y.im;
      Z.im = sg.w < 0 ? -Z.im : Z.im;
      cplx p = cmul(cmul(X, Z), Y);
      const double q = tp.atom_charge[o + a];
      p.re = q * p.re;
      p.im = q * p.im;
#pragma unroll
      for (int t = 0; t < kKSeg; ++t) {
        c[t] = c[t] + p.re;
        s[t] = s[t] + p.im;
        if (t + 1 < kKSeg) p = cmul(p, E);
      }
    }
    // the wave's segments cover consecutive vectors
    const int last = min(s0 + 63, ew.nsegs - 1) - s0;
    const int kb = __builtin_amdgcn_readfirstlane(k0);
    const int kn = __builtin_amdgcn_readlane(k0 + len, last) - kb;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
      if (lane <= last) {
#pragma unroll
        for (int t = 0; t < kKSeg; ++t)
          if (t < len) buf[k0 - kb + t] = h ? s[t] : c[t];
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
      for (int t = lane; t < kn; t += 64) (h ? sm : cm)[kb + t] = buf[t];
    }
  }
}

// The same by a sine and cosine per site and vector (ewald_direct), a vector
// per lane.
__device__ inline void ewald_direct_block(const BoxDev &b, const TopoDev &tp, const EwaldDev &ew, int m, int kb) {
  const int k = kb * blockDim.x + threadIdx.x;
  const int sp = b.species[m], f = b.first[m];
  const int n = tp.sp_natoms[sp], o = tp.sp_atom_off[sp];
  if (k >= ew.nvecs || !ewald_direct(ew, b.nmols, n)) return;
  double c = 0.0, s = 0.0;
  if (b.live[m]) {
    const double hx = ew.hx[k], hy = ew.hy[k], hz = ew.hz[k];
    for (int a = 0; a < n; ++a) {
      const double hr = hx * b.x[f + a] + hy * b.y[f + a] + hz * b.z[f + a];
      const double q = tp.atom_charge[o + a];
      double sv, cv;
      sincos(hr, &sv, &cv);
      c = c + q * cv;
      s = s + q * sv;
    }
  }
  ew.cmol[(size_t)m * ew.nvecs + k] = c;
  ew.smol[(size_t)m * ew.nvecs + k] = s;
}

// grid (nmols, parts)
__global__ void __launch_bounds__(kMaxBlock) k_ewald_mol(BoxDev b, TopoDev tp, EwaldDev ew) {
  ewald_mol_block(b, tp, ew, blockIdx.x, blockIdx.y, gridDim.y);
}

// grid (ceil(K / block), nmols)
__global__ void k_ewald_direct(BoxDev b, TopoDev tp, EwaldDev ew) {
  ewald_direct_block(b, tp, ew, blockIdx.y, blockIdx.x);
}

// stage 2: the box sums over molecules (zero for dead ones) and the energy
// term of a block of k vectors (box_vecs), written to part[kb].  The molecules
// are shared by the workgroup's waves and read several at a time: one lane per
// vector over all molecules was a chain of 512 loads on a tenth of the chip (24
// boxes of 512 waters: 0.60 ms, 0.13 here).  Few molecules are not shared: a
// block of 64 vectors leaves four times the partials to add up (one water and
// 56000 vectors: the call 31.3 us shared, 30.3 not; 15 waters not shared 43.0,
// 16 shared 41.4).
__device__ inline void ewald_box_block(const BoxDev &b, const EwaldDev &ew, int kb, double *part) {
  __shared__ double sh[2][kMaxBlock / 64][kBoxVecs];
  const bool shared = b.nmols >= kBoxShare;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int g = shared ? wave : 0, G = shared ? blockDim.x >> 6 : 1;
  const int k = shared ? kb * kBoxVecs + lane : kb * (int)blockDim.x + (int)threadIdx.x;
  double v[1] = {0.0};
  int f = 0;
  double c[4] = {0.0, 0.0, 0.0, 0.0}, s[4] = {0.0, 0.0, 0.0, 0.0};
  if (k < ew.nvecs) {
    int m = g;
    for (; m + 3 * G < b.nmols; m += 4 * G) {
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const size_t o = (size_t)(m + u * G) * ew.nvecs + k;
        c[u] = c[u] + ew.cmol[o];
        s[u] = s[u] + ew.smol[o];
      }
    }
    for (; m < b.nmols; m += G) {
      const size_t o = (size_t)m * ew.nvecs + k;
      c[0] = c[0] + ew.cmol[o];
      s[0] = s[0] + ew.smol[o];
    }
  }
  double ct = (c[0] + c[1]) + (c[2] + c[3]), st = (s[0] + s[1]) + (s[2] + s[3]);
  if (shared) {
    sh[0][wave][lane] = ct;
    sh[1][wave][lane] = st;
    __syncthreads();
    ct = st = 0.0;
    for (int u = 0; u < G; ++u) {
      ct = ct + sh[0][u][lane];
      st = st + sh[1][u][lane];
    }
  }
  if (g == 0 && k < ew.nvecs) {
    ew.cs[k] = ct;
    ew.sn[k] = st;
    v[0] = ew.cn[k] * (ct * ct + st * st);
  }
  block_reduce<1>(v, f);
  if (threadIdx.x == 0) part[kb] = v[0];
}

__global__ void k_ewald_box(BoxDev b, EwaldDev ew, double *part) { ewald_box_block(b, ew, blockIdx.x, part); }

// The two stages over many boxes: items (box, molecule * parts + part), the
// same with k blocks for parts, and (box, k block); a box's k-block terms start
// at kpart_off in kpart.
__global__ void __launch_bounds__(kMaxBlock)
    k_ewald_mol_multi(const RecomputeBox *__restrict__ boxes, TopoDev tp, const int2 *__restrict__ items) {
  const int2 it = items[blockIdx.x];
  const RecomputeBox &r = boxes[it.x];
  const int m = it.y / r.kparts;
  ewald_mol_block(r.b, tp, r.ew, m, it.y - m * r.kparts, r.kparts);
}

__global__ void k_ewald_direct_multi(const RecomputeBox *__restrict__ boxes, TopoDev tp,
                                     const int2 *__restrict__ items) {
  const int2 it = items[blockIdx.x];
  const RecomputeBox &r = boxes[it.x];
  const int m = it.y / r.kdirect;
  ewald_direct_block(r.b, tp, r.ew, m, it.y - m * r.kdirect);
}

__global__ void k_ewald_box_multi(const RecomputeBox *__restrict__ boxes, const int2 *__restrict__ items,
                                  double *kpart) {
  const int2 it = items[blockIdx.x];
  const RecomputeBox &r = boxes[it.x];
  ewald_box_block(r.b, r.ew, it.y, kpart + r.kpart_off);
}

// k_sum of every box's k-block terms, one workgroup per box: out[box].
__global__ void k_sum_multi(const RecomputeBox *__restrict__ boxes, const double *kpart, double *out) {
  const RecomputeBox &r = boxes[blockIdx.x];
  double v[1] = {0.0};
  int f = 0;
  for (size_t i = threadIdx.x; i < (size_t)r.kblk; i += blockDim.x) v[0] += kpart[r.kpart_off + i];
  block_reduce<1>(v, f);
  if (threadIdx.x == 0) out[blockIdx.x] = v[0];
}

// Update_System_Ewald_Reciprocal_Energy (energy_routines.f90:2326-2497):
// tentative sums for molecule m at new coordinates (flag: 0 translation,
// 1 rotation, 2 intra, 3 insertion, 4 deletion).  part[blk*2+{0,1}] =
// {sum Cn (C'^2+S'^2), sum Cn (2 C dC + dC^2 + 2 S dS + dS^2)}.
__global__ void k_ewald_move(TopoDev tp, EwaldDev ew, int m, int species, int flag, int n,
                             const double *__restrict__ nxyz, double *part) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  double v[2] = {0.0, 0.0};
  int f = 0;
  if (k < ew.nvecs) {
    const size_t mk = (size_t)m * ew.nvecs + k;
    const double cm = (flag == CASS_MOVE_INSERTION) ? 0.0 : ew.cmol[mk];
    const double sm = (flag == CASS_MOVE_INSERTION) ? 0.0 : ew.smol[mk];
    double c = 0.0, s = 0.0;
    if (flag != CASS_MOVE_DELETION) {
      const int o = tp.sp_atom_off[species];
      const double hx = ew.hx[k], hy = ew.hy[k], hz = ew.hz[k];
      for (int a = 0; a < n; ++a) {
        const double hr = hx * nxyz[3 * a] + hy * nxyz[3 * a + 1] + hz * nxyz[3 * a + 2];
        const double q = tp.atom_charge[o + a];
        double sv, cv;
        sincos(hr, &sv, &cv);
        c = c + q * cv;
        s = s + q * sv;
      }
    }
    const double c0 = ew.cs[k], s0 = ew.sn[k];
    double c1, s1;
    if (flag == CASS_MOVE_DELETION) {
      c1 = c0 - cm;
      s1 = s0 - sm;
    } else if (flag == CASS_MOVE_INSERTION) {
      c1 = c0 + c;
      s1 = s0 + s;
    } else {
      c1 = c0 + (c - cm);
      s1 = s0 + (s - sm);
    }
    ew.cs_new[k] = c1;
    ew.sn_new[k] = s1;
    ew.cm_new[k] = c;
    ew.sm_new[k] = s;
    const double dc = c - cm, ds = s - sm;
    v[0] = ew.cn[k] * (c1 * c1 + s1 * s1);
    v[1] = ew.cn[k] * (2.0 * c0 * dc + dc * dc + 2.0 * s0 * ds + ds * ds);
  }
  block_reduce<2>(v, f);
  if (threadIdx.x == 0) {
    part[2 * blockIdx.x] = v[0];
    part[2 * blockIdx.x + 1] = v[1];
  }
}

__global__ void k_ewald_commit(EwaldDev ew, int m) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= ew.nvecs) return;
  ew.cs[k] = ew.cs_new[k];
  ew.sn[k] = ew.sn_new[k];
  ew.cmol[(size_t)m * ew.nvecs + k] = ew.cm_new[k];
  ew.smol[(size_t)m * ew.nvecs + k] = ew.sm_new[k];
}

// Update_System_Ewald_Reciprocal_Energy_Widom (energy_routines.f90:2500-2550)
// for explicit test molecules: one block per trial, threads over k.
__global__ void k_ewald_widom(TopoDev tp, EwaldDev ew, int species, int n, const double *__restrict__ txyz,
                              double *part) {
  __shared__ double px[kMaxSites], py[kMaxSites], pz[kMaxSites], pq[kMaxSites];
  const int t = blockIdx.y;
  const int o = tp.sp_atom_off[species];
  if (threadIdx.x < n) {
    const size_t b = ((size_t)t * n + threadIdx.x) * 3;
    px[threadIdx.x] = txyz[b];
    py[threadIdx.x] = txyz[b + 1];
    pz[threadIdx.x] = txyz[b + 2];
    pq[threadIdx.x] = tp.atom_charge[o + threadIdx.x];
  }
  __syncthreads();
  double v[1] = {0.0};
  int f = 0;
  for (int k = blockIdx.x * blockDim.x + threadIdx.x; k < ew.nvecs; k += gridDim.x * blockDim.x) {
    double dc = 0.0, ds = 0.0;
    for (int a = 0; a < n; ++a) {
      const double hr = ew.hx[k] * px[a] + ew.hy[k] * py[a] + ew.hz[k] * pz[a];
      double sv, cv;
      sincos(hr, &sv, &cv);
      dc = dc + pq[a] * cv;
      ds = ds + pq[a] * sv;
    }
    const double c = ew.cs[k] + dc, s = ew.sn[k] + ds;
    v[0] += ew.cn[k] * (c * c + s * s);
  }
  block_reduce<1>(v, f);
  if (threadIdx.x == 0) part[(size_t)t * gridDim.x + blockIdx.x] = v[0];
}

// --------------------------------------------------------- Widom batch
__global__ void k_sum_widom(const double *part, const int64_t *part_ov, int n, double *out,
                            int64_t *out_ov) {
  double v[1] = {0.0};
  int f = 0;
  __shared__ int64_t sh[kMaxBlock / 64];
  int64_t c = 0;
  for (int i = threadIdx.x; i < n; i += blockDim.x) {
    v[0] += part[i];
    c += part_ov[i];
  }
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) c += __shfl_down(c, d, 64);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = c;
  block_reduce<1>(v, f);
  if (threadIdx.x == 0) {
    int64_t t = 0;
    for (int w = 0; w < (int)(blockDim.x >> 6); ++w) t += sh[w];
    *out = v[0];
    *out_ov = t;
  }
}

// ---------------------------------------------------------- instantiation
#define CASS_INSTANTIATE(P)                                                                               \
  template __global__ void k_trials<P>(BoxDev, TopoDev, PairConst<double>, PairConst<float>, int, int,    \
                                       const double *, int, int, double *, int *);                        \
  template __global__ void k_total_pairs<P>(BoxDev, TopoDev, PairConst<double>, PairConst<float>,         \
                                            double *, int *);                                             \
  template __global__ void k_total_pairs_multi<P>(const RecomputeBox *, TopoDev, const int2 *, double *, int *);
CASS_INSTANTIATE(PrecFP64)
CASS_INSTANTIATE(PrecMixed)
CASS_INSTANTIATE(PrecFP32)
#undef CASS_INSTANTIATE

}  // namespace cass
