// The step kernels: the execution policy for K envs per wavefront, the plain
// step kernel and its variant with the learned warm start.
#pragma once
#include <hip/hip_runtime.h>

#include "kbody.hpp"
#include "mlp_dev.hpp"

namespace phk {

// K environments per workgroup of one 64-lane wavefront: env g of the
// workgroup owns lanes [g * 64/K, (g + 1) * 64/K) and its own slice of the LDS.
// Loops over an env's items stride over its lanes; the dense linear algebra
// uses the first 16 of them (one DPP row).
template <int K>
struct DevXK : DevLanes {
  static constexpr int G = 64 / K;
  static constexpr int WIDTH = G;  // lanes of an env
  template <class F>
  __device__ __forceinline__ static void par(int n, F&& f) {
    for (int i = (int)(threadIdx.x % G); i < n; i += G) f(i);
    __syncthreads();
  }
  __device__ __forceinline__ static void sync() { __syncthreads(); }
  // 16-lane rows that work on one env, and which of them this lane is in
  static constexpr int ROWS = G / GL;
  __device__ __forceinline__ static int row() { return (int)(threadIdx.x % G) / GL; }
};
using DevX = DevXK<1>;

// The policy of the learned-warm-start kernel: DevXK plus the network over
// the wavefront's recorded contacts. Tile t holds contacts t * 16/K ..
// (t + 1) * 16/K - 1 of each of the K envs, one sample column per contact;
// tiles run while any env of the wavefront has contacts left.
template <int K>
struct DevXKM : DevXK<K> {
  static constexpr int G = 64 / K;
  template <class MT>
  __device__ static void mlp_tiles(const MT& M, const DState& S, int64_t e_self, int cnt) {
    constexpr int SPE = 16 / K;
    if (M.mlp.h > MLP_HMAX_STEP) {  // wider networks are trained and run in batches only
      __syncthreads();
      return;
    }
    const int lane = (int)threadIdx.x, g = lane / G, j = lane & 15, q = lane >> 4;
    const int64_t e0 = e_self - g;
    int mx = cnt;
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) mx = max(mx, __shfl_xor(mx, o));
    const int gs = j / SPE;  // env of this lane's sample column
    const int cs = __shfl(cnt, gs * G);
    const int nt = (mx + SPE - 1) / SPE;
    const bf16x4 zero = {0, 0, 0, 0};
    for (int t = 0; t < nt; t++) {
      const int c = t * SPE + j % SPE;
      const bool have = c < cs;
      const int64_t row = (e0 + gs) * MLP_CL + c;
      bf16x4 x0 = zero, x1 = zero;
      if (have) {
        const float* f = S.mlp_feat.p + row * MLP_NF;
        x0 = pack_bf4(ld_f4(f + 4 * q));
        if (q < 2) x1 = pack_bf4(ld_f4(f + 16 + 4 * q));
      }
      const f32x4 y = mlp_tile_fwd<MLP_HMAX_STEP / 16>(M.mlp, x0, x1, MlpNoSink{});
      if (q == 0 && have) st_f4(S.mlp_pred.p + row * MLP_NO, y);
    }
    __syncthreads();
  }
};

// Advance envs [begin, end) by nstep steps, K per workgroup. With ctrl_seq
// (envs x nstep x nu) the controls change every step and qpos_out
// (envs x nstep x nq) receives qpos after each step (Batch::rollout, batch.rs:46-59).
// MT is DModel (sizes and layout read at run time) or a model-specialised
// struct derived from it whose sizes and LDS layout are compile-time constants
// (spec_models.hpp, generated at build time); both read the same buffers.
template <int K, class MT>
__global__ void __launch_bounds__(64) k_step(const DModel* __restrict__ Mp, const DState* __restrict__ Sp,
                                             int64_t begin, int64_t end, int64_t nstep, const Real* ctrl_seq,
                                             Real* qpos_out) {
  const MT& M = *static_cast<const MT*>(Mp);
  const DState& S = *Sp;
  extern __shared__ double lds[];
  const int g = (int)threadIdx.x / DevXK<K>::G;
  const int64_t rel = (int64_t)blockIdx.x * K + g;
  if (begin + rel >= end) return;  // tail of the last workgroup
  Env E;
  E.s = lds + (int64_t)g * (M.L.bytes / 8);
  E.si = reinterpret_cast<int*>(E.s + M.L.ndouble);
  E.e = begin + rel;
  E.var = M.env_var[E.e];
  run_env<DevXK<K>>(M, S, E, nstep, ctrl_seq, qpos_out, rel);
}

// Persistent work-stealing variant of k_step: the grid is what the device
// holds at once, and each workgroup takes the next slot of K envs from
// *counter until the slots run out. Slot s holds envs order[s*K .. s*K+K-1]
// (offsets from begin; the identity without order). k_bucket writes an order
// that puts envs of similar cost in one wavefront, costliest first, so that a
// wavefront waits less for its slowest env and the long slots start early.
// Every env's arithmetic is the same under any order. ctrl_seq / qpos_out as
// for k_step (rows indexed by the env's offset from begin).
template <int K, class MT>
__global__ void __launch_bounds__(64) k_step_ws(const DModel* __restrict__ Mp, const DState* __restrict__ Sp,
                                                int64_t begin, int64_t end, int64_t nstep, const Real* ctrl_seq,
                                                Real* qpos_out, const int* __restrict__ order, unsigned* counter) {
  const MT& M = *static_cast<const MT*>(Mp);
  const DState& S = *Sp;
  extern __shared__ double lds[];
  const int g = (int)threadIdx.x / DevXK<K>::G;
  const int64_t n = end - begin;
  const int64_t nslots = (n + K - 1) / K;
  for (;;) {
    unsigned slot = 0;
    if (threadIdx.x == 0) slot = atomicAdd(counter, 1u);
    slot = __shfl(slot, 0);
    if ((int64_t)slot >= nslots) break;
    const int64_t idx = (int64_t)slot * K + g;
    if (idx < n) {
      const int64_t rel = order ? (int64_t)order[idx] : idx;
      Env E;
      E.s = lds + (int64_t)g * (M.L.bytes / 8);
      E.si = reinterpret_cast<int*>(E.s + M.L.ndouble);
      E.e = begin + rel;
      E.var = M.env_var[E.e];
      run_env<DevXK<K>>(M, S, E, nstep, ctrl_seq, qpos_out, rel);
    }
    __syncthreads();
  }
}

// The PGS step split around its sweeps (run_pgs_front, run_pgs_back in
// kbody.hpp), for physics step t of nstep: the front and back keep the step
// kernel's LDS working set, K envs per workgroup of one wavefront; the sweeps
// run in kernels of their own. vel and vpos hold nv doubles per env (indexed by
// env id); cap: the doubles that packed rows of one env may take
// (k_pgs_sweeps_rows), 0 for a model without packed rows.
template <int K>
__global__ void __launch_bounds__(64) k_pgs_front(const DModel* __restrict__ Mp, const DState* __restrict__ Sp,
                                                  int64_t begin, int64_t end, int64_t nstep, int64_t t,
                                                  const Real* ctrl_seq, Real* vel, Real* vpos, int64_t cap,
                                                  unsigned* counter) {
  const DModel& M = *Mp;
  const DState& S = *Sp;
  extern __shared__ double lds[];
  if (blockIdx.x == 0 && threadIdx.x == 0) *counter = 0;  // for the sweeps that follow
  const int g = (int)threadIdx.x / DevXK<K>::G;
  const int64_t rel = (int64_t)blockIdx.x * K + g;
  if (begin + rel >= end) return;
  Env E;
  E.s = lds + (int64_t)g * (M.L.bytes / 8);
  E.si = reinterpret_cast<int*>(E.s + M.L.ndouble);
  E.e = begin + rel;
  E.var = M.env_var[E.e];
  run_pgs_front<DevXK<K>>(M, S, E, nstep, t, ctrl_seq, rel, vel + E.e * M.nv, vpos + E.e * M.nv, cap);
}

// The rest of an env's sweeps in their general form, from its row `at` on:
// velocities in LDS, rows and forces in HBM (lam: the forces so far). Out of
// line: hardly any env comes here.
template <int W>
__device__ __noinline__ void pgs_sweeps_general(const DModel* Mp, const DState* Sp, int64_t e, int nr, double* v,
                                                int64_t phase_it, int64_t row_moved, Real* vpos_e) {
#if defined(__HIP_DEVICE_COMPILE__)
  using X = DevXK<4>;
  const DModel& M = *Mp;
  const DState& S = *Sp;
  const int nv = M.nv, l = (int)threadIdx.x % GL;
  const PgsAt at{(int)(phase_it >> 32), (int)(uint32_t)phase_it, (int)(row_moved >> 1), (row_moved & 1) != 0};
  Real* J = (S.gjac + e * (int64_t)M.nrmax * nv).p;
  Real* mj = (S.gmj + e * (int64_t)M.nrmax * nv).p;
  const PgsRecs rec{(S.grow + e * (int64_t)M.nrmax * 10).p};
  __threadfence_block();
  pgs_sweeps_rows<X, W>(pgs_consts(M), J, mj, rec, nr, nv, v, at, [&]() {
    for (int k = l; k < nv; k += GL) vpos_e[k] = v[k];
  });
#endif
}

// The sweeps over packed rows: four envs per wavefront, one per 16-lane row,
// with the env's rows, forces and velocities in LDS (slice doubles per env), W
// the widest row's entries. A row update is a chain (read v, W ordered adds,
// the force, write v) of about 90 instructions that the four envs share; LDS
// holds 12 or 16 envs per CU, so at most one wavefront per SIMD hides nothing of
// it and every instruction and branch counts (six-body pile, 8192 envs, a
// physics step: 2.06 ms with one env per wavefront in registers, 1.7 ms so): the terms that stay fixed over a
// phase are formed when the phase begins, normal and friction rows share one
// expression (a friction row's bias and impulse scale are 0, a normal row's
// friction coefficient 0 and its upper bound infinite), the row's record and
// the next row's entries are in flight during the sum. The four 16-lane
// rows advance independently, each from row to row, sweep to sweep and env to
// env (counter, cleared by k_pgs_front), so none waits for another's longer
// solve. The expression needs finite velocities and forces; an env that has
// others goes on in pgs_sweeps_general. EQ: the model has equalities, whose
// rows are bilateral.
template <int W, bool EQ>
__global__ void __launch_bounds__(64) k_pgs_sweeps_rows(const DModel* __restrict__ Mp, const DState* __restrict__ Sp,
                                                        int64_t begin, int64_t end, Real* vel, Real* vpos, int slice,
                                                        unsigned* counter) {
#if defined(__HIP_DEVICE_COMPILE__)
  using X = DevXK<4>;
  const DModel& M = *Mp;
  const DState& S = *Sp;
  extern __shared__ double lds[];
  // LDS by byte address (below 64 KiB)
  typedef __attribute__((address_space(3))) char LC;
  typedef __attribute__((address_space(3))) double LDd;
  LC* const lb = (LC*)lds;
  auto ld = [&](int a) -> double { return *(LDd*)(lb + a); };
  auto st = [&](int a, double x) { *(LDd*)(lb + a) = x; };
  const int g = (int)threadIdx.x / GL, l = (int)threadIdx.x % GL, l8 = 8 * l;
  const int nv = M.nv, vb = 8 * g * slice, spare = vb + 8 * nv, recb = vb + 8 * ((nv + 2) & ~1);
  constexpr int RB = 8 * PGS_REC;
  // a row's record: -inv_a times the mass scale, bias, impulse scale, friction
  // coefficient, force, and where its entries and velocities are
  enum { C0 = 0, BIAS = 8, IS = 16, MU = 24, LAM = 32, INFO = 40 };
  const PgsConsts C = pgs_consts(M);
  const int relax = pgs_relax_sweeps(C);
  const Real hi0 = pgs_tol_hi(C), lo0 = pgs_tol_lo(C), hi1 = hi0 / C.mass_scale, lo1 = lo0 / C.mass_scale;
  const int64_t n = end - begin;
  bool live = true, have = false;
  int64_t e = 0;
  int nr = 0, Jb = 0, mo = 0;  // byte address of the J entries, and from there to the M^-1 J^T entries
  int phase = 0, it = 0, r = 0, limit = 0;
  bool moved = false;
  // the current row: its record, its J entry here and that entry's address, the
  // velocity it meets, the INFO word
  int ra = recb, ja = 0, va = spare, hi_w = 0;
  Real j = 0.0;
  auto count_of = [](int hi) { return (hi >> 21) & 31; };
  auto v_addr = [&](int lo, int hi) {  // a spare slot past the row's entries
    const int base = l < ((hi >> 16) & 31) ? lo & 0xFFFF : (int)((unsigned)lo >> 16);
    return l < count_of(hi) ? base + l8 : spare;
  };
  auto info = [&](int a, int* lo, int* hi) {
    const int64_t w = *(__attribute__((address_space(3))) int64_t*)(lb + a + INFO);
    *lo = (int)w;
    *hi = (int)(w >> 32);
  };
  auto start = [&]() {  // the first row
    int lo;
    ra = recb;
    info(ra, &lo, &hi_w);
    va = v_addr(lo, hi_w);
    ja = Jb + (hi_w & 0xFFFF) * 8 + l8;
    j = ld(ja);
    j = l < count_of(hi_w) ? j : 0.0;
  };
  auto records = [&](int ph) {  // the rows' terms in phase ph
    auto rw = S.grow + e * (int64_t)M.nrmax * 10;
    for (int i = l; i < nr; i += GL) {
      const PgsRow w = pgs_row(rw[i * 10 + PR_FLAGS]);
      const Real ia = rw[i * 10 + PR_INVA], b1 = rw[i * 10 + PR_B1];
      const bool friction = w.kind == PK_FRICTION, soft = ph == 0 && !w.hard && !friction, fixed = ia == 0.0;
      const int a = recb + i * RB;
      st(a + C0, soft ? -ia * C.mass_scale : -ia);
      st(a + BIAS, !friction && (ph == 0 || w.hard) ? b1 : 0.0);
      st(a + IS, soft && !fixed ? C.impulse_scale : 0.0);
      st(a + MU, friction && !fixed ? b1 : 0.0);
      // lo: addresses of entry 0 of the lower block and of entry na of the
      // upper one less its place; hi: offset 16 bits, na 5, entries 5,
      // bilateral, unbounded above, and in 16 bytes the way back to the
      // contact's normal row's record 4
      const unsigned alo = (unsigned)(vb + 8 * w.a), blo = (unsigned)(vb + 8 * (w.count > w.na ? w.b - w.na : 0));
      const unsigned hi = (unsigned)w.off | (unsigned)w.na << 16 | (unsigned)w.count << 21 |
                          (w.kind == PK_BILATERAL ? 1u << 26 : 0u) | (!friction || fixed ? 1u << 27 : 0u) |
                          (unsigned)(w.sub * (RB / 16)) << 28;
      *(__attribute__((address_space(3))) int64_t*)(lb + a + INFO) = (int64_t)((uint64_t)hi << 32 | blo << 16 | alo);
    }
    X::order();
  };
  auto store = [&](bool forces) {
    for (int k = l; k < nv; k += GL) vel[e * nv + k] = ld(vb + 8 * k);
    auto rw = S.grow + e * (int64_t)M.nrmax * 10;
    if (forces)
      for (int i = l; i < nr; i += GL) rw[i * 10 + PR_LAM] = ld(recb + i * RB + LAM);
    have = false;
  };
  auto general = [&](int row) {  // the rest of this env's sweeps
    auto rw = S.grow + e * (int64_t)M.nrmax * 10;
    for (int i = l; i < nr; i += GL) rw[i * 10 + PR_LAM] = ld(recb + i * RB + LAM);
    pgs_sweeps_general<W>(Mp, Sp, e, nr, lds + (int64_t)g * slice, (int64_t)phase << 32 | it,
                          (int64_t)row << 1 | (moved ? 1 : 0), vpos + e * nv);
    store(false);
  };
  for (;;) {
    while (live && !have) {
      unsigned idx = 0;
      if (l == 0) idx = atomicAdd(counter, 1u);
      idx = __shfl(idx, g * GL);
      if ((int64_t)idx >= n) {
        live = false;
        break;
      }
      e = begin + idx;
      nr = S.nrows[e];
      if (S.status[e] != 0 || nr <= 0) continue;
      auto rw = S.grow + e * (int64_t)M.nrmax * 10;
      if (rw[PR_MODE] == 0.0) continue;
      const PgsRow last = pgs_row(rw[(nr - 1) * 10 + PR_FLAGS]);
      const int entries = (int)last.off + last.count;
      Jb = recb + nr * RB;
      mo = 8 * entries;
      auto gj = S.gjac + e * (int64_t)M.nrmax * nv;
      auto gm = S.gmj + e * (int64_t)M.nrmax * nv;
      bool ok = C.iterations > 0;
      for (int k = l; k < nv; k += GL) st(vb + 8 * k, vel[e * nv + k]);
      for (int i = l; i < nr; i += GL) {
        const Real ia = rw[i * 10 + PR_INVA], lm = rw[i * 10 + PR_LAM];
        st(recb + i * RB + LAM, lm);
        ok = ok && rfinite(lm) && (ia > 0x1p-900 || (ia == 0.0 && lm == 0.0));
      }
      for (int t = l; t < entries; t += GL) {
        st(Jb + 8 * t, gj[t]);
        st(Jb + mo + 8 * t, gm[t]);
      }
      st(spare, 0.0);
      st(Jb + 2 * mo + l8, 0.0);
      X::order();
      have = true;
      double* v = lds + (int64_t)g * slice;
      pgs_warm_rows<X>(v + (Jb + mo - vb) / 8, PgsRecs{rw.p}, nr, nv, v);
      for (int k = l; k < nv; k += GL) ok = ok && rfinite(ld(vb + 8 * k));
      phase = it = r = 0;
      moved = false;
      limit = C.iterations;
      if (X::ballot([&](int) { return !ok; })) {
        general(0);
        continue;
      }
      records(0);
      start();
    }
    if (__ballot(live) == 0) break;
    if (live) {
      // what the update needs, on its way during the sum; then the next row
      const Real vv = ld(va), c0 = ld(ra + C0), bias = ld(ra + BIAS), is = ld(ra + IS), mu = ld(ra + MU);
      const Real lam = ld(ra + LAM), lam_n = ld(ra - (int)(((unsigned)hi_w >> 28) << 4) + LAM), mr = ld(ja + mo);
      const bool last = r + 1 == nr;
      const int rb = last ? recb : ra + RB;
      int nlo, nhi;
      info(rb, &nlo, &nhi);
      const Real jv = X::template rowsum<W>(DLV{j * vv}, rsum0());
      const int nja = Jb + (nhi & 0xFFFF) * 8 + l8, nva = v_addr(nlo, nhi);
      const Real nj = ld(nja);
      const Real m = l < count_of(hi_w) ? mr : 0.0;
      const Real t = c0 * (jv + bias), il = is * lam, b = mu * lam_n;
      Real y = lam + (t - il);
      const Real hi = (hi_w >> 27) & 1 ? INFINITY : b;
      Real nw = rmin(rmax(y, -b), hi);
      if constexpr (EQ) {
        y = (lam + t) - il;
        nw = (hi_w >> 26) & 1 ? y : nw;
      }
      const Real dl = nw - lam, vn = vv + m * dl;
      const bool odd = __builtin_isnan(jv) || !__builtin_isfinite(vn);
      if (__ballot(odd)) {
        if (X::ballot([&](int) { return odd; })) {
          general(r);  // this row and the rest
          continue;
        }
      }
      if (__ballot(!moved && dl != 0.0)) {
        // |dl| against inv_a tol, from c0 = -inv_a or -inv_a mass_scale
        const Real size = fabs(dl), ac = fabs(c0);
        const bool soft = is != 0.0;
        const bool above = size > ac * (soft ? hi1 : hi0), below = size < ac * (soft ? lo1 : lo0);
        if (__ballot(!above && !below && dl != 0.0)) {
          if (!above && !below && dl != 0.0)
            moved = moved || pgs_reaches_tol(C, size, S.grow[e * (int64_t)M.nrmax * 10 + (int64_t)r * 10 + PR_INVA]);
        }
        moved = moved || above;
      }
      st(va, vn);
      st(ra + LAM, nw);
      X::order();
      j = l < count_of(nhi) ? nj : 0.0;
      va = nva, ja = nja, hi_w = nhi, ra = rb;
      r = last ? 0 : r + 1;
      if (last) {  // the sweep's end
        it++;
        if (!moved || it >= limit) {
          if (phase == 0) {
            for (int k = l; k < nv; k += GL) vpos[e * nv + k] = ld(vb + 8 * k);
            phase = 1;
            it = 0;
            limit = relax;
            records(1);
            start();
          } else {
            store(true);
          }
        }
        moved = false;
      }
    }
  }
#endif
}

// The sweeps over rows that are not packed (a row over 16 dofs, more rows than
// k_pgs_sweeps_rows holds, a factor that is not finite): one env per wavefront
// at a time, no LDS and few registers, so that many wavefronts share a SIMD and
// hide each other's dependent chains.
template <int K>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(5))) k_pgs_sweeps(const DModel* __restrict__ Mp, const DState* __restrict__ Sp,
                                                   int64_t begin, int64_t end, Real* vel, Real* vpos) {
#if defined(__HIP_DEVICE_COMPILE__)
  const DModel& M = *Mp;
  const DState& S = *Sp;
  const int nv = M.nv;
  const PgsConsts C = pgs_consts(M);
  for (int64_t e = begin + (int64_t)blockIdx.x; e < end; e += gridDim.x) {
    const int nr = S.nrows[e];
    if (S.status[e] != 0 || nr <= 0) continue;
    Real* rw = (S.grow + e * (int64_t)M.nrmax * 10).p;
    if ((S.grow + e * (int64_t)M.nrmax * 10)[PR_MODE] != 0.0) continue;
    Real* J = (S.gjac + e * (int64_t)M.nrmax * nv).p;
    Real* mj = (S.gmj + e * (int64_t)M.nrmax * nv).p;
    Real* v = vel + e * nv;
    Real* vp = vpos + e * nv;
    if (nr <= PGS_WAVE_ROWS) {
      const int lane = (int)threadIdx.x;
      const LaneVel r = pgs_sweeps_body(C, J, mj, rw, nr, nv, lane < nv ? v[lane] : 0.0);
      if (lane < nv) {
        v[lane] = r.v;
        vp[lane] = r.vpos;
      }
    } else if (threadIdx.x == 0) {
      pgs_sweeps_serial(C, J, mj, rw, nr, nv, v, vp);
    }
  }
#endif
}

template <int K>
__global__ void __launch_bounds__(64) k_pgs_back(const DModel* __restrict__ Mp, const DState* __restrict__ Sp,
                                                 int64_t begin, int64_t end, int64_t nstep, int64_t t, Real* qpos_out,
                                                 const Real* vel, const Real* vpos) {
  const DModel& M = *Mp;
  const DState& S = *Sp;
  extern __shared__ double lds[];
  const int g = (int)threadIdx.x / DevXK<K>::G;
  const int64_t rel = (int64_t)blockIdx.x * K + g;
  if (begin + rel >= end) return;
  Env E;
  E.s = lds + (int64_t)g * (M.L.bytes / 8);
  E.si = reinterpret_cast<int*>(E.s + M.L.ndouble);
  E.e = begin + rel;
  E.var = M.env_var[E.e];
  run_pgs_back<DevXK<K>>(M, S, E, nstep, t, qpos_out, rel, vel + E.e * M.nv, vpos + E.e * M.nv);
}

// Contact-count bucketing for k_step_ws, one workgroup: envs [begin, end)
// keyed by the Newton iterations of their last launch (summed over its steps)
// and their last contact count, grouped by key, costliest key first, into
// order (offsets from begin). Also resets the work-stealing counter for the
// launch that follows on the same stream.
constexpr int BUCKETS = 64;
static __global__ void __launch_bounds__(1024) k_bucket(const DState* __restrict__ Sp, int64_t begin, int64_t end,
                                                 int* __restrict__ order, unsigned* counter) {
  const DState& S = *Sp;
  __shared__ unsigned hist[BUCKETS];
  __shared__ unsigned off[BUCKETS];
  const int t = (int)threadIdx.x;
  const int64_t n = end - begin;
  if (t < BUCKETS) hist[t] = 0;
  __syncthreads();
  auto key = [&](int64_t e) {
    // iterations dominate an env's cost; contacts break ties within them
    int it = S.cost[e], nc = S.ncon[e];
    it = it < 0 ? 0 : (it > 31 ? 31 : it);
    nc = nc < 0 ? 0 : (nc > 1 ? 1 : nc);
    return it * 2 + nc;
  };
  for (int64_t i = t; i < n; i += blockDim.x) atomicAdd(&hist[key(begin + i)], 1u);
  __syncthreads();
  if (t == 0) {
    unsigned o = 0;
    for (int b = BUCKETS - 1; b >= 0; b--) {
      off[b] = o;
      o += hist[b];
    }
    counter[0] = 0;
  }
  __syncthreads();
  for (int64_t i = t; i < n; i += blockDim.x) {
    unsigned p = atomicAdd(&off[key(begin + i)], 1u);
    order[p] = (int)i;
  }
}

// Resets the work-stealing counter when no bucketing pass runs before k_step_ws
// (a kernel, not a memset, so that the launch sequence can be captured in a graph).
static __global__ void k_reset_counter(unsigned* counter) { counter[0] = 0; }

// The step with the learned warm start (mlp.hpp). Lane groups past the end
// stay in the loop without an env, since the network needs the whole wavefront.
template <int K, class MT>
__global__ void __launch_bounds__(64) k_step_mlp(const DModel* __restrict__ Mp, const DState* __restrict__ Sp,
                                                 int64_t begin, int64_t end, int64_t nstep, const Real* ctrl_seq,
                                                 Real* qpos_out) {
  const MT& M = *static_cast<const MT*>(Mp);
  const DState& S = *Sp;
  extern __shared__ double lds[];
  const int g = (int)threadIdx.x / DevXK<K>::G;
  const int64_t rel = (int64_t)blockIdx.x * K + g;
  const bool live = begin + rel < end;
  Env E;
  E.s = lds + (int64_t)g * (M.L.bytes / 8);
  E.si = reinterpret_cast<int*>(E.s + M.L.ndouble);
  E.e = begin + rel;
  E.var = live ? M.env_var[E.e] : 0;
  run_env_mlp<DevXKM<K>>(M, S, E, nstep, ctrl_seq, qpos_out, rel, live);
}

}  // namespace phk
