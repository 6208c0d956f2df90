// kmi_step_tb2d.hip — K time steps per launch for D2Q9 lattices (2, 4 or 8).
//
// Small 2D lattices (10^4–10^6 cells) do not fill the device: a single-step launch moves a
// few MB and its duration is the fixed cost of a dispatch (launch ramp, first-touch latency,
// the release of the written lines), 3–6 µs.  This kernel pays that cost once per K steps.
// A work-group loads its TW × TH tile plus a K-cell ring of the t populations into LDS,
// advances the whole region K steps in place (each step needs one cell less on every side),
// and writes the tile's t+K populations.  One work-item per cell of the region, so each in-LDS
// step is one dependent chain per work-item with up to 16 waves per CU to hide it; the cost is
// the ring's re-evaluation.
//
// Step s needs the (EW − 2s) × (EH − 2s) cells inside the region.  In FP64 they are dealt to the
// work-items afresh at every step, consecutive cells to consecutive lanes, so the waves that a
// step needs shrink with it: 8, 7, 6, 4, 4, 3, 2, 1 of the 9 waves of the 8×8 tile with 8 steps,
// against 9, 9, 7, 7, 7, 5, 5, 3 with active lanes, up to three on a SIMD, when every cell keeps
// its work-item (128² BGK cavity, µs per step: 2.17 kept, 1.96 dealt; 256² on 16×16 tiles with 4
// steps 3.49 and 3.30).  In FP32 the chain of one wave sets the time, and a kept cell's indices
// and wall tests stay out of the step loop: 128² F32S cavity 1.56 kept and 1.72 dealt, 512×256
// F32S Rayleigh–Bénard 4.19 and 4.63.  The second launch bound keeps 4 waves per SIMD (FP64 BGK
// 130 VGPRs without it: 256² on 8×8 tiles with 4 steps 4.37 instead of 3.72).
//
// Scope: D2Q9 BGK / TRT / MRT with periodic, wall, moving-wall and constant Zou–He
// (velocity or pressure) faces, bounce-back or inert masks and Guo forcing (constant or
// per-node), and the thermal double distribution (THM: g beside f in LDS, Dirichlet /
// adiabatic walls, Boussinesq coupling split or fused; not in FP64) — the lattices of run_cavity_2d,
// run_poiseuille_2d, run_rayleigh_benard_2d and the .krk 2D loop without per-node faces.  Per-cell arithmetic and order are the single-step kernel's (kmi_cell.h),
// and every intermediate value passes through the storage rounding, so the result is
// bit-identical to K single-step launches in every storage.
#include "kmi_cell.h"
#include "kmi_internal.h"

namespace kmi {

// LATE: the tile's own cells are stored after the step loop instead of in its last step, which
// takes 14–32 VGPRs less.  A launch whose groups spread over the CUs gains by the stores in the
// loop (2–5 %); where groups share a CU the registers decide how many do.
//   - regions of 576 cells (9 waves a group) from 257 groups on: FP32 70 VGPRs instead of 84, three
//     groups a CU instead of one or two: 900×300 BGK cavity on 16×16 tiles 5.98 instead of 8.36 µs a
//     step, on 8×8 tiles with 8 steps 14.2 instead of 19.5; thermal 90 VGPRs instead of 120, 900×300
//     Rayleigh–Bénard on 16×16 tiles 10.9 instead of 11.8.
//   - regions of 256 cells from 1025 groups on: that lattice on 8×8 tiles 8.8–9.2 instead of 9.5.
//   - tiles with two steps per launch: 64² and 128² F32 cavities on 60×12 tiles 3.12 and 3.22 instead
//     of 3.61 and 3.86, others within 1 %; the 56×8 tile in FP64: 700² 15.5 instead of 15.6.
// Whether a step writes a second buffer instead of the one it reads, which saves one of its two
// barriers: the 8×8 tile with 8 steps where its groups have a CU each (83 KB in FP64): 128² BGK
// cavity F64 1.96 → 1.89, F32S 1.56 → 1.52 µs per step.  Groups that share a CU lose more by the
// LDS (330² F32 on 16×16 tiles with 4 steps 3.9 → 4.5).
constexpr bool tb2d_two_buffers(int TW, int TH, int K, bool thm, bool late) {
  return !thm && !late && K == 8 && TW == 8 && TH == 8;
}
// Waves per SIMD the register budget is set for.
template <class R, int COLL, int TW, int TH, int K, bool THM, bool LATE>
constexpr int tb2d_waves() {
  constexpr int NE = (TW + 2 * K) * (TH + 2 * K);
  if (tb2d_two_buffers(TW, TH, K, THM, LATE)) return 3;
  if (LATE && NE < 1024 && sizeof(R) == 4) return THM ? 5 : 7;
  if (LATE && NE == 576 && COLL != KMI_BGK) return 5;
  return 4;
}

template <int ST, int COLL, int TW, int TH, int K, bool THM, bool LATE>
__global__ void __launch_bounds__((TW + 2 * K) * (TH + 2 * K),
                                  (tb2d_waves<typename Store<ST>::real, COLL, TW, TH, K, THM, LATE>()))
    k_step_tb2d(const StepArgs a) {
  using S = Store<ST>;
  using E = typename S::elem;
  using R = typename S::real;
  using GS = Store<thermal_storage(ST)>;
  using GE = typename GS::elem;
  constexpr bool SH = S::shifted;
  constexpr int EW = TW + 2 * K, EH = TH + 2 * K, NE = EW * EH;
  constexpr bool DEAL = sizeof(R) == 8;
  constexpr bool TWOBUF = tb2d_two_buffers(TW, TH, K, THM, LATE);
  constexpr int NV = (THM ? 18 : 9) * NE;
  __shared__ R lds[(TWOBUF ? 2 : 1) * NV];
  R* L = lds;
  R* G = L + 9 * NE;  // thermal populations (THM)
  const GE* __restrict__ gi = static_cast<const GE*>(a.gi);
  GE* __restrict__ go = static_cast<GE*>(a.go);
  const int nx = a.nx, ny = a.ny;
  const long long P = a.plane;
  const E* __restrict__ fi = static_cast<const E*>(a.fi);
  E* __restrict__ fo = static_cast<E*>(a.fo);
  const int ox = int(blockIdx.x) * TW - K, oy = int(blockIdx.y) * TH - K;  // LDS origin
  const int tid = threadIdx.x;
  const bool perx = a.per[0] != 0, pery = a.per[1] != 0;
  // Unwrapped coordinates overshoot the lattice by at most K + TW (K < nx, ny is required).
  auto wx = [&](int u) { return u < 0 ? u + nx : (u >= nx ? u - nx : u); };
  auto wy = [&](int u) { return u < 0 ? u + ny : (u >= ny ? u - ny : u); };
  auto inside = [&](int ux, int uy) {
    return (perx || (ux >= 0 && ux < nx)) && (pery || (uy >= 0 && uy < ny));
  };

  if (const int ux = ox + tid % EW, uy = oy + tid / EW; inside(ux, uy)) {
    const long long self = wx(ux) + (long long)nx * wy(uy);
    sfor<9>([&](auto qc) {
      constexpr int q = decltype(qc)::value;
      L[q * NE + tid] = S::ld(fi, self + q * P);
      if constexpr (THM) G[q * NE + tid] = GS::ld(gi, self + q * P);
    });
  }
  __syncthreads();

  R nv[9], gv[9];
  // the tile's own cells: step t+K straight from registers
  auto store = [&](int ux, int uy) {
    if (ux >= nx || uy >= ny) return;
    const long long self = ux + (long long)nx * uy;
    sfor<9>([&](auto qc) {
      constexpr int q = decltype(qc)::value;
      S::template st<false>(fo, self + q * P, nv[q]);
      if constexpr (THM) GS::template st<false>(go, self + q * P, gv[q]);
    });
  };
  for (int s = 1; s <= K; ++s) {
    int ex = tid % EW, ey = tid / EW;
    if constexpr (DEAL) {
      // cell tid of the step's (EW − 2s) × (EH − 2s) cells; ⌊tid / w⌋ = tid·⌈2^16/w⌉ >> 16 for
      // tid < 1024 and w ≤ 64 (tid·(w − 1) < 2^16)
      const int w = EW - 2 * s;
      unsigned m = 0;
      sfor<K>([&](auto kc) {
        constexpr int k = decltype(kc)::value + 1, wk = EW - 2 * k;
        if (s == k) m = (65536 + wk - 1) / wk;
      });
      const int row = int(unsigned(tid) * m >> 16);
      ex = s + tid - row * w;
      ey = s + row;
    }
    const int e = ex + ey * EW, ux = ox + ex, uy = oy + ey;
    const bool active = (DEAL || (ex >= s && ex < EW - s && ey >= s)) && ey < EH - s && inside(ux, uy);
    if (active) {
      const int i = wx(ux), j = wy(uy);
      const long long self = i + (long long)nx * j;
      // a link whose source lies beyond a non-periodic face bounces back (k_step's rule)
      const bool vxm = perx || i > 0, vxp = perx || i < nx - 1;
      const bool vym = pery || j > 0, vyp = pery || j < ny - 1;
      R fp[9], fr[9], gp[9], gr[9];
      sfor<9>([&](auto qc) {
        constexpr int q = decltype(qc)::value;
        constexpr int cx = Lat<9>::cx[q], cy = Lat<9>::cy[q];
        constexpr int o = Lat<9>::opp[q];
        const bool ok = (cx > 0 ? vxm : (cx < 0 ? vxp : true)) && (cy > 0 ? vym : (cy < 0 ? vyp : true));
        if constexpr (THM) gp[q] = ok ? G[q * NE + e - cx - cy * EW] : G[o * NE + e];
        R v = ok ? L[q * NE + e - cx - cy * EW] : L[o * NE + e];
        if constexpr (q != 0) {
          if (a.any_moving && !ok) {
            auto add = [&](int fid) {
              const FaceArgs& F = a.face[fid];
              if (F.kind == KMI_FACE_MOVING_WALL)
                v = v + R(six_w(Lat<9>::w[q])) * R(F.rho) * cdotu<cx, cy, 0>(R(F.u[0]), R(F.u[1]), R(F.u[2]));
            };
            if (cx > 0 && !vxm) add(KMI_WEST);
            if (cx < 0 && !vxp) add(KMI_EAST);
            if (cy > 0 && !vym) add(KMI_SOUTH);
            if (cy < 0 && !vyp) add(KMI_NORTH);
          }
        }
        fp[q] = v;
      });
      for (int n = 0; n < a.n_zh; ++n) {
        const int fid = a.zh_face[n];
        const FaceArgs& F = a.face[fid];
        if (fid == KMI_NORTH && j == ny - 1) zh_north<SH>(fp, R(F.u[0]));
        else if (fid == KMI_SOUTH && j == 0) zh_south<SH>(fp, R(F.u[0]));
        else if (fid == KMI_WEST && i == 0) {
          if (F.kind == KMI_FACE_ZOUHE_VELOCITY) zh_west<SH>(fp, R(F.u[0]));
          else zh_pressure_west<SH>(fp, R(F.rho), R(F.rho - 1.0));
        } else if (fid == KMI_EAST && i == nx - 1) {
          zh_pressure_east<SH>(fp, R(F.rho), R(F.rho - 1.0));
        }
      }
      const bool solid = a.mask != nullptr && a.mask[self] == kCellSolid;
      if constexpr (THM) {
        // the thermal step of k_step: anti-bounce-back faces, T, Boussinesq force, thermal
        // BGK with the unforced (split) or forced (fused) u, Guo collision of f
        thermal_faces<SH>(gp, a, i, j);
        const R Tl = zeroth_moment<9>(gp);
        const R m0 = zeroth_moment<9>(fp);
        const R rho = SH ? R(1) + m0 : m0;
        const R inv = R(1) / rho;
        const R jx = first_moment<9, 0>(fp);
        const R jy = first_moment<9, 1>(fp);
        const R fy = SH ? R(a.beta_g) * Tl : R(a.beta_g) * (Tl - R(a.T_ref));
        const R fx = R(0);
        R uxf, uyf, uxt, uyt;
        if (a.coupling == KMI_COUPLING_SPLIT) {
          uxt = jx * inv;
          uyt = jy * inv;
          uxf = (jx + fx / R(2)) * inv;
          uyf = (jy + fy / R(2)) * inv;
        } else {
          uxf = jx * inv;
          uyf = (jy + fy / R(2)) * inv;
          uxt = uxf;
          uyt = uyf;
        }
        collide_thermal<SH>(gp, gr, uxt, uyt, R(a.omega_T), R(a.T_ref));
        if (solid) {
          sfor<9>([&](auto qc) { fr[decltype(qc)::value] = fp[Lat<9>::opp[decltype(qc)::value]]; });
        } else {
          collide_guo<SH>(fp, fr, m0, rho, uxf, uyf, fx, fy, R(a.omega));
        }
        sfor<9>([&](auto qc) { gv[decltype(qc)::value] = gr[decltype(qc)::value]; });
      } else if (solid && a.solid_inert) {
        sfor<9>([&](auto qc) { fr[decltype(qc)::value] = SH ? R(0) : R(Lat<9>::w[decltype(qc)::value]); });
      } else if (solid) {
        sfor<9>([&](auto qc) { fr[decltype(qc)::value] = fp[Lat<9>::opp[decltype(qc)::value]]; });
      } else if constexpr (COLL == KMI_BGK) {
        if (a.forcing) {
          R fx, fy, fz;
          node_force<9>(a, self, fx, fy, fz);
          const R m0 = zeroth_moment<9>(fp);
          const R rho = SH ? R(1) + m0 : m0;
          const R inv = R(1) / rho;
          const R ux2 = (first_moment<9, 0>(fp) + fx / R(2)) * inv;
          const R uy2 = (first_moment<9, 1>(fp) + fy / R(2)) * inv;
          collide_guo<SH>(fp, fr, m0, rho, ux2, uy2, fx, fy, R(a.omega));
        } else {
          collide_bgk<9, SH>(fp, fr, R(a.omega));
        }
      } else if constexpr (COLL == KMI_TRT) {
        collide_trt<9, SH>(fp, fr, R(a.s_plus), R(a.s_minus));
      } else {
        collide_mrt<SH>(fp, fr, R(a.s_e), R(a.s_eps), R(a.s_q), R(a.s_nu));
      }
      sfor<9>([&](auto qc) {
        constexpr int q = decltype(qc)::value;
        nv[q] = fr[q];
      });
    }
    if (s == K) {
      if constexpr (!LATE)
        if (active) store(ux, uy);
      break;
    }
    if constexpr (TWOBUF) {
      L = lds + (s & 1) * NV;
      G = L + 9 * NE;
    } else {
      __syncthreads();  // every step-s read of L is done
    }
    if (active)
      sfor<9>([&](auto qc) {
        constexpr int q = decltype(qc)::value;
        L[q * NE + e] = storage_round<ST>(nv[q]);
        if constexpr (THM) G[q * NE + e] = storage_round<thermal_storage(ST)>(gv[q]);
      });
    __syncthreads();
  }
  if constexpr (LATE) {
    int ix = tid % EW - K, iy = tid / EW - K;
    if constexpr (DEAL) ix = tid % TW, iy = tid / TW;
    if (ix >= 0 && ix < TW && iy >= 0 && iy < TH) store(ox + K + ix, oy + K + iy);
  }
}

// ---- dispatch ---------------------------------------------------------------------------
// Variants: regions of 1024 cells, 1 = 28×28 tile, 2 steps; 2 = 24×24, 4 steps;
// 3 = 56×8, 4 steps; 4 = 16×16, 8 steps; 5 = 60×12, 2 steps; smaller regions, which spread
// a small lattice over more CUs: 6 = 8×8, 4 steps (256 cells); 7 = 16×16, 4 steps (576);
// 8 = 8×8, 8 steps (576).
bool tb2d_variant(int tile, int& TW, int& TH, int& K) {
  switch (tile) {
    case 1: TW = 28; TH = 28; K = 2; return true;
    case 2: TW = 24; TH = 24; K = 4; return true;
    case 3: TW = 56; TH = 8; K = 4; return true;
    case 4: TW = 16; TH = 16; K = 8; return true;
    case 5: TW = 60; TH = 12; K = 2; return true;
    case 6: TW = 8; TH = 8; K = 4; return true;
    case 7: TW = 16; TH = 16; K = 4; return true;
    case 8: TW = 8; TH = 8; K = 8; return true;
    default: return false;
  }
}

template <int ST, int COLL, int TW, int TH, int K, bool LATE>
static hipError_t launch_tb_groups(const StepArgs& a, bool th, dim3 g, hipStream_t s) {
  const dim3 b((TW + 2 * K) * (TH + 2 * K));
  if (th) {
    // the thermal chain collides f with Guo BGK; FP64 f and g exceed the registers of a
    // 1024-wide group, so FP64 thermal lattices keep single-step launches
    if constexpr (COLL == KMI_BGK && ST != KMI_STORE_F64)
      hipLaunchKernelGGL((k_step_tb2d<ST, COLL, TW, TH, K, true, LATE>), g, b, 0, s, a);
    else
      return hipErrorInvalidValue;
  } else {
    hipLaunchKernelGGL((k_step_tb2d<ST, COLL, TW, TH, K, false, LATE>), g, b, 0, s, a);
  }
  return hipGetLastError();
}

template <int ST, int COLL, int TW, int TH, int K>
static hipError_t launch_tb(const StepArgs& a, bool th, hipStream_t s) {
  const dim3 g(unsigned((a.nx + TW - 1) / TW), unsigned((a.ny + TH - 1) / TH));
  constexpr int NE = (TW + 2 * K) * (TH + 2 * K);
  if constexpr (K == 2 || (TW == 56 && ST == KMI_STORE_F64)) {
    return launch_tb_groups<ST, COLL, TW, TH, K, true>(a, th, g, s);
  } else {
    if constexpr (NE < 1024)
      if ((long long)g.x * g.y > (NE == 576 ? 256 : 1024)) return launch_tb_groups<ST, COLL, TW, TH, K, true>(a, th, g, s);
    return launch_tb_groups<ST, COLL, TW, TH, K, false>(a, th, g, s);
  }
}

template <int ST, int COLL>
static hipError_t launch_tb_tile(int tile, const StepArgs& a, bool th, hipStream_t s) {
  switch (tile) {
    case 1: return launch_tb<ST, COLL, 28, 28, 2>(a, th, s);
    case 2: return launch_tb<ST, COLL, 24, 24, 4>(a, th, s);
    case 3: return launch_tb<ST, COLL, 56, 8, 4>(a, th, s);
    case 4: return launch_tb<ST, COLL, 16, 16, 8>(a, th, s);
    case 5: return launch_tb<ST, COLL, 60, 12, 2>(a, th, s);
    case 6: return launch_tb<ST, COLL, 8, 8, 4>(a, th, s);
    case 7: return launch_tb<ST, COLL, 16, 16, 4>(a, th, s);
    case 8: return launch_tb<ST, COLL, 8, 8, 8>(a, th, s);
    default: return hipErrorInvalidValue;
  }
}

template <int ST>
static hipError_t launch_tb_coll(int coll, int tile, const StepArgs& a, bool th, hipStream_t s) {
  if (th) return launch_tb_tile<ST, KMI_BGK>(tile, a, true, s);
  if (coll == KMI_MRT) return launch_tb_tile<ST, KMI_MRT>(tile, a, false, s);
  if (coll == KMI_TRT) return launch_tb_tile<ST, KMI_TRT>(tile, a, false, s);
  return launch_tb_tile<ST, KMI_BGK>(tile, a, false, s);
}

hipError_t launch_step_tb2d(int st, int coll, int tile, bool th, const StepArgs& a, hipStream_t s) {
  switch (st) {
    case KMI_STORE_F64: return launch_tb_coll<KMI_STORE_F64>(coll, tile, a, th, s);
    case KMI_STORE_F32: return launch_tb_coll<KMI_STORE_F32>(coll, tile, a, th, s);
    case KMI_STORE_F32S: return launch_tb_coll<KMI_STORE_F32S>(coll, tile, a, th, s);
    default: return launch_tb_coll<KMI_STORE_F16S>(coll, tile, a, th, s);
  }
}

}  // namespace kmi
