// kmi_march2d.hip — four steps per launch for large D2Q9 lattices: the register march of
// kmi_march2d.h over one lattice.
//
// Scope: BGK / TRT / MRT with periodic, wall, moving-wall and constant Zou–He faces, without
// mask, forcing, cut links or thermal populations.
#include "kmi_internal.h"
#include "kmi_march2d.h"

namespace kmi {

// XREST: the x faces are periodic or resting walls, so cells off the y faces have neither a
// Ladd term nor a closure (the tests for them cost the wall strips a third of their time).
template <int ST, int COLL, bool XREST>
struct LatticeDom {
  using E = typename Store<ST>::elem;
  using R = typename Store<ST>::real;
  static constexpr bool SH = Store<ST>::shifted;
  const StepArgs& a;
  int nx, ny;
  bool perx, pery;
  KMI_DEV explicit LatticeDom(const StepArgs& args)
      : a(args), nx(args.nx), ny(args.ny), perx(args.per[0] != 0), pery(args.per[1] != 0) {}
  KMI_DEV const E* src(int q) const { return static_cast<const E*>(a.fi) + q * a.plane; }
  KMI_DEV E* dst(int q) const { return static_cast<E*>(a.fo) + q * a.plane; }
  template <int q, bool ROWS>
  KMI_DEV R ladd(R v, bool wxm, bool wxp, bool wym, bool wyp) const {
    constexpr int cx = Lat<9>::cx[q], cy = Lat<9>::cy[q];
    if constexpr (XREST && !ROWS) return v;
    if (a.any_moving) {
      auto add = [&](int fid) {
        const FaceArgs& F = a.face[fid];
        if (F.kind == KMI_FACE_MOVING_WALL)
          v = v + R(six_w(Lat<9>::w[q])) * R(F.rho) * cdotu<cx, cy, 0>(R(F.u[0]), R(F.u[1]), R(F.u[2]));
      };
      if (cx > 0 && wxm) add(KMI_WEST);
      if (cx < 0 && wxp) add(KMI_EAST);
      if (cy > 0 && wym) add(KMI_SOUTH);
      if (cy < 0 && wyp) add(KMI_NORTH);
    }
    return v;
  }
  template <bool ROWS>
  KMI_DEV void closures(R (&fp)[9], int i, int j) const {
    if constexpr (XREST && !ROWS) return;
    for (int n = 0; n < a.n_zh; ++n) {
      const int fid = a.zh_face[n];
      const FaceArgs& F = a.face[fid];
      if (ROWS && fid == KMI_NORTH && j == ny - 1) zh_north<SH>(fp, R(F.u[0]));
      else if (ROWS && fid == KMI_SOUTH && j == 0) zh_south<SH>(fp, R(F.u[0]));
      else if (fid == KMI_WEST && i == 0) {
        if (F.kind == KMI_FACE_ZOUHE_VELOCITY) zh_west<SH>(fp, R(F.u[0]));
        else zh_pressure_west<SH>(fp, R(F.rho), R(F.rho - 1.0));
      } else if (fid == KMI_EAST && i == nx - 1) {
        zh_pressure_east<SH>(fp, R(F.rho), R(F.rho - 1.0));
      }
    }
  }
  KMI_DEV void collide(const R (&fp)[9], R (&fo)[9]) const {
    if constexpr (COLL == KMI_BGK) collide_bgk<9, SH>(fp, fo, R(a.omega));
    else if constexpr (COLL == KMI_TRT) collide_trt<9, SH>(fp, fo, R(a.s_plus), R(a.s_minus));
    else collide_mrt<SH>(fp, fo, R(a.s_e), R(a.s_eps), R(a.s_q), R(a.s_nu));
  }
};

// Piece w = strip + strips · chunk; work-group b runs on XCD b mod 8 and takes four
// consecutive pieces of that XCD's band, so the columns that neighbouring strips share meet
// in one L2.
template <int ST, int COLL, int K, bool XREST>
__global__ void __launch_bounds__(256, (march_waves<ST, K>()))
    k_march2d(const StepArgs a, int rows, int pieces, int per_xcd) {
  const LatticeDom<ST, COLL, XREST> d(a);
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
  const int w = (int(blockIdx.x % 8u) * per_xcd + int(blockIdx.x / 8u)) * 4 + wave;
  if (w >= pieces) return;
  const MarchStrips st = march_strips(d.nx, K, d.perx);
  const int strip = w % st.m, chunk = w / st.m;
  const int xs = st.start(strip), xe = st.start(strip + 1);
  const int y0 = chunk * rows, y1 = min(y0 + rows, d.ny);
  if (march_inner(d.nx, d.perx, K, xs, xe)) march2d<ST, K, false>(d, xs, xe, y0, y1);
  else march2d<ST, K, true>(d, xs, xe, y0, y1);
}

static bool rests(int kind) { return kind == KMI_FACE_PERIODIC || kind == KMI_FACE_WALL; }

template <int ST, int COLL>
static hipError_t launch_march_coll(const StepArgs& a, hipStream_t s) {
  constexpr int K = 4;
  const int m = march_strips(a.nx, K, a.per[0] != 0).m;
  auto count = [&](int rows) { return (long long)m * ((a.ny + rows - 1) / rows); };
  const int rows = march_rows(a.ny, march_waves<ST, K>(), count);
  const int pieces = int(count(rows)), per_xcd = ((pieces + 3) / 4 + 7) / 8;
  const dim3 g(static_cast<unsigned>(8 * per_xcd)), b(256);
  if (rests(a.face[KMI_WEST].kind) && rests(a.face[KMI_EAST].kind))
    hipLaunchKernelGGL((k_march2d<ST, COLL, K, true>), g, b, 0, s, a, rows, pieces, per_xcd);
  else
    hipLaunchKernelGGL((k_march2d<ST, COLL, K, false>), g, b, 0, s, a, rows, pieces, per_xcd);
  return hipGetLastError();
}

template <int ST>
static hipError_t launch_march_st(int coll, const StepArgs& a, hipStream_t s) {
  if (coll == KMI_MRT) return launch_march_coll<ST, KMI_MRT>(a, s);
  if (coll == KMI_TRT) return launch_march_coll<ST, KMI_TRT>(a, s);
  return launch_march_coll<ST, KMI_BGK>(a, s);
}

// Where the march beats the 24×24 tile with four steps (k_step_tb2d).  The tile's time hardly grows up
// to 512 work-groups, two to a CU (FP64: one, 256), while a march that short of rows is bound by the
// 4 + 3 and more rows each wave evaluates in turn.  What moves the line, µs per step, tile / march:
//   - strips whose lanes are half empty between walls (channel 70×5714 F64 BGK 11.9 / 14.2): 0.7 of the groups;
//   - x faces with a closure or a Ladd term, whose tests sit in the row loop (channel F32S MRT 500² 5.6 /
//     7.5, 1024² 17.2 / 15.8, 1200² 21.7 / 19.4; F64 BGK 700² 14.6 / 11.8);
//   - F16S, whose conversions the tile hides better (BGK cavity 500² 5.4 / 6.5, 700² 9.0 / 7.6);
//   - within the tile's first round (FP64: second) the march needs, between x walls, filled strips of
//     some rows (F32 BGK box 400² 5.2 / 4.2, periodic 400² 5.2 / 3.9), and in FP32 y faces without
//     closures or Ladd terms (F32 MRT cavity 500² 5.8 / 6.2).
// Over 4,142 lattices of 165,000–4,200,000 cells (every storage; BGK, MRT; periodic, walls, lids,
// channels; squares, 32–240 wide, 32–200 high): always marching 0.862 of the tile's time and up to
// 1.8, this rule 0.827 and up to 1.16, the better of both 0.821.
bool march2d_wins(int st, int coll, const StepArgs& a) {
  if ((long long)a.nx * a.ny < 160000) return false;
  const bool f64 = st == KMI_STORE_F64, f16 = st == KMI_STORE_F16S, perx = a.per[0] != 0;
  const bool restx = rests(a.face[KMI_WEST].kind) && rests(a.face[KMI_EAST].kind);
  const bool resty = rests(a.face[KMI_SOUTH].kind) && rests(a.face[KMI_NORTH].kind);
  const bool filled = 10LL * a.nx >= 6LL * 64 * march_strips(a.nx, 4, perx).m;
  long long groups = (long long)((a.nx + 23) / 24) * ((a.ny + 23) / 24);
  if (!perx && !filled && !(f64 && restx)) groups = groups * 7 / 10;
  if (!restx) return groups > (f64 ? 840 : f16 ? 2200 : 1800);
  if (f16) return groups > (perx ? 512 : 840);
  if (groups > 512) return true;
  const bool snug = a.ny >= 64 && a.nx >= 56 && filled;
  if (perx) return snug || st != KMI_STORE_F32 || coll != KMI_MRT;
  return snug && (f64 || resty);
}

hipError_t launch_march2d(int st, int coll, const StepArgs& a, hipStream_t s) {
  switch (st) {
    case KMI_STORE_F64: return launch_march_st<KMI_STORE_F64>(coll, a, s);
    case KMI_STORE_F32: return launch_march_st<KMI_STORE_F32>(coll, a, s);
    case KMI_STORE_F32S: return launch_march_st<KMI_STORE_F32S>(coll, a, s);
    default: return launch_march_st<KMI_STORE_F16S>(coll, a, s);
  }
}

}  // namespace kmi
