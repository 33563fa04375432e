// Plane cell kernel of the matrix-free heat operator for FE degrees 1 to 3
// (gfx950). Reference: source/ThermalOperator.templates.hh:479-617.
//
// Lane layout: p+1 lanes per cell, lane s owning the x-y plane z = s of the
// cell's nodes and, after the z contraction, the x-y plane of quadrature
// points z = s. The x and y contractions run on the lane's (p+1)^2 values in
// registers; only the z direction crosses lanes, through a wave-private LDS
// buffer: one exchange for the evaluation and one for the integration
// (against six in the line-per-lane kernel). A wavefront takes a patch of
// PX x PY cells of one cell layer (7 x 3 for Q2: 63 lanes; 8 x 4 for Q1 and
// 4 x 4 for Q3: 64 lanes), so the nodes its cells share along x and y are
// summed inside the wavefront (cross-lane shuffles). Each patch then stores
// its node sums
// in its own block of a patch buffer, and a second kernel (one lane per
// node) adds the blocks of the patches that share the node, in a fixed
// order, into dst. No atomics: FP64 atomic adds to device memory are
// performed at the memory side on this chip and cost more than the whole
// computation (measured: the loads and atomic adds alone of this layout
// took 84 us per application of the 128x64x32 Q2 workload), and the result
// is the same in every run.
//
// Arithmetic: the values at the quadrature points, and so the phase state,
// equal the CPU oracle's bit for bit (S along x, y, then z with the same fma
// chains); the x and y gradients are the oracle's collocation derivatives,
// the z gradient comes from the nodal planes through DcS = Dc S. The
// integration folds each point row into the node plane at once: the x
// part through DcS^T and S^T along x, the y part through S^T along x and
// DcS^T along y, so only two planes of accumulators are live; the z part
// goes through S^T and DcS^T across the lanes. dst differs from the oracle
// by rounding only (1/(rho c_p) comes from the hardware reciprocal refined
// by two Newton steps).
//
// What bounds it: latency, not arithmetic or memory. A patch of the
// 128x64x32 Q2 workload issues for some 2,500 cycles of its wavefront; with
// the two wavefronts per SIMD that the registers allow, the chains of LDS
// reads (interval, breakpoint, coefficients), of a patch's global loads and
// of spilled registers' reloads are what it waits for. Hence:
//  - one-interval form: a wavefront whose planes are cold and lie in one
//    table interval each reads the coefficients once per plane and then runs
//    a point loop without branches or LDS reads (see there);
//  - the next patch's loads are issued a patch ahead;
//  - a row's interval look-ups advance together;
//  - the other wavefronts work in two steps with the points' properties in
//    LDS between them (see there), the heat source sits behind a call and
//    scalar constants that follow from symmetry are not held twice, so that
//    no vector register spills to memory: its reload would wait for the loads
//    in flight before it. Scalar registers do spill, to lanes of vector
//    registers (95 for Q1, 102 for Q2, 183 for Q3 with three states and merged
//    tables);
//  - the two parts of the integration share one exchange.
// 128x64x32 Q2, per application (plane + gather + face kernels): 100.4 us
// before, 76.9 us with these (71.4 with the face term in the launch); 64
// members of 64x32x16, per RK4 step: 3.17 ms before, 2.39 ms; Q1 101x67x33:
// 38.6 us before, 28.6 us (24.5). Q3 (line kernel in 8 colour launches
// before), RK4 step of 50x25x17: 433 us before, 162 us. What is left of the
// large launch is its slowest wavefront (melt under the beam: 133,000 cycles
// against a mean of 87,000). Handing patches out by a counter instead of a
// fixed share took 73 us against 77 there, but the counter's round trip cost
// the short Q1 patches 10 % and batched launches 2 %.
// Wavefronts that are solid across several intervals (one material, no
// powder, below the solidus) take a path of their own: the mixtures reduce
// to the solid value (the reference adds the other states with a zero ratio,
// which changes no bit), without the mushy-zone division. The rest update
// the phase state point by point. The heat sources run in a second pass over
// the cells a beam can reach.
#pragma once

#include "adm_kernels.hpp"

namespace adm {

template <int P>
struct PlaneLanes {
  static_assert(P >= 1 && P <= 3, "plane kernel: FE degrees 1 to 3");
  static constexpr int N = P + 1;
  static constexpr int NP = N * N;  // values per lane
  static constexpr int PX = P == 1 ? 8 : (P == 2 ? 7 : 4);
  static constexpr int PY = P == 1 ? 4 : (P == 2 ? 3 : 4);
  static constexpr int cells_per_wave = PX * PY;
  // exchange slot per lane (doubles), even so that slots stay 16-byte
  // aligned for 128-bit LDS accesses; a cell's N slots are followed by a
  // gap that spreads the cells of a 128-bit read over the banks. Q3: one
  // double more than the 16 values (64-bit accesses without conflicts; two
  // blocks of 4 wavefronts then just fit a compute unit's LDS)
  static constexpr int slot = P == 3 ? 17 : (NP + 1) & ~1;
  static constexpr int cell_slots = N * slot + (P == 1 ? 2 : 0);
  // slots of every lane's cell, including the partial cell of the lanes
  // past the last whole one (Q2: lane 63 addresses cell 21's planes)
  static constexpr int exchange = ((64 + N - 1) / N) * cell_slots;
  // two buffers: the two parts of the integration are exchanged at once.
  // Between the exchanges the same words hold values of the lane's points,
  // [point][lane]: two arrays, or three where a material is anisotropic
  static constexpr int points = 64 * NP;
  static constexpr int wave_lds = 2 * exchange;
  static constexpr int wave_lds_aniso =
      wave_lds > 3 * points ? wave_lds : 3 * points;
  static_assert(wave_lds >= 2 * points, "point arrays");
  // nodes of a patch: (P PX + 1) x (P PY + 1) per plane, N planes; the
  // patch buffer holds one double per node, [plane][y][x]
  static constexpr int patch_nx = P * PX + 1, patch_ny = P * PY + 1;
  static constexpr int patch_nodes = patch_nx * patch_ny * N;
};

// Doubles of the library's static scratch array (adm_vmult_noalloc), which
// holds the plane kernel's patch buffer there: 40 MiB per device, enough
// for the 128x64x32 Q2 workload's 4.2 million patch-buffer doubles.
constexpr size_t kNoAllocScratchDoubles = (size_t)5 << 20;

// doubles of one material's merged tables staged in LDS by the plane
// kernel: B, the coefficients of density .. thermal_conductivity_z, then
// the MergedBins record
constexpr int kPlaneMergedLds =
    kMergedLds + (int)(sizeof(MergedBins) / sizeof(double));
static_assert(sizeof(MergedBins) % sizeof(double) == 0, "bins layout");

// Quotient and remainder by a divisor used many times: with
// m = floor(2^32 / d) (2^32 - 1 for d = 1) the high word of r m is the
// quotient or one less for every r < 2^31.
struct FastDiv {
  uint32_t d, m;
  __device__ __forceinline__ explicit FastDiv(uint32_t d_)
      : d(d_), m(d_ > 1 ? (uint32_t)(0x100000000ull / d_) : 0xffffffffu) {}
  __device__ __forceinline__ uint32_t div(uint32_t r, uint32_t &rem) const {
    uint32_t q = (uint32_t)(((uint64_t)r * m) >> 32);
    rem = r - q * d;
    if (rem >= d) {
      ++q;
      rem -= d;
    }
    return q;
  }
};

// Coordinates of patch index r in a plane launch of npx x npy patches per
// cell layer and nz layers: x fastest, then y, then the cell layer; or
// (ymajor) x fastest, then the cell layer, then y -- the order in which the
// XCD-aware launch hands each XCD one contiguous range, so that every XCD
// takes a slab of patch rows through all the layers and as many of the slow
// layers (powder, melt) as the others.
struct PatchAt {
  int px, py, pz;
  __device__ __forceinline__ PatchAt(const FastDiv &by_npx,
                                     const FastDiv &by_mid, bool ymajor,
                                     int r) {
    uint32_t x, mid;
    const uint32_t t = by_npx.div((uint32_t)r, x);
    const uint32_t top = by_mid.div(t, mid);
    px = (int)x;
    py = (int)(ymajor ? top : mid);
    pz = (int)(ymajor ? mid : top);
  }
};

// 1/x from the hardware reciprocal and two Newton steps (within an ulp or
// two of the correctly rounded quotient)
__device__ __forceinline__ double recip(double x) {
  double r = __builtin_amdgcn_rcp(x);
  double e = __builtin_fma(-x, r, 1.0);
  r = __builtin_fma(r, e, r);
  e = __builtin_fma(-x, r, 1.0);
  return __builtin_fma(r, e, r);
}

// Intervals j = #{B_k <= T} of M points in a merged table by its bins
// (MergedBins). The M look-ups advance together, so that their LDS reads
// overlap. Two candidates are compared without a branch (B is padded with
// +inf, and a candidate past a bin's own breakpoints lies above T); tables
// with more breakpoints in one bin take the loop.
template <int M>
__device__ __forceinline__ void merged_bin_intervals(const double *B,
                                                     const MergedBins &mb,
                                                     const double (&T)[M],
                                                     int (&j)[M]) {
  int k0[M];
#pragma unroll
  for (int i = 0; i < M; ++i) {
    const double x = (T[i] - mb.lo) * mb.inv_w;
    int b = (int)x;  // NaN and T below lo give bin 0 after the clamp
    b = x < 0.0 ? 0 : (b > kMergedBins - 1 ? kMergedBins - 1 : b);
    k0[i] = mb.k0[b];
  }
  const int maxc = __builtin_amdgcn_readfirstlane((int)mb.maxc);
#pragma unroll
  for (int i = 0; i < M; ++i) {
    const int k1 = k0[i] + 1 < kMergedMax - 1 ? k0[i] + 1 : kMergedMax - 1;
    j[i] = k0[i] + (B[k0[i]] <= T[i] ? 1 : 0);
    j[i] += B[k1] <= T[i] ? 1 : 0;
  }
  for (int c = 2; c < maxc; ++c)
#pragma unroll
    for (int i = 0; i < M; ++i) {
      const int k = k0[i] + c < kMergedMax - 1 ? k0[i] + c : kMergedMax - 1;
      j[i] += B[k] <= T[i] ? 1 : 0;
    }
}

// One point's interval.
__device__ __forceinline__ int merged_bin_interval(const double *B,
                                                   const MergedBins &mb,
                                                   double T) {
  const double t[1] = {T};
  int j[1];
  merged_bin_intervals<1>(B, mb, t, j);
  return j[0];
}

// A uniform value pinned in scalar registers: loads from constant memory
// (kernel arguments, the constant tables) could otherwise be repeated inside
// the patch loop, and every scalar load there makes the next LDS wait a
// full one (scalar loads and LDS share one counter and scalar loads return
// out of order).
template <class T>
__device__ __forceinline__ T in_sgpr(T x) {
  asm volatile("" : "+s"(x));
  return x;
}

// Heat-source values of one lane's point plane: slot[64 q], 1/(rho c_p) of
// point q on entry, becomes source * 1/(rho c_p) * JxW. Not inlined: few
// wavefronts come here, and the exponential's constants would otherwise be
// kept in registers through the whole patch loop (28 registers that it then
// spills).
template <int P>
static __device__ __attribute__((noinline)) void plane_source(
    ADM_LDS double *slot, const ADM_LDS adm_beam_state *beams, int n_beams,
    const ADM_LDS CellConstLds *sk, const ADM_CONSTANT KConst *kc, int cx,
    int cy, int cz, int s) {
  constexpr int N = P + 1;
  const double pz = kc->origin[2] + (cz + sk->xq[s]) * kc->h[2];
#pragma unroll 1
  for (int qy = 0; qy < N; ++qy) {
    const double py = kc->origin[1] + (cy + sk->xq[qy]) * kc->h[1];
    double px[N], qs[N];
#pragma unroll
    for (int qx = 0; qx < N; ++qx) {
      px[qx] = kc->origin[0] + (cx + sk->xq[qx]) * kc->h[0];
      qs[qx] = 0.0;
    }
#pragma unroll 1
    for (int b = 0; b < n_beams; ++b)
      beam_values<N>(*(const adm_beam_state *)(beams + b), px, py, pz,
                     kc->log_01, qs);
#pragma unroll
    for (int qx = 0; qx < N; ++qx) {
      const int q = qx + N * qy;
      slot[64 * q] = (qs[qx] * slot[64 * q]) * kc->jxy[qx][qy];  // w_z: later
    }
  }
}

// wavefronts per SIMD the plane kernel is compiled for (VGPR budget). Q3
// holds 16 values per lane where Q2 holds 9: at 2 it spills 200 times per
// patch (RK4 step of 50x25x17 cells: 236 us against 193 at 1).
constexpr int plane_waves_per_eu(int p) { return p == 3 ? 1 : 2; }

template <int P, int NS, int PK>
__global__ void __launch_bounds__(256)
    __attribute__((amdgpu_waves_per_eu(plane_waves_per_eu(P))))
    plane_kernel(const CellArgs a, const double *__restrict__ src,
                 const FaceArgs fa) {
  using L = PlaneLanes<P>;
  constexpr int N = L::N, NP = L::NP, N3 = N * N * N;
  constexpr int PX = L::PX, PY = L::PY, CPW = L::cells_per_wave;
  constexpr int SL = L::slot;
  const ADM_CONSTANT MemberArgs *mb =
      a.members ? as_constant(a.members) + blockIdx.y : nullptr;
  const ADM_CONSTANT KConst &kc = *as_constant(mb ? mb->kc : a.kc);
  const MatConst &m = *(const MatConst *)&kc.mat;
  const ADM_GLOBAL uint32_t *meta_p = as_global(mb ? mb->meta : a.meta);
  const ADM_GLOBAL int32_t *slot_p =
      as_global(mb ? mb->powder_slot : a.powder_slot);
  ADM_GLOBAL double *powder_p = as_global(mb ? mb->powder : a.powder);
  ADM_GLOBAL double *liquid_p = as_global(mb ? mb->liquid : a.liquid);
  ADM_GLOBAL uint8_t *dirty_p =
      as_global(mb ? mb->liquid_dirty : a.liquid_dirty);
  const ADM_GLOBAL double *cos_p = as_global(mb ? mb->dep_cos : a.dep_cos);
  const ADM_GLOBAL double *sin_p = as_global(mb ? mb->dep_sin : a.dep_sin);
  if (mb) {
    src += (int64_t)blockIdx.y * a.member_stride;
  }
  extern __shared__ double lds[];
  // Blocks after the patches' take the face term: beside the patches instead
  // of in a launch between them and the gather pass (4.7 us of 37 per stage
  // of a 64x32x12 Q2 operator). They come last in the grid, when the large
  // launches have begun to run out of patches.
  const int n_blocks = a.plane_blocks;
  if ((int)blockIdx.x >= n_blocks) {
    face_block<P, NS, PK>(
        as_global(mb ? mb->faces : fa.faces), mb ? mb->n_faces : fa.n_faces,
        as_global(mb ? mb->face_powder : fa.face_powder),
        as_global(mb ? mb->face_out : fa.face_out),
        as_global(mb ? mb->kc : fa.kc), fa.nc[0], fa.nc[1], fa.nn[0],
        fa.nn[1], as_global(src), (ADM_LDS double *)lds,
        (int)blockIdx.x - n_blocks, blockDim.x >> 6);
    return;
  }
  __shared__ adm_beam_state sbeams[ADM_MAX_BEAMS];
  __shared__ CellConstLds sk;
  const int lext0 = in_sgpr(a.lext[0]), lext1 = in_sgpr(a.lext[1]);
  const int nc0 = in_sgpr(a.nc[0]), nc1 = in_sgpr(a.nc[1]);
  const int npx = in_sgpr(a.plane_npx), npy = in_sgpr(a.plane_npy);
  const int64_t sy = in_sgpr((int64_t)a.nn[0]);
  const int64_t sz = in_sgpr((int64_t)a.nn[0] * a.nn[1]);
  src = in_sgpr(src);
  meta_p = in_sgpr(meta_p);
  slot_p = in_sgpr(slot_p);
  powder_p = in_sgpr(powder_p);
  liquid_p = in_sgpr(liquid_p);
  dirty_p = in_sgpr(dirty_p);
  double *const patch_E =
      in_sgpr(a.plane_E + (int64_t)blockIdx.y * a.plane_E_stride);

  const int lane = threadIdx.x % 64;
  // the wavefront's index in the block, as a uniform (scalar) value
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const int cw = lane / N, s = lane % N;  // cell of the wavefront, plane
  const int ix = cw % PX, iy = cw / PX;
  // The blocks loop over the patches (persistent grid: the prologue above
  // runs once per block). Blocks are dispatched round-robin over the 8
  // XCDs (block b on XCD b % 8). One operator: each XCD takes one
  // contiguous eighth of the patches in the y-major order, a slab of patch
  // rows through every cell layer, so patches that share node lines share
  // that XCD's L2 and every XCD holds its share of the slow layers (an
  // eighth of the layers in the x-y-z order gave the top one, the powder,
  // to one XCD: 0.120 ms per application of the 128x64x32 Q2 workload,
  // against 0.100 in the plain order and 0.098 in y-major slabs). Batched
  // members (grid y): the plain order, block after block through the
  // patches (64 members of 64x32x16: 3.10 ms per RK4 step against 3.20 in
  // y-major slabs and 3.75 in layer slabs).
  const int W = blockDim.x >> 6;
  int first, stride, end;
  const bool ymajor = a.xcd_remap && n_blocks >= 8 && gridDim.y == 1;
  const int nzl = in_sgpr(a.n_rows / (npx * npy));
  if (ymajor) {
    const int x = blockIdx.x & 7, k = blockIdx.x >> 3;
    const int kx = (n_blocks - x + 7) >> 3;  // blocks on XCD x
    first = (int)((int64_t)a.n_rows * x / 8) + k * W + wave;
    end = (int)((int64_t)a.n_rows * (x + 1) / 8);
    stride = kx * W;
  } else {
    first = blockIdx.x * W + wave;
    end = a.n_rows;
    stride = n_blocks * W;
  }
  first = in_sgpr(first);
  end = in_sgpr(end);
  stride = in_sgpr(stride);
  // A patch's addresses and loads. The next patch's are issued as soon as
  // this one's values have gone through the x contraction and arrive during
  // its computation (a patch's loads take ~4,000 cycles, a fifth of the
  // time it takes).
  struct PatchLoad {
    uint32_t meta;
    int32_t pslot;
    uint8_t dirty;
    double u[NP];
  };
  const FastDiv by_npx(npx), by_mid(ymajor ? nzl : npy);
  // addresses of lanes past the mesh are those of its last cells
  auto load_patch = [&](const PatchAt &at, PatchLoad &pl) {
    const int gx = min(at.px * PX + ix, lext0 - 1);
    const int gy = min(at.py * PY + iy, lext1 - 1);
    const int64_t g = gx + (int64_t)nc0 * (gy + (int64_t)nc1 * at.pz);
    const double *sp = src + (gx * P + sy * (gy * P) + sz * (at.pz * P + s));
    pl.meta = meta_p[g];
    pl.pslot = slot_p[g];
    pl.dirty = (NS > 1 && liquid_p) ? dirty_p[g] : 0;
#pragma unroll
    for (int yy = 0; yy < N; ++yy)
#pragma unroll
      for (int xx = 0; xx < N; ++xx) pl.u[xx + N * yy] = sp[xx + sy * yy];
  };
  // What depends on the loaded cell words: the stored powder of the lane's
  // points and the cell's direction. Loaded before the stores of the patch
  // ahead, to arrive by the time of the point work.
  struct PatchMore {
    double pin[NS == 3 ? NP : 1];
    double cs, sn;
  };
  auto load_more = [&](const PatchAt &at, const PatchLoad &pl,
                       PatchMore &pm) {
    const int gx = at.px * PX + ix, gy = at.py * PY + iy;
    const bool in = cw < CPW && gx < lext0 && gy < lext1;
    const uint32_t w = in && (pl.meta & kActive) ? pl.meta : 0u;
    pm.cs = 1.0;
    pm.sn = 0.0;
    if (w & kRotated) {
      const int64_t g = gx + (int64_t)nc0 * (gy + (int64_t)nc1 * at.pz);
      pm.cs = cos_p[g];
      pm.sn = sin_p[g];
    }
#pragma unroll
    for (int q = 0; q < (NS == 3 ? NP : 1); ++q) pm.pin[q] = 0.0;
    if constexpr (NS == 3) {
      if (w & kHasPowder) {
        const ADM_GLOBAL double *sp =
            powder_p + (int64_t)pl.pslot * N3 + NP * s;
#pragma unroll
        for (int q = 0; q < NP; ++q) pm.pin[q] = sp[q];
      }
    }
  };
  PatchLoad nxt;
  PatchMore more;
  // a wavefront without a patch loads the first one's (and leaves below)
  PatchAt nat(by_npx, by_mid, ymajor, first < end ? first : 0);
  load_patch(nat, nxt);
  const int n_mat = kc.mat.n_materials;

  // Block prologue: beams, constants and merged tables into LDS. It is a
  // good part of a launch with one patch per wavefront, so its loads (after
  // the first patch's, above) are all issued before the first is waited for.
  {
    constexpr int words = sizeof(adm_beam_state) * ADM_MAX_BEAMS / 8;
    constexpr int nn = kMaxN * kMaxN, nm = ADM_MAX_MATERIALS;
    static_assert(words <= 128 && 2 * nn + 2 * kMaxN + 4 * nm <= 128,
                  "one word per lane of the smallest block");
    static_assert(sizeof(CellConstLds) ==
                      sizeof(double) * (2 * nn + 2 * kMaxN + 4 * nm),
                  "staged in the order of its members");
    const int tid = threadIdx.x;
    const adm_beam_state *bsrc = a.beams;
    int bslot = 0;
    if (a.beam_table) {
      bslot = *as_global(a.beam_slot);
      bslot = bslot < 0 ? 0
                        : (bslot < a.beam_table_len ? bslot
                                                    : a.beam_table_len - 1);
      bsrc = a.beam_table + (int64_t)bslot * ADM_MAX_BEAMS;
    }
    const uint64_t beam_word =
        reinterpret_cast<const uint64_t *>(bsrc)[min(tid, words - 1)];
    const int km = tid & (nm - 1);  // material of the lanes below
    const ADM_CONSTANT double *cp = &kc.S[0][0] + min(tid, nn - 1);
    if (tid >= nn) cp = &kc.DcS[0][0] + (tid - nn);  // Dc S (z direction)
    if (tid >= 2 * nn) cp = &kc.xq[0] + (tid - 2 * nn);
    if (tid >= 2 * nn + kMaxN) cp = &kc.wq[0] + (tid - 2 * nn - kMaxN);
    constexpr int n1d = 2 * nn + 2 * kMaxN;
    static_assert(n1d % nm == 0, "material index of a lane");
    if (tid >= n1d) cp = &kc.mat.prop[km][ADM_SOLIDUS];
    if (tid >= n1d + nm) cp = &kc.mat.prop[km][ADM_LIQUIDUS];
    if (tid >= n1d + 2 * nm) cp = &kc.mat.latent_factor[km];
    const double const_word = *cp;
    const double iso_word = kc.mat.isotropic[km] ? 1.0 : 0.0;
    double gain = 0.0, pmod = 0.0, den = 1.0;
    if (mb && tid < ADM_MAX_BEAMS) {
      gain = mb->beam_gain[tid];
      pmod = a.beam_pmod[tid];
      den = a.beam_den[tid];
      if (a.beam_pd_table) {
        const double *pd =
            a.beam_pd_table + (int64_t)bslot * 2 * ADM_MAX_BEAMS;
        pmod = pd[tid];
        den = pd[ADM_MAX_BEAMS + tid];
      }
    }
    if constexpr (PK == 2) {
      for (int mm = 0; mm < n_mat; ++mm) {
        const ADM_CONSTANT double *tab = &kc.mat.merged[mm].B[0];
        const ADM_CONSTANT double *bin =
            reinterpret_cast<const ADM_CONSTANT double *>(&kc.mat.bins[mm]) -
            kMergedLds;
        double *out = lds + mm * kPlaneMergedLds;
        constexpr int R = 4;  // words per lane and round
        for (int k0 = tid; k0 < kPlaneMergedLds; k0 += R * blockDim.x) {
          double w[R];
#pragma unroll
          for (int i = 0; i < R; ++i) {
            const int k = min(k0 + i * (int)blockDim.x, kPlaneMergedLds - 1);
            w[i] = (k < kMergedLds ? tab : bin)[k];
          }
#pragma unroll
          for (int i = 0; i < R; ++i) {
            const int k = k0 + i * (int)blockDim.x;
            if (k < kPlaneMergedLds) out[k] = w[i];
          }
        }
      }
    }
    if (tid < words) reinterpret_cast<uint64_t *>(sbeams)[tid] = beam_word;
    if (tid < n1d + 4 * nm)
      (&sk.S[0][0])[tid] = tid < n1d + 3 * nm ? const_word : iso_word;
    __syncthreads();
    if (mb) {
      if (tid < ADM_MAX_BEAMS)
        sbeams[tid].alpha =
            member_alpha(sbeams[tid], gain, pmod, den, kc.log_01);
      __syncthreads();
    }
  }
  if (first >= end) return;  // whole wavefronts
  load_more(nat, nxt, more);
  int sources_on = a.sources_on;
  if (a.beam_table) {
    sources_on = 0;
    for (int b = 0; b < a.n_beams; ++b) sources_on |= sbeams[b].on ? 1 : 0;
  }
  // uniform constants, in scalar registers for the whole patch loop:
  // in-plane shape values, collocation derivative, DcS, geometry and the
  // kernel arguments the loop reads. For Q2 the host has checked that the
  // middle Gauss point is the middle node (S row 1 = (0, 1, 0)), that S is
  // symmetric under reflection except S[2][1] and that Dc is antisymmetric
  // with Dc[1][1] = 0, bit for bit: S and Dc then take 8 scalar values
  // instead of 18, and the middle rows' products by 0 and 1 are skipped,
  // which leaves every sum as the generic chain gives it (x + 0 = x for the
  // finite temperatures here).
  double S[N][N], Dc[N][N], DS[N][N];
  if constexpr (P == 2) {
    const double s00 = in_sgpr(kc.S[0][0]), s01 = in_sgpr(kc.S[0][1]),
                 s02 = in_sgpr(kc.S[0][2]), s21 = in_sgpr(kc.S[2][1]);
    const double d00 = in_sgpr(kc.Dc[0][0]), d01 = in_sgpr(kc.Dc[0][1]),
                 d02 = in_sgpr(kc.Dc[0][2]), d10 = in_sgpr(kc.Dc[1][0]);
    S[0][0] = s00;
    S[0][1] = s01;
    S[0][2] = s02;
    S[1][0] = -0.0;
    S[1][1] = 1.0;
    S[1][2] = 0.0;
    S[2][0] = s02;
    S[2][1] = s21;
    S[2][2] = s00;
    Dc[0][0] = d00;
    Dc[0][1] = d01;
    Dc[0][2] = d02;
    Dc[1][0] = d10;
    Dc[1][1] = 0.0;
    Dc[1][2] = -d10;
    Dc[2][0] = -d02;
    Dc[2][1] = -d01;
    Dc[2][2] = -d00;
    const double e00 = in_sgpr(kc.DcS[0][0]), e01 = in_sgpr(kc.DcS[0][1]),
                 e02 = in_sgpr(kc.DcS[0][2]), e10 = in_sgpr(kc.DcS[1][0]);
    DS[0][0] = e00;
    DS[0][1] = e01;
    DS[0][2] = e02;
    DS[1][0] = e10;
    DS[1][1] = 0.0;
    DS[1][2] = -e10;
    DS[2][0] = -e02;
    DS[2][1] = -e01;
    DS[2][2] = -e00;
  } else if constexpr (P == 3) {
    // S as it is (the values at the points are the oracle's bit for bit); of
    // the derivative tables one half, made antisymmetric on the host
#pragma unroll
    for (int q = 0; q < N; ++q)
#pragma unroll
      for (int k = 0; k < N; ++k) {
        S[q][k] = in_sgpr(kc.S[q][k]);
        if (q < N / 2) {
          Dc[q][k] = in_sgpr(kc.aDc[q][k]);
          DS[q][k] = in_sgpr(kc.aDcS[q][k]);
        } else {
          Dc[q][k] = -Dc[N - 1 - q][N - 1 - k];
          DS[q][k] = -DS[N - 1 - q][N - 1 - k];
        }
      }
  } else {
#pragma unroll
    for (int q = 0; q < N; ++q)
#pragma unroll
      for (int k = 0; k < N; ++k) {
        S[q][k] = in_sgpr(kc.S[q][k]);
        Dc[q][k] = in_sgpr(kc.Dc[q][k]);
        DS[q][k] = in_sgpr(kc.DcS[q][k]);
      }
  }
  const double ihx2 = kc.inv_h2[0], ihy2 = kc.inv_h2[1],
               ihz2 = kc.inv_h2[2];
  // det w_x w_y of a point; w_z joins in the z integration. The 1-D weights
  // are symmetric (checked on the host), so few of them differ.
  double jxy[N][N];
#pragma unroll
  for (int qx = 0; qx < N; ++qx)
#pragma unroll
    for (int qy = 0; qy < N; ++qy) {
      const int x = min(qx, N - 1 - qx), y = min(qy, N - 1 - qy);
      jxy[qx][qy] = kc.jxy[min(x, y)][max(x, y)];
    }
  double *const xb = lds + (PK == 2 ? n_mat * kPlaneMergedLds : 0) +
                     wave * a.plane_wave_lds;
  double *const myslot = xb + cw * L::cell_slots + s * SL;
  // slot of plane n of this lane's cell
  auto slot_of = [&](int n) { return xb + cw * L::cell_slots + n * SL; };
  // the lane's entries of the point arrays
  double *const pa = xb + lane, *const pb = pa + L::points,
               *const pc = pb + L::points;
  // the lane's place in a patch's block of the patch buffer
  const int64_t rowlen = (int64_t)npx * L::patch_nx;
  const int64_t E_lane =
      ((int64_t)s * npy * L::patch_ny + iy * P) * rowlen + ix * P;
  for (int r = first; r < end; r += stride) {
  wave_lds_sync();  // the previous patch's exchange reads are done
  const int ppx = nat.px, ppy = nat.py, ppz = nat.pz;
  const int cx = ppx * PX + ix, cy = ppy * PY + iy, cz = ppz;
  const bool in_mesh = cw < CPW && cx < lext0 && cy < lext1;
  const int64_t c = cx + (int64_t)nc0 * (cy + (int64_t)nc1 * cz);
  const int32_t pslot32 = nxt.pslot;
  const uint32_t meta = in_mesh ? nxt.meta : 0u;
  const bool act = (meta & kActive) != 0;

  const int mid = (meta >> kMaterialShift) & 3;
  const double solidus = sk.solidus[mid], liquidus = sk.liquidus[mid];
  const double latent = sk.latent[mid];
  const bool iso = sk.iso[mid] != 0.0;
  const bool has_powder = act && (meta & kHasPowder) != 0;
  ADM_GLOBAL double *pw =
      has_powder ? powder_p + (int64_t)pslot32 * N3 + NP * s : nullptr;
  bool dirty = false;
  ADM_GLOBAL double *lq = nullptr;
  if constexpr (NS > 1) {
    if (liquid_p && act) {
      dirty = nxt.dirty != 0;
      lq = liquid_p + c * N3 + NP * s;
    }
  }
  const bool rotated = act && (meta & kRotated) != 0;
  const double cs = more.cs, sn = more.sn;
  double pin[NS == 3 ? NP : 1];
#pragma unroll
  for (int q = 0; q < (NS == 3 ? NP : 1); ++q) pin[q] = more.pin[q];

  // ---- values: S along x, then y, in registers ---------------------------
  double v[NP];
  {
    double t[NP];
#pragma unroll
    for (int yy = 0; yy < N; ++yy)
#pragma unroll
      for (int qx = 0; qx < N; ++qx) {
        if (P == 2 && qx == 1) {
          t[qx + N * yy] = nxt.u[1 + N * yy];
          continue;
        }
        double acc = S[qx][0] * nxt.u[N * yy];
#pragma unroll
        for (int k = 1; k < N; ++k)
          acc = __builtin_fma(S[qx][k], nxt.u[k + N * yy], acc);
        t[qx + N * yy] = acc;
      }
    if (r + stride < end) {
      nat = PatchAt(by_npx, by_mid, ymajor, r + stride);
      load_patch(nat, nxt);
    }
#pragma unroll
    for (int qy = 0; qy < N; ++qy)
#pragma unroll
      for (int qx = 0; qx < N; ++qx) {
        if (P == 2 && qy == 1) {
          v[qx + N * qy] = t[qx + N];
          continue;
        }
        double acc = S[qy][0] * t[qx];
#pragma unroll
        for (int k = 1; k < N; ++k)
          acc = __builtin_fma(S[qy][k], t[qx + N * k], acc);
        v[qx + N * qy] = acc;
      }
  }
  // ---- exchange 1: the cell's N planes (contracted in x and y) -----------
#pragma unroll
  for (int q = 0; q < NP; ++q) myslot[q] = v[q];
  wave_lds_sync();
  // z contraction: the value at the lane's point plane (the oracle's chain)
  // and the z derivative from the nodal planes (Dc S)
  double Tq[NP], gz[NP];
  {
    double szv[N], dzv[N];
#pragma unroll
    for (int n = 0; n < N; ++n) {
      szv[n] = sk.S[s][n];
      dzv[n] = sk.Dc[s][n];  // (Dc S)[s][n]
    }
#pragma unroll
    for (int q = 0; q < NP; ++q) {
      const double w0 = slot_of(0)[q];
      Tq[q] = szv[0] * w0;
      gz[q] = dzv[0] * w0;
    }
#pragma unroll
    for (int n = 1; n < N; ++n)
#pragma unroll
      for (int q = 0; q < NP; ++q) {
        const double wn = slot_of(n)[q];
        Tq[q] = __builtin_fma(szv[n], wn, Tq[q]);
        gz[q] = __builtin_fma(dzv[n], wn, gz[q]);
      }
  }
  wave_lds_sync();

  // ---- per-point physics, one point row (fixed y) at a time --------------
  bool near = false;
  // a patch outside the cells that a beam may reach skips the test of its
  // cells (1,500 of a cold patch's 11,000 cycles)
  const bool reach = sources_on && ppx * PX <= a.reach_hi[0] &&
                     ppx * PX + PX > a.reach_lo[0] &&
                     ppy * PY <= a.reach_hi[1] &&
                     ppy * PY + PY > a.reach_lo[1] && ppz <= a.reach_hi[2] &&
                     ppz >= a.reach_lo[2];
  if (reach && act) {
    const int cc[3] = {cx, cy, cz};
    double lo[3], hi[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      lo[d] = kc.origin[d] + cc[d] * kc.h[d];
      hi[d] = kc.origin[d] + (cc[d] + 1) * kc.h[d];
    }
#pragma unroll 1
    for (int b = 0; b < a.n_beams; ++b)
      near |= beam_may_touch(sbeams[b], lo, hi);
  }
  const double *mB = lds + mid * kPlaneMergedLds;
  const double *mC = mB + kMergedMax;
  const MergedBins &mbin =
      *reinterpret_cast<const MergedBins *>(mB + kMergedLds);
  const int mid0 = __builtin_amdgcn_readfirstlane(mid);
  // accumulators of the node plane (before the z part): Ap gathers the x
  // and y flux terms and the source, Bp the z flux
  double Ap[NP], Bp[NP];
  bool plane_liquid = false;

  // x and y gradients of point (qx, qy) by the collocation derivative (the
  // oracle's chains)
  auto grad_xy = [&](int qx, int qy, double &gxq, double &gyq) {
    gxq = Dc[qx][0] * Tq[N * qy];
    gyq = Dc[qy][0] * Tq[qx];
#pragma unroll
    for (int k = 1; k < N; ++k) {
      if (!(P == 2 && qx == 1 && k == 1))
        gxq = __builtin_fma(Dc[qx][k], Tq[k + N * qy], gxq);
      if (!(P == 2 && qy == 1 && k == 1))
        gyq = __builtin_fma(Dc[qy][k], Tq[qx + N * k], gyq);
    }
  };
  // fold a point row into the node-plane accumulators:
  //   Ap[xx, yy] += S[qy][yy] (DcS^T w0)[xx] + DcS[qy][yy] (S^T w1)[xx]
  //   Bp[xx, yy] += S[qy][yy] (S^T w2)[xx]
  auto fold_row = [&](int qy, const double (&w0)[N], const double (&w1)[N],
                      const double (&w2)[N]) {
#pragma unroll
    for (int xx = 0; xx < N; ++xx) {
      double t0 = DS[0][xx] * w0[0];
      double t1 = S[0][xx] * w1[0];
      double t2 = S[0][xx] * w2[0];
#pragma unroll
      for (int q = 1; q < N; ++q) {
        if (!(P == 2 && q == 1 && xx == 1))
          t0 = __builtin_fma(DS[q][xx], w0[q], t0);
        if (P == 2 && q == 1) {
          if (xx == 1) {
            t1 = t1 + w1[q];
            t2 = t2 + w2[q];
          }
          continue;
        }
        t1 = __builtin_fma(S[q][xx], w1[q], t1);
        t2 = __builtin_fma(S[q][xx], w2[q], t2);
      }
#pragma unroll
      for (int yy = 0; yy < N; ++yy) {
        const int o = xx + N * yy;
        if (qy == 0) {
          Ap[o] = __builtin_fma(DS[qy][yy], t1, S[qy][yy] * t0);
          Bp[o] = S[qy][yy] * t2;
        } else if (P == 2 && qy == 1) {
          if (yy == 1) {
            Ap[o] = Ap[o] + t0;
            Bp[o] = Bp[o] + t2;
          } else {
            Ap[o] = __builtin_fma(DS[qy][yy], t1, Ap[o]);
          }
        } else {
          Ap[o] = __builtin_fma(S[qy][yy], t0, Ap[o]);
          Ap[o] = __builtin_fma(DS[qy][yy], t1, Ap[o]);
          Bp[o] = __builtin_fma(S[qy][yy], t2, Bp[o]);
        }
      }
    }
  };

  // One-interval form. Most planes are cold (no point at or above the
  // solidus) and so smooth that their points lie in one interval of the
  // merged table: the interval and its coefficients are then read once per
  // plane instead of once per point, and nothing in the point loop branches
  // or waits for LDS. Taken when it holds for every lane of the wavefront
  // and every material is isotropic; without powder every point is fully
  // solid, and with powder a mixture of solid and powder.
  bool one = false;
  int j1 = 0;
  double tl = 0.0;  // left end of the plane's interval
  if constexpr (PK == 2) {
    j1 = merged_bin_interval(mB, mbin, Tq[0]);
    tl = mB[j1 > 0 ? j1 - 1 : 0];
    const double lo = j1 > 0 ? tl : -HUGE_VAL;
    double hi = j1 < kMergedMax ? mB[j1] : HUGE_VAL;
    if constexpr (NS > 1) hi = hi < solidus ? hi : solidus;
    bool ok = iso;
#pragma unroll
    for (int q = 0; q < NP; ++q) ok = ok && Tq[q] >= lo && Tq[q] < hi;
    one = !__any(act && !ok);
  }
  // wave-uniform solid path: one material, every point fully solid (no
  // powder, below the solidus)
  bool fast = false;
  if (!one) {
    bool warm = false;
    if constexpr (NS > 1) {
#pragma unroll
      for (int q = 0; q < NP; ++q) warm |= act && !(Tq[q] < solidus);
    }
    fast = !__any(warm || has_powder || (act && mid != mid0));
  }
  auto solid_again = [&]() {
    // every point solid: a liquid ratio held from the last evaluation goes
    // back to zero
    if constexpr (NS > 1) {
      if (lq && dirty) {
#pragma unroll
        for (int q = 0; q < NP; ++q) lq[q] = 0.0;
      }
    }
  };

  auto one_interval = [&](auto powder_tag) {
    constexpr bool POWDER = decltype(powder_tag)::value;
    constexpr int row = kMergedMax * ADM_MAX_STATES * 2;
    const double *cj = mC + j1 * (ADM_MAX_STATES * 2);
    const double rs0 = cj[ADM_DENSITY * row], rs1 = cj[ADM_DENSITY * row + 1];
    const double cs0 = cj[ADM_SPECIFIC_HEAT * row],
                 cs1 = cj[ADM_SPECIFIC_HEAT * row + 1];
    const double ks0 = cj[ADM_THERMAL_CONDUCTIVITY_X * row],
                 ks1 = cj[ADM_THERMAL_CONDUCTIVITY_X * row + 1];
    double rp0 = 0.0, rp1 = 0.0, cp0 = 0.0, cp1 = 0.0, kp0 = 0.0, kp1 = 0.0;
    if constexpr (POWDER) {
      rp0 = cj[ADM_DENSITY * row + 4], rp1 = cj[ADM_DENSITY * row + 5];
      cp0 = cj[ADM_SPECIFIC_HEAT * row + 4];
      cp1 = cj[ADM_SPECIFIC_HEAT * row + 5];
      kp0 = cj[ADM_THERMAL_CONDUCTIVITY_X * row + 4];
      kp1 = cj[ADM_THERMAL_CONDUCTIVITY_X * row + 5];
    }
    // isotropic: the rotation K -> k (cos^2 + sin^2) in the x-y plane
    const double rot = cs * cs + sn * sn;
    const double ax = ihx2 * rot, ay = ihy2 * rot;
    solid_again();
    static_for<0, N>([&](auto qyc) {
      constexpr int qy = decltype(qyc)::value;
      double w0[N], w1[N], w2[N];
#pragma unroll
      for (int qx = 0; qx < N; ++qx) {
        const int q = qx + N * qy;
        double gxq, gyq;
        grad_xy(qx, qy, gxq, gyq);
        const double d = Tq[q] - tl;
        double rho = __builtin_fma(d, rs1, rs0);
        double cp = __builtin_fma(d, cs1, cs0);
        double k = __builtin_fma(d, ks1, ks0);
        if constexpr (POWDER) {
          // l = 0: powder = min(powder, 1), solid = 1 - powder
          const double pv = (pin[q] < 1.0) ? pin[q] : 1.0;
          const double sv = 1.0 - pv;
          rho = sv * rho + pv * __builtin_fma(d, rp1, rp0);
          cp = sv * cp + pv * __builtin_fma(d, cp1, cp0);
          k = sv * k + pv * __builtin_fma(d, kp1, kp0);
        }
        const double irc = recip(rho * cp);
        pa[64 * q] = irc;  // for the source pass
        const double cq = ((-irc) * jxy[qx][qy]) * k;
        w0[qx] = cq * (gxq * ax);
        w1[qx] = cq * (gyq * ay);
        w2[qx] = cq * (gz[q] * ihz2);
      }
      fold_row(qy, w0, w1, w2);
    });
    if constexpr (POWDER) {
      // powder above 1 (or not a number) is cut to 1, as stored
      if (pw) {
#pragma unroll
        for (int q = 0; q < NP; ++q)
          if (!(pin[q] < 1.0) && pin[q] != 1.0) pw[q] = 1.0;
      }
    }
  };

  // General form, in two steps. First the points' properties, a row at a
  // time in a loop (the rows share one copy of the code, and the node-plane
  // accumulators are not live yet: unrolled and in one step it spills), into
  // the point arrays; then the fluxes and their folding, unrolled. The steps
  // of a row run over its points together, so that their LDS reads overlap.
  // SOLID: every point solid and material mid_ for every lane; otherwise the
  // lane's own material and the phase-state update. OUT: 1/(rho c_p) and
  // k_x (kIso), 1/(rho c_p) times the three conductivities (kAniso), or
  // 1/(rho c_p) alone (kIrc).
  constexpr int kIso = 0, kAniso = 1, kIrc = 2;
  auto points = [&](auto solid_tag, auto out_tag, int mid_, const double *mB_,
                    const double *mC_, const MergedBins &mbin_) {
    constexpr bool SOLID = decltype(solid_tag)::value;
    constexpr int OUT = decltype(out_tag)::value;
    if constexpr (SOLID) solid_again();
#pragma unroll
    for (int q = 0; q < NP; ++q) {
      if constexpr (NS == 3 && !SOLID) pa[64 * q] = pin[q];
      pb[64 * q] = Tq[q];
    }
    // polynomial coefficients of the wave's solid material: scalar loads
    const ADM_CONSTANT MatConst &mcst = kc.mat;
    constexpr bool POLY1 = PK == 0 && SOLID;
    const int order = POLY1 ? mcst.p_order : 0;
#pragma unroll 1
    for (int qy = 0; qy < N; ++qy) {
      double *const ra = pa + 64 * N * qy, *const rb = pb + 64 * N * qy,
                    *const rc = pc + 64 * N * qy;
      double Tr[N];
#pragma unroll
      for (int qx = 0; qx < N; ++qx) Tr[qx] = rb[64 * qx];
      int jr[N];
      if constexpr (PK == 2) merged_bin_intervals<N>(mB_, mbin_, Tr, jr);
      // update_state_ratios (source/ThermalOperator.templates.hh:227-317)
      double r_[N][NS], l[N];
#pragma unroll
      for (int qx = 0; qx < N; ++qx) {
        l[qx] = 0.0;
        r_[qx][0] = 1.0;
#pragma unroll
        for (int k = 1; k < NS; ++k) r_[qx][k] = 0.0;
      }
      if constexpr (!SOLID && NS > 1) {
        // the mushy division where a point of the wavefront needs it
        bool need = false;
#pragma unroll
        for (int qx = 0; qx < N; ++qx) {
          l[qx] = Tr[qx] > liquidus ? 1.0 : 0.0;
          need |= !(Tr[qx] < solidus) && !(Tr[qx] > liquidus);
        }
        if (__any(need)) {
#pragma unroll
          for (int qx = 0; qx < N; ++qx) {
            const double mushy = (Tr[qx] - solidus) / (liquidus - solidus);
            l[qx] = Tr[qx] < solidus ? 0.0
                                     : (Tr[qx] > liquidus ? 1.0 : mushy);
          }
        }
#pragma unroll
        for (int qx = 0; qx < N; ++qx) {
          const int q = qx + N * qy;
          if constexpr (NS == 2) {
            r_[qx][1] = l[qx];
            r_[qx][0] = 1.0 - l[qx];
          } else {
            const double p0 = ra[64 * qx];
            const double am = 1.0 - l[qx];
            const double pv = (p0 < am) ? p0 : am;
            r_[qx][1] = l[qx];
            r_[qx][2] = pv;
            r_[qx][0] = 1.0 - l[qx] - pv;
            if (pw && pv != p0) pw[q] = pv;
          }
          if (lq && (l[qx] != 0.0 || dirty)) lq[q] = l[qx];
          plane_liquid |= l[qx] != 0.0;
        }
      }
      // get_inv_rho_cp (source/ThermalOperator.templates.hh:415-477) and the
      // conductivities
      double rho[N], cp[N], kx[N], ky[N], kzz[N];
      if constexpr (POLY1) {
        // sum_i c_i T^i, state ratio 1
        double tp[N];
#pragma unroll
        for (int qx = 0; qx < N; ++qx) {
          tp[qx] = 1.0;
          rho[qx] = cp[qx] = kx[qx] = ky[qx] = kzz[qx] = 0.0;
        }
#pragma unroll
        for (int i = 0; i < ADM_MAX_POLY; ++i) {
          if (i > order) break;
          const auto &pcf = mcst.poly[mid_];
#pragma unroll
          for (int qx = 0; qx < N; ++qx) {
            if (i > 0) tp[qx] = tp[qx] * Tr[qx];
            rho[qx] += pcf[ADM_DENSITY][0][i] * tp[qx];
            cp[qx] += pcf[ADM_SPECIFIC_HEAT][0][i] * tp[qx];
            if constexpr (OUT != kIrc)
              kx[qx] += pcf[ADM_THERMAL_CONDUCTIVITY_X][0][i] * tp[qx];
            if constexpr (OUT == kAniso) {
              ky[qx] += pcf[ADM_THERMAL_CONDUCTIVITY_Y][0][i] * tp[qx];
              kzz[qx] += pcf[ADM_THERMAL_CONDUCTIVITY_Z][0][i] * tp[qx];
            }
          }
        }
      } else {
        auto props = [&](const auto &ev, int qx) {
          rho[qx] = ev(ADM_DENSITY, r_[qx]);
          cp[qx] = ev(ADM_SPECIFIC_HEAT, r_[qx]);
          if constexpr (OUT != kIrc)
            kx[qx] = ev(ADM_THERMAL_CONDUCTIVITY_X, r_[qx]);
          if constexpr (OUT == kAniso) {
            ky[qx] = ev(ADM_THERMAL_CONDUCTIVITY_Y, r_[qx]);
            kzz[qx] = ev(ADM_THERMAL_CONDUCTIVITY_Z, r_[qx]);
          }
        };
#pragma unroll
        for (int qx = 0; qx < N; ++qx) {
          if constexpr (PK == 2 && SOLID) {
            // the solid value alone: (0 + 1 X_s) + 0 X_l + 0 X_p = X_s
            const int j = jr[qx];
            const double d = Tr[qx] - mB_[j > 0 ? j - 1 : 0];
            const double *cj = mC_ + j * (ADM_MAX_STATES * 2);
            auto solid_ev = [&](int prop, const double(&)[NS]) {
              const double *cf = cj + prop * (kMergedMax * ADM_MAX_STATES * 2);
              return __builtin_fma(d, cf[1], cf[0]);
            };
            props(solid_ev, qx);
          } else if constexpr (PK == 2) {
            props(MergedEval(mB_, mC_, Tr[qx], jr[qx]), qx);
          } else {
            props(typename EvalOf<PK>::type(m, mid_, Tr[qx]), qx);
          }
        }
      }
#pragma unroll
      for (int qx = 0; qx < N; ++qx) {
        double c_p = cp[qx];
        if constexpr (!SOLID && NS > 1) {
          const double is_mushy = r_[qx][1] * r_[qx][0];
          if (is_mushy > 0.0) c_p += latent;
        }
        const double irc = recip(rho[qx] * c_p);
        ra[64 * qx] = OUT == kAniso ? irc * kx[qx] : irc;
        if constexpr (OUT == kIso) rb[64 * qx] = kx[qx];
        if constexpr (OUT == kAniso) {
          rb[64 * qx] = irc * ky[qx];
          rc[64 * qx] = irc * kzz[qx];
        }
      }
    }
  };
  // -(1/rho c_p) K grad T * JxW, each component with its 1/h, from the point
  // arrays
  auto fluxes = [&](auto iso_tag) {
    constexpr bool ISO = decltype(iso_tag)::value;
    // isotropic cells: the lanes that take the rotated form
    const bool turned = ISO && (fast ? __any(rotated) != 0 : rotated);
    const bool any_turned = __any(turned);
    const double ihxy = kc.inv_h[0] * kc.inv_h[1];
    static_for<0, N>([&](auto qyc) {
      constexpr int qy = decltype(qyc)::value;
      double w0[N], w1[N], w2[N];
#pragma unroll
      for (int qx = 0; qx < N; ++qx) {
        const int q = qx + N * qy;
        double gxq, gyq;
        grad_xy(qx, qy, gxq, gyq);
        if constexpr (ISO) {
          const double cq = (-pa[64 * q]) * jxy[qx][qy], k = pb[64 * q];
          w0[qx] = (cq * k) * (gxq * ihx2);
          w1[qx] = (cq * k) * (gyq * ihy2);
          w2[qx] = (cq * k) * (gz[q] * ihz2);
          if (any_turned) {
            const double ih0 = kc.inv_h[0], ih1 = kc.inv_h[1];
            const double fx = (k * cs * cs + k * sn * sn) * (gxq * ih0);
            const double fy = (k * sn * sn + k * cs * cs) * (gyq * ih1);
            w0[qx] = turned ? (cq * fx) * ih0 : w0[qx];
            w1[qx] = turned ? (cq * fy) * ih1 : w1[qx];
          }
        } else {
          const double c0 = (-pa[64 * q]) * jxy[qx][qy];
          const double c1 = (-pb[64 * q]) * jxy[qx][qy];
          const double c2 = (-pc[64 * q]) * jxy[qx][qy];
          // (c0, c1) rotated into the deposition direction
          const double cxy = ((c0 - c1) * sn * cs) * ihxy;
          w0[qx] = (c0 * cs * cs + c1 * sn * sn) * (gxq * ihx2) + cxy * gyq;
          w1[qx] = cxy * gxq + (c0 * sn * sn + c1 * cs * cs) * (gyq * ihy2);
          w2[qx] = c2 * (gz[q] * ihz2);
        }
      }
      fold_row(qy, w0, w1, w2);
    });
  };
  if (one) {
    if (NS == 3 && __any(has_powder))
      one_interval(std::integral_constant<bool, NS == 3>{});
    else
      one_interval(std::integral_constant<bool, false>{});
  } else {
    constexpr std::integral_constant<bool, true> yes{};
    constexpr std::integral_constant<bool, false> no{};
    constexpr std::integral_constant<int, kIso> iso_out{};
    constexpr std::integral_constant<int, kAniso> aniso_out{};
    // the wave's material (uniform: scalar registers, uniform LDS rows)
    const double *fB = lds + mid0 * kPlaneMergedLds;
    const MergedBins &fbin =
        *reinterpret_cast<const MergedBins *>(fB + kMergedLds);
    if (!__any(act && !iso)) {
      if (fast)
        points(yes, iso_out, mid0, fB, fB + kMergedMax, fbin);
      else
        points(no, iso_out, mid, mB, mC, mbin);
      fluxes(yes);
    } else {
      if (fast)
        points(yes, aniso_out, mid0, fB, fB + kMergedMax, fbin);
      else
        points(no, aniso_out, mid, mB, mC, mbin);
      fluxes(no);
      // the source pass needs 1/(rho c_p) alone (the state update again
      // changes nothing)
      if (reach && __any(near))
        points(no, std::integral_constant<int, kIrc>{}, mid, mB, mC, mbin);
    }
  }
  // heat sources, in a pass of their own over the cells that a beam can
  // reach (few), a point row at a time: 1/(rho c_p) from the point
  // array, then Ap[xx, yy] += S[qy][yy] (S^T val)[xx]
  if (reach && __any(near)) {
    wave_lds_sync();
    if (near) {
      plane_source<P>((ADM_LDS double *)pa,
                      (const ADM_LDS adm_beam_state *)&sbeams[0], a.n_beams,
                      (const ADM_LDS CellConstLds *)&sk, &kc, cx, cy, cz, s);
#pragma unroll
      for (int qy = 0; qy < N; ++qy)
#pragma unroll
        for (int xx = 0; xx < N; ++xx) {
          double tv = S[0][xx] * pa[64 * N * qy];
#pragma unroll
          for (int q = 1; q < N; ++q)
            tv = __builtin_fma(S[q][xx], pa[64 * (q + N * qy)], tv);
#pragma unroll
          for (int yy = 0; yy < N; ++yy)
            Ap[xx + N * yy] = __builtin_fma(S[qy][yy], tv, Ap[xx + N * yy]);
        }
    }
  }
  if constexpr (NS > 1) {
    // cell-wide "held liquid" flag over the cell's N lanes
    const uint64_t ball = __ballot(plane_liquid);
    const bool any_liquid = ((ball >> (cw * N)) & ((1ull << N) - 1)) != 0;
    if (lq && s == 0 && any_liquid != dirty) dirty_p[c] = any_liquid ? 1 : 0;
  }

  // ---- exchange 2: z part, node plane s = sum over point planes ----------
  // out = sum_qz w_qz (S[qz][s] Ap_qz + (Dc S)[qz][s] Bp_qz), the two parts
  // in a buffer each
  double out[NP];
  wave_lds_sync();
#pragma unroll
  for (int q = 0; q < NP; ++q) {
    myslot[q] = Ap[q];
    myslot[L::exchange + q] = Bp[q];
  }
  wave_lds_sync();
  {
    double sc[N], dc[N];
#pragma unroll
    for (int k = 0; k < N; ++k) {
      sc[k] = sk.S[k][s] * sk.wq[k];
      dc[k] = sk.Dc[k][s] * sk.wq[k];  // (Dc S)[k][s]
    }
#pragma unroll
    for (int q = 0; q < NP; ++q) out[q] = sc[0] * slot_of(0)[q];
#pragma unroll
    for (int k = 1; k < N; ++k)
#pragma unroll
      for (int q = 0; q < NP; ++q)
        out[q] = __builtin_fma(sc[k], slot_of(k)[q], out[q]);
#pragma unroll
    for (int k = 0; k < N; ++k)
#pragma unroll
      for (int q = 0; q < NP; ++q)
        out[q] = __builtin_fma(dc[k], slot_of(k)[L::exchange + q], out[q]);
  }
  if (!act) {
#pragma unroll
    for (int q = 0; q < NP; ++q) out[q] = 0.0;
  }

  // ---- shared nodes of the patch, then dst --------------------------------
  // x: node column P of cell (ix, iy) += column 0 of cell (ix + 1, iy)
#pragma unroll
  for (int yy = 0; yy < N; ++yy) {
    const double o = __shfl_down(out[N * yy], N);
    if (ix + 1 < PX) out[P + N * yy] += o;
  }
  // y: node row P += row 0 of cell (ix, iy + 1) (its column P already
  // holds the corner sums)
#pragma unroll
  for (int xx = 0; xx < N; ++xx) {
    const double o = __shfl_down(out[xx], N * PX);
    if (iy + 1 < PY) out[xx + N * P] += o;
  }
  // the next patch's loads have arrived by now: waiting for them here keeps
  // their wait from including the stores below
#pragma unroll
  for (int q = 0; q < NP; ++q) asm volatile("" : "+v"(nxt.u[q]));
  if (r + stride < end) load_more(nat, nxt, more);
  if (in_mesh) {
  // the patch's node sums, every node of the patch once, into its slots
  // of the patch buffer (plain stores; the gather kernel adds the slots of
  // the patches that share a node in a fixed order)
  // patch buffer layout [cell layer][plane][patch y][node y][patch x]
  // [node x]: a node row of one plane runs through the patches of a row
  // contiguously, which the gather pass reads along x
  double *E = patch_E +
              (((int64_t)ppz * N * npy + ppy) * L::patch_ny * rowlen +
               (int64_t)ppx * L::patch_nx) +
              E_lane;
#pragma unroll
  for (int yy = 0; yy < N; ++yy)
#pragma unroll
    for (int xx = 0; xx < N; ++xx) {
      if (xx == 0 && ix != 0) continue;  // summed into the left neighbour
      if (yy == 0 && iy != 0) continue;
      E[xx + rowlen * yy] = out[xx + N * yy];
    }
  }
  }  // patches
}

// Second pass of the plane kernel: one lane per node (x fastest; the
// grid's y index is the ensemble member) sums the patch-buffer slots of the
// patches that hold the node -- up to two along each axis -- in increasing
// patch order, and writes dst (or adds to it). Nodes above the launched
// cell layers get no slot: 0, or dst unchanged with add. n_nodes < 2^31.
template <int P>
__global__ void __launch_bounds__(256)
    plane_gather_kernel(const double *__restrict__ E, int64_t E_stride,
                        double *__restrict__ dst, int64_t member_stride,
                        int32_t nn0, int32_t nn1, int32_t nn2, int32_t npx,
                        int32_t npy, int32_t nz, int32_t add,
                        const FaceArgs fa, const StageArgs st) {
  using L = PlaneLanes<P>;
  constexpr int WX = P * L::PX, WY = P * L::PY;
  const int node = blockIdx.x * blockDim.x + threadIdx.x;
  if (node >= nn0 * nn1 * nn2) return;
  E += (int64_t)blockIdx.y * E_stride;
  dst += (int64_t)blockIdx.y * member_stride;
  const int row = node / nn0, X = node - row * nn0;
  const int Z = row / nn1, Y = row - Z * nn1;
  // above the top node plane of the launch's cell layers no cell or face
  // adds a term: the result is 0 (or dst as it is), and a stage update
  // leaves every vector as it is
  if (Z > P * nz) {
    if (st.kind == kStageNone && !add) dst[node] = 0.0;
    return;
  }
  const int64_t rowlen = (int64_t)npx * L::patch_nx;
  // offsets of the blocks holding the node (unused entries stay 0: in
  // bounds of E)
  int yoff[2] = {0, 0}, zoff[2] = {0, 0}, xoff[2] = {0, 0};
  int nyc = 0, nzc = 0, nxc = 0;
  const int py = Y / WY, ly = Y - py * WY;
  if (ly == 0 && py > 0) yoff[nyc++] = (py - 1) * L::patch_ny + WY;
  if (py < npy) yoff[nyc++] = py * L::patch_ny + ly;
  const int pz = Z / P, lz = Z - pz * P;
  if (lz == 0 && pz > 0 && pz - 1 < nz) zoff[nzc++] = (pz - 1) * (P + 1) + P;
  if (pz < nz) zoff[nzc++] = pz * (P + 1) + lz;
  const int px = X / WX, lx = X - px * WX;
  if (lx == 0 && px > 0) xoff[nxc++] = (px - 1) * L::patch_nx + WX;
  if (px < npx) xoff[nxc++] = px * L::patch_nx + lx;
  // up to 2 x 2 x 2 blocks: every load issued before the sums, which add
  // the blocks present in (z, y, x) order
  double v[8];
#pragma unroll
  for (int kz = 0; kz < 2; ++kz)
#pragma unroll
    for (int ky = 0; ky < 2; ++ky) {
      const double *r =
          E + ((int64_t)zoff[kz < nzc ? kz : 0] * npy * L::patch_ny +
               yoff[ky < nyc ? ky : 0]) *
                  rowlen;
#pragma unroll
      for (int kx = 0; kx < 2; ++kx) {
        const bool here = kz < nzc && ky < nyc && kx < nxc;
        v[4 * kz + 2 * ky + kx] = here ? r[xoff[kx < nxc ? kx : 0]] : 0.0;
      }
    }
  double sum = 0.0;
#pragma unroll
  for (int k = 0; k < 8; ++k)
    if (((k >> 2) < nzc) && (((k >> 1) & 1) < nyc) && ((k & 1) < nxc))
      sum += v[k];
  double r = add ? dst[node] + sum : sum;
  // the face term's slots at this node, summed in increasing face order
  // and added after the cell term (as a separate face gather pass would)
  const MemberArgs *mb = fa.members ? fa.members + blockIdx.y : nullptr;
  const int32_t *rank_p = mb ? mb->fn_rank : fa.fn_rank;
  if (rank_p && (mb ? mb->n_faces : fa.n_faces) > 0) {
    const int32_t k = rank_p[node];
    if (k >= 0) {
      const double *fo = mb ? mb->face_out : fa.face_out;
      const int32_t *off = mb ? mb->fn_offset : fa.fn_offset;
      const int32_t *slot = mb ? mb->fn_slot : fa.fn_slot;
      double fs = 0.0;
      for (int32_t e = off[k]; e < off[k + 1]; ++e) fs += fo[slot[e]];
      r += fs;
    }
  }
  // the result, or (a time step on the plane path) the stage update it
  // feeds, without storing it
  if (st.kind == kStageNone)
    dst[node] = r;
  else
    stage_apply(st, (int64_t)blockIdx.y * member_stride + node, r);
}

}  // namespace adm
