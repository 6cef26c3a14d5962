// Backward kernels of the surfel rasteriser for gfx950 (CDNA4, wave64),
// dsr/cuda_rasterizer/backward.cu:143-630.
//
//   k_blend_bwd        pass 1: per pixel, the back-to-front recurrences over
//                      the pairs it blended, storing each pair's weight,
//                      dL/dalpha and dL/ddepth (a quadrant whose pairs missed
//                      the pair store runs the whole backward here instead)
//   k_blend_bwd_grad   pass 2: per (quadrant, 64-entry chunk), each entry's 18
//                      partial gradients summed over the quadrant's pixels
//   k_preprocess_bwd   per surfel: reduces its records' partial sums over
//                      their tile instances, then the AABB-centre adjoint,
//                      dL/dT -> dL/d(mean, scale, rotation), SH backward and
//                      the densification statistic in dL_dmean2D
//
// The partial sums go to one slot per (tile-list position, quadrant) with
// plain stores and are reduced per record by the backward preprocess: no
// gradient is accumulated with global atomics, and the result does not
// depend on scheduling order.
#include "sr_device.h"
#include <type_traits>

#include "sr_internal.h"
#include "sr_pair.h"

namespace sr {

// Partial-gradient slots: 0..8 dL_dtransMat, 9..10 dL_dmean2D.xy,
// 11..13 dL_dnormal, 14 dL_dopacity, 15..17 dL_dcolors.
constexpr int kNumG = 18;
constexpr int kChainPre = 4;  // pairs of a batch in the chain pass
using V4 = float __attribute__((ext_vector_type(4)));  // a float4 the compiler keeps in registers as a whole
using V2 = float __attribute__((ext_vector_type(2)));
template <class T> SR_DEV T load8(const char* p) {  // from an 8-byte aligned place
  T v;
  __builtin_memcpy(&v, __builtin_assume_aligned(p, 8), sizeof(T));
  return v;
}
// LDS bytes from one lane's batch to the next: 16 more than its pairs, so that
// neither the quads' pieces nor the lanes' own reads share banks
template <bool kPart> constexpr int kOwnerBytes = kChainPre * PairLayout<kPart>::kBytes + 16;
constexpr unsigned kChainBlocks = 16384;  // workgroups of the chain pass at most
#ifndef SR_GRAD_GROUP
#define SR_GRAD_GROUP 4
#endif
// pixels per group in the per-pair gradient sums: an entry's partials are
// summed over each run of kGradGroup blended pixels in pixel order, and
// the runs' sums are added in order
constexpr int kGradGroup = SR_GRAD_GROUP;
static_assert(kGradGroup >= 1 && 64 % kGradGroup == 0, "groups tile the 64 pixels");

// Stores the 18 partial sums (g(k) for sum k) of a sub-list entry as five
// float4 in its slot.  Every
// entry of every sub-list sets its flag exactly once per backward and
// stores its sums when any is non-zero, so neither buffer needs clearing.
// (also: some pixel has a semantic gradient for the slot, _part variant).
template <class G>
SR_DEV void store_part(const BlendBwdArgs& a, size_t slot, G g, bool also = false) {
  bool nz = also;
#pragma unroll
  for (int k = 0; k < 18; ++k) nz |= g(k) != 0.0f;
  a.part_nz[slot] = nz ? 1 : 0;  // most entries blend no pixel of the quadrant: only a flag
  if (!nz) return;
  float4* d = reinterpret_cast<float4*>(a.part + slot * kPartStride);
  d[0] = make_float4(g(0), g(1), g(2), g(3));
  d[1] = make_float4(g(4), g(5), g(6), g(7));
  d[2] = make_float4(g(8), g(9), g(10), g(11));
  d[3] = make_float4(g(12), g(13), g(14), g(15));
  d[4] = make_float4(g(16), g(17), 0.0f, 0.0f);
}

// Per-pixel inputs of the backward blend (backward.cu:168-236).
struct PixelBwd {
  float T_final, final_A, final_D, final_D2, bg_dot;
  uint32_t last_contributor;
  int median_contributor;
  float dLp0, dLp1, dLp2, dLn0, dLn1, dLn2;
  float dL_ddepth, dL_daccum, dL_dreg, dL_dmedian;
  float dL_dmaxw;  // _part: median weight's
};

template <bool kPart>
SR_DEV PixelBwd pixel_bwd(const BlendBwdArgs& a, const ViewInfo& vi, bool inside, uint32_t pxi, uint32_t pyi) {
  PixelBwd p{};
  const size_t HW = (size_t)vi.H * vi.W, pid = (size_t)vi.W * pyi + pxi, pb = vi.pix_base;
  if (inside) {
    const float* final_T = a.final_T + 3 * pb;
    const uint32_t* n_contrib = a.n_contrib + 2 * pb;
    const float* dL_dpix = a.dL_dpix + 3 * pb;
    const float* dL_dothers = a.dL_dothers + (kPart ? 8 : 7) * pb;
    p.T_final = final_T[pid];
    p.final_D = final_T[pid + HW];
    p.final_D2 = final_T[pid + 2 * HW];
    p.last_contributor = n_contrib[pid];
    p.median_contributor = (int)n_contrib[pid + HW];
    p.dLp0 = dL_dpix[pid];
    p.dLp1 = dL_dpix[HW + pid];
    p.dLp2 = dL_dpix[2 * HW + pid];
    p.dL_ddepth = dL_dothers[pid];
    p.dL_daccum = dL_dothers[HW + pid];
    p.dLn0 = dL_dothers[2 * HW + pid];
    p.dLn1 = dL_dothers[3 * HW + pid];
    p.dLn2 = dL_dothers[4 * HW + pid];
    p.dL_dmedian = dL_dothers[5 * HW + pid];
    p.dL_dreg = dL_dothers[6 * HW + pid];
    if (kPart) p.dL_dmaxw = dL_dothers[7 * HW + pid];
  }
  p.final_A = 1.0f - p.T_final;
  float bg_dot = 0.0f;
  bg_dot += a.bg[0] * p.dLp0;
  bg_dot += a.bg[1] * p.dLp1;
  bg_dot += a.bg[2] * p.dLp2;
  p.bg_dot = bg_dot;
  return p;
}

// The back-to-front recurrences of one pixel (backward.cu:316-379): fed the
// pairs it blended in reverse order, each step yields the pair's weight
// w = alpha T, dL/dalpha and dL/ddepth, from which every per-pair gradient
// follows without further pixel state.
struct ChainBwd {
  float T;
  float acc_r0 = 0.0f, acc_r1 = 0.0f, acc_r2 = 0.0f;
  float last_c0 = 0.0f, last_c1 = 0.0f, last_c2 = 0.0f;
  float last_depth = 0.0f, accum_depth_rec = 0.0f, accum_alpha_rec = 0.0f;
  float last_n0 = 0.0f, last_n1 = 0.0f, last_n2 = 0.0f;
  float acc_n0 = 0.0f, acc_n1 = 0.0f, acc_n2 = 0.0f;
  float last_dL_dT = 0.0f, last_alpha = 0.0f;
  // nc = (normal.xyz, r); m_d, m2 = m_d * m_d, dmd_dd = distortion weight,
  // its square and its derivative
  template <bool kPart>
  SR_DEV float4 step(const PixelBwd& p, float alpha, float c_d, float m_d, float m2, float dmd_dd,
                     uint32_t contributor, const float4& nc, float g, float bl) {
    T = T / (1.0f - alpha);
    const float w = alpha * T;
    float dL_dalpha = 0.0f;
    acc_r0 = last_alpha * last_c0 + (1.0f - last_alpha) * acc_r0;
    last_c0 = nc.w;
    dL_dalpha += (nc.w - acc_r0) * p.dLp0;
    acc_r1 = last_alpha * last_c1 + (1.0f - last_alpha) * acc_r1;
    last_c1 = g;
    dL_dalpha += (g - acc_r1) * p.dLp1;
    acc_r2 = last_alpha * last_c2 + (1.0f - last_alpha) * acc_r2;
    last_c2 = bl;
    dL_dalpha += (bl - acc_r2) * p.dLp2;
    float dL_dz = 0.0f, dL_dweight = 0.0f;
    if ((int)contributor == p.median_contributor - 1) {
      dL_dz += p.dL_dmedian;
      if (kPart) dL_dweight += p.dL_dmaxw;
    }
    dL_dweight += ((p.final_D2 + m2 * p.final_A) - (2.0f * m_d) * p.final_D) * p.dL_dreg;
    dL_dalpha += dL_dweight - last_dL_dT;
    last_dL_dT = dL_dweight * alpha + (1.0f - alpha) * last_dL_dT;
    const float dL_dmd = ((2.0f * (T * alpha)) * (m_d * p.final_A - p.final_D)) * p.dL_dreg;
    dL_dz += dL_dmd * dmd_dd;
    accum_depth_rec = last_alpha * last_depth + (1.0f - last_alpha) * accum_depth_rec;
    last_depth = c_d;
    dL_dalpha += (c_d - accum_depth_rec) * p.dL_ddepth;
    accum_alpha_rec = last_alpha + (1.0f - last_alpha) * accum_alpha_rec;
    dL_dalpha += (1.0f - accum_alpha_rec) * p.dL_daccum;
    acc_n0 = last_alpha * last_n0 + (1.0f - last_alpha) * acc_n0;
    last_n0 = nc.x;
    dL_dalpha += (nc.x - acc_n0) * p.dLn0;
    acc_n1 = last_alpha * last_n1 + (1.0f - last_alpha) * acc_n1;
    last_n1 = nc.y;
    dL_dalpha += (nc.y - acc_n1) * p.dLn1;
    acc_n2 = last_alpha * last_n2 + (1.0f - last_alpha) * acc_n2;
    last_n2 = nc.z;
    dL_dalpha += (nc.z - acc_n2) * p.dLn2;
    dL_dalpha *= T;
    last_alpha = alpha;
    dL_dalpha += (-p.T_final / (1.0f - alpha)) * p.bg_dot;
    dL_dz += (alpha * T) * p.dL_ddepth;
    return make_float4(w, dL_dalpha, dL_dz, 0.0f);
  }
};
static_assert(sizeof(ChainBwd) == 18 * sizeof(float), "chain state is 18 floats");

// ChainBwd's recurrences over one segment of a run, as an affine map of the
// state entering the segment.  The seven colour, depth and normal
// accumulators and accum_alpha_rec follow x <- la l + (1 - la) x (la, l the
// alpha and value of the pair behind), last_dL_dT follows
// y <- dw alpha + (1 - alpha) y, and T <- T / (1 - alpha).  Accumulated from
// the identity over the segment's pairs (back to front), the map takes the
// entering state to the leaving one: x_out = A x_in + b, y_out = A2 y_in + b2,
// T_out = T_in / D.  Folding the maps of the later segments onto the chain's
// initial state gives the state where a segment starts without walking the
// pairs behind it; every path folds in the same order with the same
// operations, so a segment's replay starts from the same bits wherever its
// pairs come from.
struct SegMap {
  float A = 1.0f, A2 = 1.0f, b2 = 0.0f, D = 1.0f;
  float b[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};  // r, g, b, depth, n0, n1, n2, alpha
  // one pair (alpha, distortion weight m_d) after the pair behind it (la,
  // values l: r, g, b, depth, n0, n1, n2)
  template <bool kPart>
  SR_DEV void add(const PixelBwd& p, float la, const float* l, float alpha, float m_d, float m2,
                  uint32_t contributor) {
    const float om = 1.0f - la;
#pragma unroll
    for (int x = 0; x < 7; ++x) b[x] = la * l[x] + om * b[x];
    b[7] = la + om * b[7];
    A = om * A;
    float dw = ((p.final_D2 + m2 * p.final_A) - (2.0f * m_d) * p.final_D) * p.dL_dreg;
    if (kPart && (int)contributor == p.median_contributor - 1) dw = p.dL_dmaxw + dw;
    const float oa = 1.0f - alpha;
    b2 = dw * alpha + oa * b2;
    A2 = oa * A2;
    D = D * oa;
  }
  // the map applied to the recurrence part of a chain state
  SR_DEV void apply(ChainBwd& s) const {
    s.T = s.T / D;
    s.acc_r0 = A * s.acc_r0 + b[0];
    s.acc_r1 = A * s.acc_r1 + b[1];
    s.acc_r2 = A * s.acc_r2 + b[2];
    s.accum_depth_rec = A * s.accum_depth_rec + b[3];
    s.acc_n0 = A * s.acc_n0 + b[4];
    s.acc_n1 = A * s.acc_n1 + b[5];
    s.acc_n2 = A * s.acc_n2 + b[6];
    s.accum_alpha_rec = A * s.accum_alpha_rec + b[7];
    s.last_dL_dT = A2 * s.last_dL_dT + b2;
  }
  // in LDS, a lane's words 64 apart
  SR_DEV void save(float* d) const {
    d[0] = A;
    d[64] = A2;
    d[128] = b2;
    d[192] = D;
#pragma unroll
    for (int x = 0; x < 8; ++x) d[64 * (4 + x)] = b[x];
  }
  SR_DEV void load(const float* d) {
    A = d[0];
    A2 = d[64];
    b2 = d[128];
    D = d[192];
#pragma unroll
    for (int x = 0; x < 8; ++x) b[x] = d[64 * (4 + x)];
  }
};
constexpr int kSegMapFloats = 12;

// The values of a chain state that a pair sets for the next one (the "last"
// members), in SegMap's order.
SR_DEV void chain_last(const ChainBwd& s, float* l) {
  l[0] = s.last_c0;
  l[1] = s.last_c1;
  l[2] = s.last_c2;
  l[3] = s.last_depth;
  l[4] = s.last_n0;
  l[5] = s.last_n1;
  l[6] = s.last_n2;
}

// The 18 partial gradients of one pair (backward.cu:380-437) from its
// weight w, dL/dalpha and dL/ddepth and its pixel's dL/dpixel (dLp) and
// dL/dnormal (dLn), handed to add(slot, value).
template <class Add>
SR_DEV void pair_grads(float dLp0, float dLp1, float dLp2, float dLn0, float dLn1, float dLn2, const Pair& e,
                       const float4& q1, float opa, float w, float dL_dalpha, float dL_dz, float pixx, float pixy,
                       Add add) {
  add(15, w * dLp0);
  add(16, w * dLp1);
  add(17, w * dLp2);
  add(11, w * dLn0);
  add(12, w * dLn1);
  add(13, w * dLn2);
  const float G = e.G;
  const float dL_dG = opa * dL_dalpha;
  if (e.rho3d <= e.rho2d) {
    const float sx = e.sx, sy = e.sy, pz = e.pz;
    const float kx = e.kx, ky = e.ky, kz = e.kz, lx = e.lx, ly = e.ly, lz = e.lz;
    const float dL_dsx = (dL_dG * -G) * sx + dL_dz * q1.z;
    const float dL_dsy = (dL_dG * -G) * sy + dL_dz * q1.w;
    const float dsx_pz = dL_dsx / pz, dsy_pz = dL_dsy / pz;
    const float dpx = dsx_pz, dpy = dsy_pz, dpz = -(dsx_pz * sx + dsy_pz * sy);
    // dL_dk = cross(l, dL_dp), dL_dl = cross(dL_dp, k)
    const float dkx = ly * dpz - lz * dpy, dky = lz * dpx - lx * dpz, dkz = lx * dpy - ly * dpx;
    const float dlx = dpy * kz - dpz * ky, dly = dpz * kx - dpx * kz, dlz = dpx * ky - dpy * kx;
    add(0, -dkx);
    add(1, -dky);
    add(2, -dkz);
    add(3, -dlx);
    add(4, -dly);
    add(5, -dlz);
    add(6, (pixx * dkx + pixy * dlx) + dL_dz * sx);
    add(7, (pixx * dky + pixy * dly) + dL_dz * sy);
    add(8, (pixx * dkz + pixy * dlz) + dL_dz * 1.0f);
  } else {
    const float dG_ddelx = (-G * 2.0f) * e.dx;
    const float dG_ddely = (-G * 2.0f) * e.dy;
    add(9, dL_dG * dG_ddelx);
    add(10, dL_dG * dG_ddely);
    add(8, dL_dz);
  }
  add(14, G * dL_dalpha);
}

// Backward blend, pass 1 of 2: per pixel, back to front, the pairs it blended
// (the accepted pairs in front of its last contributor, exactly the
// reference's), running only the per-pixel recurrences and writing each pair's
// (w, dL/dalpha, dL/ddepth) to the pair store.  The pairs come from the store
// as one contiguous run per pixel in entry order (the forward cut it at the
// last contributor); nothing is staged, so the serial chain carries only the
// recurrences.
//
// A long run is cut into up to 16 segments, one lane each.  Each segment's lane
// first runs its pairs through SegMap (the state recurrences as an affine map,
// about a third of a step); the maps of the segments behind a segment, folded
// onto the chain's initial state, give the state where it starts; then every
// lane replays its segment with full steps from that state, so the serial
// chain of a run of n pairs is two passes over n / 16 pairs instead of one over
// n.  A wave gives its pixels as many lanes each as the quadrant's longest run
// can have segments (1 to 16, by its cost's class), and a quadrant takes as
// many waves.  300k surfels at 800 x 600: 86 us and at 400 x 300 47 (98 and 49
// with 48-byte records); with 8 lanes a pixel in every quadrant and each lane
// loading its own records 130 and 72; with the lanes by class but their own
// records still 130 and 66.
template <bool kPart>
SR_DEV void blend_bwd_stored(const BlendBwdArgs& a, int qi, int lg, int part, float4* s_buf) {
  // s_buf: a batch of every lane's pairs; between the walks the SegMaps
  float* s_map = reinterpret_cast<float*>(s_buf);
  constexpr int kBytes = PairLayout<kPart>::kBytes;
  const int B = a.vs.B, QX = B / kQuad, Q = QX * QX;
  const int tile = qi / Q, q = qi % Q;
  const ViewInfo& vi = a.vs.v[view_of_tile(a.vs, (uint32_t)tile)];
  const int lt = tile - (int)vi.tile_base;
  const int tx = lt % vi.gx, ty = lt / vi.gx;
  const int lane = threadIdx.x;
  const int npx = 64 >> lg;  // pixels of the wave
  const int ps = lane & (npx - 1), sg = lane >> (6 - lg);
  const int pxl = part * npx + ps;
  const uint32_t qxi = (uint32_t)(tx * B + (q % QX) * kQuad + (pxl & 7));
  const uint32_t qyi = (uint32_t)(ty * B + (q / QX) * kQuad + (pxl >> 3));
  const bool pin = qxi < (uint32_t)vi.W && qyi < (uint32_t)vi.H;
  const uint2 rg = pin ? a.lane_range[(size_t)qi * 64 + pxl] : make_uint2(0u, 0u);
  const int n = (int)rg.y;
  const int seg_len = chain_segment(n);
  const int nseg = (n + seg_len - 1) / seg_len;
  const PixelBwd px = pixel_bwd<kPart>(a, vi, n > 0, qxi, qyi);
  const int lo = sg * seg_len, hi = min(n, lo + seg_len) - 1;
  // alpha and values of the pair behind the segment (none behind the last)
  float la = 0.0f, l[7] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
  if (sg < nseg - 1) {
    const float* pr = reinterpret_cast<const float*>(a.ps.rec + (size_t)kBytes * (rg.x + (uint32_t)(hi + 1)));
    la = pr[2];
    l[0] = pr[4];
    l[1] = pr[5];
    l[2] = pr[6];
    l[3] = pr[3];
    l[4] = pr[7];
    l[5] = pr[8];
    l[6] = pr[9];
  }
  // Walks lane segments [lo, hi] (hi < lo: none) from the back, calling
  // fn(depth, m, alpha, position, (normal, red), green, blue) for each pair; the whole wave calls it.  A lane streaming
  // its own records would touch a cache line of its own per load, and it is
  // the line rate that bounds the pass: so the four lanes of a quad load the
  // four lanes' batches together, 64 contiguous bytes at a time, and the
  // batches change hands in LDS, the next one in flight.  Batches are whole:
  // up to kChainPre - 1 records in front of lo are read (nothing uses them;
  // the store is padded).  With kOut, fn's results go to fW the same way.
  const int ql = lane & 3, qd = lane >> 2;  // place in the quad, quad
  char* mine_at = reinterpret_cast<char*>(s_buf) + lane * kOwnerBytes<kPart>;
  auto walk = [&](auto out, int lo, int hi, auto&& fn) {
    constexpr bool kOut = decltype(out)::value;
    int left[4];     // pairs left of each of the quad's lanes
    uint32_t at[4];  // and its next batch's first record
#pragma unroll
    for (int o = 0; o < 4; ++o) {
      left[o] = __shfl(hi - lo + 1, qd * 4 + o);
      at[o] = (uint32_t)__shfl((int)(rg.x + (uint32_t)hi), qd * 4 + o) - (kChainPre - 1);
    }
    int mine = hi - lo + 1;
    // of each lane's batch: 16 bytes at 16 ql and 64 more, then the rest of
    // the four records, 8 or 16 bytes a lane
    using Rest = std::conditional_t<kPart, V4, V2>;
    V4 g[4][2] = {};
    Rest g2[4] = {};
    auto fetch = [&]() {
#pragma unroll
      for (int o = 0; o < 4; ++o) {
        if (left[o] <= 0) continue;
        const char* pr = a.ps.rec + (ptrdiff_t)kBytes * (int32_t)at[o];
        g[o][0] = load8<V4>(pr + 16 * ql);
        g[o][1] = load8<V4>(pr + 64 + 16 * ql);
        g2[o] = load8<Rest>(pr + 128 + (int)sizeof(Rest) * ql);
      }
    };
    fetch();
    while (__ballot(mine > 0) != 0ull) {
#pragma unroll
      for (int o = 0; o < 4; ++o) {
        char* d = reinterpret_cast<char*>(s_buf) + (qd * 4 + o) * kOwnerBytes<kPart>;
        *reinterpret_cast<V4*>(d + 16 * ql) = g[o][0];
        *reinterpret_cast<V4*>(d + 64 + 16 * ql) = g[o][1];
        *reinterpret_cast<Rest*>(d + 128 + (int)sizeof(Rest) * ql) = g2[o];
      }
      uint32_t was[4];
      int had[4];
#pragma unroll
      for (int o = 0; o < 4; ++o) {
        was[o] = at[o];
        had[o] = left[o];
        at[o] -= kChainPre;
        left[o] -= kChainPre;
      }
      fetch();  // in flight while this batch is used
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      float4 r[kChainPre];
#pragma unroll
      for (int k = kChainPre - 1; k >= 0; --k) {
        r[k] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if (kChainPre - 1 - k < mine) {
          const char* p = mine_at + kBytes * k;
          const V4 p0 = load8<V4>(p), p1 = load8<V4>(p + 16);
          const V2 p2 = load8<V2>(p + 32);
          const uint32_t pos = kPart ? *reinterpret_cast<const uint32_t*>(p + 40) : __float_as_uint(p0.y);
          r[k] = fn(p0.w, p0.x, p0.z, pos, make_float4(p1.w, p2.x, p2.y, p1.x), p1.y, p1.z);
        }
      }
      mine -= kChainPre;
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      if (kOut) {
        // rotated so that neither side's accesses share banks
        auto place = [&](int o, int k) { return (qd * 4 + ((o + qd) & 3)) * 4 + ((k ^ qd) & 3); };
#pragma unroll
        for (int k = 0; k < kChainPre; ++k) s_buf[place(ql, k)] = r[k];
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
        for (int o = 0; o < 4; ++o)
          if (kChainPre - 1 - ql < had[o]) {
            const float4 x = s_buf[place(o, ql)];
            a.ps.fW[was[o] + (uint32_t)ql] = PairOut{x.x, x.y, x.z};
          }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      }
    }
  };
  const bool mapped = sg >= 1 && sg < nseg;  // segment 0's map is never needed
  SegMap m;
  if (lg > 0) {  // uniform
    float pa = la, pl[7];
#pragma unroll
    for (int x = 0; x < 7; ++x) pl[x] = l[x];
    walk(std::false_type{}, lo, mapped ? hi : lo - 1,
         [&](float depth, float m_d, float alpha, uint32_t pos, const float4& nr, float g, float b) {
      m.add<kPart>(px, pa, pl, alpha, m_d, m_d * m_d, pos);
      pa = alpha;
      pl[0] = nr.w;
      pl[1] = g;
      pl[2] = b;
      pl[3] = depth;
      pl[4] = nr.x;
      pl[5] = nr.y;
      pl[6] = nr.z;
      return nr;
    });
    __syncthreads();
    if (mapped) m.save(s_map + lane);
    __syncthreads();
  }
  ChainBwd ch;
  ch.T = px.T_final;
  for (int t = nseg - 1; t > sg; --t) {
    SegMap behind;
    behind.load(s_map + t * npx + ps);
    behind.apply(ch);
  }
  __syncthreads();
  ch.last_alpha = la;
  ch.last_c0 = l[0];
  ch.last_c1 = l[1];
  ch.last_c2 = l[2];
  ch.last_depth = l[3];
  ch.last_n0 = l[4];
  ch.last_n1 = l[5];
  ch.last_n2 = l[6];
  walk(std::true_type{}, lo, hi, [&](float depth, float m_d, float alpha, uint32_t pos, const float4& nr, float g,
                                     float b) {
    return ch.step<kPart>(px, alpha, depth, m_d, m_d * m_d, dist_weight_grad<kPart>(depth), pos, nr, g, b);
  });
}

// The whole backward blend of a quadrant whose pairs missed the store: per
// chunk, the records staged, the pairs recomputed, the recurrences and the
// gradients together, each entry's sums stored as it is done.  s_buf: LDS that
// the other path sizes.
template <bool kPart>
SR_DEV void blend_bwd_missed(const BlendBwdArgs& a, int qi, float4* s_buf) {
  float4 *s_q0 = s_buf, *s_q1 = s_buf + 64, *s_q2 = s_buf + 128, *s_q3 = s_buf + 192, *s_q4 = s_buf + 256;
  uint2* s_e = reinterpret_cast<uint2*>(s_buf + 320);
  float(*s_tmp)[65] = reinterpret_cast<float(*)[65]>(s_buf + 352);
  static_assert(64 * kOwnerBytes<kPart> >= 352 * 16 + kNumG * 65 * 4 && kNumG >= kMaxSem,
                "fits the other path's LDS");
  const int cnt = (int)a.sub_count[qi];
  const int B = a.vs.B, QX = B / kQuad, Q = QX * QX;
  const int tile = qi / Q, q = qi % Q;
  const ViewInfo& vi = a.vs.v[view_of_tile(a.vs, (uint32_t)tile)];
  const int lt = tile - (int)vi.tile_base;
  const int tx = lt % vi.gx, ty = lt / vi.gx;
  const int lane = threadIdx.x, pix = lane;
  const uint32_t pxi = (uint32_t)(tx * B + (q % QX) * kQuad + (pix & 7));
  const uint32_t pyi = (uint32_t)(ty * B + (q / QX) * kQuad + (pix >> 3));
  const bool inside = pxi < (uint32_t)vi.W && pyi < (uint32_t)vi.H;
  const float pixx = pixel_centre<kPart>((int)pxi), pixy = pixel_centre<kPart>((int)pyi);
  ChainBwd ch;
  const uint32_t rbeg = a.ranges[2 * tile], ntile = a.ranges[2 * tile + 1] - rbeg;
  const uint2* list = a.sub + (size_t)Q * rbeg + (size_t)q * ntile;
  const uint64_t* masks = a.masks + mask_base(Q, rbeg, ntile, tile, q);
  const uint32_t* frag_off = a.frag_off + mask_base(Q, rbeg, ntile, tile, q);
  const PixelBwd px = pixel_bwd<kPart>(a, vi, inside, pxi, pyi);
  ch.T = px.T_final;
  // The pixel's run is cut into the stored path's segments (the forward
  // recorded how many pairs the pixel blended): while a segment's pairs go
  // through full steps, its SegMap is accumulated alongside, and where the
  // segment ends the state is reset to the maps folded onto the initial
  // state, exactly as the stored path's segment lanes start, so each pair's
  // outputs have the stored path's bits.
  ChainBwd fold = ch;  // the state the current segment started from
  SegMap seg_map;
  const int n_run = inside ? (int)a.lane_range[(size_t)qi * 64 + pix].y : 0;
  const int seg_len = chain_segment(n_run);
  int seg = (n_run + seg_len - 1) / seg_len - 1, seg_start = seg * seg_len, idx = n_run;
  const int nch = (cnt + 63) / 64;
  const bool active = inside && px.last_contributor > 0;
  for (int c = nch - 1; c >= 0; --c) {
    const ChunkRegs nx = chunk_load(masks, frag_off, a.rec, lane, c, chunk_entry(list, cnt, lane, c, nch));
    uint64_t mask = active ? nx.mask : 0ull;
    const int m = min(64, cnt - c * 64);
    __syncthreads();
    if (lane < m) {
      s_e[lane] = nx.v;
      s_q0[lane] = nx.q0;
      s_q1[lane] = nx.q1;
      s_q2[lane] = nx.q2;
      s_q3[lane] = nx.q3;
      s_q4[lane] = nx.q4;
    }
    __syncthreads();
    // this lane's entry's slot, and the entries whose sums are stored
    const uint32_t slot = lane < m ? (uint32_t)slot_of(a.pos_slot, a.pos_quads, rbeg + s_e[lane].y, q) : 0u;
    uint64_t stored = 0ull;
    if (__ballot(mask != 0ull) != 0ull) {
      // entries from last to first, the wave in step (each lane still walks
      // its own pixel's entries back to front); an entry's 18 partial
      // gradients are then summed over the pixels that blended it in pixel
      // order from 0, in runs of kGradGroup pixels whose sums are added in
      // order, exactly as the per-pair gradient pass sums a stored
      // quadrant's, so the partials have the same bits whichever quadrants
      // missed the pair store
      for (int j = 63; j >= 0; --j) {
        const bool hit = (mask >> j) & 1ull;
        if (__ballot(hit) == 0ull) continue;
        float gk[kNumG];
#pragma unroll
        for (int k = 0; k < kNumG; ++k) gk[k] = 0.0f;
        bool took = false;
        float took_w = 0.0f;
        const uint32_t contributor = s_e[j].y;  // 0-based position in the tile list
        if (hit && contributor < px.last_contributor) {
          const float4 q2 = s_q2[j];
          Pair e;  // a flagged quadrant has no stored pairs: recompute
          if (eval_pair<false>(pixx, pixy, s_q0[j], s_q1[j], q2, 0.0f, e)) {
            const float c_d = e.depth;
            const float m_d = dist_weight<kPart>(c_d), dmd_dd = dist_weight_grad<kPart>(c_d);
            const float4 q3 = s_q3[j], q4 = s_q4[j];
            --idx;  // this pair's place in the run
            if (seg >= 1) {
              float l[7];
              chain_last(ch, l);
              seg_map.add<kPart>(px, ch.last_alpha, l, e.alpha, m_d, m_d * m_d, contributor);
            }
            const float4 g = ch.step<kPart>(px, e.alpha, c_d, m_d, m_d * m_d, dmd_dd, contributor, q3, q4.x, q4.y);
            if (idx == seg_start && seg >= 1) {  // the next pair starts segment seg - 1
              seg_map.apply(fold);
              ch.T = fold.T;
              ch.acc_r0 = fold.acc_r0;
              ch.acc_r1 = fold.acc_r1;
              ch.acc_r2 = fold.acc_r2;
              ch.accum_depth_rec = fold.accum_depth_rec;
              ch.acc_n0 = fold.acc_n0;
              ch.acc_n1 = fold.acc_n1;
              ch.acc_n2 = fold.acc_n2;
              ch.accum_alpha_rec = fold.accum_alpha_rec;
              ch.last_dL_dT = fold.last_dL_dT;
              seg_map = SegMap();
              --seg;
              seg_start -= seg_len;
            }
            pair_grads(px.dLp0, px.dLp1, px.dLp2, px.dLn0, px.dLn1, px.dLn2, e, s_q1[j], q2.w, g.x, g.y, g.z,
                       pixx, pixy, [&](int k, float v) { gk[k] += v; });
            took = true;
            took_w = g.x;
          }
        }
        const uint64_t tookm = __ballot(took);
        // row `lane` of s_tmp summed over the pixels of tookm, grouped
        // exactly as the per-pair gradient pass sums
        auto grouped = [&]() {
          float acc = 0.0f, grp = 0.0f;
          int in_grp = 0;
          for (uint64_t mm = tookm; mm != 0ull; mm &= mm - 1ull) {
            grp += s_tmp[lane][__builtin_ctzll(mm)];
            if (++in_grp == kGradGroup) {
              acc += grp;
              grp = 0.0f;
              in_grp = 0;
            }
          }
          if (in_grp > 0) acc += grp;
          return acc;
        };
#pragma unroll
        for (int k = 0; k < kNumG; ++k) s_tmp[k][lane] = gk[k];
        __syncthreads();
        const float sum = lane < kNumG ? grouped() : 0.0f;
        __syncthreads();
        // the entry's slot, as store_part writes it
        const uint32_t at = (uint32_t)__shfl((int)slot, j);
        const bool sem = kPart && a.S > 0 && tookm != 0ull;
        if (__ballot(sum != 0.0f) != 0ull || sem) {
          if (lane < kPartStride) a.part[(size_t)at * kPartStride + lane] = sum;
          if (lane == 0) a.part_nz[at] = 1;
          stored |= 1ull << j;
        }
        if (sem) {  // semantics get their own gradient only
#pragma unroll
          for (int x = 0; x < kMaxSem; ++x)
            s_tmp[x][lane] = took && x < a.S ? took_w * a.dL_dsem[(size_t)a.S * vi.pix_base +
                                                                  x * ((size_t)vi.H * vi.W) + (size_t)vi.W * pyi + pxi]
                                             : 0.0f;
          __syncthreads();
          if (lane < a.S) a.sem_part[(size_t)at * a.S + lane] = grouped();
          __syncthreads();
        }
      }
    }
    if (lane < m && ((stored >> lane) & 1ull) == 0ull) a.part_nz[slot] = 0;
    __syncthreads();
  }
}

// The quadrants come in cost order, so those of a class are contiguous: work
// item w is a wave of the first class with w left.
template <bool kPart>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(3, 3))) void k_blend_bwd(BlendBwdArgs a) {
  __shared__ float4 s_buf[64 * kOwnerBytes<kPart> / 16];
  static_assert(sizeof(s_buf) >= kSegMapFloats * 64 * sizeof(float) && sizeof(s_buf) >= 64 * kChainPre * 16,
                "one map, or one batch of results, a lane");
  if (a.counters[1] & kErrCapacity) return;
  const uint32_t* end = a.counters + kCostClass;  // of the classes, in quadrants
  uint32_t items = 0;
  for (int c = 0; c <= kSegLog; ++c) items += (end[c] - (c > 0 ? end[c - 1] : 0u)) << (kSegLog - c);
  for (uint32_t w = blockIdx.x; w < items; w += gridDim.x) {
    uint32_t first = 0, at = w;
    int c = 0;
    for (; c < kSegLog && at >= (end[c] - first) << (kSegLog - c); ++c) {
      at -= (end[c] - first) << (kSegLog - c);
      first = end[c];
    }
    const int lg = kSegLog - c;
    const int qi = (int)a.q_order[first + (at >> lg)], part = (int)(at & ((1u << lg) - 1u));
    if (a.q_flag[qi] == 0u) blend_bwd_stored<kPart>(a, qi, lg, part, s_buf);
    else if (part == 0) blend_bwd_missed<kPart>(a, qi, s_buf);
    __syncthreads();
  }
}

hipError_t launch_blend_bwd(const BlendBwdArgs& a, hipStream_t s) {
  if (a.vs.T == 0) return hipSuccess;
  if (a.vs.B != 8 && a.vs.B != 16 && a.vs.B != 32) return hipErrorInvalidValue;
  const unsigned nblk = (unsigned)(a.vs.T * quads_per_tile(a.vs.B));
  const unsigned grid = nblk << kSegLog < kChainBlocks ? nblk << kSegLog : kChainBlocks;
  if (a.is_part) hipLaunchKernelGGL(k_blend_bwd<true>, dim3(grid), dim3(64), 0, s, a);
  else hipLaunchKernelGGL(k_blend_bwd<false>, dim3(grid), dim3(64), 0, s, a);
  return hipGetLastError();
}

// 64 x 64 bit-matrix transpose across a wave: lane i passes row i (bit j =
// M[i][j]) and gets column i back (bit j = M[j][i]).  Recursive block swap:
// at each of the six levels the lanes that differ in bit s exchange the
// off-diagonal s x s blocks of their 2s x 2s block.
SR_DEV uint64_t wave_transpose64(uint64_t x, int lane) {
  uint32_t lo = (uint32_t)x, hi = (uint32_t)(x >> 32);
  {
    const uint32_t plo = (uint32_t)__shfl_xor((int)lo, 32), phi = (uint32_t)__shfl_xor((int)hi, 32);
    if (lane & 32)
      lo = phi;
    else
      hi = plo;
  }
  auto level = [&](uint32_t v, int sh, uint32_t m) -> uint32_t {
    const uint32_t y = (uint32_t)__shfl_xor((int)v, sh);
    return (lane & sh) ? (((y & ~m) >> sh) | (v & ~m)) : ((v & m) | ((y & m) << sh));
  };
  lo = level(lo, 16, 0x0000FFFFu);
  hi = level(hi, 16, 0x0000FFFFu);
  lo = level(lo, 8, 0x00FF00FFu);
  hi = level(hi, 8, 0x00FF00FFu);
  lo = level(lo, 4, 0x0F0F0F0Fu);
  hi = level(hi, 4, 0x0F0F0F0Fu);
  lo = level(lo, 2, 0x33333333u);
  hi = level(hi, 2, 0x33333333u);
  lo = level(lo, 1, 0x55555555u);
  hi = level(hi, 1, 0x55555555u);
  return (uint64_t)lo | ((uint64_t)hi << 32);
}

// Backward blend, pass 2 of 2.  The per-pair gradients, balanced over the
// whole GPU on the acceptance work list: one wave per (quadrant, 64-entry
// chunk).  A pair's gradients need no pixel recurrence any more (pass 1
// stored its w, dL/dalpha and dL/ddepth).  The acceptance masks (one word
// per pixel), trimmed to the pairs in front of each pixel's last
// contributor, are transposed into one word of pixels per entry; each
// entry's pixels are cut into groups of kGradGroup in pixel order, and the
// groups of all entries are dealt over the lanes, 64 per round, so the
// lanes stay busy however unevenly the entries cover the quadrant.  A lane
// recomputes its group's pairs exactly and sums their 18 partial gradients
// in pixel order; the entry's lane then adds its group sums in order.  Each
// entry's sums go to its (position, quadrant) slot of the partial-gradient
// buffer.  The recompute path of pass 1 groups its sums the same way, so
// the partials have the same bits whichever quadrants missed the pair store.
// 88 us for 300k surfels at 800 x 600, 53 of them issuing (57 % of the lanes at
// work: the last group of an entry is rarely full).
// kSem: the _part variant's semantic channels, rounded up (0: none), whose
// gradients w dL/dsem are summed the same way into sem_part.
// The group sums change hands in rows of kGrpRow floats, 12 at a time: four a
// read instead of one, and with rows of 12 and not all 18 (20) ten KB of LDS, so
// that LDS does not hold fewer waves than registers do.  300k surfels at 800 x
// 600: 88 us with rows of 12, 90 with 8, 16, 20 or one float at a time; 1M at
// 1237 x 823 274, 280 one at a time; the _part variant with 8 channels, whose
// dL/dsem are read by four too, 126, was 144.
constexpr int kGrpRow = 12;
template <bool kPart, int kSem>
__global__ __launch_bounds__(64) void k_blend_bwd_grad(BlendBwdArgs a) {
  __shared__ uint4 s_pm[64];    // per pixel: trimmed mask (lo, hi), first stored pair of the chunk
  __shared__ float4 s_pg[64];   // per pixel: dL/dpixel (rgb), dL/dnormal.x
  __shared__ float2 s_pn[64];   // per pixel: dL/dnormal.yz
  __shared__ uint32_t s_pos[64];
  __shared__ float4 s_e0[64], s_e1[64], s_e2[64];  // per entry: record quads 0..2
  __shared__ unsigned long long s_col[64];         // per entry: the pixels that blended it
  __shared__ uint32_t s_tbase[64];                 // per entry: its first group
  __shared__ uint32_t s_head[64];
  __shared__ V4 s_grp[64][kGrpRow / 4];            // per lane: kGrpRow of its group's sums
  __shared__ V4 s_dls[kSem > 0 ? 64 : 1][kSem > 0 ? kSem / 4 : 1];  // per pixel: dL/dsem
  const int lane = threadIdx.x;
  if (a.counters[1] & kErrCapacity) return;
  const uint32_t nwork = *a.work_count;
  const int lgQ = a.vs.B == 8 ? 0 : a.vs.B == 16 ? 2 : 4;  // quadrants of a tile
  for (uint32_t w = blockIdx.x; w < nwork; w += gridDim.x) {
    const WorkItem it = unpack_work(a.work[nwork - 1u - w]);  // from the end: see work_capacity
    if (a.q_flag[it.qi] != 0u) continue;  // done by pass 1
    const ViewInfo& vi = a.vs.v[it.view];
    const int bx = it.x0, by = it.y0;
    // lane as pixel (lane & 7, lane >> 3) of the quadrant
    const int pxi = bx + (lane & 7), pyi = by + (lane >> 3);
    const bool inside = pxi < vi.W && pyi < vi.H;
    const uint32_t rbeg = a.ranges[2 * (it.qi >> lgQ)];
    const size_t mslot = it.first + 64u * (size_t)it.qi + lane;
    uint64_t mask = inside ? a.masks[mslot] : 0ull;
    const uint32_t foff = mask ? a.frag_off[mslot] : 0u;
    const size_t HW = (size_t)vi.H * vi.W, pid = (size_t)vi.W * pyi + pxi, pb = vi.pix_base;
    uint32_t lc = 0u;
    float4 pg = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    float2 pn = make_float2(0.0f, 0.0f);
    if (mask) {
      lc = a.n_contrib[2 * pb + pid];
      const float* dL_dpix = a.dL_dpix + 3 * pb;
      const float* dL_dothers = a.dL_dothers + (kPart ? 8 : 7) * pb;
      pg = make_float4(dL_dpix[pid], dL_dpix[HW + pid], dL_dpix[2 * HW + pid], dL_dothers[2 * HW + pid]);
      pn = make_float2(dL_dothers[3 * HW + pid], dL_dothers[4 * HW + pid]);
    }
    // lane as entry of the chunk
    const bool has = (uint32_t)lane < it.m;
    const uint2 v = has ? a.sub[it.first + lane] : make_uint2(0u, 0xFFFFFFFFu);
    float4 q0 = make_float4(0.0f, 0.0f, 0.0f, 0.0f), q1 = q0, q2 = q0;
    if (has) {
      const float4* r = a.rec + (size_t)kRecQuads * v.x;
      q0 = r[0];
      q1 = r[1];
      q2 = r[2];
    }
    wave_lds_fence();  // the previous item's readers are done
    s_pos[lane] = v.y;
    s_e0[lane] = q0;
    s_e1[lane] = q1;
    s_e2[lane] = q2;
    if constexpr (kSem > 0) {
      auto dls = [&](int x) { return mask && x < a.S ? a.dL_dsem[(size_t)a.S * pb + x * HW + pid] : 0.0f; };
#pragma unroll
      for (int x = 0; x < kSem; x += 4) s_dls[lane][x / 4] = V4{dls(x), dls(x + 1), dls(x + 2), dls(x + 3)};
    }
    wave_lds_fence();
    if (mask) {
      // entries in front of the last contributor: positions rise along the
      // chunk, so they are the first J, found by binary search
      int J = 0;
#pragma unroll
      for (int st = 64; st > 0; st >>= 1)
        if (J + st <= 64 && s_pos[J + st - 1] < lc) J += st;
      if (J < 64) mask &= (1ull << J) - 1ull;
    }
    s_pm[lane] = make_uint4((uint32_t)mask, (uint32_t)(mask >> 32), foff, 0u);
    s_pg[lane] = pg;
    s_pn[lane] = pn;
    const uint64_t col = wave_transpose64(mask, lane);  // bit p: pixel p blended this lane's entry
    const uint32_t ng = ((uint32_t)__popcll(col) + (kGradGroup - 1)) / kGradGroup;
    uint32_t tincl = ng;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const uint32_t y = (uint32_t)__shfl_up((int)tincl, off, 64);
      if (lane >= off) tincl += y;
    }
    const uint32_t tbase = tincl - ng, ntask = (uint32_t)__shfl((int)tincl, 63, 64);
    s_col[lane] = col;
    s_tbase[lane] = tbase;
    wave_lds_fence();
    float acc[kNumG + kSem];
#pragma unroll
    for (int k = 0; k < kNumG + kSem; ++k) acc[k] = 0.0f;
    SlotOwner owner;
    for (uint32_t base = 0; base < ntask; base += 64) {  // uniform
      const uint32_t t = base + (uint32_t)lane;
      const int j = (int)owner.at(s_head, base, tbase, ng);
      float g[kNumG + kSem];
#pragma unroll
      for (int k = 0; k < kNumG + kSem; ++k) g[k] = 0.0f;
      if (t < ntask) {
        const uint32_t gi = t - s_tbase[j];
        const uint64_t cj = s_col[j];
        // the group's pixels: the set bits of cj from the (gi kGradGroup)-th on
        const int first = select_bit(cj, gi * kGradGroup);
        uint64_t mm = cj & ~((1ull << first) - 1ull);
        const uint64_t below = (1ull << j) - 1ull;  // the entry's rank within a pixel's mask
        int pp[kGradGroup];
        PairOut fw[kGradGroup];
#pragma unroll
        for (int k = 0; k < kGradGroup; ++k) {
          pp[k] = -1;
          if (mm != 0ull) {
            const int p = __builtin_ctzll(mm);
            mm &= mm - 1ull;
            pp[k] = p;
            const uint4 pm = s_pm[p];
            const uint64_t mp = (uint64_t)pm.x | ((uint64_t)pm.y << 32);
            fw[k] = a.ps.fW[pm.z + (uint32_t)__popcll(mp & below)];
          }
        }
        const float4 r0 = s_e0[j], r1 = s_e1[j], r2 = s_e2[j];
#pragma unroll
        for (int k = 0; k < kGradGroup; ++k) {
          const int p = pp[k];
          if (p < 0) continue;
          const float4 g4 = s_pg[p];
          const float2 n2 = s_pn[p];
          const float pixx = pixel_centre<kPart>(bx + (p & 7)), pixy = pixel_centre<kPart>(by + (p >> 3));
          // the pair itself (s, G, planes) recomputed exactly as the
          // acceptance pass evaluated it: cheaper than fetching it
          Pair e;
          (void)eval_pair<false>(pixx, pixy, r0, r1, r2, 0.0f, e);
          pair_grads(g4.x, g4.y, g4.z, g4.w, n2.x, n2.y, e, r1, r2.w, fw[k].w, fw[k].dalpha, fw[k].ddepth, pixx, pixy,
                     [&](int s, float val) { g[s] += val; });
#pragma unroll
          for (int x = 0; x < kSem; x += 4) {
            const V4 d = s_dls[p][x / 4];
#pragma unroll
            for (int c = 0; c < 4; ++c) g[kNumG + x + c] += fw[k].w * d[c];
          }
        }
      }
      // the entry's lane adds its groups of this round, in order
      const uint32_t lo = max(tbase, base), hi = min(tbase + ng, base + 64u);
#pragma unroll
      for (int k0 = 0; k0 < kNumG + kSem; k0 += kGrpRow) {
        auto sums = [&](auto&& fn) {  // the row's quads, fn(place, first sum)
#pragma unroll
          for (int q = 0; q < kGrpRow / 4; ++q)
            if (k0 + 4 * q < kNumG + kSem) fn(q, k0 + 4 * q);
        };
        auto at = [&](int k) { return k < kNumG + kSem ? g[k < kNumG + kSem ? k : 0] : 0.0f; };
        sums([&](int q, int k) { s_grp[lane][q] = V4{at(k), at(k + 1), at(k + 2), at(k + 3)}; });
        wave_lds_fence();
        for (uint32_t u = lo; u < hi; ++u) {
          sums([&](int q, int k) {
            const V4 x = s_grp[u - base][q];
#pragma unroll
            for (int c = 0; c < 4; ++c)
              if (k + c < kNumG + kSem) acc[k + c] += x[c];
          });
        }
        wave_lds_fence();
      }
    }
    if (has) {
      const size_t slot = slot_of(a.pos_slot, a.pos_quads, rbeg + v.y, (int)(it.qi & ((1u << lgQ) - 1u)));
      store_part(a, slot, [&](int k) { return acc[k]; }, kSem > 0 && ng > 0u);
      if (kSem > 0 && ng > 0u) {
        float* d = a.sem_part + slot * (size_t)a.S;
#pragma unroll
        for (int x = 0; x < kSem; ++x)
          if (x < a.S) d[x] = acc[kNumG + x];
      }
    }
  }
}

hipError_t launch_blend_bwd_grad(const BlendBwdArgs& a, size_t max_items, hipStream_t s) {
  if (max_items == 0) return hipSuccess;
  const unsigned grid = (unsigned)(max_items < kChunkBlocks ? max_items : kChunkBlocks);
  if (!a.is_part) hipLaunchKernelGGL((k_blend_bwd_grad<false, 0>), dim3(grid), dim3(64), 0, s, a);
  else if (a.S == 0) hipLaunchKernelGGL((k_blend_bwd_grad<true, 0>), dim3(grid), dim3(64), 0, s, a);
  else if (a.S <= 4) hipLaunchKernelGGL((k_blend_bwd_grad<true, 4>), dim3(grid), dim3(64), 0, s, a);
  else if (a.S <= 8) hipLaunchKernelGGL((k_blend_bwd_grad<true, 8>), dim3(grid), dim3(64), 0, s, a);
  else hipLaunchKernelGGL((k_blend_bwd_grad<true, 16>), dim3(grid), dim3(64), 0, s, a);
  return hipGetLastError();
}

struct F3 {
  float x, y, z;
};
SR_DEV F3 f3(float x, float y, float z) { return F3{x, y, z}; }
SR_DEV F3 operator+(F3 a, F3 b) { return f3(a.x + b.x, a.y + b.y, a.z + b.z); }
SR_DEV F3 operator*(float s, F3 a) { return f3(s * a.x, s * a.y, s * a.z); }
SR_DEV F3 mul(F3 v, float s) { return f3(v.x * s, v.y * s, v.z * s); }
SR_DEV F3 had(F3 a, F3 b) { return f3(a.x * b.x, a.y * b.y, a.z * b.z); }
SR_DEV float dot3(F3 a, F3 b) { return (a.x * b.x + a.y * b.y) + a.z * b.z; }
SR_DEV float comp(F3 v, int i) { return i == 0 ? v.x : (i == 1 ? v.y : v.z); }

// SH backward, dsr/cuda_rasterizer/backward.cu:20-139 (same association):
// put(k, c) receives the basis value of each active coefficient k (dL/dsh_k
// = c dL/dRGB), S(k) gives coefficient k; returns dL/d(mean) through the
// view direction.
template <class Get, class Put>
SR_DEV F3 sh_backward_core(int deg, F3 dir_orig, F3 dL_dRGB, Get S, Put put) {
  const float len = sqrtf((dir_orig.x * dir_orig.x + dir_orig.y * dir_orig.y) + dir_orig.z * dir_orig.z);
  const F3 dir = f3(dir_orig.x / len, dir_orig.y / len, dir_orig.z / len);
  F3 dx = f3(0.0f, 0.0f, 0.0f), dy = dx, dz = dx;
  const float x = dir.x, y = dir.y, z = dir.z;
  put(0, kSH_C0);
  if (deg > 0) {
    put(1, -kSH_C1 * y);
    put(2, kSH_C1 * z);
    put(3, -kSH_C1 * x);
    dx = -kSH_C1 * S(3);
    dy = -kSH_C1 * S(1);
    dz = kSH_C1 * S(2);
    if (deg > 1) {
      const float xx = x * x, yy = y * y, zz = z * z, xy = x * y, yz = y * z, xz = x * z;
      put(4, kSH_C2_0 * xy);
      put(5, kSH_C2_1 * yz);
      put(6, kSH_C2_2 * ((2.0f * zz - xx) - yy));
      put(7, kSH_C2_3 * xz);
      put(8, kSH_C2_4 * (xx - yy));
      dx = dx + ((((kSH_C2_0 * y) * S(4) + ((kSH_C2_2 * 2.0f) * -x) * S(6)) + (kSH_C2_3 * z) * S(7)) +
                 ((kSH_C2_4 * 2.0f) * x) * S(8));
      dy = dy + ((((kSH_C2_0 * x) * S(4) + (kSH_C2_1 * z) * S(5)) + ((kSH_C2_2 * 2.0f) * -y) * S(6)) +
                 ((kSH_C2_4 * 2.0f) * -y) * S(8));
      dz = dz + (((kSH_C2_1 * y) * S(5) + (((kSH_C2_2 * 2.0f) * 2.0f) * z) * S(6)) + (kSH_C2_3 * x) * S(7));
      if (deg > 2) {
        put(9, (kSH_C3_0 * y) * (3.0f * xx - yy));
        put(10, (kSH_C3_1 * xy) * z);
        put(11, (kSH_C3_2 * y) * ((4.0f * zz - xx) - yy));
        put(12, (kSH_C3_3 * z) * ((2.0f * zz - 3.0f * xx) - 3.0f * yy));
        put(13, (kSH_C3_4 * x) * ((4.0f * zz - xx) - yy));
        put(14, (kSH_C3_5 * z) * (xx - yy));
        put(15, (kSH_C3_6 * x) * (xx - 3.0f * yy));
        F3 ax = mul(mul(mul(kSH_C3_0 * S(9), 3.0f), 2.0f), xy);
        ax = ax + mul(kSH_C3_1 * S(10), yz);
        ax = ax + mul(mul(kSH_C3_2 * S(11), -2.0f), xy);
        ax = ax + mul(mul(mul(kSH_C3_3 * S(12), -3.0f), 2.0f), xz);
        ax = ax + mul(kSH_C3_4 * S(13), ((-3.0f * xx + 4.0f * zz) - yy));
        ax = ax + mul(mul(kSH_C3_5 * S(14), 2.0f), xz);
        ax = ax + mul(mul(kSH_C3_6 * S(15), 3.0f), (xx - yy));
        F3 ay = mul(mul(kSH_C3_0 * S(9), 3.0f), (xx - yy));
        ay = ay + mul(kSH_C3_1 * S(10), xz);
        ay = ay + mul(kSH_C3_2 * S(11), ((-3.0f * yy + 4.0f * zz) - xx));
        ay = ay + mul(mul(mul(kSH_C3_3 * S(12), -3.0f), 2.0f), yz);
        ay = ay + mul(mul(kSH_C3_4 * S(13), -2.0f), xy);
        ay = ay + mul(mul(kSH_C3_5 * S(14), -2.0f), yz);
        ay = ay + mul(mul(mul(kSH_C3_6 * S(15), -3.0f), 2.0f), xy);
        F3 az = mul(kSH_C3_1 * S(10), xy);
        az = az + mul(mul(mul(kSH_C3_2 * S(11), 4.0f), 2.0f), yz);
        az = az + mul(mul(kSH_C3_3 * S(12), 3.0f), ((2.0f * zz - xx) - yy));
        az = az + mul(mul(mul(kSH_C3_4 * S(13), 4.0f), 2.0f), xz);
        az = az + mul(kSH_C3_5 * S(14), (xx - yy));
        dx = dx + ax;
        dy = dy + ay;
        dz = dz + az;
      }
    }
  }
  const F3 dL_ddir = f3(dot3(dx, dL_dRGB), dot3(dy, dL_dRGB), dot3(dz, dL_dRGB));
  // dnormvdv, auxiliary.h:128-138
  const F3 v = dir_orig, dv = dL_ddir;
  const float sum2 = (v.x * v.x + v.y * v.y) + v.z * v.z;
  const float invsum32 = 1.0f / sqrtf((sum2 * sum2) * sum2);
  F3 r;
  r.x = ((((sum2 - v.x * v.x) * dv.x) - (v.y * v.x) * dv.y) - (v.z * v.x) * dv.z) * invsum32;
  r.y = (((-v.x * v.y) * dv.x + (sum2 - v.y * v.y) * dv.y) - (v.z * v.y) * dv.z) * invsum32;
  r.z = (((-v.x * v.z) * dv.x - (v.y * v.z) * dv.y) + (sum2 - v.z * v.z) * dv.z) * invsum32;
  return r;
}

// SH backward of one view against memory: stores c dL_dRGB (and zeros for the
// inactive coefficients).  With 16 coefficients and 16-byte aligned rows the surfel's 48 coefficients are read and its 48
// gradients written as twelve float4 each (same values, same order of
// operations as the scalar form).
// With kRow srow is the surfel's row staged in LDS by its wave, read instead of
// sh and overwritten with the gradients (the caller stores the wave's rows)
// instead of dsh.
template <bool kRow>
SR_DEV F3 sh_backward(int deg, int M, const float* sh, F3 dir_orig, F3 dL_dRGB, float* dsh, float4* srow) {
  const int nact = (deg + 1) * (deg + 1);
  if (M == 16 && ((reinterpret_cast<uintptr_t>(sh) | reinterpret_cast<uintptr_t>(dsh)) & 15u) == 0u) {
    float shv[48];
    const float4* s4 = reinterpret_cast<const float4*>(sh);
#pragma unroll
    for (int i = 0; i < 12; ++i) {
      const float4 t = kRow ? srow[i] : s4[i];
      shv[4 * i] = t.x;
      shv[4 * i + 1] = t.y;
      shv[4 * i + 2] = t.z;
      shv[4 * i + 3] = t.w;
    }
    float cv[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) cv[k] = 0.0f;
    const F3 r = sh_backward_core(
        deg, dir_orig, dL_dRGB, [&](int k) { return f3(shv[3 * k], shv[3 * k + 1], shv[3 * k + 2]); },
        [&](int k, float c) { cv[k] = c; });
    float4* d4 = reinterpret_cast<float4*>(dsh);
#pragma unroll
    for (int i = 0; i < 12; ++i) {
      float v[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int j = 4 * i + t, k = j / 3;
        v[t] = k < nact ? cv[k] * comp(dL_dRGB, j % 3) : 0.0f;
      }
      (kRow ? srow : d4)[i] = make_float4(v[0], v[1], v[2], v[3]);
    }
    return r;
  }
  for (int k = nact; k < M; ++k) dsh[3 * k] = dsh[3 * k + 1] = dsh[3 * k + 2] = 0.0f;
  return sh_backward_core(
      deg, dir_orig, dL_dRGB, [&](int k) { return f3(sh[3 * k], sh[3 * k + 1], sh[3 * k + 2]); },
      [&](int k, float c) {
        dsh[3 * k] = c * dL_dRGB.x;
        dsh[3 * k + 1] = c * dL_dRGB.y;
        dsh[3 * k + 2] = c * dL_dRGB.z;
      });
}

// A record's colour gradient: none through a clamped channel.
SR_DEV F3 unclamped(const PreprocessBwdArgs& a, size_t r, F3 dRGB) {
  const uchar4 cl = reinterpret_cast<const uchar4*>(a.clamped)[r];
  if (cl.x) dRGB.x = 0.0f;
  if (cl.y) dRGB.y = 0.0f;
  if (cl.z) dRGB.z = 0.0f;
  return dRGB;
}

// SH backward of a surfel's only view: stores its dL_dsh row and returns the
// gradient of the mean through the view direction.
template <bool kRow>
SR_DEV F3 sh_grad(const PreprocessBwdArgs& a, int idx, size_t r, const float* campos, float m0, float m1, float m2,
                  F3 dRGB, float4* srow) {
  return sh_backward<kRow>(a.D, a.M, a.shs + (size_t)idx * a.M * 3, f3(m0 - campos[0], m1 - campos[1], m2 - campos[2]),
                           unclamped(a, r, dRGB), a.dL_dsh + (size_t)idx * a.M * 3, srow);
}

// Gradients of one surfel summed over the views that see it.
struct SurfelGrad {
  float m[3], sc[2], q[4];
};

// Record r's 18 partial gradients summed over its slots (one per instance
// and quadrant holding it, a contiguous run in instance order, quadrants in
// order): a fixed order, so the sums are the same on every run.  Four flags
// are in flight at a time, then the sums of kU slots they announce.
template <int kU>
SR_DEV void reduce_record(const PreprocessBwdArgs& a, size_t r, float (&gs)[18]) {
#pragma unroll
  for (int k = 0; k < 18; ++k) gs[k] = 0.0f;
  if (a.tiles[r] == 0 || a.part == nullptr || (a.counters[1] & kErrCapacity)) return;
  const uint2 rs = a.rslot[r];  // the record's slots: its instances in order, each one's quadrants in order
  const uint32_t s0 = rs.x, s1 = rs.x + rs.y;
  for (uint32_t s = s0; s < s1; s += 4) {
    uint8_t fl[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) fl[t] = a.part_nz[min(s + (uint32_t)t, s1 - 1u)];
#pragma unroll
    for (int t = 0; t < 4; ++t) fl[t] = s + (uint32_t)t < s1 ? fl[t] : 0;
#pragma unroll
    for (int u = 0; u < 4; u += kU) {
      V4 p[kU][5];
#pragma unroll
      for (int t = 0; t < kU; ++t) {
        if (fl[u + t] == 0) continue;
        const V4* src = reinterpret_cast<const V4*>(a.part + (size_t)(s + (uint32_t)(u + t)) * kPartStride);
#pragma unroll
        for (int k = 0; k < 5; ++k) p[t][k] = src[k];
      }
#pragma unroll
      for (int t = 0; t < kU; ++t)
#pragma unroll
        for (int k = 0; k < 18; ++k) gs[k] = fl[u + t] ? gs[k] + p[t][k / 4][k % 4] : gs[k];
    }
  }
}

// Backward preprocess of surfel idx in view v (record r),
// dsr/cuda_rasterizer/backward.cu:443-630, from the record's reduced blend
// gradients gs.  Adds the view's contributions to g and writes the record's
// outputs: dL_dtransMat (with the AABB-centre term for a precomputed T; may be
// null), dL_dmean2D (the densification statistic) and, for a single view,
// dL_dopacity, dL_dcolors and the dL_dsh row.  With several views (kMany) the
// colour gradients go to dL_dcolors for the SH pass when there are SHs.
template <bool kMany, bool kRow>
SR_DEV void preprocess_bwd_view(const PreprocessBwdArgs& a, int v, int idx, size_t r, SurfelGrad& g,
                                const float (&gs)[18], float4* srow) {
  const ViewInfo& vi = a.vs.v[v];
  const float tanx = vi.tanx, tany = vi.tany;
  const float focal_x = (float)vi.W / (2.0f * tanx);
  const float focal_y = (float)vi.H / (2.0f * tany);
  const int W = f2i((focal_x * tanx) * 2.0f);
  const int H = f2i((focal_y * tany) * 2.0f);
  const float* pm = a.pm + 16 * v;
  const float* vm = a.vm + 16 * v;
  const float* campos = a.campos + 3 * v;
  const float m0 = a.means3D[3 * idx], m1 = a.means3D[3 * idx + 1], m2 = a.means3D[3 * idx + 2];
  const bool precomp = a.tprec != nullptr;
  F3 T0, T1, T2, Rc0, Rc1;
  float qw = 0.0f, qx = 0.0f, qy = 0.0f, qz = 0.0f, scx = 0.0f, scy = 0.0f;
  float P4[3][4];
  if (precomp) {
    const float* t = a.tprec + 9 * (size_t)idx;
    T0 = f3(t[0], t[1], t[2]);
    T1 = f3(t[3], t[4], t[5]);
    T2 = f3(t[6], t[7], t[8]);
  } else {
    const float* q = a.rots + 4 * idx;
    const float q0 = q[0], q1 = q[1], q2 = q[2], q3 = q[3];
    const float n2 = ((q3 * q3 + q0 * q0) + q1 * q1) + q2 * q2;
    const float s = 1.0f / sqrtf(n2);
    qw = q0 * s;
    qx = q1 * s;
    qy = q2 * s;
    qz = q3 * s;
    const float w = qw, x = qx, y = qy, z = qz;
    Rc0 = f3(1.0f - 2.0f * (y * y + z * z), 2.0f * (x * y + w * z), 2.0f * (x * z - w * y));
    Rc1 = f3(2.0f * (x * y - w * z), 1.0f - 2.0f * (x * x + z * z), 2.0f * (y * z + w * x));
    scx = a.scales[2 * idx];
    scy = a.scales[2 * idx + 1];
    const F3 L0c = (1.0f * scx) * Rc0, L1c = (1.0f * scy) * Rc1;
    const float hw = (float)W / 2.0f, hw1 = (float)(W - 1) / 2.0f;
    const float hh = (float)H / 2.0f, hh1 = (float)(H - 1) / 2.0f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      P4[0][i] = pm[4 * i] * hw + pm[4 * i + 3] * hw1;
      P4[1][i] = pm[4 * i + 1] * hh + pm[4 * i + 3] * hh1;
      P4[2][i] = pm[4 * i + 3];
    }
    auto dotM = [&](const F3& u, float u4, int k) {
      return ((u.x * P4[k][0] + u.y * P4[k][1]) + u.z * P4[k][2]) + u4 * P4[k][3];
    };
    const F3 pc = f3(m0, m1, m2);
    T0 = f3(dotM(L0c, 0.0f, 0), dotM(L1c, 0.0f, 0), dotM(pc, 1.0f, 0));
    T1 = f3(dotM(L0c, 0.0f, 1), dotM(L1c, 0.0f, 1), dotM(pc, 1.0f, 1));
    T2 = f3(dotM(L0c, 0.0f, 2), dotM(L1c, 0.0f, 2), dotM(pc, 1.0f, 2));
  }
  F3 dT0 = f3(gs[0], gs[1], gs[2]), dT1 = f3(gs[3], gs[4], gs[5]), dT2 = f3(gs[6], gs[7], gs[8]);
  float* gm2 = a.dL_dmean2D + 3 * r;
  const float gmx = gs[9], gmy = gs[10];
  bool updated = false;
  if (gmx != 0.0f || gmy != 0.0f) {
    const F3 tv = f3(9.0f, 9.0f, -1.0f);
    const float d = (tv.x * (T2.x * T2.x) + tv.y * (T2.y * T2.y)) + tv.z * (T2.z * T2.z);
    const float invd = 1.0f / d;
    const F3 f = f3(tv.x * invd, tv.y * invd, tv.z * invd);
    const F3 dL_dT0 = had(gmx * f, T2);
    const F3 dL_dT1 = had(gmy * f, T2);
    F3 dL_dT3 = had(gmx * f, T0) + had(gmy * f, T1);
    const F3 dL_df = had(gmx * T0, T2) + had(gmy * T1, T2);
    const float dotdf = (dL_df.x * f.x + dL_df.y * f.y) + dL_df.z * f.z;
    const float dL_dd = (float)((double)dotdf * (-1.0 / (double)d));
    const F3 dd_dT3 = f3((tv.x * T2.x) * 2.0f, (tv.y * T2.y) * 2.0f, (tv.z * T2.z) * 2.0f);
    dL_dT3 = dL_dT3 + dL_dd * dd_dT3;
    dT0 = dT0 + dL_dT0;
    dT1 = dT1 + dL_dT1;
    dT2 = dT2 + dL_dT3;
    updated = precomp;
  }
  // dL_dtransMat: the blend's sums, with the AABB-centre term only for a
  // precomputed T
  const float gT2 = updated ? dT0.z : gs[2], gT5 = updated ? dT1.z : gs[5];
  if (a.dL_dtransMat != nullptr) {
    float* gT = a.dL_dtransMat + 9 * r;
    const float full[9] = {dT0.x, dT0.y, dT0.z, dT1.x, dT1.y, dT1.z, dT2.x, dT2.y, dT2.z};
#pragma unroll
    for (int k = 0; k < 9; ++k) gT[k] = updated ? full[k] : gs[k];
  }
  if (!kMany) a.dL_dopacity[r] = gs[14];
  if (!kMany || a.shs != nullptr) {
    a.dL_dcolors[3 * r] = gs[15];
    a.dL_dcolors[3 * r + 1] = gs[16];
    a.dL_dcolors[3 * r + 2] = gs[17];
  }
  if (!precomp) {
    float dM[3][3];
#pragma unroll
    for (int cc = 0; cc < 3; ++cc)
#pragma unroll
      for (int i = 0; i < 3; ++i)
        dM[cc][i] = (P4[0][i] * comp(dT0, cc) + P4[1][i] * comp(dT1, cc)) + P4[2][i] * comp(dT2, cc);
    const float gn[3] = {gs[11], gs[12], gs[13]};
    F3 dL_dtn = f3((vm[0] * gn[0] + vm[1] * gn[1]) + vm[2] * gn[2], (vm[4] * gn[0] + vm[5] * gn[1]) + vm[6] * gn[2],
                   (vm[8] * gn[0] + vm[9] * gn[1]) + vm[10] * gn[2]);
    // the camera-facing sign the forward chose (backward.cu:550-555 re-derives
    // it from p_view . normal, which the forward's FP32 test gives too; for
    // a surfel whose forward ran in FP64 the forward's decision is the one
    // its outputs used)
    const float mult = a.rec[(size_t)kRecQuads * r + 4].w > 0.0f ? 1.0f : -1.0f;
    dL_dtn = mult * dL_dtn;
    const F3 dRS0 = f3(dM[0][0], dM[0][1], dM[0][2]);
    const F3 dRS1 = f3(dM[1][0], dM[1][1], dM[1][2]);
    const F3 dR0 = f3(dRS0.x * scx, dRS0.y * scx, dRS0.z * scx);
    const F3 dR1 = f3(dRS1.x * scy, dRS1.y * scy, dRS1.z * scy);
    const F3 dR2 = dL_dtn;
    const float vR[3][3] = {{dR0.x, dR0.y, dR0.z}, {dR1.x, dR1.y, dR1.z}, {dR2.x, dR2.y, dR2.z}};
    const float w = qw, x = qx, y = qy, z = qz;
    g.q[0] += 2.0f * ((x * (vR[1][2] - vR[2][1]) + y * (vR[2][0] - vR[0][2])) + z * (vR[0][1] - vR[1][0]));
    g.q[1] += 2.0f * ((((-2.0f * x) * (vR[1][1] + vR[2][2]) + y * (vR[0][1] + vR[1][0])) + z * (vR[0][2] + vR[2][0])) +
                      w * (vR[1][2] - vR[2][1]));
    g.q[2] += 2.0f * (((x * (vR[0][1] + vR[1][0]) - (2.0f * y) * (vR[0][0] + vR[2][2])) + z * (vR[1][2] + vR[2][1])) +
                      w * (vR[2][0] - vR[0][2]));
    g.q[3] += 2.0f * (((x * (vR[0][2] + vR[2][0]) + y * (vR[1][2] + vR[2][1])) - (2.0f * z) * (vR[0][0] + vR[1][1])) +
                      w * (vR[0][1] - vR[1][0]));
    g.sc[0] += (dRS0.x * Rc0.x + dRS0.y * Rc0.y) + dRS0.z * Rc0.z;
    g.sc[1] += (dRS1.x * Rc1.x + dRS1.y * Rc1.y) + dRS1.z * Rc1.z;
    F3 dm3 = f3(dM[2][0], dM[2][1], dM[2][2]);
    if (!kMany && a.shs != nullptr)
      dm3 = dm3 + sh_grad<kRow>(a, idx, r, campos, m0, m1, m2, f3(gs[15], gs[16], gs[17]), srow);
    g.m[0] += dm3.x;
    g.m[1] += dm3.y;
    g.m[2] += dm3.z;
  } else if (!kMany && a.shs != nullptr) {
    const F3 dm3 = sh_grad<kRow>(a, idx, r, campos, m0, m1, m2, f3(gs[15], gs[16], gs[17]), srow);
    g.m[0] += dm3.x;
    g.m[1] += dm3.y;
    g.m[2] += dm3.z;
  }
  const float depth = a.rec[(size_t)kRecQuads * r + 2].x;  // Tw.z = transMat[8]
  gm2[0] = (float)(((double)(gT2 * depth) * 0.5) * (double)(float)W);
  gm2[1] = (float)(((double)(gT5 * depth) * 0.5) * (double)(float)H);
  gm2[2] = 0.0f;
}

// A surfel's outputs but dL_dsh: its records, and the sums over its views.
// Every per-surfel and per-record output is written exactly once (zeros for a
// record no view sees), so none of them needs clearing beforehand.  Returns
// whether some view saw the surfel.
template <bool kMany, bool kRow>
SR_DEV bool preprocess_bwd_surfel(const PreprocessBwdArgs& a, int idx, float4* srow) {
  SurfelGrad g{};
  bool any = false;
  float op = 0.0f, c0 = 0.0f, c1 = 0.0f, c2 = 0.0f;
  const int V = kMany ? a.vs.V : 1;
  for (int v = 0; v < V; ++v) {
    const size_t r = (size_t)v * a.P + idx;
    if (!(a.radii[r] > 0)) {
      if (a.dL_dtransMat != nullptr) {
#pragma unroll
        for (int k = 0; k < 9; ++k) a.dL_dtransMat[9 * r + k] = 0.0f;
      }
      a.dL_dmean2D[3 * r] = a.dL_dmean2D[3 * r + 1] = a.dL_dmean2D[3 * r + 2] = 0.0f;
      if (!kMany) {
        a.dL_dopacity[r] = 0.0f;
        a.dL_dcolors[3 * r] = a.dL_dcolors[3 * r + 1] = a.dL_dcolors[3 * r + 2] = 0.0f;
      }
      continue;
    }
    float gs[18];
    reduce_record<kMany ? 2 : 4>(a, r, gs);
    preprocess_bwd_view<kMany, kRow>(a, v, idx, r, g, gs, srow);
    any = true;
    op += gs[14];
    c0 += gs[15];
    c1 += gs[16];
    c2 += gs[17];
  }
  a.dL_drots[4 * idx] = g.q[0];
  a.dL_drots[4 * idx + 1] = g.q[1];
  a.dL_drots[4 * idx + 2] = g.q[2];
  a.dL_drots[4 * idx + 3] = g.q[3];
  a.dL_dscales[2 * idx] = g.sc[0];
  a.dL_dscales[2 * idx + 1] = g.sc[1];
  a.dL_dmean3D[3 * idx] = g.m[0];
  a.dL_dmean3D[3 * idx + 1] = g.m[1];
  a.dL_dmean3D[3 * idx + 2] = g.m[2];
  if (kMany) {
    a.dL_dopacity_out[idx] = op;
    a.dL_dcolors_out[3 * idx] = c0;
    a.dL_dcolors_out[3 * idx + 1] = c1;
    a.dL_dcolors_out[3 * idx + 2] = c2;
  }
  return any;
}

// Degree-3 SH in 16-byte aligned rows move through LDS: each wave loads its
// 64 surfels' rows (12 KB, contiguous) with coalesced loads and stores the
// gradient rows the same way, instead of each lane moving its 192-byte row in
// 16-byte pieces 192 bytes apart.
constexpr int kShRow = 12;  // float4 per degree-3 SH row
constexpr int kShPad = 13;  // its LDS stride where each view reads it, odd against bank conflicts
__host__ __device__ inline bool sh_rows(const PreprocessBwdArgs& a) {
  return a.shs != nullptr && a.M == 16 &&
         ((reinterpret_cast<uintptr_t>(a.shs) | reinterpret_cast<uintptr_t>(a.dL_dsh)) & 15u) == 0u;
}
// move(i, k) for the wave's rows from surfel w0 on: float4 i of their memory,
// k of the LDS rows kStride apart
template <int kStride, class Move>
SR_DEV void each_row_quad(int P, int w0, Move move) {
  const int lane = threadIdx.x & 63, n = min(64, P - w0) * kShRow;
#pragma unroll
  for (int t = 0; t < kShRow; ++t)
    if (t * 64 + lane < n) {
      const int i = t * 64 + lane, row = i / kShRow;
      move(i, row * kStride + (i - row * kShRow));
    }
}

// Runs surfel(idx, srow, rows) for the workgroup's surfels, one a thread: with
// rows, srow is the surfel's SH row staged in LDS, which it replaces by its
// dL_dsh row.
template <class Surfel>
SR_DEV void with_sh_rows(const PreprocessBwdArgs& a, Surfel surfel) {
  __shared__ float4 s_sh[256 * kShRow];
  const int idx = blockIdx.x * blockDim.x + threadIdx.x;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const bool rows = sh_rows(a);                        // uniform
  const int w0 = blockIdx.x * blockDim.x + wave * 64;  // the wave's first surfel
  float4* wrows = s_sh + wave * 64 * kShRow;
  float4* srow = wrows + lane * kShRow;
  if (rows) {
    const float4* src = reinterpret_cast<const float4*>(a.shs) + (size_t)w0 * kShRow;
    each_row_quad<kShRow>(a.P, w0, [&](int i, int k) { wrows[k] = src[i]; });
  }
  __syncthreads();
  if (idx < a.P) {
    const bool any = rows ? surfel(std::true_type{}, idx, srow) : surfel(std::false_type{}, idx, srow);
    if (!any && rows) {
      for (int k = 0; k < kShRow; ++k) srow[k] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    } else if (!any && a.shs != nullptr) {
      float* dsh = a.dL_dsh + (size_t)idx * a.M * 3;
      for (int k = 0; k < 3 * a.M; ++k) dsh[k] = 0.0f;
    }
  }
  if (rows) {
    __syncthreads();
    float4* dst = reinterpret_cast<float4*>(a.dL_dsh) + (size_t)w0 * kShRow;
    each_row_quad<kShRow>(a.P, w0, [&](int i, int k) { dst[i] = wrows[k]; });
  }
}

// Backward preprocess of a single view, one thread per surfel; three waves per
// SIMD, with the 48 KB of LDS three workgroups a CU.  Bound by the latencies in
// front of the sums as much as by memory: 300k surfels of degree 3 59 us (180
// MB, 3 TB/s), 65 with one slot's sums in flight.
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3, 8))) void k_preprocess_bwd(
    PreprocessBwdArgs a) {
  with_sh_rows(a, [&](auto row, int idx, float4* srow) {
    return preprocess_bwd_surfel<false, decltype(row)::value>(a, idx, srow);
  });
}

// Backward preprocess of several views but for the SHs: one thread per surfel,
// looping over the views.  A million surfels, 16 views: 0.91 ms and the SH pass
// 0.30, where one kernel that read and wrote the dL_dsh rows once a view, and
// 64 bytes of per-record gradients, took 3.06.
__global__ __launch_bounds__(256) void k_preprocess_bwd_views(PreprocessBwdArgs a) {
  const int idx = blockIdx.x * blockDim.x + threadIdx.x;
  if (idx < a.P) preprocess_bwd_surfel<true, false>(a, idx, nullptr);
}

// SH backward of several views, one thread per surfel: the dL_dsh row summed
// in registers over the views that see the surfel, and the mean's gradient
// through the view directions added to dL_dmean3D.
template <bool kRow>
__global__ __launch_bounds__(64) void k_sh_bwd_views(PreprocessBwdArgs a) {
  __shared__ float4 s_sh[kRow ? 64 * kShPad : 1];
  const int w0 = blockIdx.x * 64, lane = threadIdx.x, idx = w0 + lane;
  if (kRow) {
    const float4* src = reinterpret_cast<const float4*>(a.shs) + (size_t)w0 * kShRow;
    each_row_quad<kShPad>(a.P, w0, [&](int i, int k) { s_sh[k] = src[i]; });
    __syncthreads();
  }
  const bool in = idx < a.P;
  const float* row = kRow ? reinterpret_cast<const float*>(s_sh + lane * kShPad) : a.shs + (size_t)(in ? idx : 0) * a.M * 3;
  const int nact = (a.D + 1) * (a.D + 1);
  float acc[48];
#pragma unroll
  for (int k = 0; k < 48; ++k) acc[k] = 0.0f;
  F3 gm = f3(0.0f, 0.0f, 0.0f);
  const F3 m = in ? f3(a.means3D[3 * idx], a.means3D[3 * idx + 1], a.means3D[3 * idx + 2]) : gm;
  for (int v = 0; v < a.vs.V; ++v) {
    const size_t r = (size_t)v * a.P + idx;
    if (!in || !(a.radii[r] > 0)) continue;
    const F3 dRGB = unclamped(a, r, f3(a.dL_dcolors[3 * r], a.dL_dcolors[3 * r + 1], a.dL_dcolors[3 * r + 2]));
    const float* campos = a.campos + 3 * v;
    gm = gm + sh_backward_core(
                  a.D, f3(m.x - campos[0], m.y - campos[1], m.z - campos[2]), dRGB,
                  [&](int k) { return f3(row[3 * k], row[3 * k + 1], row[3 * k + 2]); },
                  [&](int k, float c) {
                    acc[3 * k] += c * dRGB.x;
                    acc[3 * k + 1] += c * dRGB.y;
                    acc[3 * k + 2] += c * dRGB.z;
                  });
  }
  if (in) {
    a.dL_dmean3D[3 * idx] += gm.x;
    a.dL_dmean3D[3 * idx + 1] += gm.y;
    a.dL_dmean3D[3 * idx + 2] += gm.z;
  }
  if (kRow) {
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kShRow; ++k)
      s_sh[lane * kShPad + k] = make_float4(acc[4 * k], acc[4 * k + 1], acc[4 * k + 2], acc[4 * k + 3]);
    __syncthreads();
    float4* dst = reinterpret_cast<float4*>(a.dL_dsh) + (size_t)w0 * kShRow;
    each_row_quad<kShPad>(a.P, w0, [&](int i, int k) { dst[i] = s_sh[k]; });
  } else if (in) {
    float* dsh = a.dL_dsh + (size_t)idx * a.M * 3;
#pragma unroll
    for (int k = 0; k < 16; ++k)
      if (k < nact) {
        dsh[3 * k] = acc[3 * k];
        dsh[3 * k + 1] = acc[3 * k + 1];
        dsh[3 * k + 2] = acc[3 * k + 2];
      }
    for (int k = 3 * nact; k < 3 * a.M; ++k) dsh[k] = 0.0f;
  }
}

hipError_t launch_preprocess_bwd(const PreprocessBwdArgs& a, hipStream_t s) {
  if (a.P == 0 || a.vs.V == 0) return hipSuccess;
  const dim3 grid((a.P + 255) / 256);
  if (a.vs.V == 1) {
    hipLaunchKernelGGL(k_preprocess_bwd, grid, dim3(256), 0, s, a);
    return hipGetLastError();
  }
  hipLaunchKernelGGL(k_preprocess_bwd_views, grid, dim3(256), 0, s, a);
  if (a.shs != nullptr) {
    const dim3 waves((a.P + 63) / 64);
    if (sh_rows(a)) hipLaunchKernelGGL(k_sh_bwd_views<true>, waves, dim3(64), 0, s, a);
    else hipLaunchKernelGGL(k_sh_bwd_views<false>, waves, dim3(64), 0, s, a);
  }
  return hipGetLastError();
}

// Backward preprocess of the _part variant (one view; dsp = submodules/
// diff-surfel-rasterization_part/cuda_rasterizer): per visible surfel the
// blend's partial gradients summed over its instances, then the AABB-centre
// adjoint added into dL_dtransMat for every visible surfel and the
// densification statistic (computeAABB, dsp/backward.cu:621-671), then the
// camera-space homography's adjoint (computeTransMat, :473-545) and the SH
// backward.  Every output is written (zeros for a culled surfel).
template <bool kRow>
SR_DEV bool part_preprocess_bwd_surfel(const PreprocessBwdArgs& a, int idx, float4* srow) {
  float* gT = a.dL_dtransMat + 9 * idx;
  float* gm2 = a.dL_dmean2D + 3 * idx;
  if (!(a.radii[idx] > 0)) {
    for (int k = 0; k < 9; ++k) gT[k] = 0.0f;
    for (int k = 0; k < 3; ++k) gm2[k] = a.dL_dmean3D[3 * idx + k] = a.dL_dcolors[3 * idx + k] = 0.0f;
    a.dL_dopacity[idx] = 0.0f;
    a.dL_dscales[2 * idx] = a.dL_dscales[2 * idx + 1] = 0.0f;
    for (int k = 0; k < 4; ++k) a.dL_drots[4 * idx + k] = 0.0f;
    return false;
  }
  float gs[18];
  reduce_record<4>(a, (size_t)idx, gs);
  const ViewInfo& vi = a.vs.v[0];
  const float tanx = vi.tanx, tany = vi.tany;
  const float fx = (float)vi.W / (2.0f * tanx), fy = (float)vi.H / (2.0f * tany);
  const float Wh = fx * tanx, Hh = fy * tany;  // "W", "H" of BACKWARD::preprocess (:685-686)
  const float4* rc = a.rec + (size_t)kRecQuads * idx;
  const float4 r0 = rc[0], r1 = rc[1], r2 = rc[2];
  const F3 T0 = f3(r0.x, r0.y, r0.z), T1 = f3(r0.w, r1.x, r1.y), T3 = f3(r1.z, r1.w, r2.x);
  F3 dT0 = f3(gs[0], gs[1], gs[2]), dT1 = f3(gs[3], gs[4], gs[5]), dT2 = f3(gs[6], gs[7], gs[8]);
  {
    const float gmx = gs[9], gmy = gs[10];
    const F3 tv = f3(1.0f, 1.0f, -1.0f);
    const float d = (tv.x * (T3.x * T3.x) + tv.y * (T3.y * T3.y)) + tv.z * (T3.z * T3.z);
    const float invd = 1.0f / d;
    const F3 f = f3(tv.x * invd, tv.y * invd, tv.z * invd);
    const F3 dL_dT0 = had(gmx * f, T3);
    const F3 dL_dT1 = had(gmy * f, T3);
    F3 dL_dT3 = had(gmx * f, T0) + had(gmy * f, T1);
    const F3 dL_df = had(gmx * T0, T3) + had(gmy * T1, T3);
    const float dotdf = (dL_df.x * f.x + dL_df.y * f.y) + dL_df.z * f.z;
    const float dL_dd = (float)((double)dotdf * (-1.0 / (double)d));
    const F3 dd_dT3 = f3((tv.x * T3.x) * 2.0f, (tv.y * T3.y) * 2.0f, (tv.z * T3.z) * 2.0f);
    dL_dT3 = dL_dT3 + dL_dd * dd_dT3;
    dT0 = dT0 + dL_dT0;
    dT1 = dT1 + dL_dT1;
    dT2 = dT2 + dL_dT3;
  }
  gT[0] = dT0.x; gT[1] = dT0.y; gT[2] = dT0.z;
  gT[3] = dT1.x; gT[4] = dT1.y; gT[5] = dT1.z;
  gT[6] = dT2.x; gT[7] = dT2.y; gT[8] = dT2.z;
  const float z = r2.x;
  gm2[0] = (dT0.z * z) * Wh;
  gm2[1] = (dT1.z * z) * Hh;
  gm2[2] = 0.0f;
  a.dL_dopacity[idx] = gs[14];
  a.dL_dcolors[3 * idx] = gs[15];
  a.dL_dcolors[3 * idx + 1] = gs[16];
  a.dL_dcolors[3 * idx + 2] = gs[17];
  const float m0 = a.means3D[3 * idx], m1 = a.means3D[3 * idx + 1], m2 = a.means3D[3 * idx + 2];
  F3 dm3 = f3(0.0f, 0.0f, 0.0f);
  if (a.tprec == nullptr) {
    const float* vm = a.vm;
    const float cx = fx * tanx, cy = fy * tany;  // intrins.zw of the backward (:596)
    const float* q = a.rots + 4 * idx;
    const float q0 = q[0], q1 = q[1], q2 = q[2], q3 = q[3];
    const float n2 = ((q3 * q3 + q0 * q0) + q1 * q1) + q2 * q2;
    const float s = 1.0f / sqrtf(n2);
    const float w = q0 * s, x = q1 * s, y = q2 * s, zq = q3 * s;
    const F3 Rc0 = f3(1.0f - 2.0f * (y * y + zq * zq), 2.0f * (x * y + w * zq), 2.0f * (x * zq - w * y));
    const F3 Rc1 = f3(2.0f * (x * y - w * zq), 1.0f - 2.0f * (x * x + zq * zq), 2.0f * (y * zq + w * x));
    const F3 Rc2 = f3(2.0f * (x * zq + w * y), 2.0f * (y * zq - w * x), 1.0f - 2.0f * (x * x + y * y));
    const float sx = a.scales[2 * idx], sy = a.scales[2 * idx + 1];
    auto Wt = [&](F3 v) {
      return f3((vm[0] * v.x + vm[1] * v.y) + vm[2] * v.z, (vm[4] * v.x + vm[5] * v.y) + vm[6] * v.z,
                (vm[8] * v.x + vm[9] * v.y) + vm[10] * v.z);
    };
    // dL_dM = (P^T dL_dT^T): column j = (fx dTu_j, fy dTv_j, (cx dTu_j + cy dTv_j) + dTw_j)
    const F3 dM0 = f3(fx * dT0.x, fy * dT1.x, (cx * dT0.x + cy * dT1.x) + dT2.x);
    const F3 dM1 = f3(fx * dT0.y, fy * dT1.y, (cx * dT0.y + cy * dT1.y) + dT2.y);
    const F3 dM2 = f3(fx * dT0.z, fy * dT1.z, (cx * dT0.z + cy * dT1.z) + dT2.z);
    const F3 dRS0 = Wt(dM0), dRS1 = Wt(dM1), dpw = Wt(dM2);
    F3 dL_dtn = Wt(f3(gs[11], gs[12], gs[13]));
    // DUAL_VISIABLE (:528-533): the sign from tn = W R[2] against p_view
    const F3 tn = f3((vm[0] * Rc2.x + vm[4] * Rc2.y) + vm[8] * Rc2.z, (vm[1] * Rc2.x + vm[5] * Rc2.y) + vm[9] * Rc2.z,
                     (vm[2] * Rc2.x + vm[6] * Rc2.y) + vm[10] * Rc2.z);
    const float pvx = ((vm[0] * m0 + vm[4] * m1) + vm[8] * m2) + vm[12];
    const float pvy = ((vm[1] * m0 + vm[5] * m1) + vm[9] * m2) + vm[13];
    const float pvz = ((vm[2] * m0 + vm[6] * m1) + vm[10] * m2) + vm[14];
    const float cosv = ((-tn.x * pvx) + (-tn.y * pvy)) + (-tn.z * pvz);
    dL_dtn = (cosv > 0.0f ? 1.0f : -1.0f) * dL_dtn;
    const F3 dR0 = f3(dRS0.x * sx, dRS0.y * sx, dRS0.z * sx);
    const F3 dR1 = f3(dRS1.x * sy, dRS1.y * sy, dRS1.z * sy);
    const float vR[3][3] = {{dR0.x, dR0.y, dR0.z}, {dR1.x, dR1.y, dR1.z}, {dL_dtn.x, dL_dtn.y, dL_dtn.z}};
    float* gq = a.dL_drots + 4 * idx;
    gq[0] = 2.0f * ((x * (vR[1][2] - vR[2][1]) + y * (vR[2][0] - vR[0][2])) + zq * (vR[0][1] - vR[1][0]));
    gq[1] = 2.0f * ((((-2.0f * x) * (vR[1][1] + vR[2][2]) + y * (vR[0][1] + vR[1][0])) + zq * (vR[0][2] + vR[2][0])) +
                    w * (vR[1][2] - vR[2][1]));
    gq[2] = 2.0f * (((x * (vR[0][1] + vR[1][0]) - (2.0f * y) * (vR[0][0] + vR[2][2])) + zq * (vR[1][2] + vR[2][1])) +
                    w * (vR[2][0] - vR[0][2]));
    gq[3] = 2.0f * (((x * (vR[0][2] + vR[2][0]) + y * (vR[1][2] + vR[2][1])) - (2.0f * zq) * (vR[0][0] + vR[1][1])) +
                    w * (vR[0][1] - vR[1][0]));
    a.dL_dscales[2 * idx] = (dRS0.x * Rc0.x + dRS0.y * Rc0.y) + dRS0.z * Rc0.z;
    a.dL_dscales[2 * idx + 1] = (dRS1.x * Rc1.x + dRS1.y * Rc1.y) + dRS1.z * Rc1.z;
    dm3 = dpw;
  } else {
    // the reference reads scales and rotations it was not given here; with
    // a precomputed T these gradients are zero
    a.dL_dscales[2 * idx] = a.dL_dscales[2 * idx + 1] = 0.0f;
    for (int k = 0; k < 4; ++k) a.dL_drots[4 * idx + k] = 0.0f;
  }
  if (a.shs != nullptr)
    dm3 = dm3 + sh_grad<kRow>(a, idx, (size_t)idx, a.campos, m0, m1, m2, f3(gs[15], gs[16], gs[17]), srow);
  a.dL_dmean3D[3 * idx] = dm3.x;
  a.dL_dmean3D[3 * idx + 1] = dm3.y;
  a.dL_dmean3D[3 * idx + 2] = dm3.z;
  return true;
}

__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3, 8))) void k_part_preprocess_bwd(
    PreprocessBwdArgs a) {
  with_sh_rows(a, [&](auto row, int idx, float4* srow) {
    return part_preprocess_bwd_surfel<decltype(row)::value>(a, idx, srow);
  });
}

// Semantic gradients: per (surfel, channel), the partials summed over the
// record's slots in the order of reduce_record, zeros for a culled surfel.  The
// channels of a surfel are neighbouring lanes, so a slot is one coalesced read:
// with this and the SH rows through LDS 79 us for 300k surfels and 8 channels,
// 92 in one kernel with a lane a surfel.
__global__ __launch_bounds__(256) void k_part_semantics_bwd(PreprocessBwdArgs a) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (size_t)a.P * a.S) return;
  const uint32_t idx = (uint32_t)(i / (uint32_t)a.S), ch = (uint32_t)(i % (uint32_t)a.S);
  float sum = 0.0f;
  if (a.radii[idx] > 0 && a.part != nullptr && a.tiles[idx] > 0 && !(a.counters[1] & kErrCapacity)) {
    const uint2 rs = a.rslot[idx];
    for (uint32_t s = rs.x, end = rs.x + rs.y; s < end; s += 4) {
      uint8_t fl[4];
      float v[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const uint32_t sl = min(s + (uint32_t)t, end - 1u);
        fl[t] = a.part_nz[sl];
        v[t] = a.sem_part[(size_t)sl * a.S + ch];  // unset, and not used, without the flag
      }
#pragma unroll
      for (int t = 0; t < 4; ++t)
        if (s + (uint32_t)t < end && fl[t] != 0) sum += v[t];
    }
  }
  a.dL_dsem[i] = sum;
}

hipError_t launch_part_preprocess_bwd(const PreprocessBwdArgs& a, hipStream_t s) {
  if (a.P == 0) return hipSuccess;
  hipLaunchKernelGGL(k_part_preprocess_bwd, dim3((a.P + 255) / 256), dim3(256), 0, s, a);
  if (a.S > 0) {
    const size_t n = (size_t)a.P * a.S;
    hipLaunchKernelGGL(k_part_semantics_bwd, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, a);
  }
  return hipGetLastError();
}

}  // namespace sr
