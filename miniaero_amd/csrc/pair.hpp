// pair.hpp -- kernels for meshes of cells with six faces each whose geometry is
// inside the bounds that find_pairs in solver.hip names (plates with cells over
// 30,000 times as long as high are outside).  Two forms: axial meshes, where a cell has
// two faces per axis, one on each side, and every area vector lies along an
// axis (box meshes, stretched or not), and skew meshes (kSkew: ramps, boxes
// whose area vectors carry rounding noise), where the slots stay in slot order
// and faces along no axis are a class of their own in the tiles' lists.
// Solvers and batches use them where every case qualifies with the same form;
// the served form does not (plan_run).
// Included by solver.hip inside its anonymous namespace.
//
// What bounds the general kernels on such meshes is the vector memory path of
// the CU, not HBM: its address unit takes 4 lanes a cycle (a wavefront's 8- or
// 16-byte loads cost 17 cycles whole and contiguous, up to 64 when every lane
// is in a line of its own; 4-byte loads 6 contiguous, about 20 otherwise), and
// with faces and slots in the reference's shuffled order most lanes are in
// lines of their own (2.1M-cell FP64 viscous plate: k_flux 739k L1 tag lookups
// in 785k busy cycles per CU, VALU 48%; batched FP32 shock tubes: VALU 64%,
// the data return busy 91%).  So the work is ordered by axis, and the arrays
// are laid out for 16-byte loads of consecutive cells:
//
//   gradients    axial: a cell's slots are (low, high) along x, y, z.  Only the two
//                faces of an axis contribute to that component of the
//                gradient, and two terms add to the same sum in either order,
//                so the reference's summation order is kept without following
//                it; a wavefront's loads of one slot are one shifted run of
//                cells.
//   flux tiles   a tile's faces are listed in chunks of 64 of one axis, so a
//                wavefront evaluates faces of one axis: the Roe and viscous
//                fluxes drop the terms of the two zero area components, and
//                both sides' loads are runs of cells.  The three axes' chunks
//                of the same 64 cells follow each other, so that the tile's
//                wavefronts read the same cells at the same time and share
//                them in L1.  Boundary faces are entries of the same lists
//                (their ghost state is built in registers), which removes the
//                boundary launch and its array.
//   arrays       five values per cell (primitives; face values per slot) are
//                two planes of 16-byte pairs and one of singles in FP64, one
//                plane of 16-byte quadruples and one of singles in FP32; the
//                20 values of a gradient record are planes of 16-byte vectors.
//                Planes are m.ns (nc rounded up to 64) long, so every
//                wavefront's access is aligned.
//
// Measured against the general kernels, microseconds per launch (k_grad,
// k_flux): FP64 viscous 256 x 128 x 64 plate 227 -> 155, 367 -> 300; FP32
// viscous 211 x 127 x 45 plate 99 -> 53, 139 -> 107; 48 batched FP32 shock
// tubes 320 -> 194, 384 -> 318; 1024-cell FP64 plate 10.5 -> 5.4, 14.5 -> 6.1;
// first-order 64 x 16 x 16 shock tube 14.1 with its boundary launch -> 5.2.
// Skew: FP64 321 x 157 x 11 ramp 126 -> 74, 120 -> 97; 4096-cell ramp 13.5 -> 7.4,
// 10.6 -> 5.8 (its boundary faces were in the gradient launch).
// At 2.1M cells the flux kernel is bound by HBM and L2: 1.39 GB fetched and 0.20
// written in 285 us, 5.5 TB/s, most of it records fetched again by the tiles
// around (96 tiles in flight per XCD against a 4 MB L2); the gradient kernel has
// its data return 86% busy.
//
// Every value the kernels keep is formed with the general kernels' operations
// in the same order, and the terms left out are +-0, so results are the same
// bits for finite values (only the sign of an exact zero can differ).

// Waves per SIMD the paired flux kernels are register-budgeted for: the FP64
// inviscid forms need a few more than the 128 registers that allow 4 unless
// told to fit.  Two for the FP64 viscous skew and first-order forms, which hold
// averaged gradients over a whole face frame or without the second order's
// ordered loads: at the 168 registers of three they spill 22 to 66 of them
// (k_flux us at 590k cells, general kernel / three waves / two: rotated box
// second order 123 / 183 / 130, first order 117 / 187 / 109; ramp 122 / 138 /
// 118, 116 / 144 / 96; plate first order 90 / 90 / 73).
template <bool kSkew, bool SO, class Visc, class T>
constexpr int kPairFluxWaves = sizeof(T) == 4 ? 5 : Visc::isViscous ? (kSkew || !SO ? 2 : 3) : 4;

constexpr int kSkewFace = 3;  // class of a tile's chunk of faces that are along no axis

constexpr int kPairMaxThreads = 384;  // flux workgroup: up to 6 wavefronts (see pair_threads)

// Plane k of a, byte offset off: a uniform base with a 32-bit lane offset
// (nc <= 2^28, so 16 c < 2^32), one address register instead of a 64-bit add
// per load.
template <class T>
__device__ __forceinline__ const T* plane(const T* a, int k, int n) {
  return a + (size_t)k * n;
}
template <class T>
__device__ __forceinline__ T at(const T* p, unsigned off) {
  return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(p) + off);
}
template <class T>
__device__ __forceinline__ void put(T* p, unsigned off, T v) {
  *reinterpret_cast<T*>(reinterpret_cast<char*>(p) + off) = v;
}

// Vector j (16 bytes: 2 doubles or 4 floats) of element i, planes of n.
template <class T>
constexpr int kVec = 16 / (int)sizeof(T);
__device__ __forceinline__ void get_vec(const double* a, int j, int n, unsigned i, double* v) {
  const double2 x = at(reinterpret_cast<const double2*>(a) + (size_t)j * n, i * 16u);
  v[0] = x.x;
  v[1] = x.y;
}
__device__ __forceinline__ void get_vec(const float* a, int j, int n, unsigned i, float* v) {
  const float4 x = at(reinterpret_cast<const float4*>(a) + (size_t)j * n, i * 16u);
  v[0] = x.x;
  v[1] = x.y;
  v[2] = x.z;
  v[3] = x.w;
}
__device__ __forceinline__ void put_vec(double* a, int j, int n, unsigned i, const double* v) {
  put(reinterpret_cast<double2*>(a) + (size_t)j * n, i * 16u, make_double2(v[0], v[1]));
}
__device__ __forceinline__ void put_vec(float* a, int j, int n, unsigned i, const float* v) {
  put(reinterpret_cast<float4*>(a) + (size_t)j * n, i * 16u, make_float4(v[0], v[1], v[2], v[3]));
}
// Five values of element i: whole vectors, then the last value's plane.
template <class T>
__device__ __forceinline__ void get_five(const T* a, int n, unsigned i, T* v) {
#pragma unroll
  for (int j = 0; j < 4 / kVec<T>; ++j) get_vec(a, j, n, i, v + j * kVec<T>);
  v[4] = at(a + (size_t)4 * n, i * (unsigned)sizeof(T));
}
template <class T>
__device__ __forceinline__ void put_five(T* a, int n, unsigned i, const T* v) {
#pragma unroll
  for (int j = 0; j < 4 / kVec<T>; ++j) put_vec(a, j, n, i, v + j * kVec<T>);
  put(a + (size_t)4 * n, i * (unsigned)sizeof(T), v[4]);
}

// Smaller and larger of two values, NaN ignored: one instruction (the
// builtins first quiet operands that could be signalling; ours come from
// arithmetic).
__device__ __forceinline__ double vmin(double a, double b) {
  double r;
  asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
__device__ __forceinline__ double vmax(double a, double b) {
  double r;
  asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
__device__ __forceinline__ float vmin(float a, float b) {
  float r;
  asm("v_min_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
__device__ __forceinline__ float vmax(float a, float b) {
  float r;
  asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}

// The range of a cell's stencil in which the quotients of grad_pair (div_by,
// quick_div) are exact: with |v| <= 2^100, density and temperature at least
// 2^-740 (FP32: 2^16 and 2^-60) and the mesh bounds find_pairs checks, no
// operand, product or remainder leaves the normal range, except where a
// velocity is neither 0 nor at least 2^-740 in magnitude (FP32: 2^-40; the sum
// of two such values is 0 or at least 2^-63, times an area of at least 2^-37).
// The front of a disturbance in a fluid at rest has such velocities for many
// steps, so they are told apart from the rest: only their own Green-Gauss
// quotients need the full division (limiter quotients are used for
// extrapolations above 1e-40 only).  NaN and infinities fail the first part: a
// cell with one has a NaN or zero temperature or an infinite density.  Cells
// are taken in one by one.  kDiv: the kernel divides by the volume (div_by);
// the FP32 record form multiplies by its reciprocal.
template <class T, bool kDiv>
struct TameCheck {
  static constexpr bool kD = sizeof(T) == 8;
  T tsum = T(0);
  int e = 0;  // smallest binary exponent of a velocity (0 for zero)
  __device__ __forceinline__ void take(const T* v) {
    tsum += v[4];
    if constexpr (kDiv) {
#pragma unroll
      for (int k = 1; k < 4; ++k) {
        if constexpr (kD) e = min(e, __builtin_amdgcn_frexp_exp(v[k]));
        else e = min(e, __builtin_amdgcn_frexp_expf(v[k]));
      }
    }
  }
  // mn, mx: the stencil's minima and maxima
  __device__ __forceinline__ bool bad(const T* mn, const T* mx) const {
    const T lo = T(kD ? 0x1p-740 : 0x1p-60), hi = T(kD ? 0x1p100 : 0x1p16);
    T big = vmax(mx[0], mx[4]);
#pragma unroll
    for (int k = 1; k < 4; ++k) big = vmax(big, vmax(mx[k], -mn[k]));
    return !(tsum <= T(8) * hi) || !(big <= hi) || !(mn[0] >= lo) || !(mn[4] >= lo);
  }
  __device__ __forceinline__ bool tiny() const { return kDiv && e < (kD ? -740 : -40); }
};

// Slot geometry of record i (m.stab): the outward area component along the
// face's axis and x_f - x_c, 4 values as whole vectors in planes of m.nsrec; on
// skew meshes the outward area vector and x_f - x_c, 6 values.  (Face geometry,
// m.ptab, planes of m.nfrec: the area component, x_f - x_left, x_f - x_right,
// 7 values; skew: the area vector in front, 9.)  Records are numbered in the
// order the kernels meet them, so the lanes of a load read consecutive records
// where they differ.
template <bool kSkew>
constexpr int kAreaVals = kSkew ? 3 : 1;
template <bool kSkew, class T>
constexpr int kSlotVecs = (kAreaVals<kSkew> + 3 + kVec<T> - 1) / kVec<T>;
template <bool kSkew, class T>
constexpr int kFaceVecs = (kAreaVals<kSkew> + 6 + kVec<T> - 1) / kVec<T>;
// vectors j0 to j1 - 1 of record i
template <class T>
__device__ __forceinline__ void slot_vecs(const DevMesh& m, unsigned i, int j0, int j1, T* q) {
#pragma unroll
  for (int j = j0; j < j1; ++j) get_vec(static_cast<const T*>(m.stab), j, m.nsrec, i, q + j * kVec<T>);
}

// A cell's neighbours (itself across a boundary face) and slot records: 3
// planes of int4, neighbours 0 to 5 then records 0 to 5 (skew meshes: with the
// cell's side of the face, 1 the right one, above kCellBits).
template <bool kSkew>
__device__ __forceinline__ void slot_ids(const DevMesh& m, const int* __restrict__ nbr, unsigned c, unsigned* nb,
                                         unsigned* ent) {
  const int4* p = reinterpret_cast<const int4*>(nbr);
  const int4 a = at(p, c * 16u), b = at(p + m.ns, c * 16u), d = at(p + (size_t)2 * m.ns, c * 16u);
  nb[0] = a.x, nb[1] = a.y, nb[2] = a.z, nb[3] = a.w, nb[4] = b.x, nb[5] = b.y;
  ent[0] = b.z, ent[1] = b.w, ent[2] = d.x, ent[3] = d.y, ent[4] = d.z, ent[5] = d.w;
  if constexpr (kSkew) {
#pragma unroll
    for (int s = 0; s < kMaxSlots; ++s) ent[s] = (unsigned)cell_of((int)ent[s]);
  }
}

// Value k of element i in five-value planes, and of a record in 20-value planes.
template <class T>
__device__ __forceinline__ size_t five_at(int k, int n, unsigned i) {
  return k == 4 ? (size_t)4 * n + i : ((size_t)(k / kVec<T>) * n + i) * kVec<T> + k % kVec<T>;
}
template <class T>
__device__ __forceinline__ size_t rec_at(int k, int n, unsigned i) {
  return ((size_t)(k / kVec<T>) * n + i) * kVec<T> + k % kVec<T>;
}

// Gradients of the velocities with full divisions, for a wavefront with tiny
// ones (TameCheck): replaces r[3] to r[11].
template <bool kSkew, class T>
__device__ __forceinline__ void tiny_gradients(const DevMesh& m, const int* __restrict__ nbr, const T* __restrict__ V,
                                               T vol, unsigned c, const T* vc, T* r) {
  unsigned ent[kMaxSlots], nb[kMaxSlots];
  slot_ids<kSkew>(m, nbr, c, nb, ent);
#pragma unroll
  for (int s = 0; s < kMaxSlots; ++s) {
    T vn[5];
    get_five(V, m.ns, nb[s], vn);
    T q[kSlotVecs<kSkew, T> * kVec<T>];
    slot_vecs(m, ent[s], 0, (kAreaVals<kSkew> + kVec<T> - 1) / kVec<T>, q);
#pragma unroll
    for (int k = 1; k < 4; ++k) {
      const T base = T(0.5) * (vc[k] + vn[k]);
#pragma unroll
      for (int d = 0; d < kAreaVals<kSkew>; ++d) {
        const T t = base * q[d];
        const T x = T(double(t) / double(vol));  // correctly rounded, as in grad_pair_slow
        T& g = r[3 * k + (kSkew ? d : s / 2)];
        g = s > (kSkew ? 0 : s / 2 * 2) ? g + x : x;
      }
    }
  }
}

// Gradient, stencil min/max and limiter of one cell whose wavefront has a
// stencil outside the tame range: one variable at a time (few registers: the
// fast path sets the kernel's occupancy), full divisions, the off-axis terms
// of the Green-Gauss sums as 0 * x.  Same values as grad_cell's general loop.
template <bool kSkew, bool SO, bool FV, class Limiter, class T>
__device__ void grad_pair_slow(const DevMesh& m, const int* __restrict__ nbr, const T* __restrict__ V,
                               T* __restrict__ rec, T* __restrict__ fv, unsigned c) {
  const int n = m.ns;
  auto id = [&](int k) { return (unsigned)nbr[((size_t)(k / 4) * n + c) * 4 + k % 4]; };  // see slot_ids
  auto record = [&](int s) { return kSkew ? (unsigned)cell_of((int)id(6 + s)) : id(6 + s); };
  const T vol = T(m.vol[c]);
  const T rvol = T(1) / vol;
#pragma unroll 1
  for (int k = 0; k < 5; ++k) {
    const T vc = V[five_at<T>(k, n, c)];
    T g[3] = {T(0), T(0), T(0)}, mn = T(1.0e300), mx = -T(1.0e300);
#pragma unroll 1
    for (int s = 0; s < kMaxSlots; ++s) {
      const T vn = V[five_at<T>(k, n, id(s))];
      T q[kSlotVecs<kSkew, T> * kVec<T>];
      slot_vecs(m, record(s), 0, (kAreaVals<kSkew> + kVec<T> - 1) / kVec<T>, q);
      // which side the cell is on: an axial mesh's low slots have it on their
      // right, and a skew mesh's order of the two decides only which of two
      // values one of which is NaN is kept, so it is looked up (a boundary
      // face's two values are the same)
      const bool left = kSkew ? !slot_of((int)id(6 + s)) : (s & 1) != 0;
      const T vl = left ? vc : vn, vr = left ? vn : vc;
      const T base = T(0.5) * (vl + vr);
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        const T gg = base * (kSkew ? q[d] : d == s / 2 ? q[0] : T(0));
        if constexpr (sizeof(T) == 8) g[d] += gg / vol;
        else if constexpr (FV) g[d] += T(double(gg) / double(vol));  // correctly rounded
        else g[d] += gg * rvol;
      }
      const T fmin = vr < vl ? vr : vl, fmax = vr > vl ? vr : vl;
      mn = ma::smin(mn, fmin);
      mx = ma::smax(mx, fmax);
    }
    T lim = SO ? T(1) : T(0);
    if constexpr (SO) {
#pragma unroll 1
      for (int s = 0; s < kMaxSlots; ++s) {
        T qs[kSlotVecs<kSkew, T> * kVec<T>];
        slot_vecs(m, record(s), 0, kSlotVecs<kSkew, T>, qs);
        const T* q = qs + kAreaVals<kSkew> - 1;
        const T dist = q[1] * q[1] + q[2] * q[2] + q[3] * q[3];
        const T du = q[1] * g[0] + q[2] * g[1] + q[3] * g[2];
        lim = ma::smin(lim, Limiter::limit(mx - vc, mn - vc, du, dist));
      }
    }
    if constexpr (FV) {
#pragma unroll 1
      for (int s = 0; s < kMaxSlots; ++s) {
        T qs[kSlotVecs<kSkew, T> * kVec<T>];
        slot_vecs(m, record(s), 0, kSlotVecs<kSkew, T>, qs);
        const T* q = qs + kAreaVals<kSkew> - 1;
        const T du = q[1] * g[0] + q[2] * g[1] + q[3] * g[2];
        fv[(size_t)5 * s * n + five_at<T>(k, n, c)] = vc + du * lim;
      }
    }
    if (!FV || rec) {
#pragma unroll
      for (int d = 0; d < 3; ++d) rec[rec_at<T>(3 * k + d, n, c)] = g[d];
      rec[rec_at<T>(15 + k, n, c)] = lim;
    }
  }
}

// Green-Gauss gradient, stencil min/max and limiter of one cell of a paired
// mesh.  rec: the gradient record (3k + d the gradient, 15 + k the limiter;
// null while stepping in the face-value scheme); FV: the extrapolated value at
// each face to fv, five values per slot.  About half the instructions of the
// general loop: 30 quotients by the volume at 3 operations from one
// reciprocal, no terms of the zero area components, one instruction per
// minimum and maximum (the minimum over the faces of min(v_L, v_R) is the
// minimum of the cell and its neighbours), short quotients in the limiter.
template <bool kSkew, bool SO, bool FV, class Limiter, class T>
__device__ __forceinline__ void grad_pair(const DevMesh& m, const int* __restrict__ nbr, const T* __restrict__ V,
                                          T* __restrict__ rec, T* __restrict__ fv, unsigned c) {
  const int n = m.ns;
  unsigned ent[kMaxSlots], nb[kMaxSlots];
  slot_ids<kSkew>(m, nbr, c, nb, ent);
  constexpr int A = kAreaVals<kSkew>, AV = (A + kVec<T> - 1) / kVec<T>, SV = kSlotVecs<kSkew, T>;
  T vc[5], geo[kMaxSlots][SV * kVec<T>], mn[5], mx[5];
  get_five(V, n, c, vc);
  const T vol = T(at(m.vol, c * 8u));
  // the reciprocal, correctly rounded (div_by needs that); the FP32 record
  // form multiplies by the 2.5-ulp one
  constexpr bool kMul = sizeof(T) == 4 && !FV;
  const T rvol = kMul ? T(1) / vol : T(1.0 / double(vol));
  T r[kRec];  // the record
  TameCheck<T, !kMul> tame;
  tame.take(vc);
#pragma unroll
  for (int k = 0; k < 5; ++k) mn[k] = mx[k] = vc[k];
#pragma unroll
  for (int s = 0; s < kMaxSlots; ++s) {
    T vn[5];
    slot_vecs(m, ent[s], 0, AV, geo[s]);
    get_five(V, n, nb[s], vn);
    tame.take(vn);
#pragma unroll
    for (int k = 0; k < 5; ++k) {
      mn[k] = vmin(mn[k], vn[k]);
      mx[k] = vmax(mx[k], vn[k]);
      const T base = T(0.5) * (vc[k] + vn[k]);
#pragma unroll
      for (int d = 0; d < A; ++d) {
        const T t = base * geo[s][d];
        const T q = kMul ? t * rvol : ma::div_by(t, vol, rvol);
        T& g = r[3 * k + (kSkew ? d : s / 2)];
        g = s > (kSkew ? 0 : s / 2 * 2) ? g + q : q;
      }
    }
  }
  if (__any(tame.bad(mn, mx))) {
    // through an opaque index: sharing loads with the fast path would keep
    // their registers over it (155 instead of 73 in the FP32 record form)
    asm volatile("" : "+v"(c));
    grad_pair_slow<kSkew, SO, FV, Limiter, T>(m, nbr, V, rec, fv, c);
    return;
  }
  if (!kMul && __any(tame.tiny())) {
    unsigned c2 = c;
    asm volatile("" : "+v"(c2));
    tiny_gradients<kSkew>(m, nbr, V, vol, c2, vc, r);
  }
  T dus[FV ? kMaxSlots : 1][5];
#pragma unroll
  for (int k = 0; k < 5; ++k) {
    r[15 + k] = SO ? T(1) : T(0);
    mx[k] = mx[k] - vc[k];
    mn[k] = mn[k] - vc[k];
  }
  if constexpr (SO) {
#pragma unroll
    for (int s = 0; s < kMaxSlots; ++s) {
      const T* q = geo[s] + A - 1;
      slot_vecs(m, ent[s], AV, SV, geo[s]);
      const T dist = q[1] * q[1] + q[2] * q[2] + q[3] * q[3];
#pragma unroll
      for (int k = 0; k < 5; ++k) {
        const T du = q[1] * r[3 * k] + q[2] * r[3 * k + 1] + q[3] * r[3 * k + 2];
        if (FV) dus[FV ? s : 0][k] = du;
        r[15 + k] = vmin(r[15 + k], Limiter::template limit<T, true>(mx[k], mn[k], du, dist));
      }
    }
  }
  if (!FV || rec) {
#pragma unroll
    for (int j = 0; j < kRec / kVec<T>; ++j) put_vec(rec, j, n, c, r + j * kVec<T>);
  }
  if constexpr (FV) {
#pragma unroll
    for (int s = 0; s < kMaxSlots; ++s) {
      T x[5];
#pragma unroll
      for (int k = 0; k < 5; ++k) x[k] = vc[k] + dus[FV ? s : 0][k] * r[15 + k];
      put_five(fv + (size_t)5 * s * n, n, c, x);
    }
  }
}

template <bool kSkew, bool SO, bool FV, class Limiter, class T>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(kGradWaves<SO, T>)))
void k_grad_pair(DevMesh m, const int* __restrict__ nbr, const T* __restrict__ V, T* __restrict__ rec,
                 T* __restrict__ fv, int per_xcd) {
  const int b = (blockIdx.x % kXcds) * per_xcd + blockIdx.x / kXcds;  // XCD-aware, see k_flux
  const int c = b * kBlock + threadIdx.x;
  if (c < m.nc) grad_pair<kSkew, SO, FV, Limiter, T>(m, nbr, V, rec, fv, (unsigned)c);
}

// State outside a boundary face of kind MA_BC_* whose area vector is p along
// axis D: the boundary policies' ghost states (Extrapolate_BC.h,
// Tangent_BC.h:86-102, Inflow_BC.h, NoSlip_BC.h:96-112), mirror_state with the
// terms of the zero components left out.
template <int D, class T>
__device__ __forceinline__ void ghost_state(int kind, const T* vc, T p, const Inflow* __restrict__ inflow, T* vr) {
  T un = vc[1 + D];
  if (kind == MA_BC_TANGENT || kind == MA_BC_NOSLIP) {
    const T an = fabs(p);
    const T ub = un * p / an;
    un = un - T(2) * ub * p / an;
  }
#pragma unroll
  for (int k = 0; k < 5; ++k) vr[k] = k == 1 + D ? un : vc[k];
  if (kind == MA_BC_INFLOW) {
    double vi[5];
    ma::primitives(inflow->U, vi);
#pragma unroll
    for (int k = 0; k < 5; ++k) vr[k] = T(vi[k]);
  }
}

// No-slip wall (NoSlip_BC.h:114-147): wall state and one-sided gradient along axis D.
template <int D, class T>
__device__ __forceinline__ void wall_gradient(const T* vc, T p, T winv, T* vf, T gf[5][3]) {
  const T s = copysign(T(1), p);
#pragma unroll
  for (int k = 0; k < 5; ++k) {
    vf[k] = k == 0 || k == 4 ? vc[k] : T(0);
#pragma unroll
    for (int d = 0; d < 3; ++d) gf[k][d] = d == D ? (vf[k] - vc[k]) * s * winv : T(0);
  }
}

// Flux of a face along axis D from its two (extrapolated) states; for a
// boundary face (kind > 0) vr comes in as the cell's state and is replaced by
// the ghost's.  gavg: face-averaged gradients (viscous; rows 1 to 4).
template <int D, bool SO, bool kWall, class Inv, class Visc, class T>
__device__ __forceinline__ void axis_flux(const T* vl, const T* vright, const T gavg[5][3], T p, int kind, T winv,
                                          const Inflow* __restrict__ inflow, const Inv& inv, const Visc& visc, T* F) {
  T vr[5];
#pragma unroll
  for (int k = 0; k < 5; ++k) vr[k] = vright[k];
  if (kind) ghost_state<D>(kind, vl, p, inflow, vr);
  // the viscous flux first: four values stay live over the Roe flux instead of
  // the averaged gradients
  T f[5];
  bool sub = false;
  if constexpr (Visc::isViscous) {
    T vf[5], gf[5][3];
#pragma unroll
    for (int k = 0; k < 5; ++k) {
      vf[k] = T(0.5) * (vl[k] + vr[k]);
#pragma unroll
      for (int d = 0; d < 3; ++d) gf[k][d] = gavg[k][d];
    }
    if (kind == MA_BC_NOSLIP) wall_gradient<D>(vl, p, winv, vf, gf);
    visc.template compute_flux_axis<D, T>(gf, vf, p, f);
    if constexpr (!SO) {
      // a NaN or infinite gradient makes every viscous component NaN, as the
      // general kernels' 0 * x terms do (second order: the extrapolated state
      // is NaN then, and with it the whole Roe flux)
      T y = T(0);
#pragma unroll
      for (int k = 1; k < 5; ++k)
#pragma unroll
        for (int d = 0; d < 3; ++d) y += T(0) * gf[k][d];
#pragma unroll
      for (int k = 1; k < 5; ++k) f[k] += y;
    }
    sub = !kind || kind == MA_BC_NOSLIP;
  } else if constexpr (kWall) {  // no-slip faces of an inviscid run: their viscous flux stays
    if (kind == MA_BC_NOSLIP) {
      const ma::NewtonianViscousFlux wallv{visc.prandtl};
      T vf[5], g[5][3];
      wall_gradient<D>(vl, p, winv, vf, g);
      wallv.template compute_flux_axis<D, T>(g, vf, p, f);
      sub = true;
    }
  }
  ma::inviscid_flux_axis<D>(inv, vl, vr, F, p);
  if constexpr (Visc::isViscous || kWall) {  // (component 0 of a viscous flux is 0)
    if (sub) {
#pragma unroll
      for (int k = 1; k < 5; ++k) F[k] -= f[k];
    }
  }
}

// Flux of a face of any area vector a (class kSkewFace of a tile's list): the
// general kernels' operations, with axis_flux's arguments.
template <bool kWall, class Inv, class Visc, class T>
__device__ __forceinline__ void skew_flux(const T* vl, const T* vright, const T gavg[5][3], const T* a, int kind,
                                          T winv, const Inflow* __restrict__ inflow, const Inv& inv,
                                          const Visc& visc, T* F) {
  const ma::FaceFrameT<T> fr = ma::frame_from_area_t<T>(a);
  T vr[5];
#pragma unroll
  for (int k = 0; k < 5; ++k) vr[k] = vright[k];
  if (kind == MA_BC_TANGENT || kind == MA_BC_NOSLIP) ma::mirror_state(vl, fr, vr);
  if (kind == MA_BC_INFLOW) {
    double vi[5];
    ma::primitives(inflow->U, vi);
#pragma unroll
    for (int k = 0; k < 5; ++k) vr[k] = T(vi[k]);
  }
  T f[5];
  bool sub = false;
  if constexpr (Visc::isViscous || kWall) {
    T vf[5], gf[5][3];
#pragma unroll
    for (int k = 0; k < 5; ++k) {
      vf[k] = T(0.5) * (vl[k] + vr[k]);
#pragma unroll
      for (int d = 0; d < 3; ++d) gf[k][d] = Visc::isViscous ? gavg[k][d] : T(0);
    }
    if (kind == MA_BC_NOSLIP) {
#pragma unroll
      for (int k = 0; k < 5; ++k) {
        vf[k] = k == 0 || k == 4 ? vl[k] : T(0);
#pragma unroll
        for (int d = 0; d < 3; ++d) gf[k][d] = (vf[k] - vl[k]) * fr.nu[d] * winv;
      }
    }
    sub = kind == MA_BC_NOSLIP || (Visc::isViscous && !kind);
    if constexpr (Visc::isViscous) visc.compute_flux(gf, vf, fr.n, f);
    else if (sub) ma::NewtonianViscousFlux{visc.prandtl}.compute_flux(gf, vf, fr.n, f);
  }
  ma::inviscid_flux(inv, vl, vr, F, fr);
  if constexpr (Visc::isViscous || kWall) {
    if (sub) {
#pragma unroll
      for (int k = 1; k < 5; ++k) F[k] -= f[k];  // (component 0 of a viscous flux is 0)
    }
  }
}

// Flux through one entry of a tile's face list along axis D (uniform over the
// wavefront): interior_flux for an internal face (cells L and Rr), the
// boundary policies for a boundary face (Rr < 0: ~Rr = boundary-face number
// << 2 | kind - 1; the cell's contribution is minus the returned flux, as on
// the left of an internal face).  kWall: the run may have no-slip faces, whose
// viscous flux is there in inviscid runs too.  Loads and extrapolation are
// common to the axes; only the flux arithmetic is per axis.  Skew meshes: D may
// be kSkewFace; Rr and gid carry the face's slots in the right and left cell
// above kCellBits.
template <bool kSkew, bool SO, bool kWall, class Inv, class Visc, class T>
__device__ __forceinline__ void pair_flux(const DevMesh& m, const T* __restrict__ V, const T* __restrict__ rec,
                                          const T* __restrict__ fv, const Inflow* __restrict__ inflow, int D,
                                          unsigned L, int Rr, int gid, const Inv& inv, const Visc& visc, T* F) {
  constexpr bool kVisc = Visc::isViscous;
  constexpr bool FV = SO && !kVisc, kRecon = SO && kVisc;
  constexpr int W = kVec<T>;
  // opaque, so that the plane bases are formed here on the scalar unit instead
  // of being kept over the face loop in more scalar registers than there are
  int n = m.ns;
  asm volatile("" : "+s"(n));
  const bool bnd = Rr < 0;
  const unsigned Rc = bnd ? L : (unsigned)(kSkew ? cell_of(Rr) : Rr);
  constexpr int A = kAreaVals<kSkew>;
  T vl[5], vr[5], geo[kFaceVecs<kSkew, T> * W];
  if constexpr (FV) {
    // the left cell's high face and the right cell's low face; a boundary
    // face's cell state
    const T* lo = fv + (size_t)(kSkew ? 5 * slot_of(bnd ? 0 : Rr) : 10 * D) * n;
    const T* hi = kSkew ? fv + (size_t)(5 * slot_of(gid)) * n : lo + (size_t)5 * n;
    if (bnd) {
      get_five(V, n, L, vl);
#pragma unroll
      for (int k = 0; k < 5; ++k) vr[k] = vl[k];
    } else {
      get_five(hi, n, L, vl);
      get_five(lo, n, Rc, vr);
    }
  } else {
    get_five(V, n, L, vl);
    get_five(V, n, Rc, vr);
  }
#pragma unroll
  for (int j = 0; j < (kRecon ? kFaceVecs<kSkew, T> : (A + W - 1) / W); ++j)
    get_vec(static_cast<const T*>(m.ptab), j, m.nfrec, (unsigned)(kSkew ? cell_of(gid) : gid), geo + j * W);
  const T* q = geo + A;  // displacements
  T gf[5][3];
  if constexpr (kVisc) {
    constexpr int j0 = kRecon ? 0 : 3 / W, j1 = kRecon ? kRec / W : (15 + W - 1) / W;  // vectors used
    T rl[kRec], rr[kRec];
#pragma unroll
    for (int j = j0; j < j1; ++j) {
      get_vec(rec, j, n, L, rl + j * W);
      get_vec(rec, j, n, Rc, rr + j * W);
    }
    if constexpr (kRecon) {
      // held here: the loads would otherwise sink into the branch below, one
      // round trip each
#pragma unroll
      for (int k = 0; k < 5; ++k) asm volatile("" : "+v"(rl[15 + k]), "+v"(rr[15 + k]));
#pragma unroll
      for (int d = 0; d < 3; ++d)
        asm volatile("" : "+v"(geo[A + d]), "+v"(geo[A + 3 + d]), "+v"(rl[d]), "+v"(rr[d]));
      if (!bnd) {
#pragma unroll
        for (int k = 0; k < 5; ++k) {
          const T tl = q[0] * rl[3 * k] + q[1] * rl[3 * k + 1] + q[2] * rl[3 * k + 2];
          const T tr = q[3] * rr[3 * k] + q[4] * rr[3 * k + 1] + q[5] * rr[3 * k + 2];
          vl[k] = vl[k] + tl * rl[15 + k];
          vr[k] = vr[k] + tr * rr[15 + k];
        }
      }
    }
#pragma unroll
    for (int k = 1; k < 5; ++k)
#pragma unroll
      for (int d = 0; d < 3; ++d) gf[k][d] = T(0.5) * (rl[3 * k + d] + rr[3 * k + d]);
  }
  const int kind = bnd ? (~Rr & 3) + 1 : 0;
  T winv = T(0);
  if (kWall && kind == MA_BC_NOSLIP) winv = T(m.fwall[m.nif + (~Rr >> 2)]);
  if (kSkew && D == kSkewFace) skew_flux<kWall>(vl, vr, gf, geo, kind, winv, inflow, inv, visc, F);
  else if (D == 0) axis_flux<0, SO, kWall>(vl, vr, gf, geo[0], kind, winv, inflow, inv, visc, F);
  else if (D == 1) axis_flux<1, SO, kWall>(vl, vr, gf, geo[kSkew ? 1 : 0], kind, winv, inflow, inv, visc, F);
  else axis_flux<2, SO, kWall>(vl, vr, gf, geo[kSkew ? 2 : 0], kind, winv, inflow, inv, visc, F);
}

// Another lane's value (byte address 4 * lane), through the LDS crossbar.
__device__ __forceinline__ float from_lane(int addr, float x) {
  return __int_as_float(__builtin_amdgcn_ds_bpermute(addr, __float_as_int(x)));
}
__device__ __forceinline__ double from_lane(int addr, double x) {
  return __hiloint2double(__builtin_amdgcn_ds_bpermute(addr, __double2hiint(x)),
                          __builtin_amdgcn_ds_bpermute(addr, __double2loint(x)));
}

// Fluxes through the three high faces of cell c of an axial mesh (viscous second
// order), list entries q0, q0 + 64 and q0 + 128: pair_flux with the cell's own
// values and gradient record loaded once instead of once per axis.
template <int D, bool kWall, class Inv, class Visc, class T>
__device__ __forceinline__ void own_face(const DevMesh& m, const T* __restrict__ V, const T* __restrict__ rec,
                                         const Inflow* __restrict__ inflow, const T* own, int mf, const T* rl, int Rr,
                                         int gid,
                                         unsigned c, unsigned c0, unsigned cells, const Inv& inv,
                                         const Visc& visc, T* F) {
  constexpr int W = kVec<T>;
  int n = m.ns;
  asm volatile("" : "+s"(n));  // see pair_flux
  const bool bnd = Rr < 0;
  const unsigned Rc = bnd ? c : (unsigned)Rr;
  T vl[5], vr[5], rr[kRec], geo[8];
#pragma unroll
  for (int k = 0; k < 5; ++k) vl[k] = own[k * mf];
#pragma unroll
  for (int j = 0; j < 8 / W; ++j)
    get_vec(static_cast<const T*>(m.ptab), j, m.nfrec, (unsigned)gid, geo + j * W);
  // a neighbour in the block (cells c0 to c0 + cells - 1) is another lane's own
  // cell; only the block's edge loads
  const bool near = Rc - c0 < cells;
  if (__any(near)) {
    const int addr = (int)(Rc - c0) * 4;
#pragma unroll
    for (int k = 0; k < 5; ++k) vr[k] = from_lane(addr, vl[k]);
#pragma unroll
    for (int k = 0; k < kRec; ++k) rr[k] = from_lane(addr, rl[k]);
  }
  if (!near) {
    get_five(V, n, Rc, vr);
#pragma unroll
    for (int j = 0; j < kRec / W; ++j) get_vec(rec, j, n, Rc, rr + j * W);
  }
#pragma unroll
  for (int k = 0; k < 5; ++k) asm volatile("" : "+v"(rr[15 + k]));
#pragma unroll
  for (int d = 0; d < 3; ++d) asm volatile("" : "+v"(geo[1 + d]), "+v"(geo[4 + d]), "+v"(rr[d]));
  if (!bnd) {
#pragma unroll
    for (int k = 0; k < 5; ++k) {
      const T tl = geo[1] * rl[3 * k] + geo[2] * rl[3 * k + 1] + geo[3] * rl[3 * k + 2];
      const T tr = geo[4] * rr[3 * k] + geo[5] * rr[3 * k + 1] + geo[6] * rr[3 * k + 2];
      vl[k] = vl[k] + tl * rl[15 + k];
      vr[k] = vr[k] + tr * rr[15 + k];
    }
  }
  T gf[5][3];
#pragma unroll
  for (int k = 1; k < 5; ++k)
#pragma unroll
    for (int d = 0; d < 3; ++d) gf[k][d] = T(0.5) * (rl[3 * k + d] + rr[3 * k + d]);
  const int kind = bnd ? (~Rr & 3) + 1 : 0;
  T winv = T(0);
  if (kWall && kind == MA_BC_NOSLIP) winv = T(m.fwall[m.nif + (~Rr >> 2)]);
  axis_flux<D, true, kWall>(vl, vr, gf, geo[0], kind, winv, inflow, inv, visc, F);
}

template <bool kWall, class Inv, class Visc, class T>
__device__ __forceinline__ void own_faces(const DevMesh& m, const TileMap& t, const T* __restrict__ V,
                                          const T* __restrict__ rec, const Inflow* __restrict__ inflow, T* lds,
                                          int list, int q0, unsigned c, unsigned c0, unsigned cells, const Inv& inv,
                                         const Visc& visc) {
  const int mf = t.max_faces;
  int R[3], g[3];
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    R[d] = t.lr[list + q0 + 64 * d].y;
    g[d] = t.fgid[list + q0 + 64 * d];
  }
  // The cell's values wait in the last face's place in LDS, its record in
  // registers: with both in registers the FP64 kernel spills 24 bytes a lane.
  T* own = lds + q0 + 128;
  T rl[kRec], F[5];
  {
    T vc[5];
    get_five(V, m.ns, c, vc);
#pragma unroll
    for (int k = 0; k < 5; ++k) own[k * mf] = vc[k];
  }
#pragma unroll
  for (int j = 0; j < kRec / kVec<T>; ++j) get_vec(rec, j, m.ns, c, rl + j * kVec<T>);
  auto keep = [&](int d) {
#pragma unroll
    for (int k = 0; k < 5; ++k) lds[k * mf + q0 + 64 * d] = F[k];
    asm volatile("" ::: "memory");  // the next axis' loads stay behind this one's arithmetic
  };
  asm volatile("" ::: "memory");  // (own is read back, not kept)
  own_face<0, kWall>(m, V, rec, inflow, own, mf, rl, R[0], g[0], c, c0, cells, inv, visc, F);
  keep(0);
  own_face<1, kWall>(m, V, rec, inflow, own, mf, rl, R[1], g[1], c, c0, cells, inv, visc, F);
  keep(1);
  own_face<2, kWall>(m, V, rec, inflow, own, mf, rl, R[2], g[2], c, c0, cells, inv, visc, F);
  keep(2);
}

// Second phase of a paired tile: every cell adds its face fluxes from LDS (5
// planes of t.max_faces) in the reference's order and takes the RK update
// (flux_tile's phase 2).
template <class T>
__device__ __forceinline__ void update_tile_pair(const DevMesh& m, const TileMap& t, int tile, int kcase, const T* lds,
                                                 const double* Uacc_in, double* Uacc_out, double* __restrict__ R,
                                                 const double* __restrict__ dt_dev, double beta,
                                                 const double* __restrict__ Un, T* __restrict__ Vnext,
                                                 double alpha_next, int last) {
  const int mf = t.max_faces;
  const int c = t.cptr[tile] + threadIdx.x;
  if (c >= t.cptr[tile + 1]) return;  // (the caller's barrier is reached by every thread)
  const int nc = m.nc;
  const unsigned off = (unsigned)c * 8u;
  // loaded before anything is stored, see flux_tile
  double uin[5], un[5];
  int ent[kMaxSlots];
#pragma unroll
  for (int s = 0; s < kMaxSlots; ++s) ent[s] = at(plane(t.slot16, s, nc), (unsigned)c * 2u);
#pragma unroll
  for (int k = 0; k < 5; ++k) uin[k] = at(Uacc_in + (size_t)k * nc, off);
  if (Vnext && !last) {
#pragma unroll
    for (int k = 0; k < 5; ++k) un[k] = at(plane(Un, k, nc), off);
  }
  const double dt = dt_dev[kcase];
  const double vol = at(m.vol, off);
  double acc[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int s = 0; s < kMaxSlots; ++s) {
    const T* x = lds + (ent[s] >> 1);
    const double sg = (ent[s] & 1) ? 1.0 : -1.0;  // sg * x is exact
#pragma unroll
    for (int k = 0; k < 5; ++k) acc[k] = __builtin_fma(sg, double(x[k * mf]), acc[k]);
  }
  const double dtv = dt / vol;
  double rr[5], unew[5];
#pragma unroll
  for (int k = 0; k < 5; ++k) {
    rr[k] = 0.0 + dtv * acc[k];
    unew[k] = uin[k] + beta * rr[k];
    put(Uacc_out + (size_t)k * nc, off, unew[k]);
  }
  if (Vnext) {
    double u[5], v[5];
    T w[5];
#pragma unroll
    for (int k = 0; k < 5; ++k) u[k] = (last ? unew[k] : un[k]) + alpha_next * rr[k];
    ma::primitives(u, v);
#pragma unroll
    for (int k = 0; k < 5; ++k) w[k] = T(v[k]);
    put_five(Vnext, m.ns, (unsigned)c, w);
  }
  if (last) {
#pragma unroll
    for (int k = 0; k < 5; ++k) put(R + (size_t)k * nc, off, rr[k]);
  }
}

// One tile of a paired mesh: flux_tile's two phases.  The face list is whole
// chunks of 64 entries of one axis each, x = left cell | axis << 28 (-1:
// padding, at the end of a chunk), y = right cell or boundary code;
// wavefront w takes chunks w, w + waves, ...  Slot entries are LDS index << 1 |
// side in the reference's summation order with the boundary faces last, in
// kind order.
template <bool kSkew, bool kOwn, bool SO, bool kWall, class Inv, class Visc, class T>
__device__ __forceinline__ void flux_tile_pair(const DevMesh& m, const TileMap& t, int tile, T* lds,
                                               const T* __restrict__ V, const T* __restrict__ rec,
                                               const T* __restrict__ fv, const Inflow* __restrict__ inflows,
                                               const double* Uacc_in, double* Uacc_out, double* __restrict__ R,
                                               const double* __restrict__ dt_dev, double beta, const Inv& inv,
                                               const Visc& visc, const double* __restrict__ Un,
                                               T* __restrict__ Vnext, double alpha_next, int last) {
  const int f0 = t.ptr[tile];
  const int n = t.ptr[tile + 1] - f0;
  const int mf = t.max_faces;
  const int kcase = t.tcase[tile];
  const Inflow* inflow = inflows + kcase;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), step = (int)blockDim.x;
  int first = wave * 64;
  if constexpr (kOwn) {
    const int c0 = t.cptr[tile], cells = t.cptr[tile + 1] - c0;
    for (int b = first; b < cells; b += step)
      if (b + lane < cells)
        own_faces<kWall>(m, t, V, rec, inflow, lds, f0, 3 * b + lane, (unsigned)(c0 + b + lane), (unsigned)(c0 + b),
                         (unsigned)min(64, cells - b), inv, visc);
    first += (cells + 63) / 64 * 192;
  }
  int2 lr = make_int2(-1, -1);
  int g = 0;
  if (first < n) {
    lr = t.lr[f0 + first + lane];
    g = t.fgid[f0 + first + lane];
  }
  for (int q = first; q < n; q += step) {
    const int2 c = lr;
    const int gc = g;
    if (q + step < n) {  // the next chunk's entries are fetched while this one is evaluated
      lr = t.lr[f0 + q + step + lane];
      g = t.fgid[f0 + q + step + lane];
    }
    const int D = __builtin_amdgcn_readfirstlane(c.x) >> kCellBits;  // (a chunk starts with a face)
    if (c.x < 0) continue;  // padding
    T F[5];
    pair_flux<kSkew, SO, kWall>(m, V, rec, fv, inflow, D, (unsigned)cell_of(c.x), c.y, gc, inv, visc, F);
#pragma unroll
    for (int k = 0; k < 5; ++k) lds[k * mf + q + lane] = F[k];
  }
  __syncthreads();
  update_tile_pair(m, t, tile, kcase, lds, Uacc_in, Uacc_out, R, dt_dev, beta, Un, Vnext, alpha_next, last);
}

// kOwn: the tile lists start with their cells' high faces (PairPlan::own), whose
// own side is loaded once for three faces.  The viscous second-order kernels
// load 25 values a side, and a tile's records alone (41 KB in FP64) exceed the
// 32 KB L1, so nearly every load goes to L2.  Keeping the own side, and taking a
// neighbour of the same 64-cell block from the lane that has it, leaves a load
// of the cell, one of its neighbour in the next block and the block's edges
// instead of 6 (L2 reads 31 -> 23 million a launch, k_flux of the 2.1M-cell FP64
// plate 338 -> 300 us, of the 1.2M-cell FP32 plate 117 -> 107), although a tile's
// low faces, which come after all blocks, load their own cell a second time: HBM
// fetches went from 1.11 to 1.39 GB.
// kWalk: fewer workgroups than tiles, each walking its XCD's run (see k_flux);
// otherwise one tile per workgroup, a form of its own because the walk's
// loop-carried values cost the FP64 viscous kernel spills and the FP64 inviscid
// one ten registers.
template <bool kSkew, bool kOwn, bool SO, bool kWall, bool kWalk, class Inv, class Visc, class T>
__global__ __launch_bounds__(kPairMaxThreads) __attribute__((amdgpu_waves_per_eu(kPairFluxWaves<kSkew, SO, Visc, T>)))
void k_flux_pair(DevMesh m, TileMap t, const T* __restrict__ V, const T* __restrict__ rec,
                 const Inflow* __restrict__ inflows, const double* Uacc_in, double* Uacc_out,
                 double* __restrict__ R, const double* __restrict__ dt_dev, double beta, Inv inv, Visc visc,
                 const double* __restrict__ Un, T* Vnext, double alpha_next, int last,
                 double* __restrict__ time_dev) {
  extern __shared__ __align__(16) unsigned char lds_raw[];
  T* lds = reinterpret_cast<T*>(lds_raw);  // 5 planes of t.max_faces
  const int xcd = blockIdx.x % kXcds;
  if constexpr (kWalk) {
    const int stride = gridDim.x / kXcds;
    for (int j = blockIdx.x / kXcds; j < t.per_xcd; j += stride) {
      const int tile = xcd * t.per_xcd + j;
      if (tile >= t.ntiles) break;  // uniform over the workgroup
      flux_tile_pair<kSkew, kOwn, SO, kWall, Inv, Visc, T>(m, t, tile, lds, V, rec, rec, inflows, Uacc_in, Uacc_out, R, dt_dev,
                                              beta, inv, visc, Un, Vnext, alpha_next, last);
      advance_time(t, tile, dt_dev, time_dev);
      __syncthreads();  // the LDS is reused by the next tile
    }
  } else {
    const int tile = xcd * t.per_xcd + blockIdx.x / kXcds;
    if (tile >= t.ntiles) return;  // uniform over the workgroup
    flux_tile_pair<kSkew, kOwn, SO, kWall, Inv, Visc, T>(m, t, tile, lds, V, rec, rec, inflows, Uacc_in, Uacc_out, R, dt_dev,
                                            beta, inv, visc, Un, Vnext, alpha_next, last);
    advance_time(t, tile, dt_dev, time_dev);
  }
}
