// kernels.hpp -- gfx950 kernels of the D3Q27 stepper (templates).
//
// Each translation unit includes this header and instantiates the launchers
// for its storage types; step_fp64.hip is compiled with -ffp-contract=off so
// the FP64 path reproduces the reference CPU arithmetic exactly, step_fp32.hip
// (FP32 and scaled-FP16 storage) lets the compiler contract to FMA.
#pragma once

#include "collision.hpp"
#include "../../include/vfx.h"

#include <hip/hip_runtime.h>
#include <cstdint>
#include <cstring>

namespace vfx {

// ------------------------------------------------------------- storage ----
// Population storage S with arithmetic type T.  _Float16 holds
// h_d = (f_d - w_d) * scale / w_d; the per-weight-class factors are kernel
// arguments (ld[c] = w_c / scale, st[c] = scale / w_c).
// Element i of a plane is addressed as plane base (wave-uniform, scalar
// registers) plus a 32-bit byte offset, so the loads and stores use the
// scalar-base + 32-bit-offset form and no 64-bit address arithmetic per lane.
// The host guarantees n_nodes * sizeof(S) < 2^32.
template <typename S> __device__ __forceinline__ const S& elem(const S* p, uint32_t i)
{
    return *(const S*)((const char*)p + i * (uint32_t)sizeof(S));
}
template <typename S> __device__ __forceinline__ S& elem(S* p, uint32_t i)
{
    return *(S*)((char*)p + i * (uint32_t)sizeof(S));
}
template <typename S, typename T> struct Storage;
template <> struct Storage<double, double> {
    static __device__ __forceinline__ double ld(const double* p, uint32_t i, float, float = 0.f) { return elem(p, i); }
    static __device__ __forceinline__ void st(double* p, uint32_t i, double v, float, float = 0.f) { elem(p, i) = v; }
    static __device__ __forceinline__ double enc(double v, float) { return v; }
    static __device__ __forceinline__ double dec(double h, float) { return h; }
};
template <> struct Storage<float, float> {
    static __device__ __forceinline__ float ld(const float* p, uint32_t i, float, float = 0.f) { return elem(p, i); }
    static __device__ __forceinline__ void st(float* p, uint32_t i, float v, float, float = 0.f) { elem(p, i) = v; }
    static __device__ __forceinline__ float enc(float v, float) { return v; }
    static __device__ __forceinline__ float dec(float h, float) { return h; }
};
// sh: offset of the stored deviation (the reference-velocity equilibrium, in
// f - w units); st takes ss = -sh * s, so both are one mixed-precision FMA
template <> struct Storage<_Float16, float> {
    // the stored half of v and the value a load gives back (one expression
    // each, shared by the memory accesses and the fused boundary conditions);
    // explicit FMAs: a contractible multiply-add would be fused in one kernel
    // and rounded twice in another, depending on the surrounding code
    static __device__ __forceinline__ _Float16 enc2(float v, float s, float ss)
    {
        return (_Float16)__builtin_fmaf(v, s, ss);
    }
    static __device__ __forceinline__ float dec2(_Float16 h, float s, float sh) { return __builtin_fmaf((float)h, s, sh); }
    static __device__ __forceinline__ float ld(const _Float16* p, uint32_t i, float s, float sh = 0.f)
    {
        return dec2(elem(p, i), s, sh);
    }
    static __device__ __forceinline__ void st(_Float16* p, uint32_t i, float v, float s, float ss = 0.f)
    {
        elem(p, i) = enc2(v, s, ss);
    }
    static __device__ __forceinline__ _Float16 enc(float v, float s) { return (_Float16)(v * s); }
    static __device__ __forceinline__ float dec(_Float16 h, float s) { return (float)h * s; }
};
// Raw buffer stores of one element type: descriptor = base address and size
// in bytes (dword 3 = 0x00020000, the gfx9-family raw-buffer format), VGPR
// byte offset + SGPR byte offset.  Used where a lane chooses between planes:
// the lane offset stays one 32-bit VGPR and the plane offset an SGPR.
typedef unsigned int vfx_u32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_rsrc(void* p, uint32_t bytes)
{
    return __builtin_amdgcn_make_buffer_rsrc(p, (short)0, (int)bytes, 0x00020000);
}
template <typename S> struct Buf;
template <> struct Buf<double> {
    static __device__ __forceinline__ void st(__amdgpu_buffer_rsrc_t r, uint32_t vo, uint32_t so, double v)
    {
        __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(vfx_u32x2, v), r, vo, so, 0);
    }
};
template <> struct Buf<float> {
    static __device__ __forceinline__ void st(__amdgpu_buffer_rsrc_t r, uint32_t vo, uint32_t so, float v)
    {
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned int, v), r, vo, so, 0);
    }
};
template <> struct Buf<_Float16> {
    static __device__ __forceinline__ void st(__amdgpu_buffer_rsrc_t r, uint32_t vo, uint32_t so, _Float16 v)
    {
        __builtin_amdgcn_raw_buffer_store_b16(__builtin_bit_cast(unsigned short, v), r, vo, so, 0);
    }
};

template <typename S> struct Compute { using T = float; };
template <> struct Compute<double> { using T = double; };

// Exact unsigned division by a run-time invariant d (Granlund & Montgomery,
// "Division by invariant integers using multiplication", PLDI 1994, fig. 4.1):
// l = ceil(log2 d), m = floor(2^32 (2^l - d) / d) + 1,
// q = (t + ((n - t) >> 1)) >> (l - 1) with t = mulhi(m, n); d = 1 is passed
// through.
struct FastDiv {
    uint32_t d, m, l;
};
inline FastDiv make_fastdiv(uint32_t d)
{
    FastDiv f{d, 0, 0};
    if (d <= 1) return f;
    uint32_t l = 0;
    while ((1ull << l) < d) ++l;
    f.l = l;
    f.m = (uint32_t)((((1ull << l) - d) << 32) / d + 1);
    return f;
}
__device__ __forceinline__ uint32_t fastdiv(uint32_t n, const FastDiv& f)
{
    if (f.d <= 1) return n;
    const uint32_t t = __umulhi(f.m, n);
    return (t + ((n - t) >> 1)) >> (f.l - 1);
}

// Device view of a vfx_lattice.
struct Lat {
    void* f;
    uint64_t N;
    uint32_t nx, ny, nz;  // direct addressing
    FastDiv div_x, div_y; // division by nx, ny
    const uint32_t* solid;
    const uint32_t* nbx;
    const uint32_t* nby;
    const uint32_t* nbz;
    const uint32_t* fluid;
    uint32_t nfluid;
    const uint32_t* types; // sparse: typeOfGridNode (nodes not GEO_SOLID/GEO_VOID collide), or NULL
    float ld[4], st[4];
    float sh[27], ss[27]; // FP16 reference-velocity offsets per direction (0 otherwise)
    void* rho;
    void* vx;
    void* vy;
    void* vz;
    int32_t write_macro;
    void* nut;             // turbulent viscosity per node (T), eddy-viscosity models
    const uint32_t* nbinv; // sparse: the node in -x-y-z (AMD model)
    void* bf[3];           // per-node body force (T), ApplyBodyForce
    double gforce[3];      // global force, unscaled
    double force_factor;
    uint32_t xrun_lg;      // 1 + log2 of the step's XCD tile run (0: built-in, step_run or xcd_run)
    uint32_t tile;         // nodes per workgroup of the direct step (0: built-in)
    const uint4* rgroups;  // sparse: per 64 work items {base node, y stride, z stride, regular}, or NULL
};

template <typename S> __device__ __forceinline__ S* plane(const Lat& L, int p) { return (S*)L.f + (uint64_t)p * L.N; }

__device__ __forceinline__ bool is_solid(const Lat& L, uint32_t k)
{
    return L.solid != nullptr && ((L.solid[k >> 5] >> (k & 31u)) & 1u);
}

// VirtualFluids node types (src/gpu/core/Calculation/Calculation.h:43-45)
constexpr uint32_t kGeoSolid = 15, kGeoVoid = 16, kGeoFluid = 19;

// sparse layout: the node of work item i (the i-th fluid node, or node i when
// typeOfGridNode selects), false if it does not collide
__device__ __forceinline__ bool sparse_node(const Lat& L, uint64_t i, uint32_t& k)
{
    if (L.types) {
        if (i >= L.N) return false;
        k = (uint32_t)i;
        const uint32_t t = L.types[k];
        return t != kGeoSolid && t != kGeoVoid;
    }
    if (i >= L.nfluid) return false;
    k = L.fluid[i];
    return k < L.N;
}
// work items of a node loop
__host__ __device__ inline uint64_t node_items(const Lat& L, int direct)
{
    return direct || L.types ? L.N : L.nfluid;
}

// The eight nodes a node's populations live on under the esoteric twist:
// kk[b], bit0 = +x, bit1 = +y, bit2 = +z (VirtualFluids ListIndices,
// KernelUtilities.h:221-245).
// interior node (no index wraps): one 24-bit multiply-add chain, then adds
// of wave-uniform strides
__device__ __forceinline__ void nbrs_interior(const Lat& L, uint32_t x, uint32_t y, uint32_t z, uint32_t (&kk)[8])
{
    const uint32_t sy = L.nx, sz = L.nx * L.ny;
    kk[0] = __umul24(__umul24(z, L.ny) + y, L.nx) + x;
    kk[1] = kk[0] + 1;
    kk[2] = kk[0] + sy;
    kk[3] = kk[2] + 1;
    kk[4] = kk[0] + sz;
    kk[5] = kk[4] + 1;
    kk[6] = kk[4] + sy;
    kk[7] = kk[6] + 1;
}
// node k of the box: its coordinates by two multiply-high divisions, the
// others by adds of one x, y and z step (1, nx, nx ny, or back across the box)
__device__ __forceinline__ void nbrs_direct(const Lat& L, uint32_t k, uint32_t (&kk)[8])
{
    const uint32_t r = fastdiv(k, L.div_x), z = fastdiv(r, L.div_y);
    const uint32_t sz = L.nx * L.ny;
    const uint32_t dx = k - r * L.nx + 1u == L.nx ? 1u - L.nx : 1u;
    const uint32_t dy = r - z * L.ny + 1u == L.ny ? L.nx - sz : L.nx;
    const uint32_t dz = z + 1u == L.nz ? sz - (uint32_t)L.N : sz;
    kk[0] = k;
    kk[1] = k + dx;
    kk[2] = k + dy;
    kk[3] = kk[1] + dy;
    kk[4] = k + dz;
    kk[5] = kk[1] + dz;
    kk[6] = kk[2] + dz;
    kk[7] = kk[3] + dz;
}
__device__ __forceinline__ void nbrs_sparse(const Lat& L, uint32_t k, uint32_t (&kk)[8])
{
    kk[0] = k;
    kk[1] = L.nbx[k];
    kk[2] = L.nby[k];
    kk[4] = L.nbz[k];
    kk[3] = L.nby[kk[1]];
    kk[5] = L.nbz[kk[1]];
    kk[6] = L.nbz[kk[2]];
    kk[7] = L.nbz[kk[3]];
}

// A wave-uniform float held in a VGPR.  FP16 loads and stores are one
// mixed-precision FMA with two lattice constants (scale and offset); a VALU
// instruction reads at most one SGPR, so the four per-class scales live in
// VGPRs (four moves per thread instead of one per access).
__device__ __forceinline__ float in_vgpr(float x)
{
    float r;
    asm("v_mov_b32 %0, %1" : "=v"(r) : "s"(x));
    return r;
}
// OUTER2: the collision hands over 2^c times the populations of weight class
// c (k17_fast<true>), so the store scales carry 2^-c (exact)
template <typename S, bool OUTER2 = false> struct Scales {
    float ld[4], st[4];
    __device__ __forceinline__ explicit Scales(const Lat& L)
    {
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            ld[c] = sizeof(S) == 2 ? in_vgpr(L.ld[c]) : L.ld[c];
            st[c] = sizeof(S) != 2 ? L.st[c] : (OUTER2 && c > 0) ? L.st[c] * (1.f / float(1 << c)) : in_vgpr(L.st[c]);
        }
    }
};

// pre-collision populations of a node in cube order
template <typename S, typename T, bool EVEN>
__device__ __forceinline__ void gather(const Lat& L, const uint32_t (&kk)[8], T (&m)[27])
{
    const Scales<S> sc(L);
#pragma unroll
    for (int s = 0; s < 27; ++s) {
        const int d = dir_at(s);
        m[s] = Storage<S, T>::ld(plane<S>(L, slot(d, EVEN)), kk[nbr(d)], sc.ld[weight_class(d)], L.sh[d]);
    }
}
// post-collision populations: the element direction d was read from receives
// the population of the opposite direction
template <typename S, typename T, bool EVEN, bool OUTER2 = false>
__device__ __forceinline__ void scatter_post(const Lat& L, const uint32_t (&kk)[8], const T (&m)[27])
{
    const Scales<S, OUTER2> sc(L);
#pragma unroll
    for (int s = 0; s < 27; ++s) {
        const int d = dir_at(s);
        const int e = inv(d);
        Storage<S, T>::st(plane<S>(L, slot(d, EVEN)), kk[nbr(d)], m[slot_of(e)], sc.st[weight_class(e)], L.ss[e]);
    }
}
// pre-collision write (initialisation, population upload)
template <typename S, typename T, bool EVEN>
__device__ __forceinline__ void scatter_pre(const Lat& L, const uint32_t (&kk)[8], const T (&m)[27])
{
#pragma unroll
    for (int s = 0; s < 27; ++s) {
        const int d = dir_at(s);
        Storage<S, T>::st(plane<S>(L, slot(d, EVEN)), kk[nbr(d)], m[s], L.st[weight_class(d)], L.ss[d]);
    }
}

// COLL: VFX_K17 / VFX_BGK in the low 4 bits, the eddy-viscosity model
// (TurbModel) of the reference-order K17 above them; FAST selects the
// reduced-operation K17 (FP32 only); OUTER2 (with FAST) leaves class-c
// populations scaled by 2^c for a scaling store.  nut: the node's turbulent
// viscosity in, the model's new value out.
constexpr int kCollBodyForce = 256;
constexpr int coll_op(int coll) { return coll & 15; }
constexpr int coll_turb(int coll) { return (coll >> 4) & 15; }
constexpr bool coll_body_force(int coll) { return (coll & kCollBodyForce) != 0; }

// runCollision with ApplyBodyForce (RunCollision.cuh:88-97): the node's force
// ((forces + bodyForce[k]) / 2) * forceFactor, then bodyForce[k] = 0
template <typename T, int COLL>
__device__ __forceinline__ void node_force(const Lat& L, uint32_t k, const Rates<T>& R, Rates<T>& Rn)
{
    if constexpr (coll_body_force(COLL)) {
        Rn = R;
        T* bx = (T*)L.bf[0];
        T* by = (T*)L.bf[1];
        T* bz = (T*)L.bf[2];
        const T ff = (T)L.force_factor;
        Rn.fx = ((T)L.gforce[0] + bx[k]) * T(0.5) * ff;
        Rn.fy = ((T)L.gforce[1] + by[k]) * T(0.5) * ff;
        Rn.fz = ((T)L.gforce[2] + bz[k]) * T(0.5) * ff;
        bx[k] = T(0);
        by[k] = T(0);
        bz[k] = T(0);
    }
}
template <typename T, int COLL, bool FAST, bool OUTER2 = false>
__device__ __forceinline__ void collide(T (&m)[27], const Rates<T>& R, T (&mv)[4], T& nut)
{
    if constexpr (coll_op(COLL) == VFX_K17) {
        if constexpr (FAST && sizeof(T) == 4) k17_fast<OUTER2, coll_turb(COLL)>(m, R, mv, nut);
        else k17<T, coll_turb(COLL)>(m, R, mv, nut);
    } else {
        bgk<T>(m, R.omega, mv);
    }
}
// runCollision's handling of the turbulent viscosity (RunCollision.cuh:116-141):
// read before the collision, stored after it; the AMD model needs the
// velocities of every node
template <typename T, int COLL> __device__ __forceinline__ T load_nut(const Lat& L, uint32_t k)
{
    if constexpr (coll_turb(COLL) != kTurbNone) return ((const T*)L.nut)[k];
    return T(0);
}
template <typename T, int COLL> __device__ __forceinline__ void store_nut(const Lat& L, uint32_t k, T nut)
{
    if constexpr (coll_turb(COLL) == kTurbSmagorinsky || coll_turb(COLL) == kTurbQR) ((T*)L.nut)[k] = nut;
}

template <typename T> __device__ __forceinline__ void write_macro(const Lat& L, uint32_t k, const T (&mv)[4])
{
    ((T*)L.rho)[k] = mv[0];
    ((T*)L.vx)[k] = mv[1];
    ((T*)L.vy)[k] = mv[2];
    ((T*)L.vz)[k] = mv[3];
}

// ------------------------------------------------------ collide + stream ----
// The command processor hands the workgroups of a launch to the 8 XCDs round
// robin (workgroup b to XCD b mod 8), and every XCD has its own L2.  Blocks
// next to each other in the lattice share cache lines at their ends (the
// +1-shifted reads of the esoteric twist, rows that do not start on a line), so
// the logical block of hardware workgroup b is chosen to give every XCD runs of
// C consecutive logical blocks: groups of 8C logical blocks, XCD x taking
// blocks x*C .. x*C+C-1 of each group (a tail shorter than 8C keeps the plain
// order).  Shared lines inside a run meet in one L2.  Runs much longer than
// this spread the XCDs over distant parts of each plane at once, which costs
// more than it saves for the 2-byte form.  xcd_run is the built-in run of the
// sparse step, step_run that of the structured one.
constexpr uint32_t kXcds = 8;
__device__ __forceinline__ uint32_t xcd_block(uint32_t b, uint32_t G, uint32_t C)
{
    const uint32_t span = kXcds * C, full = G / span * span;
    return b >= full ? b : (b / span) * span + (b % kXcds) * C + (b / kXcds) % C;
}
template <typename S> constexpr uint32_t xcd_run() { return sizeof(S) == 8 ? 256u : 16u; }
// the same for a run of 2^lg tiles (shifts only)
__device__ __forceinline__ uint32_t xcd_block_pow2(uint32_t b, uint32_t G, uint32_t lg)
{
    const uint32_t sh = lg + 3u, full = (G >> sh) << sh;
    return b >= full ? b : ((b >> sh) << sh) + ((b & (kXcds - 1u)) << lg) + ((b >> 3) & ((1u << lg) - 1u));
}
// one contiguous eighth of the blocks per XCD (a grid of a multiple of 8 blocks):
// stencils find their y and z neighbours' lines in the L2 they were read into
__device__ __forceinline__ uint32_t xcd_slab(uint32_t b, uint32_t G) { return (b % kXcds) * (G / kXcds) + b / kXcds; }

// Direct (structured) addressing: a tile is blockDim.x consecutive node
// numbers, whatever row they lie in.  The step is bound by its 27 in-place
// plane streams, so what matters is that every wavefront has 64 nodes and that
// its elements of a plane are one contiguous piece; a tile per x row leaves
// lanes idle wherever nx is no multiple of 64 (66: half the wavefronts hold 2
// nodes).  The price is a per-lane decode of the node (two multiply-high
// divisions, ~20 instructions), hidden behind the loads.  Against a tile per
// row, MI355X, us per step: FP64 66^3 36 -> 26, FP16 with AMD 224x144x120 195
// -> 175, FP16 512x256x256 736 -> 700 (with step_run), FP32 230x171x125 218 ->
// 207 (with 128-node tiles).
// Tile `block` of the lattice's `blocks`.
template <typename S, int COLL, bool EVEN, bool FAST>
__device__ __forceinline__ void step_direct_body(const Lat& L, const Rates<typename Compute<S>::T>& R, uint32_t block,
                                                 uint32_t blocks)
{
    using T = typename Compute<S>::T;
    const uint32_t blk = xcd_block_pow2(block, blocks, L.xrun_lg - 1u);
    const uint32_t k = blk * blockDim.x + threadIdx.x;
    if (k >= (uint32_t)L.N) return;
    uint32_t kk[8];
    nbrs_direct(L, k, kk);
    if (is_solid(L, kk[0])) return;
    T m[27], mv[4];
    constexpr bool O2 = FAST && coll_op(COLL) == VFX_K17 && sizeof(S) == 2;
    T nut = load_nut<T, COLL>(L, kk[0]);
    Rates<T> Rn;
    node_force<T, COLL>(L, kk[0], R, Rn);
    const Rates<T>& Ru = coll_body_force(COLL) ? Rn : R;
    gather<S, T, EVEN>(L, kk, m);
    collide<T, COLL, FAST, O2>(m, Ru, mv, nut);
    scatter_post<S, T, EVEN, O2>(L, kk, m);
    if (L.write_macro) write_macro<T>(L, kk[0], mv);
    store_nut<T, COLL>(L, kk[0], nut);
}
template <typename S, int COLL, bool EVEN, bool FAST>
__global__ void __launch_bounds__(256) k_step_direct(Lat L, Rates<typename Compute<S>::T> R)
{
    step_direct_body<S, COLL, EVEN, FAST>(L, R, blockIdx.x, gridDim.x);
}

// The eight nodes of sparse node k (as nbrs_sparse) with the second- and
// third-level neighbour reads shared across the wavefront.  VirtualFluids
// numbers a grid x-fastest, so the +x neighbour of a lane's node is mostly the
// next lane's node: where it is, nby/nbz of the +x neighbour are the next
// lane's first-level reads and nbz of the +x+y neighbour its +y neighbour's
// +z read (cross-lane shuffles instead of two dependent rounds of loads);
// the last lane reads the next node's arrays itself, and a lane whose +x
// neighbour is not the next node falls back to the loads.  `node` is the
// lane's node (0, the dummy node, for a lane without one), `next` the node of
// work item i + 1.  Same indices as nbrs_sparse.
__device__ __forceinline__ void nbrs_sparse_wave(const Lat& L, uint32_t node, uint32_t next, uint32_t (&kk)[8])
{
    const bool last = (threadIdx.x & 63u) == 63u;
    kk[0] = node;
    kk[1] = L.nbx[node];
    kk[2] = L.nby[node];
    kk[4] = L.nbz[node];
    uint32_t kn = __shfl_down(node, 1, 64), yn = __shfl_down(kk[2], 1, 64), zn = __shfl_down(kk[4], 1, 64);
    if (last) {
        kn = next;
        yn = L.nby[next];
        zn = L.nbz[next];
    }
    const bool hit = kk[1] == kn;
    kk[3] = yn;
    kk[5] = zn;
    if (!hit) {
        kk[3] = L.nby[kk[1]];
        kk[5] = L.nbz[kk[1]];
    }
    kk[6] = L.nbz[kk[2]];
    // the +x+y node's +z neighbour: the next lane's +y node's +z read
    const uint32_t z6n = __shfl_down(kk[6], 1, 64);
    kk[7] = z6n;
    if (!hit || last) kk[7] = L.nbz[kk[3]];
}

// Regular wavefronts of the sparse layout.  Where a grid is numbered x
// fastest (as VirtualFluids' generator numbers it), the 64 work items of a
// wavefront are mostly 64 consecutive nodes whose eight twist nodes are
// node + dx (j & 1) + sy ((j >> 1) & 1) + sz (j >> 2) with dx = 1 and one y
// and one z stride; at the end of a periodic row the last lane's +x neighbour
// is the row's first node, dx = 1 - sy (flag bit 1).  k_sparse_groups marks
// those wavefronts (every colliding lane checked against its index arrays,
// every formed index in bounds); the step forms their indices arithmetically
// and reads no index array.  Same indices, so the same populations, as the
// loads.
__device__ __forceinline__ void regular_nbrs(uint32_t k, uint32_t dx, uint32_t sy, uint32_t sz, uint32_t (&kk)[8])
{
#pragma unroll
    for (int j = 0; j < 8; ++j) kk[j] = k + dx * (j & 1) + sy * ((j >> 1) & 1) + sz * (j >> 2);
}
template <int = 0> __global__ void __launch_bounds__(256) k_sparse_groups(Lat L, uint4* table, uint32_t ngroups)
{
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t lane = threadIdx.x & 63u;
    uint32_t k = 0;
    const bool active = sparse_node(L, i, k);
    const bool has = L.types ? i < L.N : active;
    const uint32_t node = L.types ? (i < L.N ? (uint32_t)i : 0u) : (active ? k : 0u);
    const uint32_t k0 = __shfl(node, 0, 64);
    uint32_t sy = 0, sz = 0;
    if (lane == 0 && has) {
        sy = L.nby[node] - node;
        sz = L.nbz[node] - node;
    }
    sy = __shfl(sy, 0, 64);
    sz = __shfl(sz, 0, 64);
    bool ok = has && node == k0 + lane, okw = ok; // okw: the last lane wrapping in x
    if (ok && active) {
        uint32_t kk[8], r[8], rw[8];
        nbrs_sparse(L, node, kk);
        regular_nbrs(node, 1u, sy, sz, r);
        regular_nbrs(node, lane == 63u ? 1u - sy : 1u, sy, sz, rw);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            ok = ok && kk[j] == r[j];
            okw = okw && kk[j] == rw[j];
        }
    }
    const bool inside = (uint64_t)k0 + 64u + (uint64_t)sy + (uint64_t)sz < L.N && sy < L.N && sz < L.N;
    const bool all = __ballot(ok) == ~0ull, allw = __ballot(okw) == ~0ull;
    const uint64_t w = i >> 6;
    if (lane == 0 && w < ngroups) table[w] = make_uint4(k0, sy, sz, !inside ? 0u : all ? 1u : allw ? 3u : 0u);
}

// VirtualFluids sparse addressing over the fluid-node list
// (RunCollision.cuh:74-143 semantics).
template <typename S, int COLL, bool EVEN, bool FAST>
__global__ void __launch_bounds__(256) k_step_sparse(Lat L, Rates<typename Compute<S>::T> R)
{
    using T = typename Compute<S>::T;
    const uint32_t blk = L.xrun_lg ? xcd_block_pow2(blockIdx.x, gridDim.x, L.xrun_lg - 1u)
                                   : xcd_block(blockIdx.x, gridDim.x, xcd_run<S>());
    const uint32_t i = blk * blockDim.x + threadIdx.x;
    uint32_t kk[8], k;
    bool active;
    uint4 g = make_uint4(0u, 0u, 0u, 0u);
    if (L.rgroups) g = L.rgroups[__builtin_amdgcn_readfirstlane(i >> 6)];
    if (g.w & 1u) {
        // a regular wavefront: its nodes and their twist nodes by arithmetic
        const uint32_t lane = threadIdx.x & 63u;
        k = g.x + lane;
        active = true;
        if (L.types) {
            const uint32_t t = L.types[k];
            active = t != kGeoSolid && t != kGeoVoid;
        }
        regular_nbrs(k, (g.w & 2u) && lane == 63u ? 1u - g.y : 1u, g.y, g.z, kk);
    } else {
        active = sparse_node(L, i, k);
        // the node of work item i + 1 (the last lane of a wavefront reads its arrays)
        uint32_t next = 0;
        if ((threadIdx.x & 63u) == 63u) {
            if (L.types) next = i + 1 < L.N ? i + 1 : 0u;
            else if (i + 1 < L.nfluid) next = L.fluid[i + 1] < L.N ? L.fluid[i + 1] : 0u;
        }
        // every lane takes part in the shuffles: lanes without a node use the dummy node
        const uint32_t node = L.types ? (i < L.N ? i : 0u) : (active ? k : 0u);
        nbrs_sparse_wave(L, node, next, kk);
    }
    if (!active) return;
    T m[27], mv[4];
    constexpr bool O2 = FAST && coll_op(COLL) == VFX_K17 && sizeof(S) == 2;
    T nut = load_nut<T, COLL>(L, kk[0]);
    Rates<T> Rn;
    node_force<T, COLL>(L, kk[0], R, Rn);
    const Rates<T>& Ru = coll_body_force(COLL) ? Rn : R;
    gather<S, T, EVEN>(L, kk, m);
    collide<T, COLL, FAST, O2>(m, Ru, mv, nut);
    scatter_post<S, T, EVEN, O2>(L, kk, m);
    if (L.write_macro) write_macro<T>(L, kk[0], mv);
    store_nut<T, COLL>(L, kk[0], nut);
}

// ------------------------------------------------------------ node loops ----
// Visits every node that collides: direct -> every non-solid node of the box,
// sparse -> the fluid-node list.
struct NodeIter {
    __device__ static bool get(const Lat& L, uint64_t i, uint32_t (&kk)[8], int direct)
    {
        if (direct) {
            if (i >= L.N) return false;
            const uint32_t k = (uint32_t)i;
            if (is_solid(L, k)) return false;
            nbrs_direct(L, k, kk);
        } else {
            uint32_t k;
            if (!sparse_node(L, i, k)) return false;
            nbrs_sparse(L, k, kk);
        }
        return true;
    }
};

// shifted compressible equilibrium (InitNavierStokesCompressible_Device.cu:170-210)
template <typename T>
__device__ __forceinline__ void equilibrium(T (&m)[27], T drho, T vx1, T vx2, T vx3)
{
    const T cu_sq = T(1.5) * (vx1 * vx1 + vx2 * vx2 + vx3 * vx3);
    m[slot_of(d000)] = T(8. / 27.) * (drho - cu_sq * (T(1) + drho));
#pragma unroll
    for (int d = 1; d < 27; ++d) {
        T cu;
        if (cx(d) != 0) {
            cu = cx(d) > 0 ? vx1 : -vx1;
            if (cy(d) != 0) cu = cy(d) > 0 ? cu + vx2 : cu - vx2;
            if (cz(d) != 0) cu = cz(d) > 0 ? cu + vx3 : cu - vx3;
        } else if (cy(d) != 0) {
            cu = cy(d) > 0 ? vx2 : -vx2;
            if (cz(d) != 0) cu = cz(d) > 0 ? cu + vx3 : cu - vx3;
        } else {
            cu = cz(d) > 0 ? vx3 : -vx3;
        }
        m[slot_of(d)] = weight<T>(d) * (drho + (T(1) + drho) * (T(3) * cu + T(4.5) * cu * cu - cu_sq));
    }
}

template <typename S, bool EVEN>
__global__ void __launch_bounds__(256) k_init(Lat L, int direct, const double* drho, const double* ux, const double* uy,
                                              const double* uz)
{
    using T = typename Compute<S>::T;
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    uint32_t kk[8];
    if (!NodeIter::get(L, i, kk, direct)) return;
    const uint32_t k = kk[0];
    T m[27];
    equilibrium<T>(m, (T)drho[k], (T)ux[k], (T)uy[k], (T)uz[k]);
    scatter_pre<S, T, EVEN>(L, kk, m);
}

template <typename S, bool EVEN>
__global__ void __launch_bounds__(256) k_read(Lat L, int direct, double* out)
{
    using T = typename Compute<S>::T;
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    uint32_t kk[8];
    if (!NodeIter::get(L, i, kk, direct)) return;
    T m[27];
    gather<S, T, EVEN>(L, kk, m);
#pragma unroll
    for (int s = 0; s < 27; ++s) out[(uint64_t)kk[0] * 27 + dir_at(s)] = (double)m[s];
}

template <typename S, bool EVEN>
__global__ void __launch_bounds__(256) k_write(Lat L, int direct, const double* in)
{
    using T = typename Compute<S>::T;
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    uint32_t kk[8];
    if (!NodeIter::get(L, i, kk, direct)) return;
    T m[27];
#pragma unroll
    for (int s = 0; s < 27; ++s) m[s] = (T)in[(uint64_t)kk[0] * 27 + dir_at(s)];
    scatter_pre<S, T, EVEN>(L, kk, m);
}

// FP64 density deviation and momentum of one node (pyramid sums of
// MacroscopicQuantities.h:55-85 on the populations widened to double)
template <typename T>
__device__ __forceinline__ void node_moments(const T (&m)[27], double& r, double& jx, double& jy, double& jz)
{
    double f[27];
#pragma unroll
    for (int s = 0; s < 27; ++s) f[dir_at(s)] = (double)m[s];
    const double corners = ((f[dPPP] + f[dMMM]) + (f[dMPM] + f[dPMP])) + ((f[dMPP] + f[dPMM]) + (f[dMMP] + f[dPPM]));
    const double edges = (((f[d0MP] + f[d0PM]) + (f[d0MM] + f[d0PP])) + ((f[dM0P] + f[dP0M]) + (f[dM0M] + f[dP0P]))) +
                         ((f[dMP0] + f[dPM0]) + (f[dMM0] + f[dPP0]));
    const double faces = ((f[dM00] + f[dP00]) + (f[d0M0] + f[d0P0])) + (f[d00M] + f[d00P]);
    r = ((corners + edges) + f[d000]) + faces;
    jx = (((f[dPPP] - f[dMMM]) + (f[dPMP] - f[dMPM])) + ((f[dPMM] - f[dMPP]) + (f[dPPM] - f[dMMP]))) +
         (((f[dP0M] - f[dM0P]) + (f[dP0P] - f[dM0M])) + ((f[dPM0] - f[dMP0]) + (f[dPP0] - f[dMM0]))) +
         (f[dP00] - f[dM00]);
    jy = (((f[dPPP] - f[dMMM]) + (f[dMPM] - f[dPMP])) + ((f[dMPP] - f[dPMM]) + (f[dPPM] - f[dMMP]))) +
         (((f[d0PM] - f[d0MP]) + (f[d0PP] - f[d0MM])) + ((f[dMP0] - f[dPM0]) + (f[dPP0] - f[dMM0]))) +
         (f[d0P0] - f[d0M0]);
    jz = (((f[dPPP] - f[dMMM]) + (f[dPMP] - f[dMPM])) + ((f[dMPP] - f[dPMM]) + (f[dMMP] - f[dPPM]))) +
         (((f[d0MP] - f[d0PM]) + (f[d0PP] - f[d0MM])) + ((f[dM0P] - f[dP0M]) + (f[dP0P] - f[dM0M]))) +
         (f[d00P] - f[d00M]);
}

// macroscopic values of the pre-collision state (FP64 output)
template <typename S, bool EVEN>
__global__ void __launch_bounds__(256) k_macro(Lat L, int direct, double* drho, double* vx, double* vy, double* vz)
{
    using T = typename Compute<S>::T;
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    uint32_t kk[8];
    if (!NodeIter::get(L, i, kk, direct)) return;
    T m[27];
    gather<S, T, EVEN>(L, kk, m);
    double r, jx, jy, jz;
    node_moments<T>(m, r, jx, jy, jz);
    const double oor = 1.0 / (r + 1.0);
    const uint32_t k = kk[0];
    drho[k] = r;
    vx[k] = jx * oor;
    vy[k] = jy * oor;
    vz[k] = jz * oor;
}

// calculateMacroscopicQuantitiesCompressible_device
// (PostProcessor/MacroscopicQuantities.cu:194-237): every node's outputs are
// zeroed, then the fluid nodes get vf::lbm::getDensity, the compressible
// velocities (numerator / (rho + 1)) and getPressure (MacroscopicQuantities.h:
// 55-64, 100-115, 139-149) in the lattice's arithmetic type, in the
// reference's operation order.  LIST = 0 walks every node (direct: not solid;
// sparse with typeOfGridNode: isValidFluidNode, KernelUtilities.h:216-219, types
// 19, 5, 6, 7); LIST = 1 computes the nodes of the fluid-node list after a
// LIST = 0 pass has zeroed everything.
template <typename T> __device__ __forceinline__ void vf_macroscopic(const T (&f)[27], T& rho, T& vx, T& vy, T& vz,
                                                                     T& press)
{
    rho = ((((f[dPPP] + f[dMMM]) + (f[dMPM] + f[dPMP])) + ((f[dMPP] + f[dPMM]) + (f[dMMP] + f[dPPM]))) +
           (((f[d0MP] + f[d0PM]) + (f[d0MM] + f[d0PP])) + ((f[dM0P] + f[dP0M]) + (f[dM0M] + f[dP0P])) +
            ((f[dMP0] + f[dPM0]) + (f[dMM0] + f[dPP0]))) +
           f[d000]) +
          ((f[dM00] + f[dP00]) + (f[d0M0] + f[d0P0]) + (f[d00M] + f[d00P]));
    const T jx = ((((f[dPPP] - f[dMMM]) + (f[dPMP] - f[dMPM])) + ((f[dPMM] - f[dMPP]) + (f[dPPM] - f[dMMP]))) +
                  (((f[dP0M] - f[dM0P]) + (f[dP0P] - f[dM0M])) + ((f[dPM0] - f[dMP0]) + (f[dPP0] - f[dMM0]))) +
                  (f[dP00] - f[dM00]));
    const T jy = ((((f[dPPP] - f[dMMM]) + (f[dMPM] - f[dPMP])) + ((f[dMPP] - f[dPMM]) + (f[dPPM] - f[dMMP]))) +
                  (((f[d0PM] - f[d0MP]) + (f[d0PP] - f[d0MM])) + ((f[dMP0] - f[dPM0]) + (f[dPP0] - f[dMM0]))) +
                  (f[d0P0] - f[d0M0]));
    const T jz = ((((f[dPPP] - f[dMMM]) + (f[dPMP] - f[dMPM])) + ((f[dMPP] - f[dPMM]) + (f[dMMP] - f[dPPM]))) +
                  (((f[d0MP] - f[d0PM]) + (f[d0PP] - f[d0MM])) + ((f[dM0P] - f[dP0M]) + (f[dP0P] - f[dM0M]))) +
                  (f[d00P] - f[d00M]));
    vx = jx / (rho + T(1));
    vy = jy / (rho + T(1));
    vz = jz / (rho + T(1));
    press = (f[dP00] + f[dM00] + f[d0P0] + f[d0M0] + f[d00P] + f[d00M] +
             T(2) * (f[dPP0] + f[dMM0] + f[dPM0] + f[dMP0] + f[dP0P] + f[dM0M] + f[dP0M] + f[dM0P] + f[d0PP] +
                     f[d0MM] + f[d0PM] + f[d0MP]) +
             T(3) * (f[dPPP] + f[dMMP] + f[dPMP] + f[dMPP] + f[dPPM] + f[dMMM] + f[dPMM] + f[dMPM]) - rho -
             (vx * vx + vy * vy + vz * vz) * (T(1) + rho)) *
                T(0.5) +
            rho;
}

template <typename S, bool EVEN, int LIST>
__global__ void __launch_bounds__(256) k_macro_vf(Lat L, int direct, typename Compute<S>::T* rho,
                                                  typename Compute<S>::T* vx, typename Compute<S>::T* vy,
                                                  typename Compute<S>::T* vz, typename Compute<S>::T* press)
{
    using T = typename Compute<S>::T;
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    uint32_t k;
    bool fluid;
    if constexpr (LIST) {
        if (i >= L.nfluid) return;
        k = L.fluid[i];
        if (k >= L.N) return;
        fluid = true;
    } else {
        if (i >= L.N) return;
        k = (uint32_t)i;
        press[k] = T(0);
        rho[k] = T(0);
        vx[k] = T(0);
        vy[k] = T(0);
        vz[k] = T(0);
        if (direct) {
            fluid = !is_solid(L, k);
        } else if (L.types) {
            const uint32_t t = L.types[k];
            fluid = t == 19u || t == 5u || t == 6u || t == 7u;
        } else {
            fluid = false;
        }
    }
    if (!fluid) return;
    uint32_t kk[8];
    if (direct) nbrs_direct(L, k, kk);
    else nbrs_sparse(L, k, kk);
    T m[27];
    gather<S, T, EVEN>(L, kk, m);
    T f[27];
#pragma unroll
    for (int s = 0; s < 27; ++s) f[dir_at(s)] = m[s];
    T r, ux, uy, uz, p;
    vf_macroscopic<T>(f, r, ux, uy, uz, p);
    rho[k] = r;
    vx[k] = ux;
    vy[k] = uy;
    vz[k] = uz;
    press[k] = p;
}

// Time-averaged fields (calculateMeanCompressible_device,
// MacroscopicQuantities.cu:390-536): adds the node's density deviation and
// velocity to running sums (sum order of that kernel), and to the pressure sum
// the pressure expression evaluated with the new density and velocity sums in
// place of the node's own values, as the reference kernel does.  Every node
// of the all-node form zeroes its sums first, so only fluid nodes accumulate.
template <typename T> __device__ __forceinline__ void vf_mean_add(const T (&f)[27], T& RHO, T& VX, T& VY, T& VZ, T& PRESS)
{
#pragma clang fp contract(off)
    const T drho = ((((f[dPPP] + f[dMMM]) + (f[dMPM] + f[dPMP])) + ((f[dMPP] + f[dPMM]) + (f[dMMP] + f[dPPM]))) +
                    (((f[d0MP] + f[d0PM]) + (f[d0MM] + f[d0PP])) + ((f[dM0P] + f[dP0M]) + (f[dM0M] + f[dP0P])) +
                     ((f[dMP0] + f[dPM0]) + (f[dMM0] + f[dPP0]))) +
                    ((f[dM00] + f[dP00]) + (f[d0M0] + f[d0P0]) + (f[d00M] + f[d00P]))) +
                   f[d000];
    const T rho = T(1) + drho;
    const T r = drho + RHO;
    const T x = (((((f[dPPP] - f[dMMM]) + (f[dPMP] - f[dMPM])) + ((f[dPMM] - f[dMPP]) + (f[dPPM] - f[dMMP]))) +
                  (((f[dP0M] - f[dM0P]) + (f[dP0P] - f[dM0M])) + ((f[dPM0] - f[dMP0]) + (f[dPP0] - f[dMM0]))) +
                  (f[dP00] - f[dM00])) /
                 rho) +
                VX;
    const T y = (((((f[dPPP] - f[dMMM]) + (f[dMPM] - f[dPMP])) + ((f[dMPP] - f[dPMM]) + (f[dPPM] - f[dMMP]))) +
                  (((f[d0PM] - f[d0MP]) + (f[d0PP] - f[d0MM])) + ((f[dMP0] - f[dPM0]) + (f[dPP0] - f[dMM0]))) +
                  (f[d0P0] - f[d0M0])) /
                 rho) +
                VY;
    const T z = (((((f[dPPP] - f[dMMM]) + (f[dPMP] - f[dMPM])) + ((f[dMPP] - f[dPMM]) + (f[dMMP] - f[dPPM]))) +
                  (((f[d0MP] - f[d0PM]) + (f[d0PP] - f[d0MM])) + ((f[dM0P] - f[dP0M]) + (f[dP0P] - f[dM0M]))) +
                  (f[d00P] - f[d00M])) /
                 rho) +
                VZ;
    PRESS = (f[dP00] + f[dM00] + f[d0P0] + f[d0M0] + f[d00P] + f[d00M] +
             T(2) * (f[dPP0] + f[dMM0] + f[dPM0] + f[dMP0] + f[dP0P] + f[dM0M] + f[dP0M] + f[dM0P] + f[d0PP] +
                     f[d0MM] + f[d0PM] + f[d0MP]) +
             T(3) * (f[dPPP] + f[dMMP] + f[dPMP] + f[dMPP] + f[dPPM] + f[dMMM] + f[dPMM] + f[dMPM]) - r -
             (x * x + y * y + z * z) * (T(1) + r)) *
                T(0.5) +
            r + PRESS;
    RHO = r;
    VX = x;
    VY = y;
    VZ = z;
}

template <typename S, bool EVEN, int LIST>
__global__ void __launch_bounds__(256) k_mean_vf(Lat L, int direct, typename Compute<S>::T* vx,
                                                 typename Compute<S>::T* vy, typename Compute<S>::T* vz,
                                                 typename Compute<S>::T* rho, typename Compute<S>::T* press)
{
    using T = typename Compute<S>::T;
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    uint32_t k;
    bool fluid;
    if constexpr (LIST) {
        if (i >= L.nfluid) return;
        k = L.fluid[i];
        if (k >= L.N) return;
        fluid = true;
    } else {
        if (i >= L.N) return;
        k = (uint32_t)i;
        fluid = direct ? !is_solid(L, k) : (L.types && L.types[k] == kGeoFluid);
    }
    T P = press[k], R = rho[k], X = vx[k], Y = vy[k], Z = vz[k];
    if (!LIST) {
        press[k] = T(0);
        rho[k] = T(0);
        vx[k] = T(0);
        vy[k] = T(0);
        vz[k] = T(0);
    }
    if (!fluid) return;
    uint32_t kk[8];
    if (direct) nbrs_direct(L, k, kk);
    else nbrs_sparse(L, k, kk);
    T m[27];
    gather<S, T, EVEN>(L, kk, m);
    T f[27];
#pragma unroll
    for (int s = 0; s < 27; ++s) f[dir_at(s)] = m[s];
    vf_mean_add<T>(f, R, X, Y, Z, P);
    rho[k] = R;
    vx[k] = X;
    vy[k] = Y;
    vz[k] = Z;
    press[k] = P;
}

template <typename T> __global__ void __launch_bounds__(256) k_zero5(T* a, T* b, T* c, T* d, T* e, uint64_t n)
{
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    a[i] = T(0);
    b[i] = T(0);
    c[i] = T(0);
    d[i] = T(0);
    e[i] = T(0);
}

// ---------------------------------------------------------- reductions ----
// Deterministic two-pass FP64 sums: every block sums a fixed chunk of
// kRedBlock * kRedPerThread nodes (per-thread sequential, then a wave64
// butterfly and a fixed-order sum of the four waves); a single block then
// adds the per-block partials in index order.
constexpr int kRedBlock = 256;
constexpr int kRedPerThread = 8;
constexpr int kRedChunk = kRedBlock * kRedPerThread;

__device__ __forceinline__ double wave_sum(double v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

template <int NV> __device__ __forceinline__ void block_sum(double (&v)[NV])
{
    __shared__ double part[kRedBlock / 64][NV];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int c = 0; c < NV; ++c) {
        v[c] = wave_sum(v[c]);
        if (lane == 0) part[wave][c] = v[c];
    }
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
        for (int c = 0; c < NV; ++c) {
            double t = part[0][c];
            for (int w = 1; w < kRedBlock / 64; ++w) t += part[w][c];
            v[c] = t;
        }
    }
}

// per node: drho, jx, jy, jz (mass deviation and momentum of the pre-collision state)
template <typename S, bool EVEN, bool DIRECT>
__global__ void __launch_bounds__(kRedBlock) k_reduce_mass(Lat L, double* partial)
{
    using T = typename Compute<S>::T;
    double acc[4] = {0, 0, 0, 0};
    for (int j = 0; j < kRedPerThread; ++j) {
        const uint64_t i = (uint64_t)blockIdx.x * kRedChunk + (uint64_t)j * kRedBlock + threadIdx.x;
        uint32_t kk[8];
        if (!NodeIter::get(L, i, kk, DIRECT)) continue;
        T m[27];
        gather<S, T, EVEN>(L, kk, m);
        double r, jx, jy, jz;
        node_moments<T>(m, r, jx, jy, jz);
        acc[0] += r;
        acc[1] += jx;
        acc[2] += jy;
        acc[3] += jz;
    }
    block_sum<4>(acc);
    if (threadIdx.x == 0)
        for (int c = 0; c < 4; ++c) partial[(uint64_t)blockIdx.x * 4 + c] = acc[c];
}

template <int NV> __global__ void __launch_bounds__(kRedBlock) k_reduce_finish(const double* partial, uint32_t nblocks, double* out)
{
    double acc[NV];
#pragma unroll
    for (int c = 0; c < NV; ++c) acc[c] = 0.0;
    for (uint32_t b = threadIdx.x; b < nblocks; b += kRedBlock)
#pragma unroll
        for (int c = 0; c < NV; ++c) acc[c] += partial[(uint64_t)b * NV + c];
    block_sum<NV>(acc);
    if (threadIdx.x == 0)
#pragma unroll
        for (int c = 0; c < NV; ++c) out[c] = acc[c];
}

// The nodes up to R steps from node k along one axis of extent n and the given
// stride (periodic index wrap, also for boxes smaller than the stencil), c the
// node's coordinate.
template <int R> struct AxisNodes {
    uint32_t p[R + 1], m[R + 1];
    __device__ __forceinline__ AxisNodes(uint32_t k, uint32_t c, uint32_t n, uint32_t stride)
    {
        const uint32_t back = (n - 1u) * stride;
        uint32_t cp = c, cm = c;
        p[0] = m[0] = k;
#pragma unroll
        for (int s = 1; s <= R; ++s) {
            const bool wp = cp + 1u == n, wm = cm == 0u;
            p[s] = wp ? p[s - 1] - back : p[s - 1] + stride;
            m[s] = wm ? m[s - 1] + back : m[s - 1] - stride;
            cp = wp ? 0u : cp + 1u;
            cm = wm ? n - 1u : cm - 1u;
        }
    }
};
// order of the central difference at the node: 8, or 6 / 4 / 2 where the stencil
// meets a solid node
__device__ __forceinline__ int stencil_order(const Lat& L, const AxisNodes<4>& a)
{
    if (!L.solid) return 8;
    if (is_solid(L, a.p[2]) || is_solid(L, a.m[2])) return 2;
    if (is_solid(L, a.p[3]) || is_solid(L, a.m[3])) return 4;
    return is_solid(L, a.p[4]) || is_solid(L, a.m[4]) ? 6 : 8;
}
// 280 times the derivative of order 8; W32: the fields' byte offsets fit 32 bits
template <bool W32> __device__ __forceinline__ double derivative8(const double* v, const AxisNodes<4>& a)
{
    auto d = [&](int s) { return W32 ? elem(v, a.p[s]) - elem(v, a.m[s]) : v[a.p[s]] - v[a.m[s]]; };
    return (28.0 * 8.0) * d(1) - (7.0 * 8.0) * d(2) + (8.0 * 4.0 * (1.0 / 3.0)) * d(3) - d(4);
}
__device__ __forceinline__ double derivative(const double* v, const AxisNodes<4>& a, int order)
{
    auto d = [&](int s) { return v[a.p[s]] - v[a.m[s]]; };
    if (order == 8) return derivative8<false>(v, a) / (7.0 * 10.0 * 4.0);
    if (order == 2) return d(1) / 2.0;
    if (order == 4) return ((8.0 * v[a.p[1]] - 8.0 * v[a.m[1]]) - d(2)) / 12.0;
    return ((5.0 * 9.0) * d(1) - 9.0 * d(2) + d(3)) / (6.0 * 10.0);
}

// Kinetic energy 1/2 rho |u|^2 summed over fluid nodes whose six axis
// neighbours are fluid, and their count (KineticEnergyAnalyzer.cu:137-154).
// Enstrophy 1/2 rho |curl u|^2 on the same nodes with central differences of
// order 8, reduced to 6/4/2 where the stencil meets a wall
// (EnstrophyAnalyzer.cu:134-336).
//
// The neighbours of an axis are stepped to (compare, select, add) and shared by
// the two fields differentiated along it, and the chunks of an XCD are
// contiguous, so the enstrophy stencil's rows and planes are found in its L2.
// MI355X, 160^3: enstrophy 218 -> 97 us (one 64-bit remainder per neighbour and
// field and chunks round robin before), 48 loads of 8 bytes per node and ~41 us
// of L1 throughput; with the 64-bit offsets and order branches of the general
// form 136.  Kinetic energy 29 -> 28 us, a stream of the four fields (26 at 5 TB/s).
// PLAIN: no solid nodes and fields below 4 GiB (byte offsets of 32 bits).
template <bool ENSTROPHY, bool PLAIN>
__global__ void __launch_bounds__(kRedBlock) k_reduce_energy(Lat L, const double* rho, const double* vx, const double* vy,
                                                             const double* vz, double* partial)
{
    double acc[2] = {0, 0};
    const uint32_t full = gridDim.x / kXcds * kXcds;
    const uint32_t chunk = ENSTROPHY && blockIdx.x < full ? xcd_slab(blockIdx.x, full) : blockIdx.x;
    for (int j = 0; j < kRedPerThread; ++j) {
        const uint64_t i = (uint64_t)chunk * kRedChunk + (uint64_t)j * kRedBlock + threadIdx.x;
        if (i >= L.N) continue;
        const uint32_t k = (uint32_t)i;
        if (!PLAIN && is_solid(L, k)) continue;
        const uint32_t r = fastdiv(k, L.div_x), x = k - r * L.nx, z = fastdiv(r, L.div_y), y = r - z * L.ny;
        constexpr int R = ENSTROPHY ? 4 : 1;
        const AxisNodes<R> ax(k, x, L.nx, 1u), ay(k, y, L.ny, L.nx), az(k, z, L.nz, L.nx * L.ny);
        if (!PLAIN && L.solid &&
            (is_solid(L, ax.p[1]) || is_solid(L, ax.m[1]) || is_solid(L, ay.p[1]) || is_solid(L, ay.m[1]) ||
             is_solid(L, az.p[1]) || is_solid(L, az.m[1])))
            continue;
        acc[1] += 1.0;
        if constexpr (!ENSTROPHY) {
            acc[0] += 0.5 * (vx[k] * vx[k] + vy[k] * vy[k] + vz[k] * vz[k]) * (rho[k] + 1.0);
            continue;
        } else {
            if constexpr (!PLAIN) {
                const int ox = stencil_order(L, ax), oy = stencil_order(L, ay), oz = stencil_order(L, az);
                if (ox != 8 || oy != 8 || oz != 8) {
                    const double dyvz = derivative(vz, ay, oy), dzvy = derivative(vy, az, oz);
                    const double dzvx = derivative(vx, az, oz), dxvz = derivative(vz, ax, ox);
                    const double dxvy = derivative(vy, ax, ox), dyvx = derivative(vx, ay, oy);
                    const double wx = dyvz - dzvy, wy = dzvx - dxvz, wz = dxvy - dyvx;
                    acc[0] += 0.5 * (rho[k] + 1.0) * (wx * wx + wy * wy + wz * wz);
                    continue;
                }
            }
            // one division for the six derivatives
            const double wx = derivative8<PLAIN>(vz, ay) - derivative8<PLAIN>(vy, az);
            const double wy = derivative8<PLAIN>(vx, az) - derivative8<PLAIN>(vz, ax);
            const double wz = derivative8<PLAIN>(vy, ax) - derivative8<PLAIN>(vx, ay);
            acc[0] += 0.5 * (rho[k] + 1.0) * (wx * wx + wy * wy + wz * wz) / (280.0 * 280.0);
        }
    }
    block_sum<2>(acc);
    if (threadIdx.x == 0) {
        partial[(uint64_t)chunk * 2] = acc[0];
        partial[(uint64_t)chunk * 2 + 1] = acc[1];
    }
}

// Running FP64 sums for time averages (CalcTurbulenceIntensity,
// TurbulenceIntensity.cu:45-85): planes 0-2 sum u, planes 3-8 sum
// u_x u_x, u_y u_y, u_z u_z, u_x u_y, u_x u_z, u_y u_z.
template <typename S, bool EVEN>
__global__ void __launch_bounds__(256) k_stats(Lat L, int direct, double* sums)
{
    using T = typename Compute<S>::T;
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    uint32_t kk[8];
    if (!NodeIter::get(L, i, kk, direct)) return;
    T m[27];
    gather<S, T, EVEN>(L, kk, m);
    double r, jx, jy, jz;
    node_moments<T>(m, r, jx, jy, jz);
    const double oor = 1.0 / (r + 1.0);
    const double ux = jx * oor, uy = jy * oor, uz = jz * oor;
    const uint64_t k = kk[0], N = L.N;
    sums[k] += ux;
    sums[N + k] += uy;
    sums[2 * N + k] += uz;
    sums[3 * N + k] += ux * ux;
    sums[4 * N + k] += uy * uy;
    sums[5 * N + k] += uz * uz;
    sums[6 * N + k] += ux * uy;
    sums[7 * N + k] += ux * uz;
    sums[8 * N + k] += uy * uz;
}

// -------------------------------------------------- boundary conditions ----
// Every floating-point table of a boundary condition is of the lattice's
// arithmetic type T (double for FP64 storage, float otherwise), the `real` of
// VirtualFluids' QforBoundaryConditions; bc_at<T> reads element i.
struct BCDev {
    uint32_t n;
    const uint32_t* k;
    const void* q;         // q27[0]: 27 * n subgrid distances, SoA
    const void* vx;        // wall velocity per boundary node (NULL = 0)
    const void* vy;
    const void* vz;
    int32_t cpu_float;
    int32_t single_links;  // bounce-back, sparse: no node of the list is its own neighbour
    int32_t direct;
    double omega;          // interpolated kinds
    const void* rho;       // pressure: density deviation per boundary node
    const uint32_t* kn;    // pressure / outflow: inward neighbour of each boundary node
    int32_t normal;        // pressure / outflow: outward direction of the boundary (d000..dMMM)
    double corr;           // outflow with pressure correction: density correction factor
    // stress (wall-model) kinds, arrays of the lattice's arithmetic type
    const void* wm_normal[3];     // wall normal per boundary node
    void* wm_el[3];               // filtered velocity at the exchange location (state)
    void* wm_wall[3];             // filtered velocity at the wall node (state)
    const int32_t* wm_offset;     // sampling offset (nodes from the wall)
    const void* wm_z0;            // roughness length
    void* wm_ustar;               // monitors (NULL: none)
    void* wm_force[3];
    // precursor kinds: plane stencil per boundary node and the two plane
    // arrays (lattice's arithmetic type), blended last*(1 - tr) + current*tr
    uint32_t n_pre;
    const uint32_t* pn[4];        // precursor nodes 0PP, 0PM, 0MP, 0MM
    const void* pw[4];            // their inverse-distance weights
    const void* plast;
    const void* pcur;
    double tratio;
    double vratio;                // velocity ratio (velocity kind)
    double pu[3];                 // velocity kind: scalar velocity added to vx/vy/vz
};

template <typename T> __device__ __forceinline__ T bc_at(const void* a, uint64_t i) { return ((const T*)a)[i]; }
template <typename T> __device__ __forceinline__ T bc_q(const BCDev& B, int d, uint32_t i)
{
    return bc_at<T>(B.q, (uint64_t)d * B.n + i);
}

// The plane value at boundary node i: the four precursor nodes around it
// weighted by inverse distance, or the 0PP node alone when its weight is
// >= 1e6 (PrecursorNonReflectiveCompressible.cu:82-110,
// PrecursorDistributions.cu:95-152).  The weighted sum runs in the
// reference's order and is scaled by 1 / (sum of weights).
template <typename T> struct PlaneStencil {
    uint32_t n[4];
    T w[4];
    T inv;
    bool one;
    bool ok; // every precursor node the stencil reads lies inside the planes
};

template <typename T> __device__ __forceinline__ PlaneStencil<T> plane_stencil(const BCDev& B, uint32_t i)
{
    PlaneStencil<T> s;
    s.n[0] = B.pn[0][i];
    s.w[0] = ((const T*)B.pw[0])[i];
    s.one = !(s.w[0] < T(1e6));
    s.inv = T(0);
    s.ok = s.n[0] < B.n_pre;
    if (!s.one) {
        for (int c = 1; c < 4; ++c) {
            s.n[c] = B.pn[c][i];
            s.w[c] = ((const T*)B.pw[c])[i];
            s.ok = s.ok && s.n[c] < B.n_pre;
        }
        s.inv = T(1) / (s.w[0] + s.w[1] + s.w[2] + s.w[3]);
    }
    return s;
}

template <typename T> __device__ __forceinline__ T plane_value(const PlaneStencil<T>& s, const T* a)
{
    if (s.one) return a[s.n[0]];
    return (a[s.n[0]] * s.w[0] + a[s.n[1]] * s.w[1] + a[s.n[2]] * s.w[2] + a[s.n[3]] * s.w[3]) * s.inv;
}

// last*(1 - tr) + current*tr of plane component c (PrecursorDistributions.cu:163-171)
template <typename T> __device__ __forceinline__ T plane_blend(const BCDev& B, const PlaneStencil<T>& s, int c)
{
    const T tr = (T)B.tratio;
    const size_t off = (size_t)c * B.n_pre;
    return plane_value(s, (const T*)B.plast + off) * (T(1) - tr) + plane_value(s, (const T*)B.pcur + off) * tr;
}

// c_d . (ux, uy, uz) spelled as VirtualFluids writes it: first non-zero
// component with its sign, then the others added or subtracted in x, y, z order
template <typename T> __device__ __forceinline__ T proj(int d, T ux, T uy, T uz)
{
    T v;
    if (cx(d) != 0) {
        v = cx(d) > 0 ? ux : -ux;
        if (cy(d) != 0) v = cy(d) > 0 ? v + uy : v - uy;
        if (cz(d) != 0) v = cz(d) > 0 ? v + uz : v - uz;
    } else if (cy(d) != 0) {
        v = cy(d) > 0 ? uy : -uy;
        if (cz(d) != 0) v = cz(d) > 0 ? v + uz : v - uz;
    } else {
        v = cz(d) > 0 ? uz : -uz;
    }
    return v;
}

// 6 w_d (c_d . u) as BoundaryConditions.h:195-262 rounds it (float wall
// velocity, float component sum, double scale, float result)
template <typename T> __device__ __forceinline__ T wall_term_cpu(int d, double ux, double uy, double uz)
{
    const int n = weight_class(d);
    const double coef = n == 1 ? 4. / 9. : n == 2 ? 1. / 9. : 1. / 36.;
    const float s = proj<float>(d, (float)ux, (float)uy, (float)uz);
    return (T)(double)(float)(coef * (double)s);
}

// Moving-wall halfway bounce-back (VelocityBounceBack_Device): for every wall
// link d of a boundary node, the population leaving towards the wall comes back
// as the opposite direction, minus the wall term.  Runs between the collision
// of parity EVEN and the parity flip.
//
// fpost - 6 w_d (c_d . u): one explicit FMA in FP32, so that every kernel that
// inlines it gives the same bits; product and difference rounded apart in FP64,
// as the reference does
template <typename T>
__device__ __forceinline__ T bb_value(int d, T fpost, T ux, T uy, T uz, int cpu_float)
{
    if (cpu_float) return fpost - wall_term_cpu<T>(d, (double)ux, (double)uy, (double)uz);
    const T coef = T(weight_class(d) == 1 ? 4. / 9. : weight_class(d) == 2 ? 1. / 9. : 1. / 36.);
    const T s = proj<T>(d, ux, uy, uz);
    if constexpr (sizeof(T) == 4) return __builtin_fmaf(-coef, s, fpost);
    else return fpost - coef * s;
}

// Links DIR of entry i: every fraction is loaded first, then the populations of
// the wall links, then they are stored
template <typename S, bool EVEN, int... DIR>
__device__ __forceinline__ void bb_links(const Lat& L, const BCDev& B, uint32_t i)
{
    using T = typename Compute<S>::T;
    constexpr int G = sizeof...(DIR);
    constexpr int dir[G] = {DIR...};
    const uint32_t k = B.k[i];
    bool on[G];
    bool any = false;
#pragma unroll
    for (int j = 0; j < G; ++j) {
        const int d = dir[j];
        const T q = bc_q<T>(B, d, i);
        on[j] = q >= T(0) && q <= T(1);
        any |= on[j];
    }
    if (!any || k >= L.N) return; // malformed list entry: never touch memory outside the lattice
    uint32_t kk[8];
    if (B.direct) nbrs_direct(L, k, kk);
    else nbrs_sparse(L, k, kk);
    T ux = B.vx ? bc_at<T>(B.vx, i) : T(0), uy = B.vy ? bc_at<T>(B.vy, i) : T(0), uz = B.vz ? bc_at<T>(B.vz, i) : T(0);
    T f[G];
#pragma unroll
    for (int j = 0; j < G; ++j) {
        const int d = dir[j];
        // post-collision population of direction d sits where e was read from
        const int e = inv(d);
        if (on[j])
            f[j] = Storage<S, T>::ld(plane<S>(L, slot(e, EVEN)), kk[nbr(e)], L.ld[weight_class(d)], L.sh[d]);
    }
#pragma unroll
    for (int j = 0; j < G; ++j) {
        const int d = dir[j];
        // next step (parity !EVEN) reads direction e of node k from here
        const int e = inv(d);
        if (on[j]) {
            Storage<S, T>::st(plane<S>(L, slot(e, !EVEN)), kk[nbr(e)], bb_value<T>(d, f[j], ux, uy, uz, B.cpu_float),
                              L.st[weight_class(e)], L.ss[e]);
            // keeps the branches of a switch over links apart: with their ends
            // merged, the FMA of a half's store and its conversion (one
            // instruction, one rounding) come apart and round twice
            asm volatile("" ::"n"(dir[j]));
        }
    }
}
template <typename S, bool EVEN>
__device__ __forceinline__ void bc_velocity_bb_entry(const Lat& L, const BCDev& B, uint32_t i)
{
    if (i < B.n)
        bb_links<S, EVEN, 1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15, 16, 17, 18, 19, 20, 21, 22, 23, 24, 25, 26>(L, B, i);
}

// One thread per link (PAIRS: per link and its opposite): blockIdx.y is the
// direction, so a wavefront holds one direction of 64 boundary nodes and
// everything about the link is a constant of the switch branch it takes.  Lists
// are bound by latency: with the links of a node one after another in one thread
// each waited for the one before (its fraction, its population and its store, 26
// round trips); here the chain is fraction -> population -> store, on the sparse
// layout with up to three dependent loads of neighbour indices in between.
// MI355X, us per launch, all links of a node one after another -> one per thread:
// cavity 30^3 FP32 13.6 -> 3.6, 64^3 FP64 17.5 -> 6.2; 3, 7, 13 and 26 links per
// thread: 30^3 4.3 / 4.7 / 5.8 / 7.3, 128^3 FP16 14.4 / 14.9 / 14.9 / 15.9
// against 15.9.
//
// Where a node is its own neighbour along a link (an axis of one node), the link
// and its opposite exchange the same two elements and must share a thread, loads
// first; any other element is touched by one link only.  A structured box shows
// that by its dims; on the sparse layout the caller says that no node of the list
// is its own neighbour (single_links), otherwise pairs.  One link / one pair per
// thread, us per 6 steps: cavity 20^3 FP16 43 / 48, 66^3 FP64 190 / 187; sparse
// 62x58x56 FP16 85 / 87, 150x100x110 FP16 291 / 289, FP64 987 / 994 (one link that
// looks for its opposite's neighbour itself: 87, 303, 1005).
template <typename S, bool EVEN, bool PAIRS>
__global__ void __launch_bounds__(256) k_bc_velocity_bb(Lat L, BCDev B)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= B.n) return;
#define VFX_LINK(D) \
    case D: bb_links<S, EVEN, D>(L, B, i); break;
#define VFX_PAIR(Y, D) \
    case Y: bb_links<S, EVEN, D, inv(D)>(L, B, i); break;
    if constexpr (PAIRS) switch (blockIdx.y) {
            VFX_PAIR(0, dP00) VFX_PAIR(1, d0P0) VFX_PAIR(2, d00P) VFX_PAIR(3, dPP0) VFX_PAIR(4, dPM0) VFX_PAIR(5, dP0P)
            VFX_PAIR(6, dP0M) VFX_PAIR(7, d0PP) VFX_PAIR(8, d0PM) VFX_PAIR(9, dPPP) VFX_PAIR(10, dPPM)
            VFX_PAIR(11, dPMP) VFX_PAIR(12, dMPP)
        }
    else switch (blockIdx.y + 1) {
            VFX_LINK(1) VFX_LINK(2) VFX_LINK(3) VFX_LINK(4) VFX_LINK(5) VFX_LINK(6) VFX_LINK(7) VFX_LINK(8) VFX_LINK(9)
            VFX_LINK(10) VFX_LINK(11) VFX_LINK(12) VFX_LINK(13) VFX_LINK(14) VFX_LINK(15) VFX_LINK(16) VFX_LINK(17)
            VFX_LINK(18) VFX_LINK(19) VFX_LINK(20) VFX_LINK(21) VFX_LINK(22) VFX_LINK(23) VFX_LINK(24) VFX_LINK(25)
            VFX_LINK(26)
        }
#undef VFX_PAIR
#undef VFX_LINK
}
template <typename S> hipError_t launch_velocity_bb(const Lat& L, const BCDev& B, bool even, hipStream_t st)
{
    const bool pairs = B.direct ? L.nx == 1 || L.ny == 1 || L.nz == 1 : !B.single_links;
    auto* kernel = pairs ? (even ? k_bc_velocity_bb<S, true, true> : k_bc_velocity_bb<S, false, true>)
                         : (even ? k_bc_velocity_bb<S, true, false> : k_bc_velocity_bb<S, false, false>);
    hipLaunchKernelGGL(kernel, dim3((B.n + 255u) / 256u, pairs ? 13 : 26), dim3(256), 0, st, L, B);
    return hipGetLastError();
}

// Interpolated bounce-back family (NoSlipInterpolatedCompressible.cu:44-378,
// VelocityInterpolatedCompressible.cu:44-…, SlipCompressible.cu:45-…, formulas
// KernelUtilities.h:171-197): from the post-collision populations of the
// boundary node, density and velocity (with the sum order those kernels use),
// the symmetric equilibrium part of each wall link, and the Bouzidi-type
// interpolation with the subgrid distance q.  KIND: 1 no-slip, 2 velocity, 3 slip.
//
// The node part of the interpolated boundaries: density, velocity, rates and
// the boundary velocity of the node's post-collision populations p.
template <typename T> struct InterpNode {
    T drho, vx1, vx2, vx3, cu_sq, omega, inv1mo, VX, VY, VZ;
};
template <typename T, int KIND>
__device__ __forceinline__ InterpNode<T> interp_node(const Lat& L, const BCDev& B, uint32_t i, uint32_t k,
                                                     const T (&p)[27], int kd)
{
    // no contraction into FMAs here: which product the compiler would fuse
    // depends on the code around the inlined body (a shared subexpression
    // changes the choice), and the separate boundary kernel and the fused
    // collide-stream kernel must give the same bits
#pragma clang fp contract(off)
    InterpNode<T> n;
    const T drho = p[dPMP] + p[dMPP] + p[dPPP] + p[dMMP] + p[dPMM] + p[dMPM] + p[dPPM] + p[dMMM] + p[d0PM] + p[d0MP] +
                   p[d0PP] + p[d0MM] + p[dP0M] + p[dM0P] + p[dP0P] + p[dM0M] + p[dPM0] + p[dMP0] + p[dPP0] + p[dMM0] +
                   p[d00P] + p[d00M] + p[d0P0] + p[d0M0] + p[dP00] + p[dM00] + p[d000];
    n.drho = drho;
    // division by 1 + drho: exact in FP64 (reference order), the hardware
    // reciprocal in FP32
    const T ovr = sizeof(T) == 4 ? T(__builtin_amdgcn_rcpf(float(T(1) + drho))) : T(0);
    auto per_rho = [&](T x) -> T {
        if constexpr (sizeof(T) == 4) return x * ovr;
        else return x / (T(1) + drho);
    };
    n.vx1 = per_rho((((p[dPMP] - p[dMPM]) - (p[dMPP] - p[dPMM])) + ((p[dPPP] - p[dMMM]) - (p[dMMP] - p[dPPM])) +
                     ((p[dP0M] - p[dM0P]) + (p[dP0P] - p[dM0M])) + ((p[dPM0] - p[dMP0]) + (p[dPP0] - p[dMM0])) +
                     (p[dP00] - p[dM00])));
    n.vx2 = per_rho(((-(p[dPMP] - p[dMPM]) + (p[dMPP] - p[dPMM])) + ((p[dPPP] - p[dMMM]) - (p[dMMP] - p[dPPM])) +
                     ((p[d0PM] - p[d0MP]) + (p[d0PP] - p[d0MM])) + (-(p[dPM0] - p[dMP0]) + (p[dPP0] - p[dMM0])) +
                     (p[d0P0] - p[d0M0])));
    n.vx3 = per_rho((((p[dPMP] - p[dMPM]) + (p[dMPP] - p[dPMM])) + ((p[dPPP] - p[dMMM]) + (p[dMMP] - p[dPPM])) +
                     (-(p[d0PM] - p[d0MP]) + (p[d0PP] - p[d0MM])) + ((p[dP0P] - p[dM0M]) - (p[dP0M] - p[dM0P])) +
                     (p[d00P] - p[d00M])));
    n.cu_sq = T(1.5) * (n.vx1 * n.vx1 + n.vx2 * n.vx2 + n.vx3 * n.vx3) * (T(1) + drho);
    T omega = (T)B.omega;
    // SlipTurbulentViscosityCompressible.cu:130-134: the node's rate with its turbulent viscosity
    if constexpr (KIND == VFX_BC_SLIP_TURBULENT_VISCOSITY)
        omega = omega / (T(1) + T(3) * omega * fmax(T(0), ((const T*)L.nut)[k]));
    n.omega = omega;
    n.inv1mo = sizeof(T) == 4 ? T(1) / (T(1) - omega) : T(0);
    n.VX = n.VY = n.VZ = T(0);
    return n;
}
// the wall velocity of the velocity kinds
template <typename T> __device__ __forceinline__ void interp_wall_velocity(InterpNode<T>& n, const BCDev& B, uint32_t i, int kd)
{
    if (kd == VFX_BC_VELOCITY_INTERPOLATED || kd == VFX_BC_VELOCITY_PRESSURE_INTERPOLATED ||
        kd == VFX_BC_PRECURSOR_VELOCITY) {
        n.VX = B.vx ? bc_at<T>(B.vx, i) : T(0);
        n.VY = B.vy ? bc_at<T>(B.vy, i) : T(0);
        n.VZ = B.vz ? bc_at<T>(B.vz, i) : T(0);
    }
}

// The population re-entering along a wall link of fraction q (0 <= q <= 1):
// f, fi the node's post-collision populations of the link and its opposite,
// w the link weight, vlb = c . u of the node, vbc = c . u of the wall.
template <typename T>
__device__ __forceinline__ T interp_link_value(const InterpNode<T>& n, int kd, T w, T vlb, T vbc, T q, T f, T fi)
{
#pragma clang fp contract(off)
    const T feq = w * (n.drho + T(4.5) * vlb * vlb * (T(1) + n.drho) - n.cu_sq);
    // FP64 keeps the reference's divisions (bit parity with the CPU
    // restatement); the FP32 arithmetic of the reduced forms uses one
    // hardware reciprocal per link and 1/(1 - omega) once per node
    T a, r1q;
    if constexpr (sizeof(T) == 4) {
        r1q = __builtin_amdgcn_rcpf(T(1) + q);
        a = (T(1) - q) * r1q * (f - fi + (f + fi - T(2) * feq * n.omega) * n.inv1mo) * T(0.5);
    } else {
        r1q = T(0);
        a = (T(1) - q) / (T(1) + q) * (f - fi + (f + fi - T(2) * feq * n.omega) / (T(1) - n.omega)) * T(0.5);
    }
    T v;
    if (kd == VFX_BC_NOSLIP_INTERPOLATED) {
        if constexpr (sizeof(T) == 4) v = a + q * (f + fi) * r1q;
        else v = a + (q * (f + fi)) / (T(1) + q);
    } else {
        if constexpr (sizeof(T) == 4) v = a + (q * (f + fi) - T(6) * w * vbc) * r1q;
        else v = a + (q * (f + fi) - T(6) * w * vbc) / (T(1) + q);
        // getInterpolatedDistributionForVeloWithPressureBC (KernelUtilities.h:207-213):
        // the entering population carries the bulk pressure
        if (kd == VFX_BC_VELOCITY_PRESSURE_INTERPOLATED || kd == VFX_BC_PRECURSOR_VELOCITY) v = v - w * n.drho;
    }
    return v;
}

// The links of boundary entry i at node k from its post-collision
// populations p (indexed by direction): computes and stores the population
// re-entering along every wall link.  KIND >= 0 fixes the kind at compile
// time; KIND = -1 takes it from `kind` at run time (kinds 1, 2, 3, 5).
template <typename S, typename T, bool EVEN, int KIND>
__device__ __forceinline__ void interp_links(const Lat& L, const BCDev& B, uint32_t i, uint32_t k,
                                             const uint32_t (&kk)[8], const T (&p)[27], int kind = KIND)
{
#pragma clang fp contract(off)
    const int kd = KIND >= 0 ? KIND : kind;
    InterpNode<T> n = interp_node<T, KIND>(L, B, i, k, p, kd);
    // all link fractions first: loaded inside the link loop, each q waited for
    // the previous link's store as well (one memory counter covers both) and
    // the 26 links ran as 26 round trips
    T qs[27];
#pragma unroll
    for (int d = 1; d < 27; ++d) qs[d] = bc_q<T>(B, d, i);
    interp_wall_velocity<T>(n, B, i, kd);
    if constexpr (KIND == VFX_BC_PRECURSOR_VELOCITY) {
        // PrecursorNonReflectiveCompressible.cu:112-114: (velocityX + (1 - tr) last + tr current) / velocityRatio
        const PlaneStencil<T> s = plane_stencil<T>(B, i);
        if (!s.ok) return; // malformed plane index: never read outside the planes
        n.VX += (T)B.pu[0];
        n.VY += (T)B.pu[1];
        n.VZ += (T)B.pu[2];
        const T tr = (T)B.tratio, vr = (T)B.vratio;
        const T* last = (const T*)B.plast;
        const T* cur = (const T*)B.pcur;
        const size_t np = B.n_pre;
        n.VX = (n.VX + (T(1) - tr) * plane_value(s, last) + tr * plane_value(s, cur)) / vr;
        n.VY = (n.VY + (T(1) - tr) * plane_value(s, last + np) + tr * plane_value(s, cur + np)) / vr;
        n.VZ = (n.VZ + (T(1) - tr) * plane_value(s, last + 2 * np) + tr * plane_value(s, cur + 2 * np)) / vr;
    }
    bool fx = false, fy = false, fz = false; // slip: axes normal to a face link
#pragma unroll
    for (int d = 1; d < 27; ++d) {
        const T q = qs[d];
        if (!(q >= T(0) && q <= T(1))) continue;
        const T w = weight<T>(d);
        const T vlb = proj<T>(d, n.vx1, n.vx2, n.vx3);
        T f = p[d], fi = p[inv(d)];
        if constexpr (KIND == VFX_BC_PRECURSOR_VELOCITY) {
            // kept from PrecursorNonReflectiveCompressible.cu:383 and :392: the
            // d0PM link takes f_0PP for its opposite, the d0MP link f_0PP for its own
            if (d == d0PM) fi = p[d0PP];
            if (d == d0MP) f = p[d0PP];
        }
        T vbc = T(0);
        if (kd == VFX_BC_SLIP || kd == VFX_BC_SLIP_TURBULENT_VISCOSITY) {
            if (weight_class(d) == 1) {
                if (cx(d) != 0) fx = true;
                if (cy(d) != 0) fy = true;
                if (cz(d) != 0) fz = true;
            }
            const T sx = fx ? T(0) : n.vx1, sy = fy ? T(0) : n.vx2, sz = fz ? T(0) : n.vx3;
            vbc = proj<T>(d, sx, sy, sz);
        } else if (kd != VFX_BC_NOSLIP_INTERPOLATED) {
            vbc = proj<T>(d, n.VX, n.VY, n.VZ);
        }
        const T v = interp_link_value<T>(n, kd, w, vlb, vbc, q, f, fi);
        const int e = inv(d);
        // the precursor inlet writes with the parity's own pointers
        // (PrecursorNonReflectiveCompressible.cu:142): over the outgoing
        // population it read, which the node reads back as e two steps later
        constexpr bool WRITE_EVEN = KIND == VFX_BC_PRECURSOR_VELOCITY ? EVEN : !EVEN;
        Storage<S, T>::st(plane<S>(L, slot(e, WRITE_EVEN)), kk[nbr(e)], v, L.st[weight_class(e)], L.ss[e]);
    }
}

template <typename S, bool EVEN, int KIND>
__device__ __forceinline__ void bc_interp_entry(const Lat& L, const BCDev& B, uint32_t i, int kind = KIND)
{
    using T = typename Compute<S>::T;
    if (i >= B.n) return;
    uint32_t kk[8];
    const uint32_t k = B.k[i];
    if (k >= L.N) return;
    if (B.direct) nbrs_direct(L, k, kk);
    else nbrs_sparse(L, k, kk);
    T p[27]; // post-collision population of direction d
#pragma unroll
    for (int d = 0; d < 27; ++d) {
        const int e = inv(d);
        p[d] = Storage<S, T>::ld(plane<S>(L, slot(e, EVEN)), kk[nbr(e)], L.ld[weight_class(d)], L.sh[d]);
    }
    interp_links<S, T, EVEN, KIND>(L, B, i, k, kk, p, kind);
}

template <typename S, bool EVEN, int KIND>
__global__ void __launch_bounds__(256) k_bc_interp(Lat L, BCDev B)
{
    bc_interp_entry<S, EVEN, KIND>(L, B, blockIdx.x * blockDim.x + threadIdx.x);
}

// Precursor distributions (PrecursorDistributions.cu:44-185): post-collision,
// parity EVEN.  The nine populations with a positive x component entering
// boundary node k are the blended plane values f0..f8, written for the next
// step like the other post-collision boundary conditions.
template <typename S, bool EVEN>
__global__ void __launch_bounds__(256) k_bc_precursor_dist(Lat L, BCDev B)
{
    using T = typename Compute<S>::T;
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= B.n) return;
    const uint32_t k = B.k[i];
    if (k >= L.N) return;
    uint32_t kk[8];
    if (B.direct) nbrs_direct(L, k, kk);
    else nbrs_sparse(L, k, kk);
    const PlaneStencil<T> s = plane_stencil<T>(B, i);
    if (!s.ok) return; // malformed plane index: never read outside the planes
    constexpr int dirs[9] = {dP00, dPP0, dPM0, dP0P, dP0M, dPPP, dPMP, dPPM, dPMM};
#pragma unroll
    for (int c = 0; c < 9; ++c) {
        const int x = dirs[c];
        const T v = plane_blend(B, s, c);
        Storage<S, T>::st(plane<S>(L, slot(x, !EVEN)), kk[nbr(x)], v, L.st[weight_class(x)], L.ss[x]);
    }
}

// Non-equilibrium pressure boundary (PressureNonEquilibriumCompressible.cu:45-…):
// pre-collision, parity EVEN of the step about to run.  The populations of the
// inward neighbour keep their non-equilibrium part and get the equilibrium of
// the prescribed density; they replace the boundary node's populations of every
// direction not pointing out of the domain (c_d . normal <= 0).
template <typename T> __device__ __forceinline__ T feq_shifted(int d, T drho, T vx1, T vx2, T vx3, T cusq)
{
#pragma clang fp contract(off)
    if (d == d000) return T(8. / 27.) * (drho - (drho + T(1)) * cusq);
    const T cu = proj<T>(d, vx1, vx2, vx3);
    return weight<T>(d) * (drho + (drho + T(1)) * (T(3) * cu + T(4.5) * cu * cu - cusq));
}

// PressureNonEquilibriumCompressible.cu: density deviation and velocity v of the
// inward neighbour's populations (in cube order), and its population f of
// direction d with the equilibrium replaced by the one of the prescribed density
// rho_bc.  No FMA contraction: the same bits wherever they are inlined.
template <typename T> __device__ __forceinline__ void pressure_moments(const T (&m)[27], T (&v)[4])
{
#pragma clang fp contract(off)
#define F(d) m[slot_of(d)]
    // getCompressibleMacroscopicValues (MacroscopicQuantities.h:117-127)
    const T corners = ((F(dPPP) + F(dMMM)) + (F(dMPM) + F(dPMP))) + ((F(dMPP) + F(dPMM)) + (F(dMMP) + F(dPPM)));
    const T edges = (((F(d0MP) + F(d0PM)) + (F(d0MM) + F(d0PP))) + ((F(dM0P) + F(dP0M)) + (F(dM0M) + F(dP0P)))) +
                    ((F(dMP0) + F(dPM0)) + (F(dMM0) + F(dPP0)));
    const T faces = ((F(dM00) + F(dP00)) + (F(d0M0) + F(d0P0))) + (F(d00M) + F(d00P));
    const T drho1 = ((corners + edges) + F(d000)) + faces;
    T vx1 = (((F(dPPP) - F(dMMM)) + (F(dPMP) - F(dMPM))) + ((F(dPMM) - F(dMPP)) + (F(dPPM) - F(dMMP)))) +
            (((F(dP0M) - F(dM0P)) + (F(dP0P) - F(dM0M))) + ((F(dPM0) - F(dMP0)) + (F(dPP0) - F(dMM0)))) +
            (F(dP00) - F(dM00));
    T vx2 = (((F(dPPP) - F(dMMM)) + (F(dMPM) - F(dPMP))) + ((F(dMPP) - F(dPMM)) + (F(dPPM) - F(dMMP)))) +
            (((F(d0PM) - F(d0MP)) + (F(d0PP) - F(d0MM))) + ((F(dMP0) - F(dPM0)) + (F(dPP0) - F(dMM0)))) +
            (F(d0P0) - F(d0M0));
    T vx3 = (((F(dPPP) - F(dMMM)) + (F(dPMP) - F(dMPM))) + ((F(dMPP) - F(dPMM)) + (F(dMMP) - F(dPPM)))) +
            (((F(d0MP) - F(d0PM)) + (F(d0PP) - F(d0MM))) + ((F(dM0P) - F(dP0M)) + (F(dP0P) - F(dM0M)))) +
            (F(d00P) - F(d00M));
    const T oor = T(1) / (drho1 + T(1));
#undef F
    v[0] = drho1;
    v[1] = vx1 * oor;
    v[2] = vx2 * oor;
    v[3] = vx3 * oor;
}
template <typename T> __device__ __forceinline__ T pressure_value(int d, T f, const T (&v)[4], T rho_bc)
{
#pragma clang fp contract(off)
    const T cusq = T(1.5) * (v[1] * v[1] + v[2] * v[2] + v[3] * v[3]);
    if constexpr (sizeof(T) == 4) {
        // the two equilibria differ by w (rho_bc - drho) (1 + 3 cu + 4.5 cu^2 - cusq)
        const T cu = d == d000 ? T(0) : proj<T>(d, v[1], v[2], v[3]);
        const T e = __builtin_fmaf(__builtin_fmaf(T(4.5), cu, T(3)), cu, T(1) - cusq);
        return __builtin_fmaf(weight<T>(d) * (rho_bc - v[0]), e, f);
    }
    return (f - feq_shifted<T>(d, v[0], v[1], v[2], v[3], cusq)) + feq_shifted<T>(d, rho_bc, v[1], v[2], v[3], cusq);
}

template <typename S, bool EVEN>
__device__ __forceinline__ void bc_pressure_entry(const Lat& L, const BCDev& B, uint32_t i)
{
    using T = typename Compute<S>::T;
    if (i >= B.n) return;
    const uint32_t k = B.k[i], kn = B.kn[i];
    if (k >= L.N || kn >= L.N) return;
    uint32_t kk[8], kkn[8];
    if (B.direct) {
        nbrs_direct(L, k, kk);
        nbrs_direct(L, kn, kkn);
    } else {
        nbrs_sparse(L, k, kk);
        nbrs_sparse(L, kn, kkn);
    }
    T m[27];
    gather<S, T, EVEN>(L, kkn, m);
    T v[4];
    pressure_moments<T>(m, v);
    const T rho_bc = bc_at<T>(B.rho, i);
    const int nx = cx(B.normal), ny = cy(B.normal), nz = cz(B.normal);
#pragma unroll
    for (int d = 0; d < 27; ++d) {
        if (cx(d) * nx + cy(d) * ny + cz(d) * nz > 0) continue;
        Storage<S, T>::st(plane<S>(L, slot(d, EVEN)), kk[nbr(d)], pressure_value<T>(d, m[slot_of(d)], v, rho_bc),
                          L.st[weight_class(d)], L.ss[d]);
    }
}

template <typename S, bool EVEN>
__global__ void __launch_bounds__(256) k_bc_pressure(Lat L, BCDev B)
{
    bc_pressure_entry<S, EVEN>(L, B, blockIdx.x * blockDim.x + threadIdx.x);
}

// Several boundary groups, possibly of different lattices of one storage
// type, in one launch: block b runs the job whose block range holds b (jobs
// in increasing first_block), at that job's parity (bit j of even_mask).
// Kinds 0 (velocity bounce-back), 1, 2, 3, 5 (interpolated) and 4 (pressure),
// each entry exactly as its own kernel computes it.  The groups of one launch
// must not touch each other's elements (the post-collision groups of a step
// write wall nodes' elements only; a pressure group runs with the groups of
// its own phase).
constexpr int kMaxBCJobs = 32;
struct BCJob {
    Lat L;
    BCDev B;
    int32_t kind;
    uint32_t first_block;
};
template <typename S>
__global__ void __launch_bounds__(256) k_bc_set(const BCJob* __restrict__ jobs, uint32_t njobs, uint32_t even_mask)
{
    uint32_t j = 0;
    for (uint32_t t = 1; t < njobs; ++t)
        if (jobs[t].first_block <= blockIdx.x) j = t;
    const BCJob& J = jobs[j];
    const uint32_t i = (blockIdx.x - J.first_block) * blockDim.x + threadIdx.x;
    const bool even = (even_mask >> j) & 1u;
    switch (J.kind) {
    case VFX_BC_VELOCITY_BOUNCE_BACK:
        if (even) bc_velocity_bb_entry<S, true>(J.L, J.B, i);
        else bc_velocity_bb_entry<S, false>(J.L, J.B, i);
        break;
    case VFX_BC_PRESSURE_NEQ:
        if (even) bc_pressure_entry<S, true>(J.L, J.B, i);
        else bc_pressure_entry<S, false>(J.L, J.B, i);
        break;
    default:
        if (even) bc_interp_entry<S, true, -1>(J.L, J.B, i, J.kind);
        else bc_interp_entry<S, false, -1>(J.L, J.B, i, J.kind);
        break;
    }
}


// Wall-model (stress) boundaries (BoundaryConditions/Stress/*.cu with the
// instantaneous wall model iMEM, iMEM.cuh:43-141): post-collision, parity EVEN.
// MODE 0 StressCompressible (interpolated no-slip with pressure at the node's
// turbulent-viscosity rate, wall term / (1 + q)), 1 StressBounceBackCompressible,
// 2 StressBounceBackPressureCompressible.  The links are visited in the
// kernels' order (E W N S T B NE SW SE NW TE BW BE TW TN BS BN TS TNE BSW BNE
// TSW TSE BNW BSE TNW), which fixes the wall-momentum sums.  Kept from the
// reference: the wall model takes q of the B (00M) link, forceFactor 1 + q(B)
// in MODE 0, the NE link's pressure term in MODE 0 weighs 2/27, and the
// launcher hands velocityY in for the z velocity (Stress.cu:57-59), which the
// launch below reproduces by passing the y array twice.
__host__ __device__ constexpr int stress_link(int j)
{
    constexpr int order[26] = {1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15, 16, 17, 18, 19, 26, 23, 22, 21, 24, 25, 20};
    return order[j];
}

template <typename T>
__device__ __forceinline__ void wall_model(const BCDev& B, uint32_t i, uint32_t kN, const T* vx, const T* vy, const T* vz,
                                           T vxw, T vyw, T vzw, T rho, T q, T forceFactor, T wmx, T wmy, T wmz,
                                           T& Ux, T& Uy, T& Uz)
{
    const T* nrm[3] = {(const T*)B.wm_normal[0], (const T*)B.wm_normal[1], (const T*)B.wm_normal[2]};
    T* el[3] = {(T*)B.wm_el[0], (T*)B.wm_el[1], (T*)B.wm_el[2]};
    T* wm[3] = {(T*)B.wm_wall[0], (T*)B.wm_wall[1], (T*)B.wm_wall[2]};
    const T eps = T(0.001f);
    const T nx = nrm[0][i], ny = nrm[1][i], nz = nrm[2][i];
    T ex = eps * vx[kN] + (T(1.0) - eps) * el[0][i];
    T ey = eps * vy[kN] + (T(1.0) - eps) * el[1][i];
    T ez = eps * vz[kN] + (T(1.0) - eps) * el[2][i];
    el[0][i] = ex;
    el[1][i] = ey;
    el[2][i] = ez;
    T mx = eps * vxw + (T(1.0) - eps) * wm[0][i];
    T my = eps * vyw + (T(1.0) - eps) * wm[1][i];
    T mz = eps * vzw + (T(1.0) - eps) * wm[2][i];
    wm[0][i] = mx;
    wm[1][i] = my;
    wm[2][i] = mz;
    const T dn_el = ex * nx + ey * ny + ez * nz;
    ex -= dn_el * nx;
    ey -= dn_el * ny;
    ez -= dn_el * nz;
    const T mag_el = sqrt(ex * ex + ey * ey + ez * ez);
    const T dn_wm = mx * nx + my * ny + mz * nz;
    mx -= dn_wm * nx;
    my -= dn_wm * ny;
    mz -= dn_wm * nz;
    const T mag_wm = sqrt(mx * mx + my * my + mz * mz);
    const T dn_w = vxw * nx + vyw * ny + vzw * nz;
    const T wx = vxw - dn_w * nx, wy = vyw - dn_w * ny, wz = vzw - dn_w * nz;
    const T z = (T)B.wm_offset[i] + q;
    const T kappa = T(0.4);
    const T u_star = mag_el * kappa / (log(z / ((const T*)B.wm_z0)[i]));
    if (B.wm_ustar) ((T*)B.wm_ustar)[i] = u_star;
    const T tau_w = u_star * u_star;
    const T A = T(1.0);
    const T Fwx = (tau_w * A) * (wx / mag_wm);
    const T Fwy = (tau_w * A) * (wy / mag_wm);
    const T Fwz = (tau_w * A) * (wz / mag_wm);
    const T mdn = wmx * nx + wmy * ny + wmz * nz;
    const T Fx = Fwx - (wmx - mdn * nx) / rho;
    const T Fy = Fwy - (wmy - mdn * ny) / rho;
    const T Fz = Fwz - (wmz - mdn * nz) / rho;
    const T clip = T(2.0);
    const T cx_ = clip * ex, cy_ = clip * ey, cz_ = clip * ez;
    auto clamp = [&](T c, T F) -> T {
        const T v = T(-3.0) * F * forceFactor;
        return c > -c ? fmin(c, fmax(-c, v)) : fmax(c, fmin(-c, v));
    };
    Ux = clamp(cx_, Fx);
    Uy = clamp(cy_, Fy);
    Uz = clamp(cz_, Fz);
}

template <typename S, bool EVEN, int MODE>
__global__ void __launch_bounds__(256) k_bc_stress(Lat L, BCDev B)
{
    using T = typename Compute<S>::T;
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= B.n) return;
    const uint32_t k = B.k[i], kN = B.kn[i];
    if (k >= L.N || kN >= L.N) return;
    uint32_t kk[8];
    if (B.direct) nbrs_direct(L, k, kk);
    else nbrs_sparse(L, k, kk);
    T p[27];
#pragma unroll
    for (int d = 0; d < 27; ++d) {
        const int e = inv(d);
        p[d] = Storage<S, T>::ld(plane<S>(L, slot(e, EVEN)), kk[nbr(e)], L.ld[weight_class(d)], L.sh[d]);
    }
    const T drho = p[dPMP] + p[dMPP] + p[dPPP] + p[dMMP] + p[dPMM] + p[dMPM] + p[dPPM] + p[dMMM] + p[d0PM] + p[d0MP] +
                   p[d0PP] + p[d0MM] + p[dP0M] + p[dM0P] + p[dP0P] + p[dM0M] + p[dPM0] + p[dMP0] + p[dPP0] + p[dMM0] +
                   p[d00P] + p[d00M] + p[d0P0] + p[d0M0] + p[dP00] + p[dM00] + p[d000];
    const T vx1 = (((p[dPMP] - p[dMPM]) - (p[dMPP] - p[dPMM])) + ((p[dPPP] - p[dMMM]) - (p[dMMP] - p[dPPM])) +
                   ((p[dP0M] - p[dM0P]) + (p[dP0P] - p[dM0M])) + ((p[dPM0] - p[dMP0]) + (p[dPP0] - p[dMM0])) +
                   (p[dP00] - p[dM00])) /
                  (T(1) + drho);
    const T vx2 = ((-(p[dPMP] - p[dMPM]) + (p[dMPP] - p[dPMM])) + ((p[dPPP] - p[dMMM]) - (p[dMMP] - p[dPPM])) +
                   ((p[d0PM] - p[d0MP]) + (p[d0PP] - p[d0MM])) + (-(p[dPM0] - p[dMP0]) + (p[dPP0] - p[dMM0])) +
                   (p[d0P0] - p[d0M0])) /
                  (T(1) + drho);
    const T vx3 = (((p[dPMP] - p[dMPM]) + (p[dMPP] - p[dPMM])) + ((p[dPPP] - p[dMMM]) + (p[dMMP] - p[dPPM])) +
                   (-(p[d0PM] - p[d0MP]) + (p[d0PP] - p[d0MM])) + ((p[dP0P] - p[dM0M]) - (p[dP0M] - p[dM0P])) +
                   (p[d00P] - p[d00M])) /
                  (T(1) + drho);
    const T cu_sq = T(1.5) * (vx1 * vx1 + vx2 * vx2 + vx3 * vx3) * (T(1) + drho);
    T om = (T)B.omega;
    if constexpr (MODE == 0) {
        const T nut = L.nut ? ((const T*)L.nut)[k] : T(0);
        om = om / (T(1) + T(3) * om * fmax(T(0), nut));
    }
    T qs[27];
#pragma unroll
    for (int d = 1; d < 27; ++d) qs[d] = bc_q<T>(B, d, i);
    T fin[27] = {};
    T wmx = T(0), wmy = T(0), wmz = T(0);
#pragma unroll
    for (int j = 0; j < 26; ++j) {
        const int d = stress_link(j);
        const T q = qs[d];
        if (!(q >= T(0) && q <= T(1))) continue;
        const T f = p[d], fi = p[inv(d)];
        T v;
        if constexpr (MODE == 0) {
            const T w = weight<T>(d);
            const T vlb = proj<T>(d, vx1, vx2, vx3);
            const T feq = w * (drho + T(4.5) * vlb * vlb * (T(1) + drho) - cu_sq);
            const T wp = d == dPP0 ? T(2. / 27.) : w; // the NE link's pressure weight
            v = (T(1) - q) / (T(1) + q) * (f - fi + (f + fi - T(2) * feq * om) / (T(1) - om)) * T(0.5) +
                (q * (f + fi)) / (T(1) + q) - wp * drho;
        } else if constexpr (MODE == 1) {
            v = f;
        } else {
            v = f - weight<T>(d) * drho;
        }
        fin[inv(d)] = v;
        const T s = f + v;
        if (cx(d) > 0) wmx += s;
        if (cx(d) < 0) wmx -= s;
        if (cy(d) > 0) wmy += s;
        if (cy(d) < 0) wmy -= s;
        if (cz(d) > 0) wmz += s;
        if (cz(d) < 0) wmz -= s;
    }
    const T qB = qs[d00M];
    T Ux, Uy, Uz;
    wall_model<T>(B, i, kN, (const T*)L.vx, (const T*)L.vy, (const T*)L.vy, vx1, vx2, vx3, T(1) + drho, qB,
                  MODE == 0 ? T(1.0) + qB : T(1.0), wmx, wmy, wmz, Ux, Uy, Uz);
#pragma unroll
    for (int j = 0; j < 26; ++j) {
        const int d = stress_link(j);
        const T q = qs[d];
        if (!(q >= T(0) && q <= T(1))) continue;
        T t = T(6) * weight<T>(d) * proj<T>(d, Ux, Uy, Uz);
        if constexpr (MODE == 0) t = t / (T(1) + q);
        const int e = inv(d);
        Storage<S, T>::st(plane<S>(L, slot(e, !EVEN)), kk[nbr(e)], fin[e] - t, L.st[weight_class(e)], L.ss[e]);
        if (cx(d) > 0) wmx += -t;
        if (cx(d) < 0) wmx -= -t;
        if (cy(d) > 0) wmy += -t;
        if (cy(d) < 0) wmy -= -t;
        if (cz(d) > 0) wmz += -t;
        if (cz(d) < 0) wmz -= -t;
    }
    if (B.wm_force[0]) {
        ((T*)B.wm_force[0])[i] = wmx;
        ((T*)B.wm_force[1])[i] = wmy;
        ((T*)B.wm_force[2])[i] = wmz;
    }
}

// Non-reflecting outflow (OutflowNonReflecting.cu:44-280; with CORR
// OutflowNonReflectingPressureCorrection.cu:46-245): pre-collision, parity EVEN.
// From the node's populations f and its inward neighbour's fn, every direction
// d entering through the boundary face (c_d . normal < 0) gets
// fn[d] cs + (1 - cs) f[d] [- w_d corr drho(f)], cs = 1 / sqrtf(3), written
// into the element the next collision of the other parity reads as direction
// d of the node: slot (d, !EVEN) at the node's own neighbour index.  That
// element belongs to the node across the boundary, which does not collide, so
// the collision of parity EVEN leaves it alone.  The corrected kernel builds
// its "neighbour" indices from the boundary node, so for directions with a
// negative component fn[d] is the node's own value; kept as is.  A normal that
// is not a face direction writes nothing (the kernels' default branch).
template <typename S, bool EVEN, bool CORR>
__global__ void __launch_bounds__(256) k_bc_outflow(Lat L, BCDev B)
{
    using T = typename Compute<S>::T;
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= B.n) return;
    const uint32_t k = B.k[i], kn = B.kn[i];
    if (k >= L.N || kn >= L.N) return;
    const int nx = cx(B.normal), ny = cy(B.normal), nz = cz(B.normal);
    if (nx * nx + ny * ny + nz * nz != 1) return;
    uint32_t kk[8], kkn[8];
    if (B.direct) {
        nbrs_direct(L, k, kk);
        nbrs_direct(L, kn, kkn);
    } else {
        nbrs_sparse(L, k, kk);
        nbrs_sparse(L, kn, kkn);
    }
    T m[27], mn[27];
    gather<S, T, EVEN>(L, kk, m);
    gather<S, T, EVEN>(L, kkn, mn);
    T f[27], fn[27];
#pragma unroll
    for (int s = 0; s < 27; ++s) {
        const int d = dir_at(s);
        f[d] = m[s];
        fn[d] = (CORR && nbr(d) != 0) ? m[s] : mn[s];
    }
    T rc = T(0);
    if constexpr (CORR) {
        // vf::lbm::getDensity (MacroscopicQuantities.h:55-64)
        const T corners = ((f[dPPP] + f[dMMM]) + (f[dMPM] + f[dPMP])) + ((f[dMPP] + f[dPMM]) + (f[dMMP] + f[dPPM]));
        const T edges = (((f[d0MP] + f[d0PM]) + (f[d0MM] + f[d0PP])) + ((f[dM0P] + f[dP0M]) + (f[dM0M] + f[dP0P]))) +
                        ((f[dMP0] + f[dPM0]) + (f[dMM0] + f[dPP0]));
        const T faces = ((f[dM00] + f[dP00]) + (f[d0M0] + f[d0P0])) + (f[d00M] + f[d00P]);
        rc = (T)B.corr * (((corners + edges) + f[d000]) + faces);
    }
    const T cs = T(1) / (T)sqrtf(3.f);
#pragma unroll
    for (int d = 1; d < 27; ++d) {
        if (cx(d) * nx + cy(d) * ny + cz(d) * nz >= 0) continue;
        T v = fn[d] * cs + (T(1) - cs) * f[d];
        if constexpr (CORR) v = v - weight<T>(d) * rc;
        Storage<S, T>::st(plane<S>(L, slot(d, !EVEN)), kk[nbr(d)], v, L.st[weight_class(d)], L.ss[d]);
    }
}

// ---------------------------------------------- fused boundary conditions ----
// The non-equilibrium pressure boundary on a face normal to +-x
// (PressureNonEquilibriumCompressible, pre-collision) inside the collide-stream
// kernel of a structured (direct) lattice: on such a face every element a
// boundary node touches sits in its own cache line (x is the fastest index), so
// a boundary kernel moves ~64 times the bytes it uses.  Node k's incoming
// populations are replaced at the start of the next step from its inward
// neighbour k -+ 1, whose pre-collision populations the lane beside it has just
// gathered, instead of by a kernel after the parity flip.  The values are the
// ones that kernel would store and the collision read back (the storage round
// trip is applied), so fused and separate runs agree bit for bit.
// Node k belongs to the group iff bit k of `mask` is set; its entry is
// base[k/32] + the number of set bits below it in its word (entries sorted by
// node).
struct FusedGroup {
    const uint32_t* mask;
    const uint32_t* base;
    BCDev B;
    int32_t kind;
};

// what a store of v as direction d followed by a load gives back (the value
// the separate boundary kernels exchange through memory)
template <typename S, typename T> __device__ __forceinline__ T round_trip(T v, float st, float ss, float ld, float sh)
{
    if constexpr (sizeof(S) == 2) return Storage<S, T>::dec2(Storage<S, T>::enc2(v, st, ss), ld, sh);
    else return v;
}

// x of the lane before this one (PX) or after it, across the whole wavefront
// (DPP wave_shr / wave_shl; the end lane, which has no such lane, gets 0)
template <bool PX> __device__ __forceinline__ float lane_beside(float x)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), PX ? 0x138 : 0x130, 0xf, 0xf, true));
}
template <bool PX> __device__ __forceinline__ double lane_beside(double x)
{
    const uint64_t b = __builtin_bit_cast(uint64_t, x);
    const uint64_t lo = (uint32_t)__builtin_amdgcn_mov_dpp((int)(uint32_t)b, PX ? 0x138 : 0x130, 0xf, 0xf, true);
    const uint64_t hi = (uint32_t)__builtin_amdgcn_mov_dpp((int)(uint32_t)(b >> 32), PX ? 0x138 : 0x130, 0xf, 0xf, true);
    return __builtin_bit_cast(double, hi << 32 | lo);
}
// the boundary nodes of a wavefront take their values from the lane beside them
// (PX: outward normal +x, the inward neighbour is the lane before); every lane
// of the wavefront runs this
template <typename S, typename T, bool PX>
__device__ __forceinline__ void fused_pressure(const Lat& L, const FusedGroup& G, bool mine, T rho_bc, T (&m)[27])
{
    T own[4], v[4];
    pressure_moments<T>(m, own);
#pragma unroll
    for (int c = 0; c < 4; ++c) v[c] = lane_beside<PX>(own[c]);
#pragma unroll
    for (int s = 0; s < 27; ++s) {
        const int d = dir_at(s);
        if (PX ? cx(d) > 0 : cx(d) < 0) continue; // pointing out of the domain
        const int c = weight_class(d);
        const T f = round_trip<S, T>(pressure_value<T>(d, lane_beside<PX>(m[s]), v, rho_bc), L.st[c], L.ss[d], L.ld[c], L.sh[d]);
        m[s] = mine ? f : m[s];
    }
}

// The structured K17 step with the pressure group inside: where a wavefront
// holds boundary nodes, each takes its neighbour's populations from the lane
// beside it.  It costs its instructions (~250) and one more round trip to memory
// in the wavefronts that hold a boundary node, where a kernel of its own reads
// 27 and writes 18 cache lines per node of the face.  Every lane forms its own
// density and velocity and the lanes pass one population at a time, so no second
// set of 27 registers is live (73 VGPRs for FP16 and FP32, 6 wavefronts per SIMD,
// 122 and 4 for FP64; FP16 keeps 12 to 17 scalars in lanes of a vector register;
// held to 72 the step schedules worse, 190 us); the group's words are read before the
// populations, the entry while they arrive (after them: 150 us).  A boundary
// node whose neighbour is in another wavefront (lane 0, or 63 for -x) is left to
// k_bc_pressure_edge, launched before where the list has one.  MI355X, us per
// step, with the outlet in the step / apart / without: 288x144x144 FP16 142 / 150 /
// 128, FP32 256 / 293 / 256, FP64 524 / 582 / 511; 512x256x256 FP16 754 / 812 / 722,
// FP64 2868 / 2990 / 2785; 96x60x50 FP16 15.7 / 20.1 / 12.0; 230x130x120, 472 of
// 15104 entries in the edge launch (6.3), FP64 330 / 352 / 314, FP16 90 / 81 / 69.
template <typename S, bool EVEN>
__global__ void __launch_bounds__(256) k_step_pre(Lat L, Rates<typename Compute<S>::T> R, FusedGroup gp)
{
    using T = typename Compute<S>::T;
    constexpr bool FAST = sizeof(S) != 8;
    constexpr bool O2 = sizeof(S) == 2;
    const uint32_t blk = xcd_block_pow2(blockIdx.x, gridDim.x, L.xrun_lg - 1u);
    const uint32_t k = blk * blockDim.x + threadIdx.x;
    const bool active = k < (uint32_t)L.N && !is_solid(L, k);
    // the group's words are read before the populations, so that a boundary
    // node's entry is on its way while they arrive
    const uint32_t at = active ? k >> 5 : 0u, word = gp.mask[at], base = gp.base[at];
    uint32_t kk[8];
    nbrs_direct(L, k, kk);
    T m[27], mv[4], nut = T(0);
#pragma unroll
    for (int s = 0; s < 27; ++s) m[s] = T(0);
    if (active) gather<S, T, EVEN>(L, kk, m);
    const bool px = gp.B.normal == dP00; // outward normal +x: the inward neighbour is the lane before
    const bool member = active && ((word >> (k & 31u)) & 1u);
    if (__ballot(member)) {
        const uint32_t i = base + (uint32_t)__builtin_popcount(word & ((1u << (k & 31u)) - 1u));
        bool mine = member && i < gp.B.n && (threadIdx.x & 63u) != (px ? 0u : 63u);
        uint32_t ek = 0, ekn = 0;
        T rho_bc = T(0);
        if (mine) {
            ek = gp.B.k[i];
            ekn = gp.B.kn[i];
            rho_bc = bc_at<T>(gp.B.rho, i);
        }
        mine = mine && ek == k && ekn == (px ? k - 1u : k + 1u); // malformed tables select nothing
        if (px) fused_pressure<S, T, true>(L, gp, mine, rho_bc, m);
        else fused_pressure<S, T, false>(L, gp, mine, rho_bc, m);
    }
    if (!active) return;
    collide<T, VFX_K17, FAST, O2>(m, R, mv, nut);
    scatter_post<S, T, EVEN, O2>(L, kk, m);
}

// The entries k_step_pre leaves out: nodes in the wavefront's first lane (last,
// for an outward normal -x), chosen by the same tables and conditions.  Not
// launched for lists without such nodes (every x in a row has one k mod
// gcd(nx, 64)): 144.5 -> 143.2 us per step of the 288x144x144 channel.
template <typename S, bool EVEN>
__global__ void __launch_bounds__(256) k_bc_pressure_edge(Lat L, FusedGroup gp)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= gp.B.n) return;
    const bool px = gp.B.normal == dP00;
    const uint32_t k = gp.B.k[i];
    if ((k & 63u) != (px ? 0u : 63u) || k >= (uint32_t)L.N || is_solid(L, k)) return;
    const uint32_t word = gp.mask[k >> 5], bit = 1u << (k & 31u);
    if (!(word & bit) || gp.base[k >> 5] + (uint32_t)__builtin_popcount(word & (bit - 1u)) != i ||
        gp.B.kn[i] != (px ? k - 1u : k + 1u))
        return; // malformed tables select nothing
    bc_pressure_entry<S, EVEN>(L, gp.B, i);
}

// The coarse step and the first fine step of a nest (or any two structured
// lattices of one storage type) in one launch: the plain step's body
// (k_step_direct) per level, each level's parity a template argument.  Level
// j owns the blocks [first_j, first_j + blocks_j), first_1 a multiple of 8 so
// that the XCD-aware tile order holds per level (padding blocks exit), blocks
// of 256 nodes along x.
template <typename S> struct LevelPair {
    Lat L0, L1;
    Rates<typename Compute<S>::T> R0, R1;
    uint32_t n, blocks0, first1, blocks1;
};
template <typename S, bool E0, bool E1>
__global__ void __launch_bounds__(256) k_step_levels(LevelPair<S> P)
{
    constexpr bool FAST = sizeof(S) != 8;
    if (P.n > 1 && blockIdx.x >= P.first1) {
        if (blockIdx.x - P.first1 < P.blocks1)
            step_direct_body<S, VFX_K17, E1, FAST>(P.L1, P.R1, blockIdx.x - P.first1, P.blocks1);
    } else if (blockIdx.x < P.blocks0) {
        step_direct_body<S, VFX_K17, E0, FAST>(P.L0, P.R0, blockIdx.x, P.blocks0);
    }
}

// ------------------------------------------------------------- batched ----
// Many independent box domains (an ensemble of cavities) advanced by one launch.
// Every domain is a box of nx*ny*nz nodes whose outer layer is wall; only the
// (nx-2)(ny-2)(nz-2) interior nodes collide.  Wall links are closed by the
// moving-wall halfway bounce-back of VelocityBounceBack_Device
// (VelocityBounceBack.cu:159-184) fused into the scatter: a population leaving
// towards a wall node is written, minus the wall term, straight into the element
// the node reads the opposite direction from in the next step.  Links into the
// top plane (z = nz-1) move with the domain's lid velocity.
//
// Both destinations of a population (its streaming slot, or the bounce-back
// slot) sit at the same element of two different planes.  Every population is
// streamed unconditionally (a wall link's streaming slot belongs to the wall
// node and is never read); only the bounce-back copy of a wall link is a
// lane-masked store.  The wall layer therefore holds stale values after a
// step, which nothing reads.

// a value the caller knows to be uniform across the wavefront, as a scalar
__device__ __forceinline__ uint32_t uni(uint32_t v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ uint64_t uni64(uint64_t v)
{
    return (uint64_t)uni((uint32_t)v) | ((uint64_t)uni((uint32_t)(v >> 32)) << 32);
}

template <typename T> struct DomainDev {
    uint64_t f_off;             // element offset of the domain's 27 planes in the pool
    uint32_t N, nx, ny, nz;     // box nodes / dims (wall layer included)
    uint32_t nfx, nfy, nfluid;  // interior dims and count
    uint32_t pad;
    FastDiv div_x, div_y;       // division by nfx, nfy
    T lid_term[27];             // 6 w_e (c_e . u_lid) per direction (used where c_e,z > 0)
    Rates<T> R;
};

struct BatchDev {
    void* pool;
    const void* domains;        // DomainDev<T>[n]
    const uint2* tiles;         // (domain, first interior node) per tile
    uint32_t ntiles;
    uint32_t xcd_run;           // tiles per XCD run (xcd_block); 1 = plain order
    float ld[4], st[4];
};

// tiles and domains are read-only for the whole launch (restrict), so their
// workgroup-uniform loads become scalar loads into SGPRs and every plane
// address stays a scalar base plus a 32-bit lane offset
template <typename S, bool EVEN, bool FAST>
__global__ void __launch_bounds__(256)
    k_step_batched(BatchDev B, const uint2* __restrict__ tiles, const DomainDev<typename Compute<S>::T>* __restrict__ doms)
{
    using T = typename Compute<S>::T;
    // workgroup b starts at tile xcd_block(b): runs of xcd_run consecutive
    // tiles (which share cache lines at their ends) on one XCD, or plain order
    const uint32_t t0 = B.xcd_run > 1 ? xcd_block(blockIdx.x, gridDim.x, B.xcd_run) : blockIdx.x;
    for (uint32_t t = t0; t < B.ntiles; t += gridDim.x) {
        const uint2 tile = tiles[t];
        const DomainDev<T>& D = doms[tile.x];
        const uint32_t idx = tile.y + threadIdx.x;
        const uint32_t nfx = D.nfx, nfy = D.nfy;
        if (idx >= D.nfluid) continue;
        const uint32_t r = fastdiv(idx, D.div_x);
        const uint32_t zi = fastdiv(r, D.div_y);
        const uint32_t x = idx - r * nfx + 1, y = r - zi * nfy + 1, z = zi + 1;
        Lat L;
        L.f = (S*)B.pool + D.f_off;
        L.N = D.N;
        L.nx = D.nx;
        L.ny = D.ny;
        L.nz = D.nz;
        uint32_t kk[8];
        nbrs_interior(L, x, y, z, kk);
        T m[27], mv[4], nut = T(0);
#pragma unroll
        for (int s = 0; s < 27; ++s) {
            const int d = dir_at(s);
            m[s] = Storage<S, T>::ld(plane<S>(L, slot(d, EVEN)), kk[nbr(d)], B.ld[weight_class(d)]);
        }
        constexpr bool O2 = FAST && sizeof(S) == 2; // class-c populations come out as 2^c f
        collide<T, VFX_K17, FAST, O2>(m, D.R, mv, nut);
        // which faces of the box the node touches (lane masks: scalar logic)
        const bool xl = x == 1, xh = x == L.nx - 2, yl = y == 1, yh = y == L.ny - 2, zl = z == 1, zh = z == L.nz - 2;
        // one buffer descriptor over the domain's planes: a lane's byte offset
        // is one VGPR per neighbour node, the plane's byte offset an SGPR
        const uint32_t pb = L.N * (uint32_t)sizeof(S);
        const __amdgpu_buffer_rsrc_t rs = buffer_rsrc(L.f, 27u * pb);
        uint32_t vo[8];
#pragma unroll
        for (int b = 0; b < 8; ++b) vo[b] = kk[b] * (uint32_t)sizeof(S);
        // links into the lid plane carry the moving-wall term (only waves
        // with a lane next to the lid do the arithmetic; top = 0 leaves the
        // value unchanged exactly)
        if (__ballot(zh)) {
            const T top = zh ? T(1) : T(0);
#pragma unroll
            for (int s = 0; s < 27; ++s)
                if (cz(dir_at(s)) > 0)
                    m[s] = m[s] - (top * T(O2 ? 1 << weight_class(dir_at(s)) : 1)) * D.lid_term[dir_at(s)];
        }
        T stc[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) stc[c] = (O2 && c > 0) ? B.st[c] * (1.f / float(1 << c)) : B.st[c];
        S sv[27];
#pragma unroll
        for (int s = 0; s < 27; ++s) sv[s] = Storage<S, T>::enc(m[s], stc[weight_class(dir_at(s))]);
        // One store per population.  Streaming: population e goes to the slot
        // direction d = inv(e) was read from.  On a wall link that slot is the
        // one the wall node would read e from -- the wall layer never collides,
        // nothing reads it -- so the lane writes the bounce-back instead: the
        // slot node k reads direction d from next step, in the other parity's
        // plane at the same element (plane offset moved into the lane's offset).
#pragma unroll
        for (int s = 0; s < 27; ++s) {
            const int e = dir_at(s);
            const int d = inv(e);
            const bool wall = (cx(e) < 0 && xl) || (cx(e) > 0 && xh) || (cy(e) < 0 && yl) || (cy(e) > 0 && yh) ||
                              (cz(e) < 0 && zl) || (cz(e) > 0 && zh);
            // the lower of the two planes in the scalar offset, the lane adds a
            // non-negative distance to its plane
            const int se = slot(d, EVEN), so = slot(d, !EVEN), mn = se < so ? se : so;
            const uint32_t off = vo[nbr(d)] + (uint32_t)((wall ? so : se) - mn) * pb;
            Buf<S>::st(rs, off, (uint32_t)mn * pb, sv[s]);
        }
    }
}

// Initialise every domain's interior to the rest state f - w = 0 (both parities
// read the same zeros, walls included).
template <typename S>
__global__ void __launch_bounds__(256) k_batch_zero(void* pool, uint64_t n)
{
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) ((S*)pool)[i] = S(0);
}

} // namespace vfx

#include "refinement.hpp"

namespace vfx {

// ---------------------------------------------- VirtualFluids array export ----
// The distribution array exactly as VirtualFluids holds it (distributions.f[0]:
// 27 planes of n_nodes shifted populations at the current parity) in a chosen
// floating type: the array RestartObject::serialize/deserialize write and read
// (src/gpu/core/Restart/RestartObject.cpp:19-48).  Element j of plane p holds
// direction d = slot^-1(p) (p itself at even parity, inv(p) at odd), which
// fixes the FP16 scale and reference offset; FP32/FP64 storage is copied.
// Export writes NaN as 0, as serialize does.
// blockIdx.y is the plane: its direction, scale and offset are wave-uniform and
// no element divides its index by the node count (a 64-bit division, ~100
// instructions per element before).  MI355X, 160^3 FP32 to float, 885 MB: 201 ->
// 162 us with four elements per thread, 236 with one (432 000 workgroups).
template <typename S> struct PlaneScale {
    int d;
    float ld, st, sh, ss;
    __device__ __forceinline__ PlaneScale(const Lat& L, int p, bool even)
    {
        d = 0;
        ld = st = 1.f;
        sh = ss = 0.f;
        if constexpr (sizeof(S) == 2) {
            // constant-index selects: the kernel argument arrays stay in place
#pragma unroll
            for (int e = 0; e < 27; ++e)
                if (p == slot(e, even)) {
                    d = e;
                    ld = L.ld[weight_class(e)];
                    st = L.st[weight_class(e)];
                    sh = L.sh[e];
                    ss = L.ss[e];
                }
        }
    }
};
constexpr uint32_t kCopyPerThread = 4; // elements per thread, loaded before the first is stored
template <typename S, bool EVEN, typename O>
__global__ void __launch_bounds__(256) k_export(Lat L, O* out)
{
    using T = typename Compute<S>::T;
    const int p = (int)blockIdx.y;
    const PlaneScale<S> c(L, p, EVEN);
    const uint32_t n = (uint32_t)L.N, j0 = blockIdx.x * (256u * kCopyPerThread) + threadIdx.x;
    T v[kCopyPerThread];
#pragma unroll
    for (uint32_t u = 0; u < kCopyPerThread; ++u)
        if (j0 + u * 256u < n) v[u] = Storage<S, T>::ld(plane<S>(L, p), j0 + u * 256u, c.ld, c.sh);
#pragma unroll
    for (uint32_t u = 0; u < kCopyPerThread; ++u)
        if (j0 + u * 256u < n) (out + (uint64_t)p * L.N)[j0 + u * 256u] = v[u] != v[u] ? O(0) : (O)v[u];
}
template <typename S, bool EVEN, typename O>
__global__ void __launch_bounds__(256) k_import(Lat L, const O* in)
{
    using T = typename Compute<S>::T;
    const int p = (int)blockIdx.y;
    const PlaneScale<S> c(L, p, EVEN);
    const uint32_t n = (uint32_t)L.N, j0 = blockIdx.x * (256u * kCopyPerThread) + threadIdx.x;
    O v[kCopyPerThread];
#pragma unroll
    for (uint32_t u = 0; u < kCopyPerThread; ++u)
        if (j0 + u * 256u < n) v[u] = (in + (uint64_t)p * L.N)[j0 + u * 256u];
#pragma unroll
    for (uint32_t u = 0; u < kCopyPerThread; ++u)
        if (j0 + u * 256u < n) Storage<S, T>::st(plane<S>(L, p), j0 + u * 256u, (T)v[u], c.st, c.ss);
}

// ------------------------------------------------------- AMD viscosity ----
// Anisotropic minimum-dissipation eddy viscosity of every fluid node from the
// velocity fields the collision wrote (calcAMD,
// src/gpu/core/PostProcessor/TurbulentViscosityKernels.cu:62-113): central
// differences where both neighbours along an axis are fluid, one-sided where
// one is, zero where none is; nu_t = max(0, -C * numerator) / |grad u|^2
// (0 where the gradient vanishes).  Sparse layout: the -x/-y/-z neighbours
// come from the -x-y-z node (neighborInverse) and two + steps, fluid means
// typeOfGridNode == GEO_FLUID; direct layout: periodic index wrap, fluid =
// not solid.  Expression order as the reference's (FP64 reproduces it).
template <typename T>
__device__ __forceinline__ void amd_derivatives(uint32_t k, uint32_t km, uint32_t kp, bool fm, bool fp, const T* vx,
                                                const T* vy, const T* vz, T& dvx, T& dvy, T& dvz)
{
    const T div = (fm && fp) ? T(0.5) : T(1);
    kp = fp ? kp : k;
    km = fm ? km : k;
    dvx = (vx[kp] - vx[km]) * div;
    dvy = (vy[kp] - vy[km]) * div;
    dvz = (vz[kp] - vz[km]) * div;
}

// Bound by its reads past L2: with the blocks round robin over the XCDs the rows
// above, below, before and behind a block were in other L2s and came from memory
// again, five times the fields' bytes.  With a contiguous eighth of the lattice
// per XCD (xcd_slab) they are in its own: 224x144x120 33.6 -> 22.0 us (MI355X;
// 62 MB that it must move, 12 us).  Selecting a neighbour by its index, once for
// the three components, alone changed nothing.  (The fields are float beside
// 2-byte populations too: a 32-bit byte offset would not reach every node.)
template <typename T> __global__ void __launch_bounds__(256) k_turb_amd(Lat L, int direct, T C)
{
    const uint32_t k = xcd_slab(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
    if (k >= (uint32_t)L.N) return;
    uint32_t kp[3], km[3];
    bool fp[3] = {true, true, true}, fm[3] = {true, true, true};
    if (direct) {
        const uint32_t r = fastdiv(k, L.div_x), x = k - r * L.nx, z = fastdiv(r, L.div_y), y = r - z * L.ny;
        const uint32_t sy = L.nx, sz = L.nx * L.ny, n = (uint32_t)L.N;
        kp[0] = k + (x + 1u == L.nx ? 1u - sy : 1u);
        km[0] = k - (x == 0u ? 1u - sy : 1u);
        kp[1] = k + (y + 1u == L.ny ? sy - sz : sy);
        km[1] = k - (y == 0u ? sy - sz : sy);
        kp[2] = k + (z + 1u == L.nz ? sz - n : sz);
        km[2] = k - (z == 0u ? sz - n : sz);
        if (L.solid) {
            if (is_solid(L, k)) return;
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                fp[a] = !is_solid(L, kp[a]);
                fm[a] = !is_solid(L, km[a]);
            }
        }
    } else {
        if (L.types[k] != kGeoFluid) return;
        kp[0] = L.nbx[k];
        kp[1] = L.nby[k];
        kp[2] = L.nbz[k];
        const uint32_t w = L.nbinv[k];
        km[0] = L.nbz[L.nby[w]];
        km[1] = L.nbz[L.nbx[w]];
        km[2] = L.nby[L.nbx[w]];
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            fp[a] = L.types[kp[a]] == kGeoFluid;
            fm[a] = L.types[km[a]] == kGeoFluid;
        }
    }
    const T* vx = (const T*)L.vx;
    const T* vy = (const T*)L.vy;
    const T* vz = (const T*)L.vz;
    T dvxdx, dvxdy, dvxdz, dvydx, dvydy, dvydz, dvzdx, dvzdy, dvzdz;
    amd_derivatives<T>(k, km[0], kp[0], fm[0], fp[0], vx, vy, vz, dvxdx, dvydx, dvzdx);
    amd_derivatives<T>(k, km[1], kp[1], fm[1], fp[1], vx, vy, vz, dvxdy, dvydy, dvzdy);
    amd_derivatives<T>(k, km[2], kp[2], fm[2], fp[2], vx, vy, vz, dvxdz, dvydz, dvzdz);
    const T den = dvxdx * dvxdx + dvydx * dvydx + dvzdx * dvzdx + dvxdy * dvxdy + dvydy * dvydy + dvzdy * dvzdy +
                  dvxdz * dvxdz + dvydz * dvydz + dvzdz * dvzdz;
    const T num = (dvxdx * dvxdx + dvxdy * dvxdy + dvxdz * dvxdz) * dvxdx +
                  (dvydx * dvydx + dvydy * dvydy + dvydz * dvydz) * dvydy +
                  (dvzdx * dvzdx + dvzdy * dvzdy + dvzdz * dvzdz) * dvzdz +
                  (dvxdx * dvydx + dvxdy * dvydy + dvxdz * dvydz) * (dvxdy + dvydx) +
                  (dvxdx * dvzdx + dvxdy * dvzdy + dvxdz * dvzdz) * (dvxdz + dvzdx) +
                  (dvydx * dvzdx + dvydy * dvzdy + dvydz * dvzdz) * (dvydz + dvzdy);
    ((T*)L.nut)[k] = den != T(0) ? fmax(T(0), -C * num) / den : T(0);
}

// ------------------------------------------------------------ launchers ----
constexpr int kBlock = 256;

inline unsigned grid_for(uint64_t n, int block) { return (unsigned)((n + block - 1) / block); }
// blocks of kBlock items, a multiple of 8 of them (xcd_slab)
inline unsigned grid_slabs(uint64_t n) { return (grid_for(n, kBlock) + kXcds - 1) / kXcds * kXcds; }

// Occupancy cap of the structured step: LDS requested at launch and not
// used, so that at most 160 KiB / cap workgroups share a CU.  The FP32
// reduced-operation step (8 waves per SIMD by registers) runs fastest with at
// most 6 workgroups of 128 nodes per CU, ~3 waves per SIMD: more of them in
// flight only spread the 54 streams over more open pages (MI355X, us per step
// by tiles of 64 / 128 / 256 nodes, each at most 6 per CU: 512x256x256 1559 /
// 1359 / 1403, 230x171x125 215 / 207 / 216; 1404 without a cap); the sparse
// FP32 step, whose workgroups are 256 work items, with the same cap 1497
// against 1530.  The FP16 step is fastest at the 7
// waves its registers allow (6 or 5 waves per SIMD measured slower), FP64 and
// the reference-order kernels are limited by their registers; other
// collision templates keep the uncapped launch.
template <typename S, int COLL, bool FAST> constexpr unsigned step_lds_cap()
{
    return sizeof(S) == 4 && FAST && coll_op(COLL) == VFX_K17 && coll_turb(COLL) == kTurbNone &&
                   !coll_body_force(COLL)
               ? 24576u
               : 0u;
}

// Built-in XCD run of the structured step, by where the 54 streams' lines are
// when they are needed again.  Boxes that mostly stay in the 256 MiB last-level
// cache and all FP32 ones: 16.  FP16 from 2^23 nodes: 4.  FP64 from 2^24 nodes
// with rows of whole lines (planes and rows on the same few channels): 256, so
// that an XCD stays in its own pages.  MI355X, us per K17 step by run of 4 / 16 /
// 64 / 256 tiles of the built-in width, the rule's lines lie between:
//   FP16 128^3 53 / 43 / 43 / 43, 256x128x128 97 / 81 / 81, 160^3 83 / 82 / 81,
//     192^3 151 / 149 / 150 | 256x256x128 181 / 185, 224^3 248 / 250,
//     320x256x160 285 / 287, 384x256x256 528 / 534, 512x256x256 707 / 727 / 726 /
//     780, 512^3 2840 / 2921 / 2950
//   FP32 128^3 67 / 69, 160^3 180 / 176, 256x256x64 190 / 181, 256^3 657 / 670 /
//     674 / 717, 333x301x290 1263 / 1249 / 1243
//   FP64 160^3 372 / 357 / 359 / 369, 256x256x128 714 / 716 / 732 / 720,
//     301x257x203 1418 / 1367 / 1369 / 1379, 333^3 3550 / 3226 / 3233 / 3261 |
//     256^3 1414 / 1436 / 1449 / 1429, 512x256x256 2924 / 2921 / 2887 / 2806 (BGK
//     2905 / 2902 / 2869 / 2841), 512x512x128 2879 / 2867 / 2841 / 2815,
//     640x384x150 3363 / 3177 / 3187 / 3151
template <typename S> inline uint32_t step_run(const Lat& L)
{
    if (sizeof(S) == 2) return L.N >= (1u << 23) ? 4u : 16u;
    return sizeof(S) == 8 && L.N >= (1u << 24) && L.nx % 64u == 0 ? 256u : 16u;
}
template <typename S> inline Lat with_run(const Lat& in)
{
    Lat L = in;
    if (!L.xrun_lg) L.xrun_lg = 1u + (uint32_t)__builtin_ctz(step_run<S>(in));
    return L;
}

template <typename S, int COLL, bool EVEN, bool FAST>
hipError_t launch_step_t(const Lat& L, int direct, const Rates<typename Compute<S>::T>& R, hipStream_t st)
{
    if (direct) {
        const unsigned tile = L.tile ? L.tile : step_lds_cap<S, COLL, FAST>() ? 128u : 256u;
        hipLaunchKernelGGL((k_step_direct<S, COLL, EVEN, FAST>), dim3(grid_for(L.N, tile)), dim3(tile),
                           (step_lds_cap<S, COLL, FAST>()), st, with_run<S>(L), R);
    } else {
        const uint64_t n = node_items(L, 0);
        if (n == 0) return hipSuccess;
        hipLaunchKernelGGL((k_step_sparse<S, COLL, EVEN, FAST>), dim3(grid_for(n, kBlock)), dim3(kBlock),
                           (step_lds_cap<S, COLL, FAST>()), st, L, R);
    }
    return hipGetLastError();
}

// The reduced-operation form (FP32 arithmetic only) or the reference order.
// With an eddy-viscosity model the reduced form runs on 2-byte storage only: the
// reference order (rates of every node with IEEE divisions, ~1500 instructions)
// is bound by its arithmetic there, the reduced one by memory (MI355X, us per
// step, reference order -> reduced: Smagorinsky 224x144x120 169 -> 95,
// 384x256x200 974 -> 489; AMD with its viscosity kernel 205 -> 129, 1086 ->
// 627).  Density and velocity are the reference order's bits, the error of the
// viscosity against 64 bits is 0.91 to 1.00 of its and that of the populations,
// which is the storage's rounding, the same to four digits (one step from the
// same populations, omega 1.8 to 1.999, all models).  On 4-byte storage both are
// bound by memory (256x160x100: 185 us) and the populations of the reduced form
// are up to twice as far off (8.3e-7 against 4.4e-7 after 10 steps), so that one
// keeps the reference order.
template <typename S, int COLL>
hipError_t launch_step_p(const Lat& L, int direct, bool even, bool fast, const Rates<typename Compute<S>::T>& R,
                         hipStream_t st)
{
    if constexpr (coll_op(COLL) == VFX_K17 && (sizeof(S) == 2 || (sizeof(S) == 4 && coll_turb(COLL) == kTurbNone))) {
        if (fast) return even ? launch_step_t<S, COLL, true, true>(L, direct, R, st)
                              : launch_step_t<S, COLL, false, true>(L, direct, R, st);
    }
    return even ? launch_step_t<S, COLL, true, false>(L, direct, R, st)
                : launch_step_t<S, COLL, false, false>(L, direct, R, st);
}

// variant: 0 = default (FP64: reference operation order; FP32/FP16: reduced form), 1 = reference order;
// turb: TurbModel of the K17 collision
template <typename S> hipError_t launch_step(const Lat& L, int direct, int coll, bool even, int variant, double omega,
                                             const double* lim, const double* force, int turb, double sgs,
                                             hipStream_t st)
{
    using T = typename Compute<S>::T;
    const Rates<T> R = make_rates<T>(omega, lim, force, sgs);
    const bool bf = (coll & kCollBodyForce) != 0; // ApplyBodyForce (K17 only)
    coll &= 15;
    const bool fast = sizeof(T) == 4 && variant == 0 && coll == VFX_K17;
    constexpr int K = VFX_K17, BF = kCollBodyForce;
#define VFX_TURB(TM) \
    case TM: \
        return bf ? launch_step_p<S, K | ((TM) << 4) | BF>(L, direct, even, fast, R, st) \
                  : launch_step_p<S, K | ((TM) << 4)>(L, direct, even, fast, R, st)
    if (coll == VFX_K17) switch (turb) {
            VFX_TURB(kTurbSmagorinsky);
            VFX_TURB(kTurbAMD);
            VFX_TURB(kTurbQR);
        default:
            return bf ? launch_step_p<S, K | BF>(L, direct, even, fast, R, st)
                      : launch_step_p<S, K>(L, direct, even, fast, R, st);
        }
#undef VFX_TURB
    return launch_step_p<S, VFX_BGK>(L, direct, even, false, R, st);
}

template <typename S> hipError_t launch_bc(const Lat& L, const BCDev& B, int kind, bool even, hipStream_t st);

// K17 collide-and-stream of a structured lattice with its boundary groups: the
// pressure group inside the step (k_step_pre), the post-collision ones after it
// by their own kernels.  Inside the step a post-collision boundary node costs
// its whole wavefront the boundary code and several dependent round trips: every
// group of the 512x256x256 channel inside 1195 us against 1003 apart, the inlet
// alone +140 against +94 (FP16, MI355X).
template <typename S>
hipError_t launch_step_fused(const Lat& L, bool even, double omega, const double* lim, const double* force,
                             const FusedGroup& g0, const FusedGroup& g1, const FusedGroup& gp, int apply_pre,
                             hipStream_t st)
{
    using T = typename Compute<S>::T;
    const Rates<T> R = make_rates<T>(omega, lim, force, 0.0);
    hipError_t e = hipSuccess;
    if (gp.mask && apply_pre) {
        const dim3 edge(grid_for(gp.B.n, kBlock)), b(kBlock);
        // rows of whole wavefronts keep the pair in one (the caller's x mod 64
        // condition); apply_pre -1: the caller's list has no pair apart
        if (L.nx % 64u != 0 && apply_pre > 0) {
            if (even) hipLaunchKernelGGL((k_bc_pressure_edge<S, true>), edge, b, 0, st, L, gp);
            else hipLaunchKernelGGL((k_bc_pressure_edge<S, false>), edge, b, 0, st, L, gp);
        }
        const unsigned tile = L.tile ? L.tile : sizeof(S) == 4 ? 128u : 256u;
        const dim3 g(grid_for(L.N, tile)), t(tile);
        constexpr unsigned lds = step_lds_cap<S, VFX_K17, sizeof(S) != 8>();
        if (even) hipLaunchKernelGGL((k_step_pre<S, true>), g, t, lds, st, with_run<S>(L), R, gp);
        else hipLaunchKernelGGL((k_step_pre<S, false>), g, t, lds, st, with_run<S>(L), R, gp);
        e = hipGetLastError();
    } else {
        constexpr bool FAST = sizeof(S) != 8;
        e = even ? launch_step_t<S, VFX_K17, true, FAST>(L, 1, R, st) : launch_step_t<S, VFX_K17, false, FAST>(L, 1, R, st);
    }
    if (e == hipSuccess && g0.mask) e = launch_bc<S>(L, g0.B, g0.kind, even, st);
    if (e == hipSuccess && g1.mask) e = launch_bc<S>(L, g1.B, g1.kind, even, st);
    return e;
}

template <typename S>
hipError_t launch_bc_set(const BCJob* jobs, uint32_t njobs, uint32_t blocks, uint32_t even_mask, hipStream_t st)
{
    if (blocks == 0) return hipSuccess;
    hipLaunchKernelGGL((k_bc_set<S>), dim3(blocks), dim3(kBlock), 0, st, jobs, njobs, even_mask);
    return hipGetLastError();
}

// The levels of one launch: per level its lattice, rates inputs and parity.
struct LevelInput {
    Lat L;
    double omega;
    const double* lim;
    const double* force;
    bool even;
};
template <typename S> hipError_t launch_step_levels(const LevelInput* in, int n, hipStream_t st)
{
    using T = typename Compute<S>::T;
    constexpr bool FAST = sizeof(S) != 8;
    if (n == 1) {
        // one level: the plain step itself, in the lattice's own launch shape
        const Rates<T> R = make_rates<T>(in[0].omega, in[0].lim, in[0].force, 0.0);
        return in[0].even ? launch_step_t<S, VFX_K17, true, FAST>(in[0].L, 1, R, st)
                          : launch_step_t<S, VFX_K17, false, FAST>(in[0].L, 1, R, st);
    }
    static_assert(sizeof(LevelPair<S>) <= 4000, "kernel arguments");
    LevelPair<S> P;
    std::memset(&P, 0, sizeof(P));
    P.n = (uint32_t)n;
    Lat* L[2] = {&P.L0, &P.L1};
    Rates<T>* R[2] = {&P.R0, &P.R1};
    uint32_t* blocks[2] = {&P.blocks0, &P.blocks1};
    // one workgroup width for both levels: their own where they agree, else 256
    const uint32_t tile = in[0].L.tile == in[1].L.tile && in[0].L.tile ? in[0].L.tile : 256u;
    uint32_t first = 0;
    for (int j = 0; j < n; ++j) {
        *L[j] = with_run<S>(in[j].L);
        *R[j] = make_rates<T>(in[j].omega, in[j].lim, in[j].force, 0.0);
        *blocks[j] = grid_for(L[j]->N, tile);
        if (j == 1) P.first1 = first;
        first += (*blocks[j] + kXcds - 1) / kXcds * kXcds;
    }
    if (first == 0) return hipSuccess;
    const bool e0 = in[0].even, e1 = n > 1 ? in[1].even : e0;
    const dim3 g(first), b(tile);
    switch ((e0 ? 2 : 0) + (e1 ? 1 : 0)) {
    case 3: hipLaunchKernelGGL((k_step_levels<S, true, true>), g, b, 0, st, P); break;
    case 2: hipLaunchKernelGGL((k_step_levels<S, true, false>), g, b, 0, st, P); break;
    case 1: hipLaunchKernelGGL((k_step_levels<S, false, true>), g, b, 0, st, P); break;
    default: hipLaunchKernelGGL((k_step_levels<S, false, false>), g, b, 0, st, P); break;
    }
    return hipGetLastError();
}

// one entry per wavefront of the step's grid (4 per 256 work items)
inline uint64_t sparse_groups(const Lat& L) { return (node_items(L, 0) + kBlock - 1) / kBlock * (kBlock / 64); }
inline hipError_t launch_sparse_groups(const Lat& L, uint4* table, uint32_t ngroups, hipStream_t st)
{
    const uint64_t items = (uint64_t)ngroups * 64u;
    hipLaunchKernelGGL((k_sparse_groups<0>), dim3(grid_for(items, kBlock)), dim3(kBlock), 0, st, L, table, ngroups);
    return hipGetLastError();
}

template <typename S> hipError_t launch_turb_amd(const Lat& L, int direct, double sgs, hipStream_t st)
{
    using T = typename Compute<S>::T;
    hipLaunchKernelGGL((k_turb_amd<T>), dim3(grid_slabs(L.N)), dim3(kBlock), 0, st, L, direct, (T)sgs);
    return hipGetLastError();
}

template <typename S> hipError_t launch_init(const Lat& L, int direct, bool even, const double* drho, const double* ux,
                                             const double* uy, const double* uz, hipStream_t st)
{
    const uint64_t n = node_items(L, direct);
    if (n == 0) return hipSuccess;
    if (even) hipLaunchKernelGGL((k_init<S, true>), dim3(grid_for(n, kBlock)), dim3(kBlock), 0, st, L, direct, drho, ux, uy, uz);
    else hipLaunchKernelGGL((k_init<S, false>), dim3(grid_for(n, kBlock)), dim3(kBlock), 0, st, L, direct, drho, ux, uy, uz);
    return hipGetLastError();
}

template <typename S> hipError_t launch_rw(const Lat& L, int direct, bool even, double* out, const double* in, hipStream_t st)
{
    const uint64_t n = node_items(L, direct);
    if (n == 0) return hipSuccess;
    const dim3 g(grid_for(n, kBlock)), b(kBlock);
    if (out) {
        if (even) hipLaunchKernelGGL((k_read<S, true>), g, b, 0, st, L, direct, out);
        else hipLaunchKernelGGL((k_read<S, false>), g, b, 0, st, L, direct, out);
    } else {
        if (even) hipLaunchKernelGGL((k_write<S, true>), g, b, 0, st, L, direct, in);
        else hipLaunchKernelGGL((k_write<S, false>), g, b, 0, st, L, direct, in);
    }
    return hipGetLastError();
}

// out_fp64: the VirtualFluids array in double (else float); exactly one of
// out / in is non-null
template <typename S>
hipError_t launch_vf_array(const Lat& L, bool even, bool fp64, void* out, const void* in, hipStream_t st)
{
    const dim3 g(grid_for(L.N, kBlock * kCopyPerThread), 27), b(kBlock);
    if (out) {
        if (fp64) {
            if (even) hipLaunchKernelGGL((k_export<S, true, double>), g, b, 0, st, L, (double*)out);
            else hipLaunchKernelGGL((k_export<S, false, double>), g, b, 0, st, L, (double*)out);
        } else {
            if (even) hipLaunchKernelGGL((k_export<S, true, float>), g, b, 0, st, L, (float*)out);
            else hipLaunchKernelGGL((k_export<S, false, float>), g, b, 0, st, L, (float*)out);
        }
    } else {
        if (fp64) {
            if (even) hipLaunchKernelGGL((k_import<S, true, double>), g, b, 0, st, L, (const double*)in);
            else hipLaunchKernelGGL((k_import<S, false, double>), g, b, 0, st, L, (const double*)in);
        } else {
            if (even) hipLaunchKernelGGL((k_import<S, true, float>), g, b, 0, st, L, (const float*)in);
            else hipLaunchKernelGGL((k_import<S, false, float>), g, b, 0, st, L, (const float*)in);
        }
    }
    return hipGetLastError();
}

template <typename S> hipError_t launch_macro(const Lat& L, int direct, bool even, double* r, double* vx, double* vy,
                                              double* vz, hipStream_t st)
{
    const uint64_t n = node_items(L, direct);
    if (n == 0) return hipSuccess;
    const dim3 g(grid_for(n, kBlock)), b(kBlock);
    if (even) hipLaunchKernelGGL((k_macro<S, true>), g, b, 0, st, L, direct, r, vx, vy, vz);
    else hipLaunchKernelGGL((k_macro<S, false>), g, b, 0, st, L, direct, r, vx, vy, vz);
    return hipGetLastError();
}

template <typename S>
hipError_t launch_macro_vf(const Lat& L, int direct, bool even, void* rho, void* vx, void* vy, void* vz, void* press,
                           hipStream_t st)
{
    using T = typename Compute<S>::T;
    T *r = (T*)rho, *x = (T*)vx, *y = (T*)vy, *z = (T*)vz, *p = (T*)press;
    const dim3 b(kBlock);
    if (even) hipLaunchKernelGGL((k_macro_vf<S, true, 0>), dim3(grid_for(L.N, kBlock)), b, 0, st, L, direct, r, x, y, z, p);
    else hipLaunchKernelGGL((k_macro_vf<S, false, 0>), dim3(grid_for(L.N, kBlock)), b, 0, st, L, direct, r, x, y, z, p);
    if (!direct && !L.types && L.nfluid) {
        if (even) hipLaunchKernelGGL((k_macro_vf<S, true, 1>), dim3(grid_for(L.nfluid, kBlock)), b, 0, st, L, direct, r, x, y, z, p);
        else hipLaunchKernelGGL((k_macro_vf<S, false, 1>), dim3(grid_for(L.nfluid, kBlock)), b, 0, st, L, direct, r, x, y, z, p);
    }
    return hipGetLastError();
}

template <typename S>
hipError_t launch_mean_vf(const Lat& L, int direct, bool even, void* vx, void* vy, void* vz, void* rho, void* press,
                          hipStream_t st)
{
    using T = typename Compute<S>::T;
    T *x = (T*)vx, *y = (T*)vy, *z = (T*)vz, *r = (T*)rho, *p = (T*)press;
    const dim3 b(kBlock);
    if (direct || L.types) {
        if (even) hipLaunchKernelGGL((k_mean_vf<S, true, 0>), dim3(grid_for(L.N, kBlock)), b, 0, st, L, direct, x, y, z, r, p);
        else hipLaunchKernelGGL((k_mean_vf<S, false, 0>), dim3(grid_for(L.N, kBlock)), b, 0, st, L, direct, x, y, z, r, p);
    } else if (L.nfluid) {
        if (even) hipLaunchKernelGGL((k_mean_vf<S, true, 1>), dim3(grid_for(L.nfluid, kBlock)), b, 0, st, L, direct, x, y, z, r, p);
        else hipLaunchKernelGGL((k_mean_vf<S, false, 1>), dim3(grid_for(L.nfluid, kBlock)), b, 0, st, L, direct, x, y, z, r, p);
    }
    return hipGetLastError();
}

template <typename T> hipError_t launch_zero5(uint64_t n, void* a, void* b, void* c, void* d, void* e, hipStream_t st)
{
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL((k_zero5<T>), dim3(grid_for(n, kBlock)), dim3(kBlock), 0, st, (T*)a, (T*)b, (T*)c, (T*)d, (T*)e, n);
    return hipGetLastError();
}

template <typename S>
hipError_t launch_batched(const BatchDev& B, bool even, int variant, unsigned block, unsigned grid, hipStream_t st)
{
    using T = typename Compute<S>::T;
    const bool fast = sizeof(T) == 4 && variant == 0;
    const dim3 g(grid), b(block);
    if (fast) {
        if (even) hipLaunchKernelGGL((k_step_batched<S, true, true>), g, b, 0, st, B, B.tiles, (const DomainDev<T>*)B.domains);
        else hipLaunchKernelGGL((k_step_batched<S, false, true>), g, b, 0, st, B, B.tiles, (const DomainDev<T>*)B.domains);
    } else {
        if (even) hipLaunchKernelGGL((k_step_batched<S, true, false>), g, b, 0, st, B, B.tiles, (const DomainDev<T>*)B.domains);
        else hipLaunchKernelGGL((k_step_batched<S, false, false>), g, b, 0, st, B, B.tiles, (const DomainDev<T>*)B.domains);
    }
    return hipGetLastError();
}

template <typename S> hipError_t launch_batch_zero(void* pool, uint64_t n, hipStream_t st)
{
    if (n == 0) return hipSuccess;
    const uint64_t g = (n + kBlock - 1) / kBlock;
    hipLaunchKernelGGL((k_batch_zero<S>), dim3((unsigned)(g < 65536 ? g : 65536)), dim3(kBlock), 0, st, pool, n);
    return hipGetLastError();
}

inline uint32_t reduce_blocks(uint64_t n) { return (uint32_t)((n + kRedChunk - 1) / kRedChunk); }

template <typename S> hipError_t launch_reduce_mass(const Lat& L, int direct, bool even, double* ws, double* out, hipStream_t st)
{
    const uint64_t n = node_items(L, direct);
    const uint32_t nb = reduce_blocks(n ? n : 1);
    auto* kernel = direct ? (even ? k_reduce_mass<S, true, true> : k_reduce_mass<S, false, true>)
                          : (even ? k_reduce_mass<S, true, false> : k_reduce_mass<S, false, false>);
    hipLaunchKernelGGL(kernel, dim3(nb), dim3(kRedBlock), 0, st, L, ws);
    hipLaunchKernelGGL((k_reduce_finish<4>), dim3(1), dim3(kRedBlock), 0, st, ws, nb, out);
    return hipGetLastError();
}

template <typename S> hipError_t launch_stats(const Lat& L, int direct, bool even, double* sums, hipStream_t st)
{
    const uint64_t n = node_items(L, direct);
    if (n == 0) return hipSuccess;
    const dim3 g(grid_for(n, kBlock)), b(kBlock);
    if (even) hipLaunchKernelGGL((k_stats<S, true>), g, b, 0, st, L, direct, sums);
    else hipLaunchKernelGGL((k_stats<S, false>), g, b, 0, st, L, direct, sums);
    return hipGetLastError();
}

// One thread per boundary node.  A node of a face normal to x touches a cache
// line per element, and those of a workgroup queue at one CU: lists that leave
// CUs idle with workgroups of 256 (below 256 of them) run workgroups of 64.
// MI355X, us per launch, workgroups of 256 / 64: interpolated inlet of 2784 nodes
// 8.4 / 5.6, 5304 12.0 / 6.6, 8836 12.3 / 7.9, 20164 16.1 / 15.8, 64516 53 / 53;
// pressure outlet of 5304 12.4 / 5.7, 8836 13.0 / 7.0, 20164 16.9 / 16.3; no-slip
// walls of 22284 6.3 / 5.7, 48254 6.5 / 6.1, 97214 7.0 / 8.1, 518878 20 / 25 (FP32;
// 64516 and 518878 FP16).  Channel 96x60x50 FP32 per step, outlet in the step:
// 37.6 -> 30.2 (33.2 with the interpolated kinds in the step as well).
template <typename S> hipError_t launch_bc(const Lat& L, const BCDev& B, int kind, bool even, hipStream_t st)
{
    if (B.n == 0) return hipSuccess;
    const unsigned w = B.n < 256u * kBlock ? 64u : kBlock;
    const dim3 g(grid_for(B.n, w)), b(w);
    switch (kind) {
    case VFX_BC_VELOCITY_BOUNCE_BACK: return launch_velocity_bb<S>(L, B, even, st);
    case VFX_BC_NOSLIP_INTERPOLATED:
        if (even) hipLaunchKernelGGL((k_bc_interp<S, true, VFX_BC_NOSLIP_INTERPOLATED>), g, b, 0, st, L, B);
        else hipLaunchKernelGGL((k_bc_interp<S, false, VFX_BC_NOSLIP_INTERPOLATED>), g, b, 0, st, L, B);
        break;
    case VFX_BC_VELOCITY_INTERPOLATED:
        if (even) hipLaunchKernelGGL((k_bc_interp<S, true, VFX_BC_VELOCITY_INTERPOLATED>), g, b, 0, st, L, B);
        else hipLaunchKernelGGL((k_bc_interp<S, false, VFX_BC_VELOCITY_INTERPOLATED>), g, b, 0, st, L, B);
        break;
    case VFX_BC_SLIP:
        if (even) hipLaunchKernelGGL((k_bc_interp<S, true, VFX_BC_SLIP>), g, b, 0, st, L, B);
        else hipLaunchKernelGGL((k_bc_interp<S, false, VFX_BC_SLIP>), g, b, 0, st, L, B);
        break;
    case VFX_BC_PRESSURE_NEQ:
        if (even) hipLaunchKernelGGL((k_bc_pressure<S, true>), g, b, 0, st, L, B);
        else hipLaunchKernelGGL((k_bc_pressure<S, false>), g, b, 0, st, L, B);
        break;
    case VFX_BC_VELOCITY_PRESSURE_INTERPOLATED:
        if (even) hipLaunchKernelGGL((k_bc_interp<S, true, VFX_BC_VELOCITY_PRESSURE_INTERPOLATED>), g, b, 0, st, L, B);
        else hipLaunchKernelGGL((k_bc_interp<S, false, VFX_BC_VELOCITY_PRESSURE_INTERPOLATED>), g, b, 0, st, L, B);
        break;
    case VFX_BC_SLIP_TURBULENT_VISCOSITY:
        if (even) hipLaunchKernelGGL((k_bc_interp<S, true, VFX_BC_SLIP_TURBULENT_VISCOSITY>), g, b, 0, st, L, B);
        else hipLaunchKernelGGL((k_bc_interp<S, false, VFX_BC_SLIP_TURBULENT_VISCOSITY>), g, b, 0, st, L, B);
        break;
    case VFX_BC_STRESS_INTERPOLATED:
        if (even) hipLaunchKernelGGL((k_bc_stress<S, true, 0>), g, b, 0, st, L, B);
        else hipLaunchKernelGGL((k_bc_stress<S, false, 0>), g, b, 0, st, L, B);
        break;
    case VFX_BC_STRESS_BOUNCE_BACK:
        if (even) hipLaunchKernelGGL((k_bc_stress<S, true, 1>), g, b, 0, st, L, B);
        else hipLaunchKernelGGL((k_bc_stress<S, false, 1>), g, b, 0, st, L, B);
        break;
    case VFX_BC_STRESS_BOUNCE_BACK_PRESSURE:
        if (even) hipLaunchKernelGGL((k_bc_stress<S, true, 2>), g, b, 0, st, L, B);
        else hipLaunchKernelGGL((k_bc_stress<S, false, 2>), g, b, 0, st, L, B);
        break;
    case VFX_BC_PRECURSOR_VELOCITY:
        if (even) hipLaunchKernelGGL((k_bc_interp<S, true, VFX_BC_PRECURSOR_VELOCITY>), g, b, 0, st, L, B);
        else hipLaunchKernelGGL((k_bc_interp<S, false, VFX_BC_PRECURSOR_VELOCITY>), g, b, 0, st, L, B);
        break;
    case VFX_BC_PRECURSOR_DISTRIBUTIONS:
        if (even) hipLaunchKernelGGL((k_bc_precursor_dist<S, true>), g, b, 0, st, L, B);
        else hipLaunchKernelGGL((k_bc_precursor_dist<S, false>), g, b, 0, st, L, B);
        break;
    case VFX_BC_OUTFLOW_NON_REFLECTING:
        if (even) hipLaunchKernelGGL((k_bc_outflow<S, true, false>), g, b, 0, st, L, B);
        else hipLaunchKernelGGL((k_bc_outflow<S, false, false>), g, b, 0, st, L, B);
        break;
    case VFX_BC_OUTFLOW_NON_REFLECTING_PRESSURE_CORRECTION:
        if (even) hipLaunchKernelGGL((k_bc_outflow<S, true, true>), g, b, 0, st, L, B);
        else hipLaunchKernelGGL((k_bc_outflow<S, false, true>), g, b, 0, st, L, B);
        break;
    default:
        return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

#define VFX_INSTANTIATE_LAUNCHERS(S)                                                                                   \
    template hipError_t launch_step<S>(const Lat&, int, int, bool, int, double, const double*, const double*, int,      \
                                       double, hipStream_t);                                                           \
    template hipError_t launch_step_fused<S>(const Lat&, bool, double, const double*, const double*, const FusedGroup&, \
                                             const FusedGroup&, const FusedGroup&, int, hipStream_t); \
    template hipError_t launch_turb_amd<S>(const Lat&, int, double, hipStream_t);                                      \
    template hipError_t launch_bc_set<S>(const BCJob*, uint32_t, uint32_t, uint32_t, hipStream_t);                    \
    template hipError_t launch_step_levels<S>(const LevelInput*, int, hipStream_t);                                    \
    template hipError_t launch_init<S>(const Lat&, int, bool, const double*, const double*, const double*,             \
                                       const double*, hipStream_t);                                                    \
    template hipError_t launch_rw<S>(const Lat&, int, bool, double*, const double*, hipStream_t);                      \
    template hipError_t launch_vf_array<S>(const Lat&, bool, bool, void*, const void*, hipStream_t);                  \
    template hipError_t launch_macro<S>(const Lat&, int, bool, double*, double*, double*, double*, hipStream_t);       \
    template hipError_t launch_macro_vf<S>(const Lat&, int, bool, void*, void*, void*, void*, void*, hipStream_t);     \
    template hipError_t launch_mean_vf<S>(const Lat&, int, bool, void*, void*, void*, void*, void*, hipStream_t);      \
    template hipError_t launch_bc<S>(const Lat&, const BCDev&, int, bool, hipStream_t);                            \
    template hipError_t launch_reduce_mass<S>(const Lat&, int, bool, double*, double*, hipStream_t);              \
    template hipError_t launch_stats<S>(const Lat&, int, bool, double*, hipStream_t);                             \
    template hipError_t launch_batched<S>(const BatchDev&, bool, int, unsigned, unsigned, hipStream_t);           \
    template hipError_t launch_batch_zero<S>(void*, uint64_t, hipStream_t);                                        \
    template hipError_t launch_scale<S>(const Lat&, const Lat&, const ICellsDev&, bool, bool, bool, double, double,     \
                                        hipStream_t);                                                                  \
    template hipError_t launch_scale_both<S>(const Lat&, const Lat&, const ICellsDev&, const ICellsDev&, bool, bool,     \
                                             double, double, hipStream_t);

#define VFX_EXTERN_LAUNCHERS(S)                                                                                        \
    extern template hipError_t launch_step<S>(const Lat&, int, int, bool, int, double, const double*, const double*,   \
                                              int, double, hipStream_t);                                               \
    extern template hipError_t launch_step_fused<S>(const Lat&, bool, double, const double*, const double*,            \
                                                    const FusedGroup&, const FusedGroup&, const FusedGroup&,           \
                                                    int, hipStream_t);                                                 \
    extern template hipError_t launch_turb_amd<S>(const Lat&, int, double, hipStream_t);                               \
    extern template hipError_t launch_bc_set<S>(const BCJob*, uint32_t, uint32_t, uint32_t, hipStream_t);             \
    extern template hipError_t launch_step_levels<S>(const LevelInput*, int, hipStream_t);                             \
    extern template hipError_t launch_init<S>(const Lat&, int, bool, const double*, const double*, const double*,      \
                                              const double*, hipStream_t);                                             \
    extern template hipError_t launch_rw<S>(const Lat&, int, bool, double*, const double*, hipStream_t);               \
    extern template hipError_t launch_vf_array<S>(const Lat&, bool, bool, void*, const void*, hipStream_t);           \
    extern template hipError_t launch_macro<S>(const Lat&, int, bool, double*, double*, double*, double*, hipStream_t); \
    extern template hipError_t launch_macro_vf<S>(const Lat&, int, bool, void*, void*, void*, void*, void*, hipStream_t); \
    extern template hipError_t launch_mean_vf<S>(const Lat&, int, bool, void*, void*, void*, void*, void*, hipStream_t); \
    extern template hipError_t launch_bc<S>(const Lat&, const BCDev&, int, bool, hipStream_t);                     \
    extern template hipError_t launch_reduce_mass<S>(const Lat&, int, bool, double*, double*, hipStream_t);       \
    extern template hipError_t launch_stats<S>(const Lat&, int, bool, double*, hipStream_t);                      \
    extern template hipError_t launch_batched<S>(const BatchDev&, bool, int, unsigned, unsigned, hipStream_t);    \
    extern template hipError_t launch_batch_zero<S>(void*, uint64_t, hipStream_t);                                 \
    extern template hipError_t launch_scale<S>(const Lat&, const Lat&, const ICellsDev&, bool, bool, bool, double,     \
                                               double, hipStream_t);                                                   \
    extern template hipError_t launch_scale_both<S>(const Lat&, const Lat&, const ICellsDev&, const ICellsDev&, bool,   \
                                                    bool, double, double, hipStream_t);

} // namespace vfx
