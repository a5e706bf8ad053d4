// HIP kernels of the MI355X residual engine (gfx950, wave64, FP64).
//
// Numerics follow the reference operation by operation so that, compiled
// with -ffp-contract=off, every result matches the CPU oracle bit for bit:
//   - TENO reconstruction: face_reconstruction.cpp:866-1039
//   - Riemann fluxes:      riemann_solver.h:205-519
//   - flux functors / BCs: flux_functor.h:124-178, boundary_*.cpp
//   - residual assembly:   solver_rhs.cpp:44-55 (canonical one-thread order)
//   - SSP-RK / RK4 / FE:   time_integrator.cpp:57-163
//   - spectral radius, dt: solver.cpp:580-742
#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "ddpow.hpp"
#include "device.hpp"
#include "indicator.hpp"
#include "riemann.hpp"

namespace mlr::dev {

namespace {

constexpr uint32_t kBoundaryBit = 1u << 3;

struct D4 {
    double v[4];
};

__device__ inline D4 ld4(const double* __restrict__ p, size_t i) {
    const double2* q = reinterpret_cast<const double2*>(p + 4 * i);
    const double2 a = q[0], b = q[1];
    return D4{{a.x, a.y, b.x, b.y}};
}
__device__ inline void st4(double* __restrict__ p, size_t i, const D4& x) {
    double2* q = reinterpret_cast<double2*>(p + 4 * i);
    q[0] = make_double2(x.v[0], x.v[1]);
    q[1] = make_double2(x.v[2], x.v[3]);
}

// Correctly rounded x^6 (double-double product, exact FMA residuals); equals
// glibc's pow(x, 6.0) wherever that is correctly rounded.
__device__ inline double pow6_cr(double x) {
    const double h2 = x * x;
    const double l2 = __builtin_fma(x, x, -h2);
    const double p3 = h2 * x;
    const double e3 = __builtin_fma(h2, x, -p3) + l2 * x;
    const double h3 = p3 + e3;
    const double l3 = e3 - (h3 - p3);
    const double p6 = h3 * h3;
    const double e6 = __builtin_fma(h3, h3, -p6) + 2.0 * h3 * l3;
    return p6 + e6;
}

__device__ inline double pressure_raw(double gamma, const double* u) {
    return (gamma - 1.0) * (u[3] - 0.5 * (u[1] * u[1] + u[2] * u[2]) / u[0]);
}

// The largest step tt in [0, 1] from the cell mean Uc toward the face state u
// that keeps density and pressure at or above eps (Zhang & Shu 2010, the
// pressure by bisection), in the oracle's order.
__device__ inline double point_limit(double gamma, const double* Uc, const double* u, double eps) {
    double wv[4];
    double tt = 1.0;
    if (u[0] < eps) tt = (Uc[0] - eps) / (Uc[0] - u[0]);
#pragma unroll
    for (int k = 0; k < 4; ++k) wv[k] = Uc[k] + tt * (u[k] - Uc[k]);
    if (pressure_raw(gamma, wv) < eps) {
        double lo = 0.0, hi = tt;
        for (int it = 0; it < 40; it++) {
            const double mid = 0.5 * (lo + hi);
#pragma unroll
            for (int k = 0; k < 4; ++k) wv[k] = Uc[k] + mid * (u[k] - Uc[k]);
            if (pressure_raw(gamma, wv) < eps) hi = mid;
            else lo = mid;
        }
        tt = lo;
    }
    return tt;
}

// ------------------------------------------------------------ quad exchange
// The 4 lanes of a quad serve one cell. DPP quad permutations move values
// between them in registers (no LDS, so occupancy is set by VGPRs alone).
template <int CTRL>
__device__ inline double qperm(double x) {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(x), CTRL, 0xF, 0xF, false);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(x), CTRL, 0xF, 0xF, false);
    return __hiloint2double(hi, lo);
}
// quad_perm controls: lane j of a quad reads lane (j - r) & 3, r = 1, 2, 3;
// (kRot2 is also lane j ^ 2)
constexpr int kRot1 = 0x93, kRot2 = 0x4E, kRot3 = 0x39;

__device__ inline double sel4(const double* x, int i) {
    return i == 0 ? x[0] : (i == 1 ? x[1] : (i == 2 ? x[2] : x[3]));
}
// 4 x 4 transpose across a quad: out[j] = x[q] of quad lane j (q = own lane).
__device__ inline void quad_transpose(const double* x, double* out, int q) {
    double r[4];
    r[0] = sel4(x, q);
    r[1] = qperm<kRot1>(sel4(x, (q + 1) & 3));
    r[2] = qperm<kRot2>(sel4(x, (q + 2) & 3));
    r[3] = qperm<kRot3>(sel4(x, (q + 3) & 3));
#pragma unroll
    for (int j = 0; j < 4; ++j) out[j] = sel4(r, (q - j) & 3);
}
// ------------------------------------------------------------ derived tables
// The target cell's frame: node 0 and the inverse of the Jacobian of its
// map from the reference triangle, as the precompute forms them.
struct TriFrame {
    double w0x, w0y, j0, j1, j2, j3;
};
__device__ inline TriFrame tri_frame(double x0, double y0, double x1, double y1, double x2, double y2) {
    TriFrame F;
    F.w0x = x0;
    F.w0y = y0;
    const double J0 = x1 - x0, J1 = x2 - x0, J2 = y1 - y0, J3 = y2 - y0;
    const double det = J0 * J3 - J1 * J2;
    const double id = 1.0 / det;
    F.j0 = J3 * id;
    F.j1 = -J1 * id;
    F.j2 = -J2 * id;
    F.j3 = J0 * id;
    return F;
}
// a point in the frame: Ji (x - w0)
__device__ inline void to_frame(const TriFrame& F, double x, double y, double& a, double& b) {
    const double tx = x - F.w0x, ty = y - F.w0y;
    a = F.j0 * tx + F.j1 * ty;
    b = F.j2 * tx + F.j3 * ty;
}
// area in the frame of the triangle with nodes (x0, y0), (x1, y1), (x2, y2)
__device__ inline double frame_area(const TriFrame& F, double x0, double y0, double x1, double y1, double x2,
                                    double y2) {
    double a0, b0, a1, b1, a2, b2;
    to_frame(F, x0, y0, a0, b0);
    to_frame(F, x1, y1, a1, b1);
    to_frame(F, x2, y2, a2, b2);
    return 0.5 * fabs(a0 * (b1 - b2) + a1 * (b2 - b0) + a2 * (b0 - b1));
}
// Legendre P_p(x) for p <= 2, terms combined as the basis evaluator does:
// P_2 = 0.5 ((3 x) x - 1)
__device__ inline double legendre_le2(int p, double x) {
    const double p2 = 0.5 * ((3.0 * x) * x - 1.0);
    return p == 0 ? 1.0 : (p == 1 ? x : p2);
}

// ------------------------------------------------------------ streamed tables
template <int I, int N, typename F>
__device__ __forceinline__ void each_index_from(F&& f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        each_index_from<I + 1, N>(f);
    }
}
template <int N, typename F>
__device__ __forceinline__ void each_index(F&& f) {
    each_index_from<0, N>(f);
}

// A wave's member tables through LDS. For each member the wave's 64 lanes (16
// cells x 4 stencils) need KP rows of A+, one of areas and one of positions,
// each 64 consecutive entries. Loads that write LDS directly (16 bytes a
// lane, two rows an instruction) fetch SD members ahead without holding
// registers, so the loads in flight do not compete with the accumulators.
// A wave reads only its own slots: it waits for its own loads (they complete
// in order), and for its reads of a slot before that slot is loaded again.
template <int KP, int MP, typename IdxT, int SD>
struct MemberStream {
    static constexpr int kRows = KP + 1;                            // A+ rows and the areas
    static constexpr int kSlot = kRows * 512 + 64 * (int)sizeof(IdxT);
    static constexpr int kLoads = kRows / 2 + 1;                    // instructions per member
    // the next member to load: the wave's A+ rows and positions, and this
    // lane's part of the last two rows (an A+ row for the lower half of the
    // lanes, the areas for the upper)
    const unsigned char *rows, *pos, *last;
    uint32_t lane_rows, lane_pos, last_step;
    unsigned char *base, *next;

    __device__ __forceinline__ void init(const Teno& t, uint32_t lb, unsigned char* slots) {
        static_assert(SD == 0 || kRows % 2 == 0, "row pairs");
        const uint32_t lane = threadIdx.x & 63u, w = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
        base = slots + (size_t)w * SD * kSlot;
        next = base;
        const bool upper = lane >= 32;
        rows = reinterpret_cast<const unsigned char*>(t.A + teno_a_off(lb, MP, KP, 0, 0, 16 * w, 0));
        lane_rows = (lane >> 5) * 2048 + (lane & 31) * 16;
        last = upper ? reinterpret_cast<const unsigned char*>(t.ta + teno_mem_off(lb, MP, 0, 16 * w, 0)) +
                           (lane & 31) * 16
                     : rows + (kRows / 2 - 1) * 4096 + lane * 16;
        last_step = upper ? 2048 : KP * 2048;
        const unsigned char* loc = sizeof(IdxT) == 1 ? t.loc8 : reinterpret_cast<const unsigned char*>(t.loc16);
        pos = loc + teno_mem_off(lb, MP, 0, 16 * w, 0) * sizeof(IdxT);
        lane_pos = lane * 16;
    }
    __device__ __forceinline__ unsigned char* slot(int i) const { return base + (i % SD) * kSlot; }
    static __device__ __forceinline__ void load16(const unsigned char* src, unsigned char* dst) {
        __builtin_amdgcn_global_load_lds(const_cast<unsigned char*>(src),
                                         (__attribute__((address_space(3))) void*)dst, 16, 0, 0);
    }
    __device__ __forceinline__ void issue() {
#pragma unroll
        for (int n = 0; n < kRows / 2 - 1; ++n) load16(rows + n * 4096 + lane_rows, next + n * 1024);
        load16(last, next + (kRows / 2 - 1) * 1024);
        if (lane_pos < 64 * sizeof(IdxT)) load16(pos + lane_pos, next + kRows * 512);
        rows += KP * 2048;
        last += last_step;
        pos += 256 * sizeof(IdxT);
        next = next == base + (SD - 1) * kSlot ? base : next + kSlot;
    }
    // member I's loads are complete: all but those of the members issued after it
    template <int I>
    __device__ __forceinline__ void wait() const {
        constexpr int kAfter = MP - 1 - I < SD - 1 ? MP - 1 - I : SD - 1;
        static_assert(SD * kLoads <= 63, "the counter holds every load in flight");
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kAfter * kLoads) : "memory");
    }
    // the reads of a slot are complete
    __device__ __forceinline__ void release() const { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }
};

// ------------------------------------------------------------ TENO kernel
// 64 cells per 256-thread block, 4 lanes (a quad) per cell.
// Phase A: quad lane s owns stencil s: stencil-major loads of ids, areas and
// A+, gathers of the members' states, a = A+ b, smoothness, raw weight.
// Quad transposes then hand lane v the 4 stencils' coefficients and weights
// of conserved variable v. Phase B: cut-off, weights and the face-point sums
// in the reference's stencil-then-dof order; with the corrected weighting the
// quad then scales its face states toward the cell mean for positivity.
// KP = n_dof - 1, MP = members per stencil after the target (0: runtime),
// FQ = face points per cell; IdxT is the width of the in-tile positions and
// TILE the LDS capacity in cells. The block first stages the states of every
// cell its stencils read (the tile list) in LDS, so each neighbour state is
// fetched once per block instead of once per stencil member. Blocks are
// mapped so that each of the 8 XCDs walks one contiguous range of the
// space-filling-curve order.
// GM: 0 plain TENO; 1 the learned gate evaluates the network and records
// its decisions; 2 the gate takes the recorded decisions (no network code).
// Split passes (no full-TENO code in the gated kernels, so they keep few
// registers): 3 evaluates like 1 and 4 reuses like 2, but both reconstruct
// only the gated cells and mark the waves holding ungated ones; 5 then
// reconstructs only the ungated cells, in the marked blocks.
// CT: compact tables (corrected weighting): A carries the member areas and
// the face-point basis values come from the small per-edge table t.fbc, so
// neither ta nor the per-cell face basis is read.
// DV: derived face basis (p = 2, Legendre basis, one face point per face):
// the face-point basis values are recomputed from the cell's node
// coordinates with the precompute's operations in its order, so they equal
// the table bit for bit, and the per-cell face basis is not read.
// SD: stream depth (plain pass, unrolled members, odd KP): the member tables
// come through LDS (see MemberStream), in SD slots per wave from sh_net on.
// TIGHT: the loads of a member are not moved above the member before it. At
// the 80 registers of 6 waves per SIMD the loads in flight push accumulators
// to scratch: 2,097,152 cells 1,682 us, 69 registers spilled (1,405 and 34
// before the face points' limits took the quad's lanes); kept apart 1,254 us
// and 23. With 96 registers (5 waves) it only takes loads out of flight:
// 1,115 us, kept apart 1,221.
template <int KP, int MP, int FQ, typename IdxT, int TILE, int GM, bool CT = false, bool DV = false, int SD = 0,
          bool TIGHT = false>
__device__ __forceinline__ void teno_block(const Geom& g, const Teno& t, const double* __restrict__ U,
                                           double* __restrict__ fs, uint8_t* __restrict__ dec, const Physics& ph,
                                           uint32_t lb, double2* sh_u, unsigned char* sh_net) {
    constexpr bool kEval = GM == 1 || GM == 3;
    constexpr bool kReuse = GM == 2 || GM == 4 || GM == 5;
    constexpr bool kLinOnly = GM == 3 || GM == 4;
    constexpr bool kFullOnly = GM == 5;
    const uint32_t N = g.N;
    if (lb * 64u >= N) return;  // whole block past the end (uniform)
    // the block's wave marks as one word (uniform)
    [[maybe_unused]] uint32_t marks = 0xFFFFFFFFu;
    if constexpr (kFullOnly) {
        marks = reinterpret_cast<const uint32_t*>(t.blk_mixed)[lb];
        if (marks == 0u) return;
    }
    using Stream = MemberStream<KP, MP, IdxT, SD>;
    [[maybe_unused]] Stream stream;
    [[maybe_unused]] bool streams = true;  // (uniform in a wave)
    if constexpr (SD > 0) {
        // every lane of a wave takes part in its loads, so a streamed pass
        // runs whole waves: those that hold a cell it reconstructs
        static_assert((GM == 0 || GM == 5) && MP > 0 && !CT, "streamed tables: a full pass at a compiled stencil size");
        const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
        if (kFullOnly) streams = ((marks >> (8 * w)) & 0xFFu) != 0u;
        if (streams) {
            stream.init(t, lb, sh_net);
#pragma unroll
            for (int i = 0; i < (SD < MP ? SD : MP); ++i) stream.issue();
        }
    }
    {
        const uint32_t t0 = t.blk_off[lb], nloc = t.blk_off[lb + 1] - t0;
        const double2* U2 = reinterpret_cast<const double2*>(U);
        for (uint32_t j = threadIdx.x; j < 2 * nloc; j += blockDim.x)
            sh_u[j] = U2[2 * (size_t)t.blk_ids[t0 + (j >> 1)] + (j & 1u)];
        if (kEval && t.gate) ind::stage_net(t.net, sh_net);  // the network, once per block
    }
    __syncthreads();
    if (SD > 0 && !streams) return;
    const IdxT* __restrict__ loc = sizeof(IdxT) == 1 ? reinterpret_cast<const IdxT*>(t.loc8)
                                                     : reinterpret_cast<const IdxT*>(t.loc16);
    const int q = threadIdx.x & 3;
    const uint32_t c = lb * 64u + (threadIdx.x >> 2);
    const bool valid = c < N;
    const uint32_t cc = valid ? c : 0;
    const int Mp = MP > 0 ? MP : t.M - 1;

    // ---- learned gate: the MLP judges each cell from its central stencil
    // (features from the LDS tile, one MFMA column per cell); a smooth cell
    // skips its directional stencils and takes the central one.
    bool smooth = false;
    if (kReuse && t.gate) {
        // the decisions the network recorded earlier in the step
        smooth = valid && t.gate_dec[c] != 0;
        if constexpr (!kFullOnly) {
            const uint64_t bal = __ballot(smooth && q == 0);
            if ((threadIdx.x & 63) == 0 && bal) t.gated[lb * 4u + (threadIdx.x >> 6)] += (uint32_t)__popcll(bal);
        }
    } else if (kEval && t.gate) {
        const int lane = threadIdx.x & 63, gq = lane >> 4;
        const uint32_t cm = lb * 64u + (threadIdx.x >> 6) * 16u + (lane & 15);
        const bool vm = cm < N;
        const D4 Uo = ld4(U, vm ? cm : 0);
        const ind::CellRef r = ind::cell_ref_col(t.gamma, Uo.v, gq, lane & 15);
        // lane (column cell, group gq) holds members 4 kc + gq, kc = 0..2
        double d[3][4], smax[4] = {0.0, 0.0, 0.0, 0.0};
        bool ok = r.ok;
#pragma unroll
        for (int kc = 0; kc < 3; ++kc) {
            const int m = 4 * kc + gq;
            if (m == 0) continue;
            const uint32_t pos = loc[teno_mem_off(lb, Mp, m - 1, cm & 63u, 0)];  // stencil 0
            const double2 u01 = sh_u[2 * pos], u23 = sh_u[2 * pos + 1];
            const double Um[4] = {u01.x, u01.y, u23.x, u23.y};
            ok = ind::member_diff(t.gamma, r, Um, d[kc]) && ok;
#pragma unroll
            for (int v = 0; v < 4; ++v) smax[v] = fmax(smax[v], fabs(d[kc][v]));
        }
        // stencil-wide maxima and validity: the 4 lanes of a column
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            smax[v] = fmax(smax[v], __shfl_xor(smax[v], 16));
            smax[v] = fmax(smax[v], __shfl_xor(smax[v], 32));
        }
        int okc = ok ? 1 : 0;
        okc &= __shfl_xor(okc, 16);
        okc &= __shfl_xor(okc, 32);
        // the 4 reciprocals of the maxima: lane gq takes variable gq's
        double is[4];
        const double is_mine = ind::inv_scale(sel4(smax, gq));
#pragma unroll
        for (int v = 0; v < 4; ++v) is[v] = __shfl(is_mine, (lane & 15) + 16 * v);
        ind::v4s xb[3];
#pragma unroll
        for (int kc = 0; kc < 3; ++kc) {
            const int m = 4 * kc + gq;
            double x[4];
#pragma unroll
            for (int v = 0; v < 4; ++v)
                x[v] = !okc ? 0.0 : (m == 0 ? ind::scale_feature(smax[v]) : ind::pattern_feature(d[kc][v], is[v]));
            xb[kc] = ind::pack_feats(x);
        }
        const float z = ind::mlp_wave(ind::lds_net(t.net, sh_net), xb, lane);
        const int sm = (vm && okc && z >= t.net.logit_threshold) ? 1 : 0;
        if (vm && gq == 0) t.gate_dec[cm] = (uint8_t)sm;
        const uint64_t bal = __ballot(sm && gq == 0);
        if (lane == 0 && bal) t.gated[lb * 4u + (threadIdx.x >> 6)] += (uint32_t)__popcll(bal);
        if constexpr (GM == 3) {
            // mark the wave when a valid cell of it was not gated
            const uint64_t ung = __ballot(vm && !sm && gq == 0);
            if (lane == 0) t.blk_mixed[lb * 4u + (threadIdx.x >> 6)] = ung ? 1 : 0;
        }
        smooth = __shfl(sm, lane >> 2) != 0;
    }

    const uint32_t info0 = g.info[cc];
    const D4 uc = ld4(U, cc);
    const uint32_t cl = c & 63u;
    // Quad exchanges of the plain pass and of the gated passes that keep no
    // network in LDS (reuse, ungated cells), with 8-bit tiles, go through LDS: 4
    // planes of 258 doubles per block (the 2-double pad puts the 4 lanes of
    // a quad on distinct banks when they read one plane), 8 LDS instructions
    // per 4 x 4 transpose instead of the DPP form's selects and moves. A
    // wave reads only its own lanes' entries, and a wave's LDS accesses run
    // in order, so wave-scope fences (compiler ordering) suffice.
    // A streamed pass takes them through its own wave's slots, which hold
    // nothing any more then.
    constexpr bool kLdsX = ((GM == 0 || GM == 4 || GM == 5) && TILE == 256) || SD > 0;
    constexpr int kXs = SD > 0 ? 66 : 258;
    __shared__ double xbuf_block[kLdsX && SD == 0 ? 4 * kXs : 1];
    double* xbuf = xbuf_block;
    if constexpr (SD > 0) {
        static_assert(4 * kXs * 8 <= SD * Stream::kSlot, "the exchange fits the wave's slots");
        xbuf = reinterpret_cast<double*>(stream.base);
    }
    auto wave_sync = []() {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    // out[j] = x[q] of quad lane j
    auto exchange = [&](const double* x, double* out) {
        if constexpr (kLdsX) {
            const uint32_t tid = SD > 0 ? threadIdx.x & 63u : threadIdx.x, base = tid & ~3u;
#pragma unroll
            for (int i = 0; i < 4; ++i) xbuf[i * kXs + tid] = x[i];
            wave_sync();
#pragma unroll
            for (int j = 0; j < 4; ++j) out[j] = xbuf[q * kXs + base + j];
            wave_sync();
        } else {
            quad_transpose(x, out, q);
        }
    };
    // the member update a += A+_i (ta_i (u_i - u_c)) of member i of this
    // lane's stencil q; a wave's 64 lanes read 64 consecutive entries
    auto member = [&](int i, double (&a)[KP][4]) {
        const size_t o = teno_mem_off(lb, Mp, i, cl, q);
        const uint32_t pos = loc[o];
        const double2 u01 = sh_u[2 * pos], u23 = sh_u[2 * pos + 1];
        const D4 un = {{u01.x, u01.y, u23.x, u23.y}};
        double b[4];
        if constexpr (CT) {
#pragma unroll
            for (int v = 0; v < 4; ++v) b[v] = un.v[v] - uc.v[v];
        } else {
            const double tt = t.ta[o];
#pragma unroll
            for (int v = 0; v < 4; ++v) b[v] = tt * (un.v[v] - uc.v[v]);
        }
        const double* Ai = t.A + teno_a_off(lb, Mp, KP, i, 0, cl, q);
        if constexpr (MP == 0 && KP == 9) {
            // a member's 9 rows all loaded before the first is used: left to
            // itself the compiler saves registers by loading them one at a
            // time, each waited for. 320,000 cells, 24 members 921 -> 548 us
            // (882 with the schedule that it chose before the face points'
            // limits took the quad's lanes), ensembles 834 -> 490. At 5 rows
            // it loads ahead by itself and this costs 4%.
            double Ak[KP];
#pragma unroll
            for (int k = 0; k < KP; ++k) Ak[k] = Ai[(size_t)k * 256];
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int k = 0; k < KP; ++k)
#pragma unroll
                for (int v = 0; v < 4; ++v) a[k][v] = a[k][v] + Ak[k] * b[v];
        } else {
#pragma unroll
            for (int k = 0; k < KP; ++k) {
                const double Ak = Ai[(size_t)k * 256];
#pragma unroll
                for (int v = 0; v < 4; ++v) a[k][v] = a[k][v] + Ak * b[v];
            }
        }
        if constexpr (TIGHT) __builtin_amdgcn_sched_barrier(0);
    };

    const double ucv = sel4(uc.v, q);  // lane-dependent pick by selects, not a stack array
    double f[FQ];
    bool central = false;
    // the central stencil's linear reconstruction through its precombined
    // operator (gated cells): quad lane q sums face points q and q + 4 for
    // all 4 variables over the members, a quad transpose hands lane v its
    // variable's face points
    auto linear_faces = [&]() {
        double acc[2][4] = {{0.0, 0.0, 0.0, 0.0}, {0.0, 0.0, 0.0, 0.0}};
        const bool has0 = q < FQ, has1 = q + 4 < FQ;
        if (valid && has0) {
            auto add = [&](int i) {
                const double* Lw = t.lin + teno_lin_off(lb, Mp, i, cl, FQ, q);
                const uint32_t pos = loc[teno_mem_off(lb, Mp, i, cl, 0)];  // central stencil
                const double2 u01 = sh_u[2 * pos], u23 = sh_u[2 * pos + 1];
                const double d[4] = {u01.x - uc.v[0], u01.y - uc.v[1], u23.x - uc.v[2], u23.y - uc.v[3]};
                const double w0 = Lw[0];
#pragma unroll
                for (int v = 0; v < 4; ++v) acc[0][v] = acc[0][v] + w0 * d[v];
                if (has1) {
                    const double w1 = Lw[4];
#pragma unroll
                    for (int v = 0; v < 4; ++v) acc[1][v] = acc[1][v] + w1 * d[v];
                }
            };
            if constexpr (MP > 0) {
#pragma unroll
                for (int i = 0; i < MP; ++i) add(i);
            } else {
                for (int i = 0; i < Mp; ++i) add(i);
            }
        }
        double y[4];
        exchange(acc[0], y);
#pragma unroll
        for (int fq = 0; fq < (FQ < 4 ? FQ : 4); ++fq) f[fq] = ucv + y[fq];
        if constexpr (FQ > 4) {
            exchange(acc[1], y);
#pragma unroll
            for (int fq = 4; fq < FQ; ++fq) f[fq] = ucv + y[fq - 4];
        }
        central = true;
    };

    // full TENO for this cell (the plain path)
    auto full_teno = [&]() {
        const bool active = valid && ((info0 >> (20 + q)) & 1u);

        // ---- phase A: lane q = stencil
        double a[KP][4];
#pragma unroll
        for (int k = 0; k < KP; ++k)
#pragma unroll
            for (int v = 0; v < 4; ++v) a[k][v] = 0.0;
        double w[4] = {0.0, 0.0, 0.0, 0.0};
        if constexpr (SD > 0) {
            // every lane runs along (a lane without a stencil reads table
            // entries of no meaning and the tile's first cell) and is cleared after
            each_index<MP>([&](auto ic) __attribute__((always_inline)) {
                constexpr int i = decltype(ic)::value;
                stream.template wait<i>();
                const unsigned char* m = stream.slot(i);
                const int lane = threadIdx.x & 63;
                const uint32_t p = reinterpret_cast<const IdxT*>(m + Stream::kRows * 512)[lane];
                const uint32_t pos = active ? p : 0u;
                const double* Am = reinterpret_cast<const double*>(m) + lane;
                const double tt = Am[KP * 64];
                const double2 u01 = sh_u[2 * pos], u23 = sh_u[2 * pos + 1];
                const double b[4] = {tt * (u01.x - uc.v[0]), tt * (u01.y - uc.v[1]), tt * (u23.x - uc.v[2]),
                                     tt * (u23.y - uc.v[3])};
#pragma unroll
                for (int k = 0; k < KP; ++k) {
                    const double Ak = Am[k * 64];
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        a[k][v] = a[k][v] + Ak * b[v];
                        // summed here: sunk to the sums' uses the products' operands would all stay live
                        asm volatile("" : "+v"(a[k][v]));
                    }
                }
                if constexpr (i + SD < MP) {
                    stream.release();
                    stream.issue();
                }
            });
            if (!active) {
#pragma unroll
                for (int k = 0; k < KP; ++k)
#pragma unroll
                    for (int v = 0; v < 4; ++v) a[k][v] = 0.0;
            }
        }
        [[maybe_unused]] const auto* oi = (const __attribute__((address_space(4))) double*)t.oi;
        if (active) {
            if constexpr (SD > 0) {
            } else if constexpr (MP > 0) {
#pragma unroll
                for (int i = 0; i < MP; ++i) member(i, a);
            } else {
                for (int i = 0; i < Mp; ++i) member(i, a);
            }
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                double si = 0.0;
#pragma unroll
                for (int k = 0; k < KP; ++k) {
                    double oia = 0.0;
#pragma unroll
                    for (int j = 0; j < KP; ++j) oia = oia + (SD > 0 ? oi[k * KP + j] : t.OI[k * KP + j]) * a[j][v];
                    si = si + a[k][v] * oia;
                }
                w[v] = 1.0 / pow6_cr(si + 1.0e-12);
            }
        }

        // ---- exchange: lane q = variable
        double ws[4];
        double at[4][KP];
        exchange(w, ws);
#pragma unroll
        for (int k = 0; k < KP; ++k) {
            double x[4] = {a[k][0], a[k][1], a[k][2], a[k][3]}, y[4];
            exchange(x, y);
#pragma unroll
            for (int st = 0; st < 4; ++st) at[st][k] = y[st];
        }

        // ---- phase B: cut-off (face_reconstruction.cpp:948-981)
        constexpr int G = 4;
        const double CT1 = 1.0e-7, CT2 = 1.0e-5;
        double sd = 0.0;
#pragma unroll
        for (int st = 1; st < G; ++st) sd += ws[st];
        if (ws[0] / (sd + ws[0]) > CT1) {
            central = true;
            ws[0] = 1.0;
#pragma unroll
            for (int st = 1; st < G; ++st) ws[st] = 0.0;
        } else {
            if (t.variant != 0) ws[0] = 0.0;
#pragma unroll
            for (int st = 1; st < G; ++st) {
                if (ws[st] / sd > CT2) ws[st] = (1.0 / t.K);
                else if (t.variant != 0) ws[st] = 0.0;
            }
            double s2 = 0.0;
#pragma unroll
            for (int st = 1; st < G; ++st) s2 += ws[st];
#pragma unroll
            for (int st = 1; st < G; ++st) ws[st] /= s2;
        }
        double pw[G][KP];
#pragma unroll
        for (int st = 0; st < G; ++st)
#pragma unroll
            for (int k = 0; k < KP; ++k) pw[st][k] = ws[st] * at[st][k];

        // face points (face_reconstruction.cpp:985-1031)
        if constexpr (CT) {
            // keep the small table's loads here: hoisted to the kernel's
            // start (their addresses are known from info0) they would hold
            // 30 registers through the stencil loop
            __asm__ volatile("" ::: "memory");
        }
#pragma unroll
        for (int fq = 0; fq < FQ; ++fq) {
            double bk[KP];
            if constexpr (CT) {
                static_assert(FQ == 3, "compact tables: one face point per face");
                // the face's reference edge, from the slot-0 info word
                const double* B = t.fbc + ((info0 >> (24 + 2 * fq)) & 3u) * KP;
#pragma unroll
                for (int k = 0; k < KP; ++k) bk[k] = B[k];
            } else if constexpr (DV) {
                static_assert(FQ == 3 && KP == 5, "derived tables: p = 2, one face point per face");
                // face slot fq runs from cell node ia to node ib: the edge
                // (lo, hi) from bits 24 + 2 fq, its direction from the flip bit
                const double2* cv = reinterpret_cast<const double2*>(t.cvert) + 3 * (size_t)cc;
                const double2 n0 = cv[0], n1 = cv[1], n2 = cv[2];
                const TriFrame F = tri_frame(n0.x, n0.y, n1.x, n1.y, n2.x, n2.y);
                const uint32_t e = (info0 >> (24 + 2 * fq)) & 3u;
                const bool flip = ((info0 >> face_flip_shift(fq)) & 1u) != 0u;
                const uint32_t lo = e == 1u ? 1u : 0u, hi = e == 0u ? 1u : 2u;
                const uint32_t ia = flip ? hi : lo, ib = flip ? lo : hi;
                const double xa = ia == 0u ? n0.x : (ia == 1u ? n1.x : n2.x);
                const double ya = ia == 0u ? n0.y : (ia == 1u ? n1.y : n2.y);
                const double xb = ib == 0u ? n0.x : (ib == 1u ? n1.x : n2.x);
                const double yb = ib == 0u ? n0.y : (ib == 1u ? n1.y : n2.y);
                double ax, ay, bx, by;
                to_frame(F, xa, ya, ax, ay);
                to_frame(F, xb, yb, bx, by);
                const double s = (t.qf + 1.0) * 0.5;
                const double xq = s * (bx - ax) + ax, yq = s * (by - ay) + ay;
                // the reference weighting adds ipt_k over the cell's own area in its frame
                const double ta0 = t.variant != 0 ? 1.0 : frame_area(F, n0.x, n0.y, n1.x, n1.y, n2.x, n2.y);
#pragma unroll
                for (int k = 0; k < KP; ++k) {
                    const double psi =
                        legendre_le2(t.poly[2 * k + 2], xq) * legendre_le2(t.poly[2 * k + 3], yq);
                    bk[k] = t.variant != 0 ? psi - t.ipt[k + 1] : psi + (t.ipt[k + 1] / ta0);
                }
            } else {
                const double* B = t.fbasis + (((size_t)lb * FQ + fq) * KP) * 64 + (c & 63u);
#pragma unroll
                for (int k = 0; k < KP; ++k) bk[k] = B[k * 64];
            }
            double acc = ucv;
#pragma unroll
            for (int st = 0; st < G; ++st) {
                if (ws[st] == 0.0) continue;
                acc = acc + (ws[st] * 0.0) * t.basis0;
#pragma unroll
                for (int k = 0; k < KP; ++k) acc = acc + pw[st][k] * bk[k];
            }
            f[fq] = acc;
        }
    };
    // a cell another pass of the split reconstructs: the cell average
    // stands in (positivity leaves it alone) and nothing is stored
    auto skip = [&]() {
#pragma unroll
        for (int fq = 0; fq < FQ; ++fq) f[fq] = ucv;
    };

    if constexpr (SD > 0) {
        full_teno();  // of gated cells too: nothing of theirs is stored
    } else if constexpr (kFullOnly) {
        if (smooth) skip();
        else full_teno();
    } else if (GM != 0 && t.gate && __all(smooth || !valid)) {
        // every cell of the wave takes its central stencil
        smooth = true;  // lanes past the end too: they store nothing
        linear_faces();
    } else if (GM != 0 && smooth) {
        linear_faces();  // a gated cell in a wave with ungated ones
    } else if constexpr (kLinOnly) {
        skip();
    } else {
        full_teno();
    }
    const int v = q;

    if (t.variant != 0) {
        // positivity scaling of the cell's face states (Zhang & Shu 2010):
        // quad lane q takes the limits of face points q and q + 4 (the
        // 40-step bisection is a serial chain, and the quad's four chains
        // run side by side), the smallest holds for the cell
        const double pc = pressure_raw(ph.gamma, uc.v);
        const double eps = fmin(1.0e-13, fmin(uc.v[0], pc));
        double limit = 1.0;
#pragma unroll
        for (int h = 0; h < FQ; h += 4) {
            double x[4], u[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) x[j] = h + j < FQ ? f[h + j < FQ ? h + j : 0] : 0.0;
            exchange(x, u);
            if (h + q < FQ) limit = fmin(limit, point_limit(ph.gamma, uc.v, u, eps));
        }
        const double other = fmin(qperm<kRot1>(limit), fmin(qperm<kRot2>(limit), qperm<kRot3>(limit)));
        const double theta = fmin(limit, other);
        if (theta < 1.0)
#pragma unroll
            for (int fq = 0; fq < FQ; ++fq) f[fq] = ucv + theta * (f[fq] - ucv);
    }
    const uint64_t cmask = __ballot(central);
    if (valid && (kLinOnly ? smooth : kFullOnly ? !smooth : true)) {
#pragma unroll
        for (int fq = 0; fq < FQ; ++fq) fs[((size_t)fq * N + c) * 4 + v] = f[fq];
        if (dec && v == 0) dec[c] = (uint8_t)((cmask >> ((threadIdx.x & 63u) & ~3u)) & 0xFu);
    }
}

// TIGHT (see teno_block): the plain pass at the 6-wave target. The gated
// passes spill less there and the compact tables' pass holds no areas
constexpr bool keep_members_apart(int gm, int occ, bool ct) { return gm == 0 && occ == 6 && !ct; }

// OCC: waves per SIMD the register allocation targets (0: the compiler's
// own choice); an autotuner picks it per mesh, results are identical
template <int KP, int MP, int FQ, typename IdxT, int TILE, int GM, int OCC, bool CT = false, bool DV = false>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(OCC == 0 ? 1 : OCC, OCC == 0 ? 8 : OCC)))
void teno_kernel(Geom g, Teno t, const double* __restrict__ U,
                                                   double* __restrict__ fs, uint8_t* __restrict__ dec,
                                                   Physics ph, uint32_t blocks_per_xcd) {
    // dynamic LDS: the tile's states (TILE cells), then the network when gated
    extern __shared__ __align__(16) unsigned char teno_smem[];
    const uint32_t lb = (blockIdx.x & 7u) * blocks_per_xcd + (blockIdx.x >> 3);
    teno_block<KP, MP, FQ, IdxT, TILE, GM, CT, DV, 0, keep_members_apart(GM, OCC, CT)>(
        g, t, U, fs, dec, ph, lb, reinterpret_cast<double2*>(teno_smem), teno_smem + TILE * 32);
}

// The ungated cells of a split gated pass (mode 5), block by block from the
// list of marked blocks. Few blocks are marked (400 of 8,192 at 524,288
// cells), so the pass is one block's chain, most of it waiting for tables no
// cache holds: streaming them two members ahead takes 43 us to 24. The list
// keeps the other blocks from being started: with a grid over every block
// 64 us streamed and 34 not; at 8,388,608 cells 47 us against 123 for the
// grid without streaming. Four members ahead and two blocks a CU: the same.
// A list of every block costs: with no cell gated the three passes of a step
// of 2,097,152 cells take 1,131 us each instead of 1,110.
constexpr uint32_t kUngatedBlocks = 2048;  // two of the chip's fill; each walks its share of the list
constexpr int kUngatedDepth = 2;
template <bool CT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4, 4)))
void teno_ungated_kernel(Geom g, Teno t, const double* __restrict__ U, double* __restrict__ fs,
                         uint8_t* __restrict__ dec, Physics ph) {
    extern __shared__ __align__(16) unsigned char teno_smem[];
    // each XCD takes one contiguous eighth of the list
    const uint32_t count = t.mixed_list[0], chunk = (count + 7u) >> 3, lo = (blockIdx.x & 7u) * chunk;
    const uint32_t hi = lo + chunk < count ? lo + chunk : count;
    for (uint32_t k = lo + (blockIdx.x >> 3); k < hi; k += gridDim.x >> 3) {
        teno_block<5, 11, 3, uint8_t, 256, 5, CT, false, CT ? 0 : kUngatedDepth>(
            g, t, U, fs, dec, ph, t.mixed_list[1 + k], reinterpret_cast<double2*>(teno_smem), teno_smem + 256 * 32);
        __syncthreads();  // the next block's tile reuses the LDS
    }
}

// The marked blocks in ascending order: one block scans 4,096 marks a round.
__global__ __launch_bounds__(1024) void list_mixed_kernel(const uint32_t* __restrict__ marks, uint32_t n,
                                                          uint32_t* __restrict__ list) {
    __shared__ uint32_t wave_sum[2][16];
    const uint32_t lane = threadIdx.x & 63u, w = threadIdx.x >> 6;
    uint32_t total = 0;
    auto load = [&](uint32_t i, uint32_t (&m)[4]) {
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) m[k] = i + k < n ? marks[i + k] : 0u;
    };
    uint32_t m[4], next[4];
    load(4 * threadIdx.x, m);
    for (uint32_t base = 0, round = 0; base < n; base += 4096, round ^= 1u) {
        load(base + 4096 + 4 * threadIdx.x, next);
        uint32_t mine = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) mine += m[k] ? 1u : 0u;
        uint32_t incl = mine;
        for (uint32_t off = 1; off < 64; off <<= 1) {
            const uint32_t o = __shfl_up(incl, off);
            if (lane >= off) incl += o;
        }
        if (lane == 63) wave_sum[round][w] = incl;
        __syncthreads();
        uint32_t at = total + incl - mine, sum = 0;
        for (uint32_t k = 0; k < 16; ++k) {
            const uint32_t s = wave_sum[round][k];
            if (k < w) at += s;
            sum += s;
        }
        total += sum;
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) {
            if (m[k]) list[1 + at++] = base + 4 * threadIdx.x + k;
            m[k] = next[k];
        }
    }
    if (threadIdx.x == 0) list[0] = total;
}

// the plain pass with streamed member tables: dynamic LDS holds the tile
// (tile_bytes) and the waves' slots
template <int KP, int MP, int FQ, typename IdxT, int SD, int OCC>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(OCC, OCC)))
void teno_stream_kernel(Geom g, Teno t, const double* __restrict__ U, double* __restrict__ fs,
                        uint8_t* __restrict__ dec, Physics ph, uint32_t tile_bytes, uint32_t blocks_per_xcd) {
    extern __shared__ __align__(16) unsigned char teno_smem[];
    const uint32_t lb = (blockIdx.x & 7u) * blocks_per_xcd + (blockIdx.x >> 3);
    teno_block<KP, MP, FQ, IdxT, 0, 0, false, false, SD>(
        g, t, U, fs, dec, ph, lb, reinterpret_cast<double2*>(teno_smem), teno_smem + tile_bytes);
}

__device__ inline const double* case_buf(const CaseBufs& c, int role) {
    return role == kBufUn ? c.Un : (role == kBufUa ? c.Ua : c.Ub);
}
__device__ inline double* case_buf_w(const CaseBufs& c, int role) {
    return role == kBufUn ? c.Un : (role == kBufUa ? c.Ua : (role == kBufUb ? c.Ub : nullptr));
}

// The TENO pass of every case of an ensemble in one launch: the grid covers
// all cases' 64-cell blocks (XCD-aware order over the whole grid), each
// block looks its case up and runs that case's block.
template <int KP, int MP, int FQ, typename IdxT, int TILE, int GM, int OCC, bool DV = false>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(OCC == 0 ? 1 : OCC, OCC == 0 ? 8 : OCC)))
void teno_batch_kernel(const CaseBufs* __restrict__ cases, const uint32_t* __restrict__ teno_case, int in_role,
                                                         uint32_t total, Physics ph, uint32_t blocks_per_xcd) {
    extern __shared__ __align__(16) unsigned char teno_smem[];
    const uint32_t gb = (blockIdx.x & 7u) * blocks_per_xcd + (blockIdx.x >> 3);
    if (gb >= total) return;
    const CaseBufs& cs = cases[teno_case[gb]];
    teno_block<KP, MP, FQ, IdxT, TILE, GM, false, DV, 0, keep_members_apart(GM, OCC, false)>(
        cs.g, cs.t, case_buf(cs, in_role), cs.fs, cs.dec, ph, gb - cs.blk_teno0, reinterpret_cast<double2*>(teno_smem),
        teno_smem + TILE * 32);
}

// ------------------------------------------------------------ viscous terms
// Navier-Stokes extension (no reference counterpart). Sutherland viscosity.
__device__ inline double viscosity(const Physics& ph, double T) {
    if (ph.S_mu < 0.0) return ph.mu_ref;
    const double t = T / ph.T_mu;
    return ph.mu_ref * (t * sqrt(t)) * ((ph.T_mu + ph.S_mu) / (T + ph.S_mu));
}

// Values of (u, v, T) a boundary face holds for the gradients: no-slip wall
// (u, v) = 0; slip wall and symmetry the tangential velocity; fixed (u, p, T)
// its values; extrapolation and p_out the cell's own (no contribution).
__device__ inline void boundary_uvT(const BCParam& b, double n0, double n1, const double* c, double* f) {
    if (b.type == 5) {
        f[0] = 0.0; f[1] = 0.0; f[2] = c[2];
    } else if (b.type == 0 || b.type == 2) {
        const double un = c[0] * n0 + c[1] * n1;
        f[0] = c[0] - un * n0; f[1] = c[1] - un * n1; f[2] = c[2];
    } else if (b.type == 3) {
        f[0] = b.u0; f[1] = b.u1; f[2] = b.T;
    } else {
        f[0] = c[0]; f[1] = c[1]; f[2] = c[2];
    }
}

// One thread per cell: (u, v, T, mu) of the state and the weighted
// least-squares gradients of u, v and T over the face neighbours (weights
// 1/|d|^2, d from the centroid to the neighbour's centroid or to the boundary
// face's midpoint), exact for linear fields.
__global__ __launch_bounds__(256) void viscous_grad_kernel(Geom g, const double* __restrict__ U, Physics ph,
                                                           double* __restrict__ vp, double* __restrict__ vg,
                                                           uint32_t blocks_per_xcd) {
    const uint32_t lb = (blockIdx.x & 7u) * blocks_per_xcd + (blockIdx.x >> 3);
    const uint32_t c = lb * blockDim.x + threadIdx.x;
    if (c >= g.N) return;
    double Wc[5];
    const D4 uc = ld4(U, c);
    prims(ph, uc.v, Wc);
    const double pc[3] = {Wc[0], Wc[1], Wc[3]};
    double a11 = 0.0, a12 = 0.0, a22 = 0.0, b[3][2] = {{0.0, 0.0}, {0.0, 0.0}, {0.0, 0.0}};
    for (uint32_t l = 0; l < g.S; ++l) {
        const size_t o = (size_t)l * g.N + c;
        const uint32_t inf = g.info[o];
        const double dx = g.dcx[o], dy = g.dcy[o];
        double pf[3];
        if (!(inf & kBoundaryBit)) {
            double Wn[5];
            const D4 un = ld4(U, (uint32_t)g.nb[o]);
            prims(ph, un.v, Wn);
            pf[0] = Wn[0]; pf[1] = Wn[1]; pf[2] = Wn[3];
        } else {
            boundary_uvT(g.bc[(inf >> 4) & 0xFu], g.nx[o], g.ny[o], pc, pf);
        }
        const double w = 1.0 / (dx * dx + dy * dy);
        a11 += w * dx * dx;
        a12 += w * dx * dy;
        a22 += w * dy * dy;
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const double dp = w * (pf[k] - pc[k]);
            b[k][0] += dx * dp;
            b[k][1] += dy * dp;
        }
    }
    const double id = 1.0 / (a11 * a22 - a12 * a12);
    double gr[6];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        gr[2 * k] = (a22 * b[k][0] - a12 * b[k][1]) * id;
        gr[2 * k + 1] = (a11 * b[k][1] - a12 * b[k][0]) * id;
    }
    st4(vp, c, D4{{pc[0], pc[1], pc[2], viscosity(ph, pc[2])}});
    double2* G2 = reinterpret_cast<double2*>(vg + 6 * (size_t)c);
    G2[0] = make_double2(gr[0], gr[1]);
    G2[1] = make_double2(gr[2], gr[3]);
    G2[2] = make_double2(gr[4], gr[5]);
}

// Viscous flux through a face, in the face's orientation (unit normal n from
// its side-0 cell L, slot sL, to R, slot sR): G = (0, tau n, (u tau + k grad T) n). Face
// gradients are the mean of the two cells' gradients with the directional
// derivative along d = x_R - x_L replaced by (phi_R - phi_L) / |d|; the face
// velocity is the mean of both cells' linear extrapolations to the face
// midpoint. On a boundary face the cell's gradient is corrected toward the
// boundary value along the centroid-to-midpoint vector. All of it is exact
// for linear fields.
__device__ inline void viscous_face(const Physics& ph, const Geom& g, const StageArgs& a, uint32_t L, uint32_t sL,
                                    uint32_t R, uint32_t sR, bool bnd, uint32_t bc, double n0, double n1, double* G) {
    G[0] = 0.0; G[1] = 0.0; G[2] = 0.0; G[3] = 0.0;
    int bt = -1;
    if (bnd) {
        bt = g.bc[bc].type;
        if (bt == 0 || bt == 2) return;  // symmetry, slip wall: no viscous stress or heat flux
    }
    const size_t oL = (size_t)sL * g.N + L;
    const D4 pL = ld4(a.vp, L);
    const double2* gL2 = reinterpret_cast<const double2*>(a.vg + 6 * (size_t)L);
    const double2 gL0 = gL2[0], gL1 = gL2[1], gL3 = gL2[2];
    const double dx = g.dcx[oL], dy = g.dcy[oL];
    const double il = 1.0 / sqrt(dx * dx + dy * dy);
    const double tx = dx * il, ty = dy * il;
    double gx[3], gy[3], uf, vf, mu;
    const double phL[3] = {pL.v[0], pL.v[1], pL.v[2]};
    if (!bnd) {
        const D4 pR = ld4(a.vp, R);
        const double2* gR2 = reinterpret_cast<const double2*>(a.vg + 6 * (size_t)R);
        const double2 gR0 = gR2[0], gR1 = gR2[1], gR3 = gR2[2];
        gx[0] = 0.5 * (gL0.x + gR0.x); gy[0] = 0.5 * (gL0.y + gR0.y);
        gx[1] = 0.5 * (gL1.x + gR1.x); gy[1] = 0.5 * (gL1.y + gR1.y);
        gx[2] = 0.5 * (gL3.x + gR3.x); gy[2] = 0.5 * (gL3.y + gR3.y);
        const double phR[3] = {pR.v[0], pR.v[1], pR.v[2]};
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const double corr = (phR[k] - phL[k]) * il - (gx[k] * tx + gy[k] * ty);
            gx[k] += corr * tx;
            gy[k] += corr * ty;
        }
        const size_t oR = (size_t)sR * g.N + R;
        // centroid-to-midpoint vectors
        const double mLx = g.mfx[oL], mLy = g.mfy[oL], mRx = g.mfx[oR], mRy = g.mfy[oR];
        uf = 0.5 * ((pL.v[0] + (gL0.x * mLx + gL0.y * mLy)) + (pR.v[0] + (gR0.x * mRx + gR0.y * mRy)));
        vf = 0.5 * ((pL.v[1] + (gL1.x * mLx + gL1.y * mLy)) + (pR.v[1] + (gR1.x * mRx + gR1.y * mRy)));
        mu = 0.5 * (pL.v[3] + pR.v[3]);
    } else {
        gx[0] = gL0.x; gy[0] = gL0.y;
        gx[1] = gL1.x; gy[1] = gL1.y;
        gx[2] = gL3.x; gy[2] = gL3.y;
        double pf[3];
        boundary_uvT(g.bc[bc], n0, n1, phL, pf);
        if (bt != 1 && bt != 4) {  // a prescribed value: correct toward it
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                const double corr = (pf[k] - phL[k]) * il - (gx[k] * tx + gy[k] * ty);
                gx[k] += corr * tx;
                gy[k] += corr * ty;
            }
        }
        uf = pf[0];
        vf = pf[1];
        mu = pL.v[3];
    }
    const double div = gx[0] + gy[1];
    const double txx = mu * (2.0 * gx[0] - (2.0 / 3.0) * div);
    const double tyy = mu * (2.0 * gy[1] - (2.0 / 3.0) * div);
    const double txy = mu * (gy[0] + gx[1]);
    G[1] = txx * n0 + txy * n1;
    G[2] = txy * n0 + tyy * n1;
    // adiabatic no-slip wall: u = 0 and no heat flux
    if (bt == 5) return;
    const double k = mu * ph.cp / ph.Pr;
    G[3] = uf * G[1] + vf * G[2] + k * (gx[2] * n0 + gy[2] * n1);
}

// ------------------------------------------------------------ flux + update
// The fluxes of a block of cells, then the residual and the stage update of
// each cell. A block of bs cells takes every face of its cells once (the
// face lists of its 64-cell blocks), one face per thread and round, and leaves
// area times flux in LDS; after a barrier one thread per cell sums its faces
// in the canonical order, divides by the volume and applies the stage's
// SSP-RK update (no atomics). A flux has the same bits for both cells of its
// face, so the sums equal a serial run's in the one-thread order.
// What bounds it: on a full chip FP64 issue (8,388,608 cells: 2,586 VALU
// instructions per wave, the SIMDs issuing 77% of the launch, 1.75 GB moved
// where one thread per cell and its three faces moved 3.07 GB); on small
// meshes the chain of divisions, square roots and powers in one flux.
// Evaluating a face once per block instead of once per cell takes 1.7
// evaluations per cell instead of 3, and reads 58 B of face lists instead of
// 96 B of slot arrays per cell. HLLC on a flow with waves everywhere (rocprof;
// one thread per cell -> faces once -> with the leaner powers of
// riemann.hpp): 8,388,608 cells 1,161 -> 973 -> 871 us on one machine,
// 524,288 72.8 -> 51.9 -> 49.5 us, 2,048 26.4 -> 9 -> 8.5 us. Faces once
// alone: with the limiter, 73,006 cells 35 -> 16 us; viscous Roe, 99,700
// cells 22.8 -> 16 us. Holding the registers (about 100 for HLLC, 4 waves
// per SIMD) to 5 waves costs time: 8,388,608 cells 957 us against 895, at 6
// waves 1,110 us. So does pooling the faces that take the two-rarefaction
// estimate, its three powers 550 of a flux's 1,300 instructions, onto the
// block's first threads through LDS: 524,288 cells 57.4 us against 50.1, the
// two barriers and the 28 more registers cost more than the idle lanes.
// RS: Riemann solver (compile-time, so each instantiation carries one
// solver's code and registers). PP: the positivity-preserving flux limiter
// (pp_limit) on every face, for the stage updates (not the residual-only
// operator, which has no dt). VISC: the viscous fluxes.
template <int RS, bool PP, bool VISC>
__device__ __forceinline__ void face_flux(const Geom& g, const StageArgs& a, const Physics& ph, uint32_t e,
                                          [[maybe_unused]] double pdt, double* out) {
    const uint32_t N = g.N, Q = g.Q;
    const uint32_t meta = g.face_meta[e], c0 = g.face_c0[e], c1 = g.face_c1[e];
    const uint32_t s0 = meta & 3u, s1 = (meta >> kFaceSlot1Shift) & 3u, bc = (meta >> kFaceBcShift) & 0xFu;
    const bool bnd = (meta & kFaceBoundary) != 0;
    const double n0 = g.face_nx[e], n1 = g.face_ny[e], ar = g.face_area[e];
    double F[4] = {0.0, 0.0, 0.0, 0.0};
    for (uint32_t q = 0; q < Q; ++q) {
        D4 L, R;
        if (a.fo) {
            L = ld4(a.Uin, c0);
            R = ld4(a.Uin, c1);
        } else {
            L = ld4(a.fs, (size_t)(s0 * Q + q) * N + c0);
            // on a boundary (c1 = c0) the state an extrapolation boundary
            // copies into its ghost: the face state itself
            // (boundary_extrapolation.cpp:38-55), or in the corrected variant
            // the cell mean
            if (!bnd) R = ld4(a.fs, (size_t)(s1 * Q + q) * N + c1);
            else R = a.corrected ? ld4(a.Uin, c0) : L;
        }
        double Ft[4];
        point_flux(ph, g.bc, RS, a.corrected, bnd, bc, n0, n1, L.v, R.v, Ft);
        const double wq = g.qw[q];
#pragma unroll
        for (int i = 0; i < 4; i++) F[i] += wq * Ft[i];
    }
#pragma unroll
    for (int i = 0; i < 4; i++) F[i] *= 0.5;
    if constexpr (PP) {
        const D4 U0 = ld4(a.Uin, c0), U1 = ld4(a.Uin, c1);
        const double Sd = (double)g.S;
        pp_limit(ph, g.bc, bnd, bc, n0, n1, F, U0.v, Sd * pdt * ar / g.volume[c0], U1.v,
                 Sd * pdt * ar / g.volume[c1]);
    }
    if constexpr (VISC) {
        double G[4];
        viscous_face(ph, g, a, c0, s0, c1, s1, bnd, bc, n0, n1, G);
#pragma unroll
        for (int i = 1; i < 4; i++) F[i] -= G[i];
    }
#pragma unroll
    for (int i = 0; i < 4; i++) out[i] = ar * F[i];
}

// The stage's update of cell c with its residual r.
__device__ __forceinline__ void stage_update(const StageArgs& a, const Physics& ph, uint32_t c, double dt,
                                             const double* r) {
    if (a.op == kRhsOnly) {
        st4(a.rhs, c, D4{{r[0], r[1], r[2], r[3]}});
        return;
    }
    const D4 un = ld4(a.Un, c);
    D4 out, wa;
    bool final_stage = false;
    switch (a.op) {
    case kFE:
        for (int i = 0; i < 4; i++) out.v[i] = un.v[i] + dt * r[i];
        st4(a.Uout, c, out);
        final_stage = true;
        break;
    case kSSP1: {
        const double c0 = dt * (1.0 / 6.0);
        for (int i = 0; i < 4; i++) { out.v[i] = un.v[i] + dt * r[i]; wa.v[i] = un.v[i] + c0 * r[i]; }
        st4(a.Uout, c, out);
        st4(a.W, c, wa);
        break;
    }
    case kSSP2: {
        const D4 u1 = ld4(a.Uin, c);
        const D4 w0 = ld4(a.W, c);
        const double c1 = dt * (1.0 / 6.0), d4 = dt / 4.0;
        for (int i = 0; i < 4; i++) {
            const double y = 3.0 / 4.0 * un.v[i] + 1.0 / 4.0 * u1.v[i];
            out.v[i] = y + d4 * r[i];
            wa.v[i] = w0.v[i] + c1 * r[i];
        }
        st4(a.Uout, c, out);
        st4(a.W, c, wa);
        break;
    }
    case kSSP3: {
        const D4 w0 = ld4(a.W, c);
        const double c2 = dt * (2.0 / 3.0);
        for (int i = 0; i < 4; i++) out.v[i] = w0.v[i] + c2 * r[i];
        st4(a.Uout, c, out);
        final_stage = true;
        break;
    }
    case kRK4_1: case kRK4_2: case kRK4_3: {
        const double half = dt / 2.0;
        const double cs = a.op == kRK4_1 ? dt * (1.0 / 6.0) : dt * (1.0 / 3.0);
        const double step = a.op == kRK4_3 ? dt : half;
        D4 w0 = un;
        if (a.op != kRK4_1) w0 = ld4(a.W, c);
        for (int i = 0; i < 4; i++) { out.v[i] = un.v[i] + step * r[i]; wa.v[i] = w0.v[i] + cs * r[i]; }
        st4(a.Uout, c, out);
        st4(a.W, c, wa);
        break;
    }
    case kRK4_4: {
        const D4 w0 = ld4(a.W, c);
        const double c3 = dt * (1.0 / 6.0);
        for (int i = 0; i < 4; i++) out.v[i] = w0.v[i] + c3 * r[i];
        st4(a.Uout, c, out);
        final_stage = true;
        break;
    }
    default: break;
    }
    if (final_stage && a.prims) {
        double W5[5];
        prims(ph, out.v, W5);
        st4(a.prims, c, D4{{W5[0], W5[1], W5[2], W5[3]}});
        a.h[c] = W5[4];
    }
}

// JOIN: the pass is a step's first and finds the time step. Every block joins
// the block maxima of the radii (at most kJoinBlocks over its threads: 2 each
// of 512 to 16 each of the 64 of a large ensemble's smallest blocks; loaded
// before the faces and joined at the barrier after them), so the step has no
// launch of one block for it: 4.5 us of 82 at 8,192 cells, while a block's join
// adds under 1 us. Above kJoinBlocks maxima one block joins them in its own
// launch.
__device__ inline unsigned long long wave_max(unsigned long long m) {
    for (int off = 32; off > 0; off >>= 1) {
        const unsigned long long o = __shfl_xor(m, off);
        m = o > m ? o : m;
    }
    return m;
}

// lb: flux block of bs cells; sf: LDS for 4 planes of its face-list entries
template <int RS, bool PP, bool VISC, bool JOIN>
__device__ __forceinline__ void flux_block(const Geom& g, const StageArgs& a, const Physics& ph, uint32_t lb,
                                           uint32_t bs, double* sf, const DtJoin& jn) {
    const uint32_t N = g.N, first = lb * bs;
    if (first >= N) return;  // whole block past the end (uniform)
    const uint32_t last = N - first < bs ? N : first + bs;
    const uint32_t f0 = g.face_off[first >> 6], nf = g.face_off[(last + 63u) >> 6] - f0;
    __shared__ unsigned long long sh_max[JOIN ? 8 : 1];  // a wave each
    unsigned long long m = 0ull;
    auto share = [&]() {
        m = wave_max(m);
        if ((threadIdx.x & 63u) == 0u) sh_max[threadIdx.x >> 6] = m;
    };
    auto joined = [&]() {
        for (uint32_t w = 0; w < (blockDim.x >> 6); ++w) m = sh_max[w] > m ? sh_max[w] : m;
        return jn.fixed_dt > 0.0 ? jn.fixed_dt : jn.cfl / __longlong_as_double((long long)m);
    };
    double dt = 0.0;
    if constexpr (JOIN) {
        if (!(jn.fixed_dt > 0.0))
            for (uint32_t i = threadIdx.x; i < jn.n_blk; i += blockDim.x) m = jn.lam_blk[i] > m ? jn.lam_blk[i] : m;
        if constexpr (PP) {  // the limiter needs it at the faces
            share();
            __syncthreads();
            dt = joined();
        }
    } else if (a.op != kRhsOnly) {
        dt = *a.dt;
    }
    for (uint32_t i = threadIdx.x; i < nf; i += blockDim.x) {
        if (a.parts != 3 && !(a.parts & (g.face_meta[f0 + i] & kFaceBoundary ? 2 : 1))) continue;
        double F[4];
        face_flux<RS, PP, VISC>(g, a, ph, f0 + i, dt, F);
#pragma unroll
        for (int k = 0; k < 4; ++k) sf[k * nf + i] = F[k];
    }
    if constexpr (JOIN && !PP) share();
    __syncthreads();
    if constexpr (JOIN) {
        if constexpr (!PP) dt = joined();
        if (lb == 0 && threadIdx.x == 0) {
            *jn.dt = dt;
            if (jn.dt_hist) jn.dt_hist[*jn.step % jn.hist_cap] = dt;
            *jn.step += 1;
        }
    }
    for (uint32_t c = first + threadIdx.x; c < last; c += blockDim.x) {
        const uint32_t slots = g.cell_faces[c], sum = g.cell_sum[c];
        const uint32_t base = g.face_off[c >> 6] - f0, count = (sum >> kSumCountShift) & 0x7u;
        double r[4] = {0.0, 0.0, 0.0, 0.0};
        for (uint32_t rk = 0; rk < count; ++rk) {
            const uint32_t l = (sum >> (2 * rk)) & 3u;
            if (!(a.parts & ((sum >> (kSumBoundaryShift + l)) & 1u ? 2 : 1))) continue;
            const uint32_t i = base + ((slots >> (8 * l)) & 0xFFu);
            const bool side = ((sum >> (kSumSideShift + l)) & 1u) != 0;
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const double f = sf[k * nf + i];
                r[k] += side ? f : -f;
            }
        }
        const double vol = g.volume[c];
#pragma unroll
        for (int k = 0; k < 4; k++) r[k] /= vol;
        stage_update(a, ph, c, dt, r);
    }
}

template <int RS, bool PP, bool VISC, bool JOIN>
__global__ __launch_bounds__(512) void flux_update_kernel(Geom g, StageArgs a, Physics ph, uint32_t bs,
                                                          uint32_t blocks_per_xcd, DtJoin jn) {
    extern __shared__ __align__(16) unsigned char flux_smem[];
    const uint32_t lb = (blockIdx.x & 7u) * blocks_per_xcd + (blockIdx.x >> 3);
    flux_block<RS, PP, VISC, JOIN>(g, a, ph, lb, bs, reinterpret_cast<double*>(flux_smem), jn);
}

__device__ inline StageArgs case_stage(const CaseBufs& cs, int op, int riemann, int fo, int corrected, int in,
                                       int out) {
    StageArgs a{};
    a.op = op;
    a.riemann = riemann;
    a.fo = fo;
    a.corrected = corrected;
    a.parts = 3;
    a.Uin = case_buf(cs, in);
    a.Un = cs.Un;
    a.Uout = case_buf_w(cs, out);
    a.W = cs.W;
    a.prims = cs.prims;
    a.h = cs.h;
    a.rhs = cs.rhs;
    a.fs = cs.fs;
    a.dt = cs.dt;
    return a;
}

// The flux + stage update of every case in one launch (blocks of bs cells;
// the case table's block offsets count blocks of that size).
template <int RS, bool PP, bool JOIN>
__global__ __launch_bounds__(256) void flux_batch_kernel(const CaseBufs* __restrict__ cases,
                                                         const uint32_t* __restrict__ flux_case, BatchStage st,
                                                         uint32_t total, Physics ph, uint32_t bs,
                                                         uint32_t blocks_per_xcd) {
    extern __shared__ __align__(16) unsigned char flux_smem[];
    const uint32_t gb = (blockIdx.x & 7u) * blocks_per_xcd + (blockIdx.x >> 3);
    if (gb >= total) return;
    const CaseBufs& cs = cases[flux_case[gb]];
    const StageArgs a = case_stage(cs, st.op, RS, st.fo, st.corrected, st.in, st.out);
    DtJoin jn{};
    if constexpr (JOIN)
        jn = DtJoin{cs.lam_blk, (cs.g.N + bs - 1) / bs, st.cfl, st.fixed_dt, cs.dt, cs.dt_hist, st.hist_cap, cs.step};
    flux_block<RS, PP, false, JOIN>(cs.g, a, ph, gb - cs.blk_flux0, bs, reinterpret_cast<double*>(flux_smem), jn);
}

// ------------------------------------------------------------ dt
// solver.cpp:592-706: per-cell spectral radius over the cell's faces in
// local order; the block's maximum, joined over the blocks by
// finalize_dt_kernel.
__device__ __forceinline__ void spectral_block(const Geom& g, const double* __restrict__ Un,
                                               const double* __restrict__ pr, const Physics& ph,
                                               double* __restrict__ lam_cell, unsigned long long* __restrict__ lam_blk,
                                               uint32_t lb) {
    const uint32_t N = g.N;
    const uint32_t c = lb * blockDim.x + threadIdx.x;
    double lam = 0.0;
    bool ok = false;
    if (c < N) {
        const D4 wc = ld4(pr, c);
        const double rc = Un[4 * (size_t)c];
        const double sc = sqrt(ph.gamma * wc.v[2] / rc);
        double conv = 0.0, acou = 0.0;
        const uint32_t S = g.S;
        for (uint32_t l = 0; l < S; ++l) {
            const size_t o = (size_t)l * N + c;
            const uint32_t nbc = (uint32_t)g.nb[o];
            const double n0 = g.nx[o], n1 = g.ny[o], dxn = g.dxn[o];
            const D4 wn = ld4(pr, nbc);
            const double rn = Un[4 * (size_t)nbc];
            const double sn = sqrt(ph.gamma * wn.v[2] / rn);
            const double sf = 0.5 * (sc + sn);
            const double uf0 = 0.5 * (wc.v[0] + wn.v[0]), uf1 = 0.5 * (wc.v[1] + wn.v[1]);
            const double un = fabs(uf0 * n0 + uf1 * n1);
            conv += un / dxn;
            const double qq = sf / dxn;
            acou += qq * qq;
        }
        const double gf = 3.0 / S;
        conv *= 1.37 * gf;
        acou = 1.37 * sqrt(gf * acou);
        lam = conv + acou;
        if (ph.viscous) {
            // viscous radius max(4/3, gamma/Pr) (mu / rho) sum_f (A_f / V)^2
            const double V = g.volume[c];
            double s2 = 0.0;
            for (uint32_t l = 0; l < S; ++l) {
                const double q = g.area[(size_t)l * N + c] / V;
                s2 += q * q;
            }
            lam += fmax(4.0 / 3.0, ph.gamma / ph.Pr) * (viscosity(ph, wc.v[3]) / rc) * s2;
        }
        lam_cell[c] = lam;
        ok = lam == lam;  // NaN radii are ignored by the reference's max join
    }
    // non-negative doubles order like their bit patterns
    unsigned long long bits = ok ? (unsigned long long)__double_as_longlong(lam) : 0ull;
    for (int off = 32; off > 0; off >>= 1) {
        const unsigned long long o2 = __shfl_xor(bits, off);
        bits = o2 > bits ? o2 : bits;
    }
    __shared__ unsigned long long sh[4];
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = bits;
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long m = sh[0];
        for (int i = 1; i < (int)(blockDim.x >> 6); ++i) m = sh[i] > m ? sh[i] : m;
        lam_blk[lb] = m;  // the block's maximum; the step's first flux pass or the finalize kernel joins them
    }
}

// max over n per-block maxima (bit patterns of non-negative doubles) by one
// block; every thread returns the result
__device__ inline unsigned long long join_blocks(const unsigned long long* __restrict__ lam_blk, uint32_t n) {
    unsigned long long m = 0ull;
    const uint32_t st = blockDim.x;
    uint32_t i = threadIdx.x;
    // 8 loads in flight per thread (the max is order-free)
    for (; i + 7 * st < n; i += 8 * st) {
        unsigned long long v[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) v[k] = lam_blk[i + k * st];
#pragma unroll
        for (int k = 0; k < 8; ++k) m = v[k] > m ? v[k] : m;
    }
    for (; i < n; i += st) m = lam_blk[i] > m ? lam_blk[i] : m;
    for (int off = 32; off > 0; off >>= 1) {
        const unsigned long long o2 = __shfl_xor(m, off);
        m = o2 > m ? o2 : m;
    }
    __shared__ unsigned long long sh[16];
    __syncthreads();
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = m;
    __syncthreads();
    m = sh[0];
    for (int i = 1; i < (int)(blockDim.x >> 6); ++i) m = sh[i] > m ? sh[i] : m;
    return m;
}

__global__ __launch_bounds__(256) void spectral_kernel(Geom g, const double* __restrict__ Un,
                                                       const double* __restrict__ pr, Physics ph,
                                                       double* __restrict__ lam_cell,
                                                       unsigned long long* __restrict__ lam_blk,
                                                       uint32_t blocks_per_xcd) {
    // each XCD walks one contiguous range of blocks (its neighbours' states stay in its L2)
    const uint32_t lb = (blockIdx.x & 7u) * blocks_per_xcd + (blockIdx.x >> 3);
    if (lb * blockDim.x >= g.N) return;  // past the last block (uniform)
    spectral_block(g, Un, pr, ph, lam_cell, lam_blk, lb);
}

// spectral radii of every case in one launch (each block inside one case, so
// the block max goes to that case's maximum)
__global__ __launch_bounds__(256) void spectral_batch_kernel(const CaseBufs* __restrict__ cases,
                                                             const uint32_t* __restrict__ flux_case,
                                                             uint32_t total, Physics ph, uint32_t blocks_per_xcd) {
    const uint32_t gb = (blockIdx.x & 7u) * blocks_per_xcd + (blockIdx.x >> 3);
    if (gb >= total) return;
    const CaseBufs& cs = cases[flux_case[gb]];
    spectral_block(cs.g, cs.Un, cs.prims, ph, cs.lam_cell, cs.lam_blk, gb - cs.blk_flux0);
}

// dt = cfl / max lambda over the per-block maxima (one block of 1024 threads)
// or the fixed dt; its history entry and the step counter
__global__ __launch_bounds__(1024) void finalize_dt_kernel(const unsigned long long* __restrict__ lam_blk,
                                                           uint32_t n_blk, double cfl, double fixed_dt, double* dt,
                                                           double* dt_hist, int64_t hist_cap, int64_t* step) {
    const unsigned long long m = fixed_dt > 0.0 ? 0ull : join_blocks(lam_blk, n_blk);
    if (threadIdx.x != 0) return;
    const double d = fixed_dt > 0.0 ? fixed_dt : cfl / __longlong_as_double((long long)m);
    *dt = d;
    if (dt_hist && step) dt_hist[*step % hist_cap] = d;
    if (step) *step += 1;
}

// one case's dt from its per-block maxima (blocks of bs cells), its history
// entry and step counter; every thread of the block takes part
__device__ inline void finalize_case(const CaseBufs& cs, double cfl, double fixed_dt, int64_t hist_cap, uint32_t bs) {
    const unsigned long long m = fixed_dt > 0.0 ? 0ull : join_blocks(cs.lam_blk, (cs.g.N + bs - 1) / bs);
    if (threadIdx.x != 0) return;
    const double d = fixed_dt > 0.0 ? fixed_dt : cfl / __longlong_as_double((long long)m);
    *cs.dt = d;
    cs.dt_hist[*cs.step % hist_cap] = d;
    *cs.step += 1;
}

// per-case dt of an ensemble: block k finalises case k
__global__ __launch_bounds__(256) void finalize_batch_kernel(const CaseBufs* __restrict__ cases, int n_cases,
                                                             double cfl, double fixed_dt, int64_t hist_cap,
                                                             uint32_t bs) {
    const int k = blockIdx.x;
    if (k >= n_cases) return;
    finalize_case(cases[k], cfl, fixed_dt, hist_cap, bs);
}

// ------------------------------------------------------------ persistent ensemble step
// The whole step of every case in one cooperative launch: the spectral radii
// and each case's dt, then per stage the TENO face states and the flux +
// stage update, with a grid-wide barrier between phases. The grid holds as
// many blocks as fit on the GPU at once; each phase's work items (64-cell
// TENO blocks, 256-cell flux / spectral blocks, over all cases through the
// offset table) are dealt out so that each XCD walks one contiguous eighth,
// as the per-phase kernels do. Every item runs the per-phase kernels' own
// per-cell code, so results are bit-identical to them.
// Grid-wide barrier of the persistent launch (every block resident: the
// cooperative launch guarantees it). Each wave first waits for its own
// stores to reach its XCD's L2; then one thread per block releases them past
// that L2 (each XCD has its own), arrives on a counter and waits for the
// generation the last arrival advances, and drops stale lines of its L2 once
// through. The waits poll with relaxed loads and no invalidation, so blocks
// that arrive early leave the L2 of those still working alone. A wait longer
// than spin_ticks of the device wall clock gives up and raises bar->err (the
// launch then still ends; the host reports the error and resets the state).
__device__ inline void grid_barrier(StepBarrier* bar, uint32_t n_blocks, long long spin_ticks) {
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (threadIdx.x == 0) {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
        const uint32_t g = __hip_atomic_load(&bar->gen, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (__hip_atomic_fetch_add(&bar->count, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == n_blocks - 1) {
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");  // every arrival's release is ordered before
            __hip_atomic_store(&bar->count, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(&bar->gen, g + 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
        } else {
            const long long t0 = wall_clock64();
            while (__hip_atomic_load(&bar->gen, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == g) {
                __builtin_amdgcn_s_sleep(8);
                if (wall_clock64() - t0 > spin_ticks) {
                    __hip_atomic_store(&bar->err, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    break;
                }
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    }
    __syncthreads();
}

template <int RS, bool TENO>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4, 8)))
void ensemble_step_kernel(const CaseBufs* __restrict__ cases, int n_cases, const uint32_t* __restrict__ teno_case,
                          const uint32_t* __restrict__ flux_case, uint32_t teno_total, uint32_t flux_total,
                          PersistentStep ps, Physics ph) {
    extern __shared__ __align__(16) unsigned char step_smem[];
    const uint32_t G = gridDim.x, xcd = blockIdx.x & 7u, rank = blockIdx.x >> 3;
    const uint32_t on_xcd = (G + 7u - xcd) >> 3;
    auto stamp = [&](int i) {
        if (ps.clocks && blockIdx.x == 0 && threadIdx.x == 0) ps.clocks[i] = wall_clock64();
    };
    stamp(0);
    auto each = [&](uint32_t total, auto&& f) {
        const uint32_t per = (total + 7u) >> 3, lo = xcd * per, hi = lo + per < total ? lo + per : total;
        for (uint32_t w = lo + rank; w < hi; w += on_xcd) {
            f(w);
            __syncthreads();  // the next item reuses the block's LDS
        }
    };
    if (ps.use_cfl) {
        each(flux_total, [&](uint32_t gb) {
            const CaseBufs& cs = cases[flux_case[gb]];
            spectral_block(cs.g, cs.Un, cs.prims, ph, cs.lam_cell, cs.lam_blk, gb - cs.blk_flux0);
        });
        grid_barrier(ps.bar, G, ps.spin_ticks);
    }
    stamp(1);
    for (int k = (int)blockIdx.x; k < n_cases; k += (int)G) {
        finalize_case(cases[k], ps.cfl, ps.fixed_dt, ps.hist_cap, 256u);
        __syncthreads();
    }
    grid_barrier(ps.bar, G, ps.spin_ticks);
    stamp(2);
#pragma unroll 1
    for (int st = 0; st < ps.n_stages; ++st) {
        if constexpr (TENO) {
            each(teno_total, [&](uint32_t gb) {
                const CaseBufs& cs = cases[teno_case[gb]];
                teno_block<5, 11, 3, uint8_t, 256, 0>(cs.g, cs.t, case_buf(cs, ps.in[st]), cs.fs, cs.dec, ph,
                                                      gb - cs.blk_teno0, reinterpret_cast<double2*>(step_smem),
                                                      step_smem + 256 * 32);
            });
            grid_barrier(ps.bar, G, ps.spin_ticks);
        }
        stamp(3 + 2 * st);
        each(flux_total, [&](uint32_t gb) {
            const CaseBufs& cs = cases[flux_case[gb]];
            const StageArgs a = case_stage(cs, ps.op[st], RS, ps.fo, ps.corrected, ps.in[st], ps.out[st]);
            flux_block<RS, false, false, false>(cs.g, a, ph, gb - cs.blk_flux0, blockDim.x,
                                                reinterpret_cast<double*>(step_smem), DtJoin{});
        });
        if (st + 1 < ps.n_stages || ps.clocks) grid_barrier(ps.bar, G, ps.spin_ticks);
        stamp(4 + 2 * st);
    }
}

__global__ void copy_kernel(const double* __restrict__ s, double* __restrict__ d, size_t n) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) d[i] = s[i];
}

// Streaming probes: the bandwidth HBM delivers to a plain access pattern
// (16 B per lane, grid-stride, 4 loads in flight per lane), the practical
// ceiling the gather kernels are compared with.
__global__ __launch_bounds__(256) void stream_copy_kernel(const double2* __restrict__ s, double2* __restrict__ d,
                                                          size_t n) {
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    for (; i + 3 * stride < n; i += 4 * stride) {
        const double2 a = s[i], b = s[i + stride], c = s[i + 2 * stride], e = s[i + 3 * stride];
        d[i] = a;
        d[i + stride] = b;
        d[i + 2 * stride] = c;
        d[i + 3 * stride] = e;
    }
    for (; i < n; i += stride) d[i] = s[i];
}

__global__ __launch_bounds__(256) void stream_read_kernel(const double2* __restrict__ s, double* __restrict__ out,
                                                          size_t n) {
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    double acc0 = 0.0, acc1 = 0.0;
    for (; i + 3 * stride < n; i += 4 * stride) {
        const double2 a = s[i], b = s[i + stride], c = s[i + 2 * stride], e = s[i + 3 * stride];
        acc0 += (a.x + b.x) + (c.x + e.x);
        acc1 += (a.y + b.y) + (c.y + e.y);
    }
    for (; i < n; i += stride) acc0 += s[i].x + s[i].y;
    out[(size_t)blockIdx.x * blockDim.x + threadIdx.x] = acc0 + acc1;
}

// Two more read patterns for the same ceiling: 64 contiguous bytes per lane
// per iteration (four 16-byte loads from one lane's own run), and 16-byte
// non-temporal loads (no reuse expected in the caches).
__global__ __launch_bounds__(256) void stream_read_wide_kernel(const double2* __restrict__ s,
                                                               double* __restrict__ out, size_t n) {
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    double acc0 = 0.0, acc1 = 0.0;
    for (; 4 * i + 3 < n; i += stride) {
        const double2 a = s[4 * i], b = s[4 * i + 1], c = s[4 * i + 2], e = s[4 * i + 3];
        acc0 += (a.x + b.x) + (c.x + e.x);
        acc1 += (a.y + b.y) + (c.y + e.y);
    }
    for (size_t j = 4 * i; j < n && j < 4 * i + 4; ++j) acc0 += s[j].x + s[j].y;
    out[(size_t)blockIdx.x * blockDim.x + threadIdx.x] = acc0 + acc1;
}

typedef double v2d __attribute__((ext_vector_type(2)));
__global__ __launch_bounds__(256) void stream_read_nt_kernel(const double2* __restrict__ s2, double* __restrict__ out,
                                                             size_t n) {
    const v2d* s = reinterpret_cast<const v2d*>(s2);
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    double acc0 = 0.0, acc1 = 0.0;
    for (; i + 3 * stride < n; i += 4 * stride) {
        const v2d a = __builtin_nontemporal_load(s + i), b = __builtin_nontemporal_load(s + i + stride);
        const v2d c = __builtin_nontemporal_load(s + i + 2 * stride);
        const v2d e = __builtin_nontemporal_load(s + i + 3 * stride);
        acc0 += (a.x + b.x) + (c.x + e.x);
        acc1 += (a.y + b.y) + (c.y + e.y);
    }
    for (; i < n; i += stride) acc0 += s[i].x + s[i].y;
    out[(size_t)blockIdx.x * blockDim.x + threadIdx.x] = acc0 + acc1;
}

// Device math probes for the parity tests (sqrt, division, pow, pow6).
__global__ void probe_kernel(const double* x, const double* y, double* out, int n, int which) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    switch (which) {
    case 0: out[i] = sqrt(x[i]); break;
    case 1: out[i] = x[i] / y[i]; break;
    case 2: out[i] = ddpow::pow_dd(x[i], y[i]); break;
    case 4: out[i] = pow(x[i], y[i]); break;
    case 3: out[i] = pow6_cr(x[i]); break;
    default: out[i] = 0.0;
    }
}

}  // namespace

hipError_t list_mixed(const Teno& t, uint32_t N, hipStream_t stream) {
    hipLaunchKernelGGL(list_mixed_kernel, dim3(1), dim3(1024), 0, stream,
                       reinterpret_cast<const uint32_t*>(t.blk_mixed), (N + 63) / 64, t.mixed_list);
    return hipGetLastError();
}

hipError_t teno_faces(const Geom& g, const Teno& t, const double* U, double* fs, uint8_t* dec,
                      const Physics& ph, int occ, int gate_reuse, hipStream_t stream) {
    const int Kp = t.K - 1, Mp = t.M - 1;
    const uint32_t FQ = g.S * g.Q;
    if (g.S != 3 || (FQ != 3 && FQ != 6) || Mp < 1) return hipErrorInvalidValue;
    if (occ != 0 && occ != 4 && occ != 5 && occ != 6) return hipErrorInvalidValue;
    const uint32_t nblk = (g.N + 63) / 64, per_xcd = (nblk + 7) / 8;
    const dim3 grid(8 * per_xcd), block(256);
    const bool small = t.loc8 != nullptr;
    if (!small && t.loc16 == nullptr) return hipErrorInvalidValue;
    const size_t net_lds = (t.gate && !gate_reuse) ? ind::kNetInferBytes : 0;
    // small: 8-bit tile positions (tiles of <= 256 cells); O: occupancy target
#define MLR_TENO_S(KP, MP, FQV, G, O)                                                                       \
    hipLaunchKernelGGL((teno_kernel<KP, MP, FQV, uint8_t, 256, G, O>), grid, block, 256 * 32 + net_lds, stream, \
                       g, t, U, fs, dec, ph, per_xcd)
#define MLR_TENO_L(KP, MP, FQV, G)                                                                         \
    hipLaunchKernelGGL((teno_kernel<KP, MP, FQV, uint16_t, 1024, G, 0>), grid, block, 1024 * 32 + net_lds,   \
                       stream, g, t, U, fs, dec, ph, per_xcd)
#define MLR_TENO_G(KP, MP, FQV, G)                  \
    do {                                            \
        if (small) MLR_TENO_S(KP, MP, FQV, G, 0);   \
        else MLR_TENO_L(KP, MP, FQV, G);            \
    } while (0)
    // the gated kernels exist where the central stencil has the network's 12 members or more
#define MLR_TENO(KP, MP, FQV)                              \
    do {                                                   \
        if (!t.gate) MLR_TENO_G(KP, MP, FQV, 0);           \
        else if (gate_reuse) MLR_TENO_G(KP, MP, FQV, 2);   \
        else MLR_TENO_G(KP, MP, FQV, 1);                   \
    } while (0)
    if (t.gate && Mp < ind::kMembers - 1) return hipErrorInvalidValue;
    // the second part of a split gated pass: the marked blocks, listed anew
    // after each evaluation
    auto ungated = [&](bool compact) {
        if (!gate_reuse)
            if (const hipError_t e = list_mixed(t, g.N, stream); e != hipSuccess) return e;
        const dim3 ug(8 * per_xcd < kUngatedBlocks ? 8 * per_xcd : kUngatedBlocks);
        const size_t tile = 256 * 32, slots = 4 * kUngatedDepth * (6 * 512 + 64);
        if (compact)
            hipLaunchKernelGGL((teno_ungated_kernel<true>), ug, block, tile, stream, g, t, U, fs, dec, ph);
        else
            hipLaunchKernelGGL((teno_ungated_kernel<false>), ug, block, tile + slots, stream, g, t, U, fs, dec, ph);
        return hipGetLastError();
    };
    if (t.derived) {
        // derived face basis: plain TENO at p = 2 with the default stencil
        // size and 8-bit tile positions
        if (!(FQ == 3 && Kp == 5 && Mp == 11 && small) || t.cvert == nullptr || t.compact || t.gate)
            return hipErrorInvalidValue;
        const size_t lds = 256 * 32;
        if (occ == 4)
            hipLaunchKernelGGL((teno_kernel<5, 11, 3, uint8_t, 256, 0, 4, false, true>), grid, block, lds, stream, g,
                               t, U, fs, dec, ph, per_xcd);
        else if (occ == 5)
            hipLaunchKernelGGL((teno_kernel<5, 11, 3, uint8_t, 256, 0, 5, false, true>), grid, block, lds, stream, g,
                               t, U, fs, dec, ph, per_xcd);
        else if (occ == 0)
            hipLaunchKernelGGL((teno_kernel<5, 11, 3, uint8_t, 256, 0, 0, false, true>), grid, block, lds, stream, g,
                               t, U, fs, dec, ph, per_xcd);
        else
            return hipErrorInvalidValue;
        return hipGetLastError();
    }
    if (t.compact) {
        // compact tables: p = 2 with the default stencil size, 8-bit tile
        // positions, the compiler's occupancy
        if (!(FQ == 3 && Kp == 5 && Mp == 11 && small) || t.fbc == nullptr) return hipErrorInvalidValue;
        const size_t lds = 256 * 32;
        if (t.gate && t.blk_mixed) {
            // split gated pass: the gated cells (linear operators, no tables),
            // then the ungated cells of the marked blocks on compact tables
            if (gate_reuse) MLR_TENO_S(5, 11, 3, 4, 0);
            else MLR_TENO_S(5, 11, 3, 3, 0);
            if (const hipError_t e = hipGetLastError(); e != hipSuccess) return e;
            return ungated(true);
        } else if (!t.gate) {
            if (occ == 5)
                hipLaunchKernelGGL((teno_kernel<5, 11, 3, uint8_t, 256, 0, 5, true>), grid, block, lds, stream, g, t,
                                   U, fs, dec, ph, per_xcd);
            else if (occ == 6)
                hipLaunchKernelGGL((teno_kernel<5, 11, 3, uint8_t, 256, 0, 6, true>), grid, block, lds, stream, g, t,
                                   U, fs, dec, ph, per_xcd);
            else
                hipLaunchKernelGGL((teno_kernel<5, 11, 3, uint8_t, 256, 0, 0, true>), grid, block, lds, stream, g, t,
                                   U, fs, dec, ph, per_xcd);
        } else if (gate_reuse) {
            hipLaunchKernelGGL((teno_kernel<5, 11, 3, uint8_t, 256, 2, 0, true>), grid, block, lds, stream, g, t, U,
                               fs, dec, ph, per_xcd);
        } else {
            hipLaunchKernelGGL((teno_kernel<5, 11, 3, uint8_t, 256, 1, 0, true>), grid, block, lds + net_lds, stream,
                               g, t, U, fs, dec, ph, per_xcd);
        }
        return hipGetLastError();
    }
    if (FQ == 6 && Kp == 9 && Mp == 19 && !t.gate) {
        // plain p = 3 at the default stencil size: streamed member tables.
        // 36 accumulators a lane leave the plain loop 3 waves per SIMD that
        // wait on memory 82% of the time (or 4 that spill); with two members
        // ahead in LDS (51 KB a block, 3 blocks a CU) the pass runs at 95% of
        // what the tables' bytes allow: 524,288 cells 1,124 -> 695 us, 80,000
        // 205 -> 118. Three members ahead (2 blocks a CU) 720, 4 waves 760.
        // At p = 2, where the plain loop keeps 4 waves busy, streaming gains
        // nothing (1,048,576 cells: 1,141 against 1,127 us) and the smallest
        // meshes lose 3 us.
        constexpr int kDepth = 2;
        const uint32_t tile = t.tile_max * 32;
        const size_t slots = 4 * kDepth * (10 * 512 + 64 * (small ? 1 : 2));
        if (small)
            hipLaunchKernelGGL((teno_stream_kernel<9, 19, 6, uint8_t, kDepth, 3>), grid, block, tile + slots, stream, g,
                               t, U, fs, dec, ph, tile, per_xcd);
        else
            hipLaunchKernelGGL((teno_stream_kernel<9, 19, 6, uint16_t, kDepth, 3>), grid, block, tile + slots, stream,
                               g, t, U, fs, dec, ph, tile, per_xcd);
        return hipGetLastError();
    }
    // the default stencil size (factor 2: M = 2K) is compiled with the member
    // loop unrolled up to p = 2, there in three occupancy targets; other sizes
    // and gated p = 3 take the runtime loop
    if (FQ == 3) {
        switch (Kp) {
        case 2: if (Mp == 5) MLR_TENO_G(2, 5, 3, 0); else MLR_TENO_G(2, 0, 3, 0); break;
        case 5:
            if (Mp == 11 && small && t.gate && t.blk_mixed) {
                // split gated pass: the gated cells (modes 3 / 4, no
                // full-TENO code), then the ungated ones of the marked
                // blocks (mode 5). The evaluate pass targets 6 waves per
                // SIMD (77 VGPRs, no spill; the compiler's own choice, 75
                // VGPRs + 8 AGPRs, gives 5); the others run at the
                // compiler's occupancy (the tune's target does not apply)
                if (gate_reuse) MLR_TENO_S(5, 11, 3, 4, 0);
                else MLR_TENO_S(5, 11, 3, 3, 6);
                if (const hipError_t e = hipGetLastError(); e != hipSuccess) return e;
                return ungated(false);
            } else if (Mp == 11 && small) {
                const int gm = !t.gate ? 0 : (gate_reuse ? 2 : 1);
#define MLR_TENO_O(GMV)                                       \
    do {                                                      \
        if (occ == 5) MLR_TENO_S(5, 11, 3, GMV, 5);           \
        else if (occ == 6) MLR_TENO_S(5, 11, 3, GMV, 6);      \
        else MLR_TENO_S(5, 11, 3, GMV, 0);                    \
    } while (0)
                if (gm == 0) MLR_TENO_O(0);
                else if (gm == 1) MLR_TENO_O(1);
                else MLR_TENO_O(2);
#undef MLR_TENO_O
            } else if (Mp == 11) {
                MLR_TENO(5, 11, 3);
            } else {
                MLR_TENO(5, 0, 3);
            }
            break;
        case 9: MLR_TENO(9, 0, 3); break;
        default: return hipErrorInvalidValue;
        }
    } else {
        switch (Kp) {
        case 2: MLR_TENO_G(2, 0, 6, 0); break;
        case 5: MLR_TENO(5, 0, 6); break;
        // gated p = 3 at the default stencil size too: the loop unrolled took
        // 256 registers, 1 wave per SIMD (320,000 cells 1,258 us, 540 here)
        case 9: MLR_TENO(9, 0, 6); break;
        default: return hipErrorInvalidValue;
        }
    }
#undef MLR_TENO_S
#undef MLR_TENO_L
#undef MLR_TENO_G
#undef MLR_TENO
    return hipGetLastError();
}

namespace {
// Threads of a flux block of bs cells, whose faces number about 1.7 bs on
// triangles and 2.2 bs on quads. While the whole mesh's faces fit the chip at
// once (4 waves per SIMD hold 262,144 threads), a kernel lasts as long as one
// thread's chain, and two threads per cell halve it: HLLC residual of 8,192
// triangles 8.9 us against 14.1 us with one thread per cell, 131,072
// triangles 16.3 against 18.2. On larger meshes the second half of the block
// idles in the cell sums: 2,097,152 triangles 174 us with one thread per
// cell, 190 with two; they cross near 262,144 (30.6 us both). Blocks of 256
// cells, of which a CU holds half as many, cross between 131,072 and 245,000:
// HLLC stage of 8,192 triangles 16.0 -> 13.6 us, 90,000 quads 22.9 -> 19.1,
// Rusanov of 1,000 quads 11.6 -> 10.3; 245,000 triangles 27.2 -> 27.6, with
// Roe 20.1 -> 21.4. An ensemble's blocks have at most 256 threads.
uint32_t flux_threads(uint32_t bs, uint64_t cells) {
    return cells <= (bs < 256 ? 1u << 18 : 1u << 17) ? 2 * bs : bs;
}
int face_size(uint32_t bs) { return bs == 64 ? 0 : (bs == 128 ? 1 : 2); }
}  // namespace

hipError_t flux_update(const Geom& g, const StageArgs& a, const Physics& ph, uint32_t bs, hipStream_t stream,
                       const DtJoin* join) {
    if (bs != 64 && bs != 128 && bs != 256) return hipErrorInvalidValue;
    const uint32_t nblk = (g.N + bs - 1) / bs, per_xcd = (nblk + 7) / 8;
    const dim3 grid(8 * per_xcd), block(flux_threads(bs, g.N));
    const size_t lds = (size_t)g.face_max[face_size(bs)] * 32;
    const bool pp = a.pp && a.op != kRhsOnly;
    if (a.parts != 3 && a.op != kRhsOnly) return hipErrorInvalidValue;
    if (join && (a.op == kRhsOnly || join->n_blk > kJoinBlocks)) return hipErrorInvalidValue;
    const DtJoin jn = join ? *join : DtJoin{};
#define MLR_FK(RSV, PPV, VV)                                                                                       \
    do {                                                                                                           \
        if (join)                                                                                                  \
            hipLaunchKernelGGL((flux_update_kernel<RSV, PPV, VV, true>), grid, block, lds, stream, g, a, ph, bs,   \
                               per_xcd, jn);                                                                       \
        else                                                                                                       \
            hipLaunchKernelGGL((flux_update_kernel<RSV, PPV, VV, false>), grid, block, lds, stream, g, a, ph, bs,  \
                               per_xcd, jn);                                                                       \
    } while (0)
#define MLR_FU(RSV)                               \
    do {                                          \
        if (ph.viscous) MLR_FK(RSV, false, true); \
        else if (pp) MLR_FK(RSV, true, false);    \
        else MLR_FK(RSV, false, false);           \
    } while (0)
    switch (a.riemann) {
    case 0: MLR_FU(0); break;
    case 1: MLR_FU(1); break;
    case 2: MLR_FU(2); break;
    case 3: MLR_FU(3); break;
    default: return hipErrorInvalidValue;
    }
#undef MLR_FU
#undef MLR_FK
    return hipGetLastError();
}

hipError_t spectral_radius(const Geom& g, const double* Un, const double* prims, const Physics& ph,
                           double* lam_cell, unsigned long long* lam_blk, uint32_t bs, hipStream_t stream) {
    if (bs != 64 && bs != 128 && bs != 256) return hipErrorInvalidValue;
    const uint32_t nblk = (g.N + bs - 1) / bs, per_xcd = (nblk + 7) / 8;
    hipLaunchKernelGGL(spectral_kernel, dim3(8 * per_xcd), dim3(bs), 0, stream, g, Un, prims, ph, lam_cell, lam_blk,
                       per_xcd);
    return hipGetLastError();
}

hipError_t finalize_dt(const unsigned long long* lam_blk, uint32_t n_blk, double cfl, double fixed_dt, double* dt,
                       double* dt_hist, int64_t hist_cap, int64_t* step, hipStream_t stream) {
    hipLaunchKernelGGL(finalize_dt_kernel, dim3(1), dim3(1024), 0, stream, lam_blk, n_blk, cfl, fixed_dt, dt, dt_hist,
                       hist_cap, step);
    return hipGetLastError();
}

hipError_t teno_batch(const CaseBufs* cases, const uint32_t* block_case, uint32_t total_blocks, int in_role, int K,
                      int M, int FQ, bool small, bool gated, int occ, int gate_reuse, bool split, bool derived,
                      const Physics& ph, hipStream_t stream) {
    const int Kp = K - 1, Mp = M - 1;
    const size_t net_lds = (gated && !gate_reuse) ? ind::kNetInferBytes : 0;
    if ((FQ != 3 && FQ != 6) || Mp < 1) return hipErrorInvalidValue;
    const uint32_t per_xcd = (total_blocks + 7) / 8;
    const dim3 grid(8 * per_xcd), block(256);
    if (derived) {
        // derived face basis: plain p = 2 with the default stencil size and
        // 8-bit tile positions in every case (each case's Teno::cvert set)
        if (!(FQ == 3 && Kp == 5 && Mp == 11 && small) || gated) return hipErrorInvalidValue;
        if (occ == 4)
            hipLaunchKernelGGL((teno_batch_kernel<5, 11, 3, uint8_t, 256, 0, 4, true>), grid, block, 256 * 32,
                               stream, cases, block_case, in_role, total_blocks, ph, per_xcd);
        else if (occ == 5)
            hipLaunchKernelGGL((teno_batch_kernel<5, 11, 3, uint8_t, 256, 0, 5, true>), grid, block, 256 * 32,
                               stream, cases, block_case, in_role, total_blocks, ph, per_xcd);
        else if (occ == 0)
            hipLaunchKernelGGL((teno_batch_kernel<5, 11, 3, uint8_t, 256, 0, 0, true>), grid, block, 256 * 32,
                               stream, cases, block_case, in_role, total_blocks, ph, per_xcd);
        else
            return hipErrorInvalidValue;
        return hipGetLastError();
    }
    if (occ != 0 && occ != 5 && occ != 6) return hipErrorInvalidValue;
#define MLR_TB_S(KP, MP, FQV, G, O)                                                                             \
    hipLaunchKernelGGL((teno_batch_kernel<KP, MP, FQV, uint8_t, 256, G, O>), grid, block, 256 * 32 + net_lds,   \
                       stream, cases, block_case, in_role, total_blocks, ph, per_xcd)
#define MLR_TB_G(KP, MP, FQV, G)                                                                               \
    do {                                                                                                       \
        if (small)                                                                                             \
            MLR_TB_S(KP, MP, FQV, G, 0);                                                                       \
        else                                                                                                   \
            hipLaunchKernelGGL((teno_batch_kernel<KP, MP, FQV, uint16_t, 1024, G, 0>), grid, block,              \
                               1024 * 32 + net_lds, stream, cases, block_case, in_role, total_blocks, ph, per_xcd); \
    } while (0)
#define MLR_TB(KP, MP, FQV)                              \
    do {                                                 \
        if (!gated) MLR_TB_G(KP, MP, FQV, 0);            \
        else if (gate_reuse) MLR_TB_G(KP, MP, FQV, 2);   \
        else MLR_TB_G(KP, MP, FQV, 1);                   \
    } while (0)
    if (gated && Mp < ind::kMembers - 1) return hipErrorInvalidValue;
    if (FQ == 3 && Kp == 5 && Mp == 11 && small && gated && split) {
        // split gated pass (teno_faces' modes 3 / 4, then 5)
        if (gate_reuse) MLR_TB_S(5, 11, 3, 4, 0);
        else MLR_TB_S(5, 11, 3, 3, 6);  // the evaluate pass at 6 waves per SIMD, as teno_faces
        if (const hipError_t e = hipGetLastError(); e != hipSuccess) return e;
        hipLaunchKernelGGL((teno_batch_kernel<5, 11, 3, uint8_t, 256, 5, 0>), grid, block, 256 * 32, stream, cases,
                           block_case, in_role, total_blocks, ph, per_xcd);
    } else if (FQ == 3 && Kp == 5 && Mp == 11 && small) {
        const int gm = !gated ? 0 : (gate_reuse ? 2 : 1);
#define MLR_TB_O(GMV)                                     \
    do {                                                  \
        if (occ == 5) MLR_TB_S(5, 11, 3, GMV, 5);         \
        else if (occ == 6) MLR_TB_S(5, 11, 3, GMV, 6);    \
        else MLR_TB_S(5, 11, 3, GMV, 0);                  \
    } while (0)
        if (gm == 0) MLR_TB_O(0);
        else if (gm == 1) MLR_TB_O(1);
        else MLR_TB_O(2);
#undef MLR_TB_O
    } else if (FQ == 3 && Kp == 5 && Mp == 11) MLR_TB(5, 11, 3);
    else if (FQ == 3 && Kp == 5) MLR_TB(5, 0, 3);
    else if (FQ == 3 && Kp == 2) MLR_TB_G(2, 0, 3, 0);
    else if (FQ == 6 && Kp == 9) MLR_TB(9, 0, 6);
    else return hipErrorInvalidValue;
#undef MLR_TB_S
#undef MLR_TB_G
#undef MLR_TB
    return hipGetLastError();
}

hipError_t flux_batch(const CaseBufs* cases, const uint32_t* block_case, uint32_t total_blocks, const BatchStage& st,
                      int riemann, const Physics& ph, uint32_t bs, uint32_t face_max, hipStream_t stream) {
    if (bs != 64 && bs != 128 && bs != 256) return hipErrorInvalidValue;
    const uint32_t per_xcd = (total_blocks + 7) / 8;
    const dim3 grid(8 * per_xcd), block(bs < 256 ? flux_threads(bs, (uint64_t)total_blocks * bs) : bs);
    const size_t lds = (size_t)face_max * 32;
#define MLR_FBK(RSV, PPV)                                                                                           \
    do {                                                                                                           \
        if (st.join)                                                                                               \
            hipLaunchKernelGGL((flux_batch_kernel<RSV, PPV, true>), grid, block, lds, stream, cases, block_case,   \
                               st, total_blocks, ph, bs, per_xcd);                                                 \
        else                                                                                                       \
            hipLaunchKernelGGL((flux_batch_kernel<RSV, PPV, false>), grid, block, lds, stream, cases, block_case,  \
                               st, total_blocks, ph, bs, per_xcd);                                                 \
    } while (0)
#define MLR_FB(RSV)                      \
    do {                                 \
        if (st.pp) MLR_FBK(RSV, true);   \
        else MLR_FBK(RSV, false);        \
    } while (0)
    switch (riemann) {
    case 0: MLR_FB(0); break;
    case 1: MLR_FB(1); break;
    case 2: MLR_FB(2); break;
    case 3: MLR_FB(3); break;
    default: return hipErrorInvalidValue;
    }
#undef MLR_FB
#undef MLR_FBK
    return hipGetLastError();
}

hipError_t spectral_batch(const CaseBufs* cases, const uint32_t* block_case, uint32_t total_blocks, const Physics& ph,
                          uint32_t bs, hipStream_t stream) {
    if (bs != 64 && bs != 128 && bs != 256) return hipErrorInvalidValue;
    const uint32_t per_xcd = (total_blocks + 7) / 8;
    hipLaunchKernelGGL(spectral_batch_kernel, dim3(8 * per_xcd), dim3(bs), 0, stream, cases, block_case, total_blocks,
                       ph, per_xcd);
    return hipGetLastError();
}

hipError_t finalize_batch(const CaseBufs* cases, int n_cases, double cfl, double fixed_dt, int64_t hist_cap,
                          uint32_t bs, hipStream_t stream) {
    if (bs != 64 && bs != 128 && bs != 256) return hipErrorInvalidValue;
    hipLaunchKernelGGL(finalize_batch_kernel, dim3(n_cases), dim3(256), 0, stream, cases, n_cases, cfl, fixed_dt,
                       hist_cap, bs);
    return hipGetLastError();
}

namespace {
template <int RS, bool TENO>
hipError_t launch_step_persistent(const CaseBufs* cases, int n_cases, const uint32_t* teno_case,
                                  const uint32_t* flux_case, uint32_t teno_total, uint32_t flux_total,
                                  const PersistentStep& ps, uint32_t face_max, const Physics& ph, hipStream_t stream,
                                  int* grid_out) {
    const void* fn = reinterpret_cast<const void*>(&ensemble_step_kernel<RS, TENO>);
    // a block holds a TENO tile or a flux block's face fluxes
    const size_t flux_lds = (size_t)face_max * 32;
    const size_t lds = TENO && flux_lds < 256 * 32 ? 256 * 32 : flux_lds;
    int per_cu = 0, dev = 0, cus = 0;
    if (hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, fn, 256, lds); e != hipSuccess) return e;
    if (hipError_t e = hipGetDevice(&dev); e != hipSuccess) return e;
    if (hipError_t e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev); e != hipSuccess)
        return e;
    const int grid = per_cu * cus;  // every block resident at once: the grid barrier needs it
    if (grid < 8) return hipErrorInvalidConfiguration;  // each XCD's range needs a block
    if (grid_out) *grid_out = grid;
    const CaseBufs* c = cases;
    int n = n_cases;
    uint32_t tt = teno_total, ft = flux_total;
    PersistentStep p = ps;
    Physics h = ph;
    const uint32_t *tc = teno_case, *fc = flux_case;
    void* args[] = {&c, &n, &tc, &fc, &tt, &ft, &p, &h};
    return hipLaunchCooperativeKernel(fn, dim3(grid), dim3(256), args, (unsigned)lds, stream);
}
}  // namespace

hipError_t ensemble_step(const CaseBufs* cases, int n_cases, const uint32_t* teno_case, const uint32_t* flux_case,
                         uint32_t teno_total, uint32_t flux_total,
                         const PersistentStep& ps, int riemann, bool teno, uint32_t face_max, const Physics& ph,
                         hipStream_t stream, int* grid_out) {
    if (n_cases < 1 || ps.n_stages < 1 || ps.n_stages > 4) return hipErrorInvalidValue;
#define MLR_STEP(RSV)                                                                                          \
    return teno ? launch_step_persistent<RSV, true>(cases, n_cases, teno_case, flux_case, teno_total, flux_total, ps, \
                                                    face_max, ph, stream, grid_out)                                 \
                : launch_step_persistent<RSV, false>(cases, n_cases, teno_case, flux_case, teno_total, flux_total,  \
                                                     ps, face_max, ph, stream, grid_out)
    switch (riemann) {
    case 0: MLR_STEP(0);
    case 1: MLR_STEP(1);
    case 2: MLR_STEP(2);
    case 3: MLR_STEP(3);
    default: return hipErrorInvalidValue;
    }
#undef MLR_STEP
}

hipError_t viscous_grad(const Geom& g, const double* U, const Physics& ph, double* vp, double* vg, uint32_t bs,
                        hipStream_t stream) {
    if (bs != 64 && bs != 128 && bs != 256) return hipErrorInvalidValue;
    const uint32_t nblk = (g.N + bs - 1) / bs, per_xcd = (nblk + 7) / 8;
    hipLaunchKernelGGL(viscous_grad_kernel, dim3(8 * per_xcd), dim3(bs), 0, stream, g, U, ph, vp, vg, per_xcd);
    return hipGetLastError();
}

hipError_t copy_state(const double* src, double* dst, uint32_t N, hipStream_t stream) {
    const size_t n = 4 * (size_t)N;
    hipLaunchKernelGGL(copy_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream, src, dst, n);
    return hipGetLastError();
}

uint32_t stream_probe_threads(size_t bytes) {
    const size_t n = bytes / 16;
    const size_t blocks = (n + 255) / 256;
    return (uint32_t)(blocks < 16384 ? blocks : 16384) * 256u;
}

hipError_t stream_probe(int kind, const void* src, void* dst, size_t bytes, hipStream_t stream) {
    const size_t n = bytes / 16;
    const uint32_t threads = stream_probe_threads(bytes);
    if (threads == 0) return hipErrorInvalidValue;
    const dim3 grid(threads / 256), block(256);
    switch (kind) {
    case 0:
        hipLaunchKernelGGL(stream_copy_kernel, grid, block, 0, stream, static_cast<const double2*>(src),
                           static_cast<double2*>(dst), n);
        break;
    case 1:
        hipLaunchKernelGGL(stream_read_kernel, grid, block, 0, stream, static_cast<const double2*>(src),
                           static_cast<double*>(dst), n);
        break;
    case 2: return hipMemcpyAsync(dst, src, bytes / 16 * 16, hipMemcpyDeviceToDevice, stream);
    case 3:
        hipLaunchKernelGGL(stream_read_wide_kernel, grid, block, 0, stream, static_cast<const double2*>(src),
                           static_cast<double*>(dst), n);
        break;
    case 4:
        hipLaunchKernelGGL(stream_read_nt_kernel, grid, block, 0, stream, static_cast<const double2*>(src),
                           static_cast<double*>(dst), n);
        break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t probe_math(const double* x, const double* y, double* out, int n, int which, hipStream_t stream) {
    hipLaunchKernelGGL(probe_kernel, dim3((n + 255) / 256), dim3(256), 0, stream, x, y, out, n, which);
    return hipGetLastError();
}

}  // namespace mlr::dev
