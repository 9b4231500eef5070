// A whole n-qubit state in the registers of one workgroup of 2^W waves: the
// gates, permutations and inner products of one layer (2 <= n <= 13; 14 for psi
// alone, and for psi and lambda in two halves that differ in the top wire).
//
// Why registers: a layer rotates every wire, so a state kept in LDS is read
// and written once per group of wires (three or four times a layer for psi
// and for lambda).  In registers a layer moves each array through LDS once
// for the ring CNOT and, with more than one wave, once more to bring the
// wires of the wave index into registers; everything else stays in the
// lane.  At 13 qubits psi and lambda take 128 of the 256 VGPRs of 512 threads.
//
// Storage position s = lane + 64 r + 64 A wave (r < A = 2^R: register).  In
// layout 1 wires 0..5 sit on the lane, 6..5+R on r, the W highest on the wave;
// wire 2 pairs lanes l and l ^ 7 (the others l ^ 1, 2, 8, 16, 32), because a
// row of 16 lanes can be exchanged by xor 1, 2, 7 and 8 in one DPP move but
// not by xor 4.  So logical low bits = lane ^ 3 where lane bit 2 is set.
// One layer of the adjoint sweep, from layout 1:
//   register wires: pairs in registers;
//   wires 0..3: the partner by a DPP move (signed on the way);
//   wires 5, 4: v_permlane32/16_swap exchanges the lane bit with a register
//     bit (one instruction per register pair and 32 bits; no LDS), then they
//     are register wires;
//   the W wave wires: exchanged with W register bits through LDS.
// That ends in layout 2, from which the next ring CNOT reads back into
// layout 1.  The forward sweep runs the same steps mirrored, 2 to 1, so a
// layer's RZ phases meet layout 1 in both directions.
//
// RY in tangent form, [[1, -t], [t, 1]] with |t| <= 1, one FMA per output
// component and no branch: where |sin| > |cos| of the half angle,
// RY(theta) = (X Z) RY(theta') with t = -cos / sin, the Z joins the layer's
// phases and the X only flips the label of the wire, a bit of the mask f
// (logical index = storage index ^ f) that the ring CNOT maps like any index.
// A flipped label negates t and the wire's gradients and reads the other entry
// of a phase table.  The factors cos or sin of a layer multiply its phase
// table.  RZ as diag(1, e^{i phi}): the global phase cancels in energies and
// gradients, and between the sweep there and back.
#pragma once

#include <type_traits>

#include "rie_kernels.hpp"

namespace rie {

// Per-layer record (doubles): tangents t[w] (w < 14), [14] the factor of the
// dphi sums, [15] the mask k of flipped wires (as a double), [16 + w] the factor of wire
// w's dtheta sum, then complex tables: [32] phases of wires 0..2 times the
// layer's scale, [48] of wires 3..5, [64] of the register wires (2^R), then
// of the wave wires (2^W).
constexpr int kRecDphi = 14;
constexpr int kRecFlips = 15;
constexpr int kRecG = 16;
constexpr int kRecLa = 32;
constexpr int kRecLb = 48;
constexpr int kRecReg = 64;

// Eight amplitudes a lane at 12 qubits (512 threads): with sixteen (256 threads,
// one wave per SIMD) the adjoint layer spills and hides no latency, 14.0 us a
// layer against 10.6.
__host__ __device__ constexpr int reg_bits(int n) {
    return n <= 6 ? 0 : n == 7 ? 1 : n <= 10 ? 2 : n <= 12 ? 3 : 4;  // 13, 14: 4
}
__host__ __device__ constexpr int wave_bits(int n) { return n <= 8 ? 0 : n - 6 - reg_bits(n); }
__host__ __device__ constexpr int record_doubles(int n) {
    return kRecReg + 2 * (1 << reg_bits(n)) + 2 * (1 << wave_bits(n));
}

__host__ __device__ constexpr uint32_t ring_fwd_c(uint32_t i, int n) {
    uint32_t p = i;
    p ^= p << 1;
    p ^= p << 2;
    p ^= p << 4;
    p ^= p << 8;
    p &= (1u << n) - 1u;
    uint32_t par = i >> 1;
    par ^= par >> 8;
    par ^= par >> 4;
    par ^= par >> 2;
    par ^= par >> 1;
    return (p & ~1u) | (par & 1u);
}
__host__ __device__ constexpr uint32_t ring_inv_c(uint32_t i, int n) {
    return ((i ^ (i << 1)) & ((1u << n) - 1u)) ^ (((i >> (n - 1)) & 1u) ? 3u : 0u);
}

// Order fence for LDS traffic inside one wave: a wave's LDS operations execute
// in program order, so only the compiler has to keep them.
__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_wave_barrier();
    asm volatile("" ::: "memory");
}

__device__ __forceinline__ void swap_regs32(double &a, double &b) {
    const auto lo = __builtin_amdgcn_permlane32_swap((unsigned)__double2loint(a),
                                                     (unsigned)__double2loint(b), false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap((unsigned)__double2hiint(a),
                                                     (unsigned)__double2hiint(b), false, false);
    a = __hiloint2double((int)hi[0], (int)lo[0]);
    b = __hiloint2double((int)hi[1], (int)lo[1]);
}

__device__ __forceinline__ void swap_regs16(double &a, double &b) {
    const auto lo = __builtin_amdgcn_permlane16_swap((unsigned)__double2loint(a),
                                                     (unsigned)__double2loint(b), false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap((unsigned)__double2hiint(a),
                                                     (unsigned)__double2hiint(b), false, false);
    a = __hiloint2double((int)hi[0], (int)lo[0]);
    b = __hiloint2double((int)hi[1], (int)lo[1]);
}

// v of the lane that pairs with this one on lane wire w, its sign flipped
// where neg is the sign bit (0 or 0x80000000).
template <int w>
__device__ __forceinline__ double lane_partner(double v, uint32_t neg) {
    if constexpr (w < 4) {
        constexpr int ctrl = w == 0 ? 0xB1 : w == 1 ? 0x4E : w == 2 ? 0x141 : 0x128;
        const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), ctrl, 0xf, 0xf, true);
        const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), ctrl, 0xf, 0xf, true);
        return __hiloint2double(hi ^ (int)neg, lo);
    } else {
        double a = v;
        double b = v;
        if constexpr (w == 4) {
            swap_regs16(a, b);
        } else {
            swap_regs32(a, b);
        }
        // a holds the wire's 0 half in both halves, b its 1 half
        const double p = ((threadIdx.x >> w) & 1u) ? a : b;
        return __hiloint2double(__double2hiint(p) ^ (int)neg, __double2loint(p));
    }
}

// First step of the sums of two values over a wave: lanes with logical bit 0
// clear keep v0, the others v1, each with its partner's share.
__device__ __forceinline__ double fold_pair(double v0, double v1, uint32_t x) {
    const bool b = (x & 1u) != 0;
    return (b ? v1 : v0) + lane_partner<0>(b ? v0 : v1, 0u);
}

// The other steps, for NP = 2, 4 or 8 folded pairs at once: transpose and add
// over the other row wires, then the four rows.  The lane whose low logical
// bits are j (mod 2 NP) returns value j's total, v[m] holding pair (2m, 2m+1).
template <int NP>
__device__ __forceinline__ double wave_sums(double (&v)[NP], uint32_t x) {
    int have = NP;
    auto step = [&](auto wc) {
        constexpr int w = decltype(wc)::value;
        if (have > 1) {
            const bool b = ((x >> w) & 1u) != 0;
#pragma unroll
            for (int m = 0; m < NP / 2; ++m) {
                if (2 * m + 1 < have) {
                    const double keep = b ? v[2 * m + 1] : v[2 * m];
                    const double send = b ? v[2 * m] : v[2 * m + 1];
                    v[m] = keep + lane_partner<w>(send, 0u);
                }
            }
            have >>= 1;
        } else {
            v[0] += lane_partner<w>(v[0], 0u);
        }
    };
    step(std::integral_constant<int, 1>{});
    step(std::integral_constant<int, 2>{});
    step(std::integral_constant<int, 3>{});
    double a = v[0];
    double b = v[0];
    swap_regs16(a, b);
    a += b;
    b = a;
    swap_regs32(a, b);
    return a + b;
}

// Keeps the compiler from moving work across: without it the scheduler pulls
// the partners and table entries of many amplitudes ahead and spills at 12 and
// 13 qubits, where psi and lambda already take half the registers.
__device__ __forceinline__ void hold_schedule() { __builtin_amdgcn_sched_barrier(0); }

// Order in which the adjoint sweep un-rotates the wires: the register wires,
// 0..3, 5, 4, then the wave wires.
__host__ __device__ constexpr int adjoint_order(int w, int R) {
    return w >= 6 + R ? w : w >= 6 ? w - 6 : w < 4 ? R + w : w == 5 ? R + 4 : R + 5;
}

// O = 1: one half (top wire n fixed, `outer`) of an (n + 1)-qubit state.
template <int n, int O = 0>
struct RegState {
    static constexpr int R = reg_bits(n);
    static constexpr int W = wave_bits(n);
    static constexpr int A = 1 << R;
    static constexpr int kWaves = 1 << W;
    static constexpr int kThreads = 64 << W;
    static constexpr int kLaneWires = n < 6 ? n : 6;
    static constexpr int kRec = record_doubles(n + O);
    static constexpr uint32_t kAmps = 1u << n;
    // LDS amplitudes of one exchange buffer (lanes beyond 2^n use theirs too)
    static constexpr uint32_t kBuf = kAmps < 64u ? 64u : kAmps;
    // 256 KB at 14 qubits: the exchanges move re and im in turn
    static constexpr bool kPlanes = n > kRegMaxQubits;
    static constexpr size_t kExchangeBytes = (kPlanes ? 8 : 16) * (size_t)kBuf;
    static_assert(n >= 2 && n <= 14 && W <= R, "register layouts");
    static_assert(O == 0 || (n == 13 && reg_bits(14) == R && wave_bits(14) == W + 1),
                  "halves of 14 qubits");

    // storage bit of wire w in layout 1 (w itself) and in layout 2
    static constexpr int pos2(int w) {
        int pos[16] = {};
        for (int k = 0; k < n; ++k) {
            pos[k] = k;
        }
        auto swap_bits = [&](int a, int b) {
            for (int k = 0; k < n; ++k) {
                pos[k] = pos[k] == a ? b : pos[k] == b ? a : pos[k];
            }
        };
        if (R == 1) {
            swap_bits(5, 6);
            swap_bits(4, 6);
        } else if (R >= 2) {
            swap_bits(5, 6);
            swap_bits(4, 7);
        }
        for (int k = 0; k < W; ++k) {
            swap_bits(6 + k, 6 + R + k);
        }
        return pos[w];
    }
    // layout 1 and its inverse: the lane frame of wire 2
    static constexpr __host__ __device__ uint32_t frame(uint32_t s) {
        return s ^ (((s >> 2) & 1u) * 3u);
    }
    // logical index of a layout-2 storage position, and back
    static constexpr __host__ __device__ uint32_t logical2(uint32_t s) {
        const uint32_t x = frame(s);
        uint32_t i = 0;
        for (int w = 0; w < n; ++w) {
            i |= ((x >> pos2(w)) & 1u) << w;
        }
        return i;
    }
    static constexpr __host__ __device__ uint32_t storage2(uint32_t i) {
        uint32_t s = 0;
        for (int w = 0; w < n; ++w) {
            s |= ((i >> w) & 1u) << pos2(w);
        }
        return frame(s);
    }

    // Exchanges through LDS: every amplitude is written at its storage
    // position and read from a linear image of the reader's.
    //   kind 0: forward ring CNOT, layout 1 -> 2    kind 1: the same, 1 -> 1
    //   kind 2: inverse ring CNOT, layout 2 -> 1    kind 3: the same, 1 -> 1
    static constexpr __host__ __device__ uint32_t image(int kind, uint32_t s) {
        return kind == 0   ? frame(ring_inv_c(logical2(s), n))
               : kind == 1 ? frame(ring_inv_c(frame(s), n))
               : kind == 2 ? storage2(ring_fwd_c(frame(s), n))
                           : frame(ring_fwd_c(frame(s), n));
    }

    uint32_t lane;   // 0..63
    uint32_t wave;   // 0..2^W-1
    uint32_t x;      // logical low bits of the lane (layout 1)
    uint32_t own;    // storage position of r = 0
    uint32_t from[4];
    bool active;     // lane holds an amplitude (n < 6: lanes below 2^n)
    uint32_t outer = 0;  // the half (O = 1)

    __device__ __forceinline__ void setup(uint32_t lane_, uint32_t wave_) {
        lane = lane_;
        wave = wave_;
        x = frame(lane);
        own = lane + ((uint32_t)(64 * A) * wave);
        active = n >= 6 || lane < kAmps;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            from[k] = active ? image(k, own) : lane;
        }
    }

    // sign bit where this lane's wire w (layout 1, w < 6) is 1
    __device__ __forceinline__ uint32_t sign_of(int w) const { return (x << (31 - w)) & 0x80000000u; }

    static __device__ __forceinline__ void sync() {
        if constexpr (W == 0) {
            wave_lds_fence();
        } else {
            __syncthreads();
        }
    }

    __device__ __forceinline__ void put(double2 *buf, const double2 (&a)[A]) const {
#pragma unroll
        for (int r = 0; r < A; ++r) {
            buf[own + 64u * r] = a[r];
        }
    }

    // kinds 0..3 (see image), 4: wave bits <-> the W low register bits
    template <int kind, typename T, typename F>
    __device__ __forceinline__ void read(const T *buf, F &&store) const {
        if constexpr (kind < 4) {
            uint32_t base = from[kind];
            // formed here each time: A addresses held across the layers would
            // spill at 12 and 13 qubits
            asm volatile("" : "+v"(base));
#pragma unroll
            for (int r = 0; r < A; ++r) {
                store(r, buf[base ^ image(kind, 64u * r)]);
            }
        } else {
            constexpr uint32_t m = (1u << W) - 1u;
#pragma unroll
            for (uint32_t r = 0; r < (uint32_t)A; ++r) {
                store((int)r, buf[lane + 64u * ((r & ~m) | wave) + 64u * A * (r & m)]);
            }
        }
    }

    template <int kind>
    __device__ __forceinline__ void get(const double2 *buf, double2 (&a)[A]) const {
        read<kind>(buf, [&](int r, double2 v) { a[r] = v; });
    }

    // One array through LDS, after a barrier for earlier reads of buf.
    template <int kind>
    __device__ __forceinline__ void exchange(double2 *buf, double2 (&a)[A]) const {
        if constexpr (kPlanes) {
            double *plane = reinterpret_cast<double *>(buf);
            sync();
#pragma unroll
            for (int r = 0; r < A; ++r) {
                plane[own + 64u * r] = a[r].x;
            }
            sync();
            read<kind>(plane, [&](int r, double v) { a[r].x = v; });
            sync();
#pragma unroll
            for (int r = 0; r < A; ++r) {
                plane[own + 64u * r] = a[r].y;
            }
            sync();
            read<kind>(plane, [&](int r, double v) { a[r].y = v; });
        } else {
            sync();
            put(buf, a);
            sync();
            get<kind>(buf, a);
        }
    }

    // Two arrays, through one buffer in turn (kSplit) or two at once.
    template <int kind, bool kSplit>
    __device__ __forceinline__ void exchange2(double2 *buf, double2 (&a)[A],
                                              double2 (&b)[A]) const {
        if constexpr (kSplit) {
            exchange<kind>(buf, a);
            exchange<kind>(buf, b);
        } else {
            sync();
            put(buf, a);
            put(buf + kBuf, b);
            sync();
            get<kind>(buf, a);
            get<kind>(buf + kBuf, b);
        }
    }

    // ---- RY on one wire of one array, tangent form without its factor ----

    template <bool kInv>
    static __device__ __forceinline__ void rot_reg(double2 (&a)[A], int bit, double t) {
        const double u = kInv ? t : -t;
#pragma unroll
        for (int r = 0; r < A; ++r) {
            if (((r >> bit) & 1) == 0) {
                double2 &a0 = a[r];
                double2 &a1 = a[r | (1 << bit)];
                const double x0 = fma(u, a1.x, a0.x);
                const double y0 = fma(u, a1.y, a0.y);
                a1.x = fma(-u, a0.x, a1.x);
                a1.y = fma(-u, a0.y, a1.y);
                a0.x = x0;
                a0.y = y0;
            }
        }
    }

    // the other amplitude of wire w, negated on the side that RY subtracts it
    template <bool kInv, int w>
    __device__ __forceinline__ double2 signed_partner(double2 v) const {
        const uint32_t neg = kInv ? sign_of(w) : sign_of(w) ^ 0x80000000u;
        return make_double2(lane_partner<w>(v.x, neg), lane_partner<w>(v.y, neg));
    }

    static __device__ __forceinline__ double2 rot_with(double2 v, double2 p, double t) {
        return make_double2(fma(t, p.x, v.x), fma(t, p.y, v.y));
    }

    template <bool kInv, int w>
    __device__ __forceinline__ void rot_lane(double2 (&a)[A], double t) const {
#pragma unroll
        for (int r = 0; r < A; ++r) {
            a[r] = rot_with(a[r], signed_partner<kInv, w>(a[r]), t);
        }
    }

    // lane bit 5 or 4 <-> register bit
    template <int lane_bit>
    static __device__ __forceinline__ void swap_lane(double2 (&a)[A], int bit) {
#pragma unroll
        for (int r = 0; r < A; ++r) {
            if (((r >> bit) & 1) == 0) {
                double2 &a0 = a[r];
                double2 &a1 = a[r | (1 << bit)];
                if constexpr (lane_bit == 5) {
                    swap_regs32(a0.x, a1.x);
                    swap_regs32(a0.y, a1.y);
                } else {
                    swap_regs16(a0.x, a1.x);
                    swap_regs16(a0.y, a1.y);
                }
            }
        }
    }

    // ---- records ----

    // One layer's record in LDS with the label mask f its gates meet.
    struct Rec {
        const double *p;
        uint32_t f;
        // wire w's tangent for storage order
        __device__ __forceinline__ double t(int w) const {
            const double v = p[w];
            const uint32_t neg = (f << (31 - w)) & 0x80000000u;
            return __hiloint2double(__double2hiint(v) ^ (int)neg, __double2loint(v));
        }
        __device__ __forceinline__ double2 c(int at) const {
            return *reinterpret_cast<const double2 *>(p + at);
        }
        __device__ __forceinline__ double2 reg_phase(int r) const {
            return c(kRecReg + 2 * (r ^ (int)((f >> 6) & (uint32_t)(A - 1))));
        }
    };

    // the wires whose labels a layer flips
    static __device__ __forceinline__ uint32_t flips(const double *p) {
        return (uint32_t)__builtin_amdgcn_readfirstlane((int)p[kRecFlips]);
    }

    // phase of this lane's wires (and the wave's), times the layer's scale
    __device__ __forceinline__ double2 lane_phase(const Rec &k) const {
        double2 z = k.c(kRecLa + 2 * (int)((x ^ k.f) & 7u));
        if constexpr (n > 3) {
            z = cmul(z, k.c(kRecLb + 2 * (int)(((x ^ k.f) >> 3) & 7u)));
        }
        if constexpr (W + O > 0) {
            constexpr uint32_t m = (1u << (W + O)) - 1u;
            const uint32_t v = wave | (outer << W);
            z = cmul(z, k.c(kRecReg + 2 * A + 2 * (int)(v ^ ((k.f >> (6 + R)) & m))));
        }
        return z;
    }

    // ---- forward: layer 0 on |0...0>, and one further layer ----

    // real product of (1, t) per wire, times the layer's phases (f = 0)
    __device__ __forceinline__ void product_state(const Rec &k, double2 (&a)[A]) const {
        double lanes = active ? 1.0 : 0.0;
        const uint32_t hi = x | (wave << (6 + R));
#pragma unroll
        for (int w = 0; w < n; ++w) {
            if (w < 6 || w >= 6 + R) {
                lanes *= ((hi >> w) & 1u) != 0 ? k.t(w) : 1.0;
            }
        }
        const double2 z = lane_phase(k);
#pragma unroll
        for (int r = 0; r < A; ++r) {
            double v = lanes;
#pragma unroll
            for (int j = 0; j < R; ++j) {
                if (((r >> j) & 1) != 0) {
                    v *= k.t(6 + j);
                }
            }
            const double2 q = R == 0 ? z : cmul(z, k.reg_phase(r));
            a[r] = make_double2(v * q.x, v * q.y);
        }
    }

    // from layout 2 to layout 1, the layer's gates and phases applied
    __device__ __forceinline__ void forward_layer(const Rec &k, double2 (&a)[A],
                                                  double2 *buf) const {
        if constexpr (W > 0) {
#pragma unroll
            for (int j = 0; j < W; ++j) {
                rot_reg<false>(a, j, k.t(6 + R + j));
            }
            exchange<4>(buf, a);
        }
        if constexpr (R == 1) {
            rot_reg<false>(a, 0, k.t(4));
            swap_lane<4>(a, 0);
            rot_reg<false>(a, 0, k.t(5));
            swap_lane<5>(a, 0);
        } else if constexpr (R >= 2) {
            rot_reg<false>(a, 1, k.t(4));
            rot_reg<false>(a, 0, k.t(5));
            swap_lane<4>(a, 1);
            swap_lane<5>(a, 0);
        } else {
            if constexpr (n > 4) {
                rot_lane<false, 4>(a, k.t(4));
            }
            if constexpr (n > 5) {
                rot_lane<false, 5>(a, k.t(5));
            }
        }
        rot_lane<false, 0>(a, k.t(0));
        rot_lane<false, 1>(a, k.t(1));
        if constexpr (n > 2) {
            rot_lane<false, 2>(a, k.t(2));
        }
        if constexpr (n > 3) {
            rot_lane<false, 3>(a, k.t(3));
        }
#pragma unroll
        for (int j = 0; j < R; ++j) {
            rot_reg<false>(a, j, k.t(6 + j));
        }
        const double2 z = lane_phase(k);
#pragma unroll
        for (int r = 0; r < A; ++r) {
            a[r] = cmul(a[r], R == 0 ? z : cmul(z, k.reg_phase(r)));
        }
    }

    // ---- adjoint: one layer on (c, l) from layout 1 to layout 2 ----

    // The place of wire w in that order (the records' dtheta factors use it).
    static constexpr __host__ __device__ int record_order(int w) { return adjoint_order(w, R); }

    // kRotate: leave both arrays un-rotated (false: layer 0's gradients only).
    // Per-wave sums go to red: [w] the dtheta sums, [16 + w] the dphi sums of
    // the lane wires, [22] of the whole wave, [24 + j] of register wire j.
    // kSplit: psi and lambda pass through one buffer in turn.
    template <bool kRotate, bool kSplit>
    __device__ __forceinline__ void adjoint_layer(const Rec &k, double2 (&c)[A], double2 (&l)[A],
                                                  double2 *buf, double *red) const {
        constexpr int NP = n <= 4 ? 2 : n <= 8 ? 4 : 8;
        double dt[NP];    // folded pairs of dtheta sums
        double first[NP]; // the half of a pair that came first
#pragma unroll
        for (int j = 0; j < NP; ++j) {
            dt[j] = 0.0;
            first[j] = 0.0;
        }
        auto emit = [&](int w, double v) {
            const int o = w ^ 1;
            if (o < n && record_order(w) < record_order(o)) {
                first[w >> 1] = v;
            } else {
                const double u = o < n ? first[w >> 1] : 0.0;
                dt[w >> 1] = (w & 1) ? fold_pair(u, v, x) : fold_pair(v, u, x);
            }
        };
        {
            const double2 z = lane_phase(k);
#pragma unroll
            for (int r = 0; r < A; ++r) {
                const double2 q = R == 0 ? z : cmul(z, k.reg_phase(r));
                const double2 zc = make_double2(q.x, -q.y);
                c[r] = cmul(c[r], zc);
                l[r] = cmul(l[r], zc);
                if (A >= 8 && (r & 3) == 3) {
                    hold_schedule();
                }
            }
        }
        // dphi of every wire from Im(l* c): phase-free and unchanged by the
        // rotations of other wires
        {
            double q[A];
#pragma unroll
            for (int r = 0; r < A; ++r) {
                q[r] = l[r].x * c[r].y - l[r].y * c[r].x;
            }
            double dp[4] = {0.0, 0.0, 0.0, 0.0};  // register wires
#pragma unroll
            for (int j = R - 1; j >= 0; --j) {
                // signed sum over register bit j of what is left
#pragma unroll
                for (int r = 0; r < (1 << j); ++r) {
                    dp[j] += q[r] - q[r | (1 << j)];
                    q[r] += q[r | (1 << j)];
                }
            }
            if constexpr (R > 0) {
                double pairs[2] = {fold_pair(dp[0], dp[1], x), fold_pair(dp[2], dp[3], x)};
                const double v = wave_sums<2>(pairs, x);
                if (lane < 4) {
                    red[24 + (int)(x & 3u)] = v;
                }
            }
            // Walsh transform over the lane wires: the lane with one logical
            // bit w holds wire w's signed sum, lane 0 the plain one
            double v = q[0];
            auto step = [&](auto wc) {
                constexpr int w = decltype(wc)::value;
                if constexpr (w < kLaneWires) {
                    const double s = __hiloint2double(
                        __double2hiint(v) ^ (int)sign_of(w), __double2loint(v));
                    v = lane_partner<w>(v, 0u) + s;
                }
            };
            step(std::integral_constant<int, 0>{});
            step(std::integral_constant<int, 1>{});
            step(std::integral_constant<int, 2>{});
            step(std::integral_constant<int, 3>{});
            step(std::integral_constant<int, 4>{});
            step(std::integral_constant<int, 5>{});
            if (x < kAmps && (x & (x - 1u)) == 0) {  // x = 0 or a power of two
                red[16 + (x == 0 ? 6 : __builtin_ctz(x))] = v;
            }
        }
        // Ends a wire: nothing of the next one may start before it.  Without
        // rotations no data dependence orders the wires, so psi passes
        // through an empty statement there.
        auto next_wire = [&]() {
            if constexpr (A >= 8) {
                hold_schedule();
                if constexpr (!kRotate) {
#pragma unroll
                    for (int r = 0; r < A; ++r) {
                        asm volatile("" : "+v"(c[r].x), "+v"(c[r].y));
                    }
                }
            }
        };
        auto reg_wire = [&](int bit, int w) {
            double s0 = 0.0;
            double s1 = 0.0;
#pragma unroll
            for (int r = 0; r < A; ++r) {
                if (((r >> bit) & 1) == 0) {
                    const int o = r | (1 << bit);
                    s0 += l[r].x * c[o].x + l[r].y * c[o].y;
                    s1 += l[o].x * c[r].x + l[o].y * c[r].y;
                }
            }
            if constexpr (kRotate) {
                rot_reg<true>(c, bit, k.t(w));
                rot_reg<true>(l, bit, k.t(w));
            }
            emit(w, s0 - s1);
            next_wire();
        };
        auto lane_wire = [&](auto wc) {
            constexpr int w = decltype(wc)::value;
            double s = 0.0;
            const double t = k.t(w);
#pragma unroll
            for (int r = 0; r < A; ++r) {
                const double2 p = signed_partner<true, w>(c[r]);
                s += l[r].x * p.x + l[r].y * p.y;
                if constexpr (kRotate) {
                    c[r] = rot_with(c[r], p, t);
                    l[r] = rot_with(l[r], signed_partner<true, w>(l[r]), t);
                }
                if (A >= 8 && (r & 3) == 3) {
                    hold_schedule();
                }
            }
            emit(w, s);
            next_wire();
        };
#pragma unroll
        for (int j = 0; j < R; ++j) {
            reg_wire(j, 6 + j);
        }
        lane_wire(std::integral_constant<int, 0>{});
        lane_wire(std::integral_constant<int, 1>{});
        if constexpr (n > 2) {
            lane_wire(std::integral_constant<int, 2>{});
        }
        if constexpr (n > 3) {
            lane_wire(std::integral_constant<int, 3>{});
        }
        if constexpr (R == 1) {
            swap_lane<5>(c, 0);
            swap_lane<5>(l, 0);
            reg_wire(0, 5);
            swap_lane<4>(c, 0);
            swap_lane<4>(l, 0);
            reg_wire(0, 4);
        } else if constexpr (R >= 2) {
            swap_lane<5>(c, 0);
            swap_lane<5>(l, 0);
            swap_lane<4>(c, 1);
            swap_lane<4>(l, 1);
            reg_wire(0, 5);
            reg_wire(1, 4);
        } else {
            if constexpr (n > 5) {
                lane_wire(std::integral_constant<int, 5>{});
            }
            if constexpr (n > 4) {
                lane_wire(std::integral_constant<int, 4>{});
            }
        }
        if constexpr (W > 0) {
            exchange2<4, kSplit>(buf, c, l);
#pragma unroll
            for (int j = 0; j < W; ++j) {
                reg_wire(j, 6 + R + j);
            }
        }
        const double v = wave_sums<NP>(dt, x);
        if (lane < (uint32_t)(2 * NP)) {
            red[x & (uint32_t)(2 * NP - 1)] = v;
        }
    }

    // Gradient entry i = 2 w + {0: dtheta, 1: dphi} of a layer from the
    // per-wave sums (red: 32 doubles per wave).  f: the layer's label mask, k:
    // the flips its RY leaves.  all_scaled: no wire was un-rotated, so every
    // sum carries the whole layer's scale.
    static __device__ __forceinline__ double gradient_entry(int i, const double *rec,
                                                            const double *red, uint32_t f,
                                                            uint32_t k, bool all_scaled) {
        // one address and sign rule per lane, so that the waves' sums are all
        // read at once (a branch per wave cost 1 to 2 us a layer at 13 qubits)
        const int w = i >> 1;
        const bool phi = (i & 1) != 0;
        const bool wave_wire = phi && w >= 6 + R;
        const int at = !phi ? w : w < 6 ? 16 + w : wave_wire ? 22 : 24 + (w - 6);
        const int bit = wave_wire ? w - 6 - R : 31;
        double acc = 0.0;
#pragma unroll
        for (int v = 0; v < kWaves; ++v) {
            const double q = red[32 * v + at];
            acc += (((uint32_t)v >> bit) & 1u) ? -q : q;
        }
        acc *= rec[phi || all_scaled ? kRecDphi : kRecG + w];
        const uint32_t flip = phi ? (f ^ k) >> w : ~(f >> w);
        return (flip & 1u) ? -acc : acc;
    }

    // ---- lambda = H psi in layout 1; returns this lane's share of <psi|H|psi> ----

    __device__ __forceinline__ double hamiltonian(double field, uint32_t f_mask,
                                                  const double2 (&c)[A], double2 (&l)[A],
                                                  double2 *buf) const {
        sync();
        put(buf, c);
        sync();
        return hamiltonian_of(field, f_mask, c, l, buf, nullptr);
    }

    // The same from a copy of psi in storage order (and, O = 1, of the other
    // half's).
    __device__ __forceinline__ double hamiltonian_of(double field, uint32_t f_mask,
                                                     const double2 (&c)[A], double2 (&l)[A],
                                                     const double2 *buf,
                                                     const double2 *other) const {
        double e = 0.0;
#pragma unroll
        for (int r = 0; r < A; ++r) {
            double2 f = make_double2(0.0, 0.0);
            auto add = [&](double2 v) {
                f.x += v.x;
                f.y += v.y;
            };
            auto lane_add = [&](auto wc) {
                constexpr int w = decltype(wc)::value;
                if constexpr (w < kLaneWires) {
                    add(make_double2(lane_partner<w>(c[r].x, 0u), lane_partner<w>(c[r].y, 0u)));
                }
            };
            lane_add(std::integral_constant<int, 0>{});
            lane_add(std::integral_constant<int, 1>{});
            lane_add(std::integral_constant<int, 2>{});
            lane_add(std::integral_constant<int, 3>{});
            if constexpr (kLaneWires > 4) {
                add(buf[(own ^ 16u) + 64u * r]);
            }
            if constexpr (kLaneWires > 5) {
                add(buf[(own ^ 32u) + 64u * r]);
            }
#pragma unroll
            for (int j = 0; j < R; ++j) {
                add(c[r ^ (1 << j)]);
            }
#pragma unroll
            for (int j = 0; j < W; ++j) {
                add(buf[(own ^ ((uint32_t)(64 * A) << j)) + 64u * r]);
            }
            if constexpr (O > 0) {
                add(other[own + 64u * r]);
            }
            const uint32_t i =
                (x | ((uint32_t)r << 6) | (wave << (6 + R)) | (outer << n)) ^ f_mask;
            const double d = ham_diag((uint64_t)i, n + O);
            l[r] = make_double2(d * c[r].x - field * f.x, d * c[r].y - field * f.y);
            if (!active) {
                l[r] = make_double2(0.0, 0.0);
            }
            e += c[r].x * l[r].x + c[r].y * l[r].y;
        }
        return e;
    }
};

// A value that every lane holds, in scalar registers.  The job's fields come
// through a pointer that the compiler cannot tell apart from per-lane data;
// left there, the layer loop runs under an execution mask and keeps its
// counters and label masks in vector registers.
template <typename T>
__device__ __forceinline__ T uniform(T v) {
    static_assert(sizeof(T) % 4 == 0, "whole words");
    uint32_t w[sizeof(T) / 4];
    __builtin_memcpy(w, &v, sizeof(T));
#pragma unroll
    for (int i = 0; i < (int)(sizeof(T) / 4); ++i) {
        w[i] = (uint32_t)__builtin_amdgcn_readfirstlane((int)w[i]);
    }
    __builtin_memcpy(&v, w, sizeof(T));
    return v;
}

// Records of the sweep's layers 0 .. L-1 and back L-1 .. 0, three in LDS: the
// one in use, the next, and one whose readers may lag a barrier behind.  Two
// more are in flight in registers, so a record read from another XCD's L2 or
// from HBM has two layers' time to arrive.
template <int kRec>
struct RecordRing {
    double (*slots)[kRec];
    const double *base;
    int layers;
    int steps;
    bool loads;    // this wave moves the records
    int at;        // this lane's two doubles (the last lanes repeat the end)
    int next = 0;  // step of the next load
    int slot = 0;
    double2 p1 = {0.0, 0.0};
    double2 p2 = {0.0, 0.0};

    __device__ __forceinline__ double2 load() {
        const int q = next < steps ? next : steps - 1;
        const int l = q < layers ? q : 2 * layers - 1 - q;
        ++next;
        return *reinterpret_cast<const double2 *>(base + (size_t)l * kRec + at);
    }
    __device__ __forceinline__ void store(int s, double2 v) {
        *reinterpret_cast<double2 *>(&slots[s][at]) = v;
    }
    __device__ __forceinline__ void start() {
        if (loads) {
            store(0, load());
            p1 = load();
            p2 = load();
        }
    }
    // the current step's record; stages the next one (visible to other waves
    // after the step's barriers)
    __device__ __forceinline__ const double *advance() {
        const double *cur = slots[slot];
        slot = slot == 2 ? 0 : slot + 1;
        if (loads) {
            store(slot, p1);
            p1 = p2;
            p2 = load();
        }
        return cur;
    }
};

}  // namespace rie
