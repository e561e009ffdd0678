// Channels-last time steps that are no whole vectors (C no multiple of the lane's VEC channels), moved in whole ones.
//
// A lane owns the same VEC channels at every time step, so where C is no multiple of VEC its elements start at another
// component of memory's aligned vectors from step to step. ClSteps (RAGGED) loads and stores them where they are, at
// any element: every such access straddles vectors, a wave's accesses straddle one more line than they have, and the
// stores that leave are parts of lines. Here every load and all stores but those of a step's first and last lane are
// aligned vectors, and the elements move between neighbouring lanes in registers: a step that starts `phase` elements
// into an aligned vector is loaded from that vector's border, and each lane takes its last elements from the lane
// above (a DPP move by one lane and at most one funnel shift per register); on the way out each lane puts the last
// elements of the lane below in front of its own.
//
// The phase of step t is (first + t * C) mod VEC. Scan positions are counted from a virtual origin k0 < VEC steps before
// the tensor's, chosen so that the phase there is 0; a wave's span of S steps (S a multiple of VEC) then has the same
// phases whichever span it is, known at compile time from M = C mod VEC: no shift amount is ever a register. The
// virtual steps are the identity, like those past the end.
//
// fp32 [64, 2048, 1001], 4 waves of 8 steps, forward / backward: 346 / 573 us at any element, 299 / 505 us here (bf16 197 / 344 ->
// 158 / 263 us; GPU time, buffers in rotation), where the bytes take 275 / 435 us at C = 1024. Reads are those of the algorithm
// to 0.1 % and writes 3 % more (FETCH_SIZE, WRITE_SIZE); a wave issues 1.3 / 1.5 times the vector instructions. What is left is
// the wave's accesses, still nine lines for the bytes of eight (C = 992, on whole lines, takes 289 / 493 us as well). Loads go
// through the caches' normal policy, because the line that two channel groups share is in the L2 when the second one asks for it
// (in one run with 304 / 509 us: 313 / 528 with non-temporal ones); stores of whole vectors are non-temporal in fp32 (there 341
// / 565 with cached loads and stores) and fp64 and cached in 16 bits (bf16 in one run 164 / 286 -> 155 / 270 us). Loading a tile
// ahead is level in fp32 (there 298 / 519).
//
// The vector after a group's last one is needed too, so a wave owns at most 63 vectors of channels per step. Vectors that
// hold foreign elements are only ever read, and only those with an element of the tensor in them (the host sends dense
// tensors whose bases lie on vector borders).
#pragma once

#include <utility>

#include "scan_kernels.hpp"

namespace scanscam {

// Element moves across two neighbouring vectors: the vector that starts SHIFT elements into (first, second).
template <typename ST, int VEC, int SHIFT>
__device__ __forceinline__ typename Vec<ST, VEC>::raw_t cl_funnel(typename Vec<ST, VEC>::raw_t first, typename Vec<ST, VEC>::raw_t second)
{
    constexpr int D = (int)sizeof(ST) * VEC / 4;
    struct Words { uint32_t w[D]; };
    const Words f = __builtin_bit_cast(Words, first), s = __builtin_bit_cast(Words, second);
    constexpr int q = SHIFT * (int)sizeof(ST) / 4, r = SHIFT * (int)sizeof(ST) % 4 * 8;
    auto word = [&](int i) { return i < D ? f.w[i < D ? i : 0] : s.w[i - D < D ? i - D : 0]; };
    Words out;
#pragma unroll
    for (int i = 0; i < D; i++) {
        if constexpr (r == 0) out.w[i] = word(i + q);
        else out.w[i] = __builtin_amdgcn_alignbit(word(i + q + 1), word(i + q), r);
    }
    return __builtin_bit_cast(typename Vec<ST, VEC>::raw_t, out);
}

// The same vector of the next / previous lane (lanes without one keep their own: nobody uses it). Only the words that
// are used are moved.
template <int CTRL, typename raw_t> __device__ __forceinline__ raw_t cl_neighbour(raw_t v)
{
    constexpr int D = (int)sizeof(raw_t) / 4;
    struct Words { uint32_t w[D]; };
    Words x = __builtin_bit_cast(Words, v);
#pragma unroll
    for (int i = 0; i < D; i++) x.w[i] = (uint32_t)__builtin_amdgcn_update_dpp((int)x.w[i], (int)x.w[i], CTRL, 0xf, 0xf, false);
    return __builtin_bit_cast(raw_t, x);
}

// ClSteps with the same phases (issue, fold, apply) on aligned vectors.
template <typename ST, int VEC, int S, bool REV, int M, typename CT, bool SPLIT>
struct ClShiftSteps {
    static_assert(M > 0 && M < VEC && S % VEC == 0 && VEC * sizeof(ST) >= 8, "");
    using V = Vec<ST, VEC>;
    using raw_t = typename V::raw_t;
    static constexpr bool BUF = cl_buffered<ST, VEC, S, REV, SPLIT>();
    using BV = ClAccess<ST, VEC, BUF>;
    using Base = typename BV::Base;
    static constexpr int E = (int)sizeof(ST);

    CT g[S][VEC], v[S][VEC];
    raw_t rh[REV ? S : 1];
    raw_t ra[S], rx[S];  // what issue() brought; dead once fold() has run
    raw_t n_rh[REV ? S : 1];
    int first, n_first;  // scan position of the first step (negative: virtual steps)
    int tb, n_tb;        // time step the bases point at

    // Phase of step s (memory's step, off by `d` steps in time), an element count below VEC.
    static constexpr int phase(int s, int d = 0)
    {
        const int k = REV ? (s - d) * (VEC - M) : (s + d) * M;
        return ((k % VEC) + VEC) % VEC;
    }
    // A tensor's base for a span whose first step is t lies `lead` elements before that step: on the vector border before it
    // for buffer instructions; for global ones, whose base may be any address, a constant number that keeps every offset
    // from being negative (one scalar addition fewer per access: bf16 [64, 2048, 1001] backward in one run 280 -> 265 us).
    static __device__ __forceinline__ int phase_at(const ClLane<ST> &ln, int t) { return (ln.phase0 + t % VEC * M) % VEC; }
    static __device__ __forceinline__ int lead_at(const ClLane<ST> &ln, int t)
    {
        if constexpr (BUF) return phase_at(ln, t);
        else return VEC - 1;
    }
    template <typename P> static __device__ __forceinline__ P base(P p, const ClLane<ST> &ln, int t)
    {
        return p + ((int64_t)t * ln.pa - lead_at(ln, t));
    }

    // The lane's vector of a step that starts `ph` elements after a vector border; the lane after the group's last loads one
    // more where the group's elements reach into it.
    static __device__ __forceinline__ unsigned lane_off(const ClLane<ST> &ln, int ph)
    {
        return ph == 0 ? ln.c : (ph <= VEC - M ? ln.c_few : ln.c_all);
    }

    __device__ __forceinline__ void issue(const ClLane<ST> &ln, int T, int first_step)
    {
        n_first = first_step - ln.k0;
        const int lowest = REV ? T - 1 - (n_first + S - 1) - 1 : n_first;
        // At most T - 2: a step that does not exist reads step tb from its border on, which ends at most two vectors past it.
        n_tb = lowest < 0 ? 0 : (lowest > T - 2 ? T - 2 : lowest);
        const int tb_ = n_tb, pitch = ln.pa;
        const Base res_a = BV::base(base(ln.a, ln, tb_)), res_x = BV::base(base(ln.x, ln, tb_)), res_h = BV::base(base(ln.h, ln, tb_));
        const int lead = lead_at(ln, tb_);
        const unsigned none = (unsigned)((lead - phase_at(ln, tb_)) * E);
        auto off = [&](int t, int ph) { return (unsigned)((t - tb_) * pitch + (lead - ph)) * (unsigned)E; };
#pragma unroll
        for (int s = 0; s < S; s++) {
            const int tau = n_first + s;
            const int t = REV ? T - 1 - tau : tau;
            const bool in = (unsigned)t < (unsigned)T;
            const bool a_in = in && (!REV || t + 1 < T), h_in = in && t > 0;
            const int pa = phase(s, REV ? 1 : 0), px = phase(s), ph = phase(s, -1);
            ra[s] = BV::template load<0>(res_a, lane_off(ln, pa), a_in ? off(REV ? t + 1 : t, pa) : none);
            rx[s] = BV::template load<0>(res_x, lane_off(ln, px), in ? off(t, px) : none);
            if (REV) n_rh[s] = BV::template load<0>(res_h, lane_off(ln, ph), h_in ? off(t - 1, ph) : none);
        }
    }
    static constexpr bool CACHED_STORES = sizeof(ST) == 2;

    // This lane's elements of a step that was loaded from the border `PH` elements before it.
    template <int PH> static __device__ __forceinline__ raw_t own(raw_t r)
    {
        if constexpr (PH == 0) return r;
        else return cl_funnel<ST, VEC, PH>(r, cl_neighbour<0x130>(r));
    }
    template <int I> struct Const { static constexpr int value = I; };
    template <typename F, int... I> static __device__ __forceinline__ void each(F &&f, std::integer_sequence<int, I...>) { (f(Const<I>{}), ...); }
    template <typename F> static __device__ __forceinline__ void each_step(F &&f) { each(f, std::make_integer_sequence<int, S>{}); }

    __device__ __forceinline__ void fold(int T, CT (&A)[VEC], CT (&B)[VEC], int = 0)
    {
        first = n_first;
        tb = n_tb;
        if (REV) {
#pragma unroll
            for (int s = 0; s < S; s++) rh[s] = n_rh[s];
        }
#pragma unroll
        for (int k = 0; k < VEC; k++) {
            A[k] = CT(1);
            B[k] = CT(0);
        }
        each_step([&](auto c) {
            constexpr int s = decltype(c)::value;
            const int tau = first + s;
            const int t = REV ? T - 1 - tau : tau;
            const bool in = (unsigned)t < (unsigned)T, a_in = in && (!REV || t + 1 < T);
            CT fa[VEC], fx[VEC];
            V::unpack(own<phase(s, REV ? 1 : 0)>(ra[s]), fa);
            V::unpack(own<phase(s)>(rx[s]), fx);
#pragma unroll
            for (int k = 0; k < VEC; k++) {
                g[s][k] = in ? (a_in ? fa[k] : CT(0)) : CT(1);
                v[s][k] = in ? fx[k] : CT(0);
                B[k] = fma_(g[s][k], B[k], v[s][k]);
                A[k] = A[k] * g[s][k];
            }
        });
    }

    __device__ __forceinline__ void load_fold(const ClLane<ST> &ln, int T, int first_step, CT (&A)[VEC], CT (&B)[VEC])
    {
        issue(ln, T, first_step);
        fold(T, A, B);
    }

    // A step's elements to memory, PH elements after a vector border: whole vectors from the lanes whose vector is theirs
    // and the lane below's, the first and the last VEC elements of the step as they are.
    template <int PH> static __device__ __forceinline__ void put(raw_t r, Base res, ST *p, const ClLane<ST> &ln, unsigned off)
    {
        typedef raw_t raw_elem_aligned_t __attribute__((aligned(sizeof(ST))));
        char *at = reinterpret_cast<char *>(p) + off;  // the border
        const raw_t below = PH == 0 && !ln.tail ? r : cl_neighbour<0x138>(r);
        raw_t whole = r;
        if constexpr (PH != 0) whole = cl_funnel<ST, VEC, VEC - PH>(below, r);
        // Whole vectors: up to the group's last, of which a tail group (M elements in the last lane) holds only so many.
        const int whole_end = ln.tail && PH < VEC - M ? ln.last : ln.last + 1;
        if (ln.lane >= (PH == 0 ? 0 : 1) && ln.lane < whole_end) {
            if constexpr (CACHED_STORES && !BUF) BV::store_cached_elem_aligned(whole, res, ln.c, off);  // (no resource: see lead_at)
            else if constexpr (CACHED_STORES) BV::store_cached(whole, res, ln.c, off);
            else BV::store(whole, res, ln.c, off);
        }
        if (PH != 0 || ln.tail) {
            raw_t end = r;
            int back = 0;
            if (ln.tail && ln.lane == ln.last) {
                end = cl_funnel<ST, VEC, M>(below, r);
                back = VEC - M;
            }
            if ((PH != 0 && ln.lane == 0) || ln.lane == ln.last)
                *reinterpret_cast<raw_elem_aligned_t *>(at + (ln.c + (unsigned)(PH * E)) - back * E) = end;
        }
    }

    __device__ __forceinline__ void apply(const ClLane<ST> &ln, int T, CT (&mine)[VEC])
    {
        const int pitch = ln.pa;
        const int lead = lead_at(ln, tb);
        ST *const y0 = base(ln.y0, ln, tb), *const y1 = base(ln.y1, ln, tb);
        const Base res_y0 = BV::base(y0), res_y1 = BV::base(y1);
        each_step([&](auto c) {
            constexpr int s = decltype(c)::value;
            const int tau = first + s;
            const int t = REV ? T - 1 - tau : tau;
            const bool in = (unsigned)t < (unsigned)T, h_in = in && t > 0;
            const unsigned off = (unsigned)((t - tb) * pitch + (lead - phase(s))) * (unsigned)E;
            CT out[VEC];
#pragma unroll
            for (int k = 0; k < VEC; k++) {
                mine[k] = fma_(g[s][k], mine[k], v[s][k]);
                out[k] = mine[k];
            }
            if constexpr (!REV) {
                if (in) put<phase(s)>(V::pack(out), res_y0, y0, ln, off);
            } else {
                CT fh[VEC], ga[VEC];
                V::unpack(own<phase(s, -1)>(rh[s]), fh);
#pragma unroll
                for (int k = 0; k < VEC; k++) ga[k] = out[k] * (h_in ? fh[k] : CT(0));
                if (in) {
                    put<phase(s)>(V::pack(out), res_y0, y0, ln, off);
                    put<phase(s)>(V::pack(ga), res_y1, y1, ln, off);
                }
            }
        });
    }
};

}  // namespace scanscam
