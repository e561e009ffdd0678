// Channels-last scan of contiguous tiles staged through LDS: dense tensors of few or odd channel counts.
//
// The kernels of scan_cl_kernels.hpp give every lane a fixed run of channels of one time step, so what a wave
// moves per instruction is that step's bytes: few channels leave lanes idle or need the recurrence to run
// across lanes, and steps that are no whole 16-byte vectors are loaded and stored element-aligned. Here memory
// and arithmetic each get the mapping that suits them. A workgroup owns all channels of one batch element and
// walks time in tiles of `rows` steps, each a contiguous run of memory:
//   load    the run comes in as aligned 16-byte vectors, consecutive lanes on consecutive vectors, into
//           registers, and goes to LDS as it is. The next tile's loads are issued as soon as this tile is in
//           LDS, so they are in flight while this tile is computed.
//   fold    a thread owns one channel and `seg` consecutive steps and folds them to one affine pair,
//           reading LDS at the time stride; consecutive threads are consecutive channels, then
//           consecutive spans of time.
//   carry   the pairs of a channel's spans are exchanged through LDS; the carry from tile to tile stays in
//           registers.
//   replay  every thread runs its steps again from its carry and writes the results over the tile's inputs.
//   store   the results leave as aligned 16-byte vectors, the mapping of the load; a run's first and last
//           vector, where they hold foreign bytes, are stored element by element.
// The aligned vector that holds a run's first or last element may also hold bytes that are not the run's: at most
// 15, of the same 16-byte block, never used. The host sends only tensors whose base is a 16-byte border, so no
// block begins before the tensor and corresponding runs of all tensors have one phase against the border.
//
// In a kernel trace 53 to 65 % of 8 TB/s (bf16 [2048, 512, 40] 48.5 / 83.8 us forwards / backwards, fp32 [1000, 1023, 17] 44.0 /
// 82.2 us), at 1.01 to 1.03 times the bytes it has to move. Bound by a tile's chain of four barriers and two LDS passes
// against the workgroups in flight: the waves wait half of their cycles and another quarter to third for an instruction to
// issue; bank conflicts are 23 to 29 % of the LDS cycles. Registers allow 6 workgroups per CU forwards and 4 backwards in
// fp32, 4 and 4 in 16-bit storage (3 backwards in parts), 8 and 5 in fp64 (7 and 4). Two vectors per thread (8 KiB tiles),
// because with four the registers halve the workgroups per CU (bf16 [851, 467, 27] 16.6 / 27.7 us against 24.5 / 37.9), and
// one 16-bit channel per thread, not two, because that halves the spans each thread folds its carry over ([1024, 2048, 16]
// 39.0 / 65.4 us against 41.9 / 68.3). Pieces of a time step (wider C, strided views) staged the same way were slower
// than the walk throughout (fp32 [64, 2048, 1001] 359 / 659 us at best against 359 / 610) and are not built.
//
// The arithmetic is that of scan_kernels.hpp (src/scanscam_cpu.hpp:17-27, 64-77 of the reference): fp32 (fp64
// for double), every output one chain of FMAs from the carry into the thread's steps.
#pragma once

#include "scan_cl_kernels.hpp"

namespace scanscam {

struct StagedArgs {
    const void *a;  // gates                       [B, T, C]
    const void *x;  // forward: b      backward: gh
    const void *h;  // forward: unused backward: saved forward output
    void *y0;       // forward: h      backward: gb
    void *y1;       // forward: unused backward: ga
    int32_t T;
    int32_t C;
    int32_t rows;   // time steps per tile
    int32_t seg;    // time steps per thread and tile
    int32_t spans;  // spans of `seg` steps in a tile, at most kStagedThreads / C
    int32_t parts;  // parts of a batch element's tiles, one workgroup each (1: the whole)
    int32_t tiles;  // tiles per part
    uint64_t *ws;   // workspace, or null where a call in one part has none: two words, the second of them the flag of
                    // an expired wait (kTimeoutWord), then, parts > 1, the parts' affine pairs, [B, parts, C]
};
constexpr int kStagedHeader = 2;  // words of the workspace before the pairs

// What a launch does: all of a batch element in one workgroup; or, with time in parts over workgroups, first every
// part's affine pairs (kReduce), then the scan of every part from the composition of the pairs before it (kApply).
enum StagedPass { kWhole, kReduce, kApply };

constexpr int kStagedThreads = 256;
constexpr int kStagedVectors = 2;  // 16-byte vectors per thread, tile and tensor
// Time steps per thread and tile, at most: 256 threads fill a tile of 2 vectors each with 32 / E steps; one less
// leaves room for the run's phase and makes the stride from span to span odd, so that the lanes of a wave that sit in
// different spans meet in different LDS banks.
constexpr int staged_steps(int esize) { return 16 * kStagedVectors / esize - 1; }

// A product of a part's gates spans any number of steps, so it is kept as m * 2^e. In fp32 alone 1.02 to the 8000th is
// infinite, and infinity times a carry of zero NaN where the recurrence itself stays finite (the other kernels compose
// at most about a thousand steps before they go on from a value). Scaling by a power of two rounds nothing, so where fp32
// holds the product, results have the bits they would have with it. It costs 1 to 5 % of a call in parts, 6 to 14 % with
// two or three channels, whose tiles have the most spans (forward / backward, us: fp32 [14, 13990, 24] 21.2 / 29.7 ->
// 21.5 / 29.9, [1, 250000, 8] 19.1 / 24.8 -> 20.2 / 25.7, [1, 1000000, 2] 36.0 / 47.6 -> 40.9 / 51.0).
__device__ __forceinline__ float frexp_m(float v) { return __builtin_amdgcn_frexp_mantf(v); }
__device__ __forceinline__ double frexp_m(double v) { return __builtin_amdgcn_frexp_mant(v); }
__device__ __forceinline__ int frexp_e(float v) { return __builtin_amdgcn_frexp_expf(v); }
__device__ __forceinline__ int frexp_e(double v) { return __builtin_amdgcn_frexp_exp(v); }
__device__ __forceinline__ float scale2(float v, int e) { return __builtin_ldexpf(v, e); }
__device__ __forceinline__ double scale2(double v, int e) { return __builtin_ldexp(v, e); }

template <typename CT>
struct GateProduct {
    static constexpr int FAR = 1 << 22;  // nothing but zero survives 2^FAR, and no sum of a few hundred leaves 32 bits
    CT m;  // |m| <= 1 (or not finite) while gates are multiplied onto it: no product of it and a gate overflows
    int e;
    __device__ __forceinline__ void times(CT g)
    {
        const CT v = m * g;
        m = frexp_m(v);
        e += frexp_e(v);
    }
    __device__ __forceinline__ void bound() { e = e < -FAR ? -FAR : (e > FAR ? FAR : e); }
    __device__ __forceinline__ void normalise()  // 1 <= |m| < 2, or zero times 2^0
    {
        e += frexp_e(m) - 1;
        m = CT(2) * frexp_m(m);
        bound();
        if (m == CT(0)) e = 0;
    }
};

// What a part does to the value entering it: B + m * 2^e * value, m normalised (so that the scaled value overflows only
// where the product does, and is subnormal only where the product is below twice the smallest normal number).
template <typename CT>
struct PartPair {
    CT m, B;
    int e;
    __device__ __forceinline__ CT after(CT value) const { return fma_(m, scale2(value, e), B); }
};

template <typename ST, bool REV, int PASS>
__global__ __launch_bounds__(kStagedThreads) void scan_cl_staged_kernel(const StagedArgs p)
{
    using CT = typename ComputeOf<ST>::type;
    using V = Vec<ST, 16 / (int)sizeof(ST)>;
    using raw_t = typename V::raw_t;
    using W = Vec<ST, 1>;
    using word_t = typename W::raw_t;  // one element as it is stored
    constexpr int NT = kStagedThreads, U = kStagedVectors, E = (int)sizeof(ST), VEC = 16 / E, SEG = staged_steps(E);
    constexpr int NS = REV && PASS != kReduce ? 3 : 2;  // tensors in: a, x, h
    struct Pair { CT A, B; };
    using Part = PartPair<CT>;
    __shared__ raw_t stage[NS][NT * U];
    __shared__ Pair ex[NT];
    __shared__ int ex_e[PASS == kApply ? NT : 1];

    const int tid = threadIdx.x;
    const int C = p.C, Q = p.spans;
    const int q = tid / C, c = tid - q * C;  // this thread's span and channel
    const bool active = q < Q;
    const int64_t batch = PASS == kWhole ? blockIdx.x : blockIdx.x / p.parts;
    const int part = PASS == kWhole ? 0 : (int)(blockIdx.x % p.parts);
    // No workgroup waits for another here, so the flag says so, whatever the workspace held before.
    if (PASS != kApply && p.ws && blockIdx.x == 0 && tid == 0) p.ws[kTimeoutWord] = 0;
    if (PASS == kReduce && part == (REV ? 0 : p.parts - 1)) return;  // no part comes after it in scan order
    const int64_t start = batch * p.T * p.C * E;  // first byte of the batch element
    const int step = p.C * E;             // bytes from time step to time step
    const int all_tiles = (p.T + p.rows - 1) / p.rows;
    const int tile0 = PASS == kWhole ? 0 : part * p.tiles;  // tiles [tile0, tile1) are this workgroup's
    const int tile1 = PASS == kWhole || all_tiles - tile0 < p.tiles ? all_tiles : tile0 + p.tiles;

    auto widen = [](word_t w) { CT f[1]; W::unpack(w, f); return f[0]; };
    auto narrow = [](CT v) { const CT f[1] = {v}; return W::pack(f); };
    const word_t zero = narrow(CT(0)), one = narrow(CT(1));

    raw_t reg[NS][U];
    word_t edge_h;  // backwards: h just before the tile (0 before the start), for the threads of its first steps
    auto load = [&](int tile) {
        const int t0 = tile * p.rows, n = p.T - t0 < p.rows ? p.T - t0 : p.rows;
        const int64_t at = start + (int64_t)t0 * step;
        const int low = (int)(at & 15), end = low + n * step;
#pragma unroll
        for (int s = 0; s < NS; s++) {
            const char *base = static_cast<const char *>(s == 0 ? p.a : (s == 1 ? p.x : p.h)) + (at - low);
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int off = (tid + u * NT) * 16;
                reg[s][u] = V::load(reinterpret_cast<const ST *>(base + (off < end ? off : 0)));
            }
        }
        if (NS == 3) {
            edge_h = zero;
            if (q == 0 && t0 > 0)
                edge_h = reinterpret_cast<const word_t *>(static_cast<const char *>(p.h) + (at - step))[c];
        }
    };

    CT carry = CT(0);
    GateProduct<CT> product = {CT(1), 0};  // kReduce: of all gates
    word_t a_next = zero;  // backwards: a of the step just after the tile (0 past the end)
    if (REV && PASS != kWhole && active && tile1 < all_tiles)
        a_next = reinterpret_cast<const word_t *>(static_cast<const char *>(p.a) + start + (int64_t)tile1 * p.rows * step)[c];
    load(REV ? tile1 - 1 : tile0);
    if (PASS == kApply) {
        // The carry into this part: the pairs of the parts before it in scan order, in as many runs as there are threads
        // for each channel.
        const int before = REV ? p.parts - 1 - part : part;
        const int runs = NT / C, run = (before + runs - 1) / runs;
        const Part *pairs = reinterpret_cast<const Part *>(p.ws + kStagedHeader) + batch * p.parts * C + c;
        GateProduct<CT> gates = {CT(1), 0};
        CT value = CT(0);
        if (q < runs) {
            const int last = (q + 1) * run < before ? (q + 1) * run : before;
            for (int i = q * run; i < last; i += 4) {
                Part e[4];
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    const int n = i + k < last ? i + k : last - 1;
                    e[k] = pairs[(int64_t)(REV ? p.parts - 1 - n : n) * C];
                }
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    if (i + k < last) {
                        value = e[k].after(value);
                        gates.m *= e[k].m;
                        gates.e += e[k].e;
                    }
                }
                gates.normalise();
            }
        }
        ex[tid] = Pair{gates.m, value};
        ex_e[tid] = gates.e;
        __syncthreads();
        for (int i = 0; i < runs; i++) {
            const Pair e = ex[i * C + c];
            carry = Part{e.A, e.B, ex_e[i * C + c]}.after(carry);
        }
        // (ex is written again after the barriers of the first tile.)
    }
    auto to_lds = [&]() {
#pragma unroll
        for (int s = 0; s < NS; s++)
#pragma unroll
            for (int u = 0; u < U; u++) stage[s][tid + u * NT] = reg[s][u];
    };

    to_lds();
    __syncthreads();
    const int ntiles = tile1 - tile0;
    for (int it = 0; it < ntiles; it++) {
        const int tile = REV ? tile1 - 1 - it : tile0 + it;
        const int t0 = tile * p.rows, n = p.T - t0 < p.rows ? p.T - t0 : p.rows;
        const word_t edge0 = NS == 3 ? edge_h : zero;
        if (it + 1 < ntiles) load(REV ? tile - 1 : tile + 1);

        // Byte of this thread's channels at step r of the tile, the same in every slot.
        const int64_t first = start + (int64_t)t0 * step;
        const int low = (int)(first & 15);
        char *lds = reinterpret_cast<char *>(stage) + low + c * E;
        constexpr int SLOT = NT * U * 16;
        auto at = [&](int s, int r) -> word_t * { return reinterpret_cast<word_t *>(lds + s * SLOT + r * step); };

        const int r0 = q * p.seg < n ? q * p.seg : n;
        const int r1 = !active ? r0 : (r0 + p.seg < n ? r0 + p.seg : n);
        const int cnt = r1 - r0;
        // The thread's steps in scan order, packed as they are stored: gate (backwards a of the step after) and
        // value, the identity past `cnt`, and backwards h of the step before. All reads are under way before the
        // first is used, and are kept for the replay.
        word_t wa[SEG], wx[SEG], wh[NS == 3 ? SEG : 1];
        if (cnt == SEG) {
#pragma unroll
            for (int i = 0; i < SEG; i++) {
                const int r = REV ? r1 - 1 - i : r0 + i;
                if (!REV) wa[i] = *at(0, r);
                else if (i > 0) wa[i] = *at(0, r + 1);
                wx[i] = *at(1, r);
                if (NS == 3 && i + 1 < SEG) wh[i] = *at(2, r - 1);
            }
        } else {
#pragma unroll
            for (int i = 0; i < SEG; i++) {
                wa[i] = one;
                wx[i] = zero;
                if (NS == 3) wh[i] = zero;
                if (i < cnt) {
                    const int r = REV ? r1 - 1 - i : r0 + i;
                    if (!REV) wa[i] = *at(0, r);
                    else if (i > 0) wa[i] = *at(0, r + 1);
                    wx[i] = *at(1, r);
                    if (NS == 3 && i + 1 < cnt) wh[i] = *at(2, r - 1);
                }
            }
        }
        if (REV && active) {
            // The neighbours' steps: a just after the last step, h just before the first one, and for the next tile
            // a of this tile's first step.
            if (cnt > 0) {
                wa[0] = r1 < n ? *at(0, r1) : a_next;
                const word_t before = NS == 3 && r0 > 0 ? *at(2, r0 - 1) : edge0;
                if (NS < 3) {
                } else if (cnt == SEG) {
                    wh[SEG - 1] = before;
                } else {
#pragma unroll
                    for (int i = 0; i < SEG; i++)
                        if (i == cnt - 1) wh[i] = before;
                }
            }
            a_next = *at(0, 0);
        }
        CT A = CT(1), B = CT(0);
#pragma unroll
        for (int i = 0; i < SEG; i++) {
            const CT g = widen(wa[i]);
            B = fma_(g, B, widen(wx[i]));
            A = A * g;
        }

        CT mine = carry;
        if (Q > 1) {
            ex[tid] = Pair{A, B};
            __syncthreads();
            if (PASS != kReduce || q == 0) {  // (kReduce: only the threads that write the part's pair)
                for (int i = 0; i < Q; i++) {
                    const int qq = REV ? Q - 1 - i : i;
                    const Pair e = ex[qq * C + c];
                    if (qq == q) mine = carry;
                    carry = fma_(e.A, carry, e.B);
                    if (PASS == kReduce) product.times(e.A);
                }
            }
        } else {
            carry = fma_(A, carry, B);
            if (PASS == kReduce) product.times(A);
        }
        if (PASS == kReduce) {
            product.bound();
            __syncthreads();
            if (it + 1 < ntiles) to_lds();
            __syncthreads();
            continue;
        }

        // Backwards the results of a step go over gh and h of that step; the neighbours' border steps were read before
        // the barrier above (Q == 1: there is no neighbour).
#pragma unroll
        for (int i = 0; i < SEG; i++) {
            mine = fma_(widen(wa[i]), mine, widen(wx[i]));
            if (cnt == SEG || i < cnt) {
                const int r = REV ? r1 - 1 - i : r0 + i;
                *at(1, r) = narrow(mine);
                if (NS == 3) *at(2, r) = narrow(mine * widen(wh[i]));
            }
        }
        __syncthreads();

        // The results leave LDS before the next tile enters it, and leave for memory after that: the wait for the next
        // tile's loads then finds no younger stores in front of it.
        raw_t res[REV ? 2 : 1][U];
#pragma unroll
        for (int s = 0; s < (REV ? 2 : 1); s++)
#pragma unroll
            for (int u = 0; u < U; u++) res[s][u] = stage[1 + s][tid + u * NT];
        __syncthreads();
        if (it + 1 < ntiles) to_lds();
        const int end = low + n * step;
#pragma unroll
        for (int s = 0; s < (REV ? 2 : 1); s++) {
            char *base = static_cast<char *>(s == 0 ? p.y0 : p.y1) + (first - low);
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int off = (tid + u * NT) * 16;
                ST *dst = reinterpret_cast<ST *>(base + off);
                if (off >= low && off + 16 <= end) {
                    V::store(dst, res[s][u]);
                } else if (off < end) {
                    const Elems<ST, VEC> e = __builtin_bit_cast(Elems<ST, VEC>, res[s][u]);
#pragma unroll
                    for (int k = 0; k < VEC; k++)
                        if (off + k * E >= low && off + k * E < end) dst[k] = e.e[k];
                }
            }
        }
        __syncthreads();
    }
    if (PASS == kReduce && q == 0) {
        product.normalise();
        reinterpret_cast<Part *>(p.ws + kStagedHeader)[(batch * p.parts + part) * C + c] = Part{product.m, carry, product.e};
    }
}

}  // namespace scanscam
