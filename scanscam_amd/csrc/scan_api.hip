// C ABI of libscanscam_hip.so (declared in include/scanscam_hip.h): argument
// checks, the choice of kernel family and launch shape, and the launches.
#include "scanscam_hip.h"

#include "scan_launch.hpp"
#include "scan_cl_plan.hpp"

#include <mutex>

// Look-back scratch of scanscam_scan_fwd_noalloc: a fixed array in every GPU's memory that the library
// runs on, held until the process ends. Host code never uses this name as an address -- it is a
// host-side stand-in for the symbol; noalloc_scratch() asks the runtime where the current device keeps
// its copy and hands that pointer to the kernels.
static __device__ __align__(256) unsigned char scratch[SCANSCAM_NOALLOC_SCRATCH_BYTES];

namespace {

using scanscam::kCounterStride;
using scanscam::kMaxCounters;
using scanscam::kSuper;
using scanscam::kModeFlat;
using scanscam::kModeLookback;
using scanscam::kModeRow;
using scanscam::kModeSmall;
using scanscam::kModeStaged;
using scanscam::kWave;
using scanscam::Launch;
using scanscam::ScanArgs;

// Prepares the look-back workspace (a kernel, not a memset, so that a caller may capture the launch
// sequence in a HIP graph): the ticket counters and the time-out flag (the first `zero_words` words) are
// zeroed, every descriptor word after them is set to all ones, the kernels' "not yet".
__global__ __launch_bounds__(256) void scan_ws_clear_kernel(uint64_t *ws, int64_t words, int64_t zero_words)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < words) ws[i] = i < zero_words ? 0ull : ~0ull;
}

hipError_t clear_workspace(uint64_t *ws, int64_t words, int64_t zero_words, hipStream_t stream)
{
    void *params[] = {&ws, &words, &zero_words};
    return hipLaunchKernel(reinterpret_cast<const void *>(scan_ws_clear_kernel), dim3((unsigned)((words + 255) / 256)),
                           dim3(256), params, 0, stream);
}

constexpr int64_t kLastLevelCache = int64_t(256) << 20;  // bytes

constexpr int64_t kMaxT = (int64_t(1) << 31) - (int64_t(1) << 20);

int elem_size(int dtype)
{
    switch (dtype) {
    case SCANSCAM_F32: return 4;
    case SCANSCAM_BF16:
    case SCANSCAM_F16: return 2;
    case SCANSCAM_F64: return 8;
    default: return 0;
    }
}

// 64-bit words per value published in the look-back workspace (one per 32-bit half), and per tile (its
// aggregate pair) and super-tile (its pair and its end value) of the row layout's look-back kernel, whose
// fp32 pairs are one word (scanscam::kTileWords, kSuperWords).
int value_words(int dtype) { return dtype == SCANSCAM_F64 ? 2 : 1; }
int tile_words(int dtype) { return dtype == SCANSCAM_F64 ? scanscam::kTileWords<double> : scanscam::kTileWords<float>; }
int super_words(int dtype) { return dtype == SCANSCAM_F64 ? scanscam::kSuperWords<double> : scanscam::kSuperWords<float>; }

// Bytes of the arithmetic type behind a storage type.
int compute_size(int dtype) { return dtype == SCANSCAM_F64 ? 8 : 4; }


int pow2_ceil(int64_t v)
{
    int p = 1;
    while (p < v) p <<= 1;
    return p;
}

bool unroll_ok(int vec, int full, int unroll)
{
    if (vec == full) return unroll == 1 || unroll == 2 || unroll == 3 || unroll == 4 || unroll == 8;
    return unroll == 1 || unroll == 4;
}

struct Resolved {
    Launch l;
    int nch;
    int tiles_per_row;
    int counters;
    int row_major;       // a counter's tickets walk its rows one after the other (see resolve)
    int line_shift;      // chunks laid out from the 128-byte line border before each row's start (see resolve)
    int64_t super_base;  // word offset of the super-tile descriptors
    size_t ws_bytes;
};

// Look-back tiles in chunks (8 waves x 4 chunks per wave) and the ticket order of the look-back kernel.
// Tile-major: a counter's tickets visit tile 0 of each of its rows, then tile 1 of each, ...; few tiles of a
// row are in flight together, so carries arrive with little waiting, at the price of as many separate spans of
// memory being streamed at once as there are rows. Row-major: a counter's tickets finish one row before the
// next, so the tiles in flight sweep memory in address order, which the memory system serves 5-8 points
// faster (measured with scan-free streaming kernels in both orders), while all tiles of a row are in flight together and wait for each other:
// worth it when a row is only a few tiles long.
constexpr int kTileChunks = 32;
constexpr int kRowMajorCounters = 4;

bool row_major_order(int64_t rows, int tiles_per_row) { return rows >= 256 && tiles_per_row <= 16; }

// Many rows of moderate length: from two tiles per row on, the look-back kernel in row-major order beats one
// workgroup walking each row, which streams as many separate spans as there are rows in flight, leaves CUs
// idle in its last round of workgroups, and whose 16-wave steps seldom divide a row. Measured at 16 M to 128 M
// elements, fp32 and bf16, with tiles fitted to the row (resolve): 2 to 15 tiles per row gain +2 to +20 % forward
// and +9 to +30 % backward, also where the row kernel's workgroups come out in full rounds of 256; rows of 8
// tiles (4 exact steps of the row kernel) tie forward. At 16 tiles the forward pass of the row kernel (8 exact
// steps) is 5-8 % faster and keeps the shape unless its rounds do not come out; the backward pass still gains
// 4-6 %. A problem of fewer than 2048 tiles is too small to hide the extra launch that clears the workspace.
// Rows of more than 16 tiles go to the look-back kernel (in tile-major order) only where the row kernel's
// rounds do not come out.
constexpr int kComputeUnits = 256;  // MI355X

bool prefer_lookback_for_many_rows(int64_t rows, int nch, bool rev, int esize)
{
    const int tpr = (nch + kTileChunks - 1) / kTileChunks;
    if (rows < 256 || tpr < 2 || rows * tpr < 2048) return false;
    // Two tiles of up to 24 chunks, 4- and 8-byte elements, forward: one workgroup of up to 12 waves per row is
    // faster (fp32, 34-48 chunks: 72 against 63 % of peak at 16 M elements, 78-80 against 76 % at 64 M; from 52
    // chunks on, and backward, the look-back kernel; 16-bit storage: the look-back kernel, 70 against 60-64 %).
    if (!rev && esize >= 4 && tpr == 2 && nch <= 48) return false;
    const int64_t rounds = (rows + kComputeUnits - 1) / kComputeUnits;
    const bool ragged_rounds = rows * 100 < rounds * kComputeUnits * 93;  // the row kernel's CUs idle > 7 % of the time
    if (rev && tpr <= 16) return true;
    if (tpr <= 15) return true;
    return ragged_rounds;
}

// Turns (shape, alignment, direction, optional user plan) into a launch. `aligned128` says whether every
// row of every tensor starts on a 128-byte line border; `aligned16` says
// whether every tensor base is 16-byte aligned.
int gcd_int(int a, int b) { return b == 0 ? a : gcd_int(b, a % b); }

// Rows the flat kernel can take of `rows` rows of length T: the largest count whose elements are a whole
// number of 16-byte vectors (the few rows left over go to the other kernels).
int64_t flat_rows(int64_t rows, int64_t T, int full) { return rows - rows % (full / gcd_int((int)(T % full), full)); }

// Short rows that start at any element, or whose vectors do not fill the SMALL kernel's power-of-two group of
// lanes: the flat kernel, where the tensors allow it (dense, 16-byte aligned bases). Measured at 32 M and 64 M
// elements, forward / backward, % of peak: fp32 flat 80-83 / 76-79 at every T from 4 to 256, SMALL the same
// where T / 4 is a power of two and 64-77 / 63-77 elsewhere (T = 70: 64 / 64, 132: 70 / 67, 36: 74 / 72); float64
// alike. 16-bit storage: flat 72-73 / 66-68 at every T (the three-component scan costs its instruction-bound
// backward pass 8-10 points), SMALL 70-77 / 68-78 on vector-aligned rows that fill at least 0.6 of their group,
// 57-68 / 55-67 otherwise (T = 100, 136, 264, 500).
bool prefer_flat(int64_t T, int full, int esize)
{
    if (T % full != 0) return true;
    const int nv = (int)(T / full), group = pow2_ceil(nv);
    if (esize == 2) return nv * 10 < group * 6;
    return nv != group;
}

// `flat_ok`: the tensors are dense [rows, T] arrays on 16-byte aligned bases (what the flat kernel needs).
int resolve(const scanscam_plan *user, int64_t rows, int64_t T, int dtype, bool aligned16, bool aligned128, bool rev,
            Resolved *out, bool flat_ok = false)
{
    const int esize = elem_size(dtype);
    if (esize == 0) return SCANSCAM_EDTYPE;
    if (rows < 0 || T < 0 || T >= kMaxT) return SCANSCAM_EINVAL;
    const int full = 16 / esize;
    scanscam_plan u = {0, 0, 0, 0, 0, 0};
    if (user) u = *user;

    Launch &l = out->l;
    l = Launch{0, 0, 0, 0, 1, 64, 0, false, 1};
    const bool flat_possible = flat_ok && T >= full && T <= (int64_t)kWave * full && flat_rows(rows, T, full) > 0;
    // Up to 32 MiB per tensor the flat kernel's larger workgroups (16 chunks each, a halo chunk and an LDS exchange
    // per workgroup) cost more than the few lanes it still fills gain: rows of four vectors or more stay with the small kernel's
    // element-aligned vectors there (fp32 [16513, 127] forward 9.2 -> 7.4 us, bf16 [33554, 250] 15.6 -> 12.7 us over 200
    // launches; [8224, 255], 64 vectors per row, 6.7 against 7.0 us; at 100 MB, [200000, 127], the flat kernel is
    // ahead, 49 against 58 us).
    // (Only where the rows fill nine tenths of their lane group: at bf16 [119837, 70], 9 vectors in 16 lanes, the flat
    // kernel is 15 / 38 % ahead at 16 MB too.)
    const int64_t row_vectors = (T + full - 1) / full;
    const bool small_problem = rows * T * esize <= (int64_t(1) << 25) && T >= 4 * full &&
                               row_vectors * 10 >= (int64_t)pow2_ceil((int)row_vectors) * 9;
    if (u.mode == kModeFlat ||
        (u.mode == SCANSCAM_MODE_AUTO && flat_possible && !u.vec && (u.unroll == 0 || u.unroll == 2 || u.unroll == 4) &&
         !small_problem && prefer_flat(T, full, esize))) {
        if (!flat_possible) return SCANSCAM_EPLAN;
        if (u.vec && u.vec != full) return SCANSCAM_EPLAN;
        l.mode = kModeFlat;
        l.vec = full;
        // 4 waves x 4 chunks; 16-bit storage (twice the registers per chunk) 8 waves x 2 chunks -- from 16 MiB per
        // tensor on: below, 4 x 4 there too (bf16 [119837, 70] forward 16.0 -> 14.3 us, [27962, 300] 12.7 -> 11.2 us).
        const bool halves = esize == 2 && rows * T * esize > (int64_t(1) << 24);
        l.unroll = u.unroll ? u.unroll : (halves ? 2 : 4);
        l.waves = u.waves ? u.waves : (halves ? 8 : 4);
        if ((l.unroll != 2 && l.unroll != 4) || l.waves < 1 || l.waves > scanscam::kMaxWaves) return SCANSCAM_EPLAN;
        out->nch = 1;
        out->tiles_per_row = 0;
        out->counters = 1;
        out->row_major = 0;
        out->line_shift = 0;
        out->super_base = 0;
        out->ws_bytes = 0;
        return SCANSCAM_OK;
    }
    // The full 16-byte vector needs rows that start on 16-byte borders -- or the element-aligned ("ragged")
    // variants of the kernels: ROW and LOOKBACK for rows of at least nine tenths of a chunk (on shorter rows
    // most of their lanes would idle), SMALL for rows of 4 vectors to one chunk (shorter ones lose nothing
    // with one element per lane).
    const bool vec_aligned = aligned16 && (T % full == 0);
    const bool small_rows = u.mode == kModeSmall || (u.mode == SCANSCAM_MODE_AUTO && T <= (int64_t)kWave * full);
    const bool ragged_possible = full > 1 && (small_rows ? (T >= 4 * full && T <= (int64_t)kWave * full)
                                                         : T * 10 >= (int64_t)kWave * full * 9);
    l.vec = u.vec ? u.vec : ((vec_aligned || ragged_possible) ? full : 1);
    if (l.vec != 1 && l.vec != full) return SCANSCAM_EPLAN;
    l.ragged = l.vec == full && full != 1 && !vec_aligned;
    if (l.ragged && !ragged_possible) return SCANSCAM_EPLAN;

    const int64_t chunk = (int64_t)kWave * l.vec;
    // Rows that start inside a 128-byte line, longer than one chunk: the ROW and LOOKBACK kernels lay their
    // chunks out from the line border before each row's start, so that a wave's loads and stores cover
    // whole lines (fp32 [23140, 2900], rows 16-byte aligned only: 129 / 220 us, 136 / 250 us without). A row
    // then takes up to one line's worth of vector slots more, which is not worth a fifth chunk for rows of
    // up to four (one wave per row: [67108, 1000] 128 us forward without, 150 with).
    // (Element-aligned rows: the border is counted in elements, and the vectors then sit on 16-byte borders.)
    const int64_t lead = l.ragged ? 128 / esize - 1 : 128 / ((int64_t)l.vec * esize) - 1;
    const int64_t nvec = l.ragged ? (T + lead + l.vec - 1) / l.vec : (T + l.vec - 1) / l.vec + lead;
    const int64_t nch_plain = (T + chunk - 1) / chunk, nch_lines = (nvec + kWave - 1) / kWave;
    // Rows of up to 4 chunks take one wave with 1, 2 or 4 chunks (2 or 4 when element-aligned): no shift
    // either where it would double that count and leave half the wave's slots empty (bf16 [33520, 1001], two
    // chunks: 38 / 57 us without the shift, 51 / 87 us with it in a wave of 4).
    // (Element-aligned 16-bit rows of three chunks take a wave of exactly three, below.)
    auto chunks_of_one_wave = [&](int64_t n) { return (l.ragged && esize == 2 && n == 3) ? 3 : pow2_ceil(l.ragged && n < 2 ? 2 : n); };
    const bool same_wave_shape =
        nch_plain > 4 || (nch_lines <= 4 && chunks_of_one_wave(nch_lines) == chunks_of_one_wave(nch_plain));
    out->line_shift = (!aligned128 && !small_rows && (T > chunk || l.ragged) && same_wave_shape) ? 1 : 0;
    const int64_t nch64 = out->line_shift ? nch_lines : nch_plain;
    const int nch = (int)nch64;
    out->nch = nch;
    out->tiles_per_row = 0;
    out->counters = 1;
    out->row_major = 0;
    out->super_base = 0;
    out->ws_bytes = 0;
    if (rows == 0 || T == 0) return SCANSCAM_OK;

    l.mode = u.mode;
    if (l.mode == SCANSCAM_MODE_AUTO) {
        if (T <= chunk) l.mode = kModeSmall;  // (line_shift is 0 here)
        // From 256 rows on, one 16-wave workgroup per row fills the chip as well as tiles over
        // workgroups do and needs no carry hand-off between workgroups.
        else if (nch >= 64 && rows < 256) l.mode = kModeLookback;
        else if (prefer_lookback_for_many_rows(rows, nch, rev, esize)) l.mode = kModeLookback;
        else l.mode = kModeRow;
    }

    if (l.mode == kModeSmall) {
        if (T > chunk) return SCANSCAM_EPLAN;
        l.group = pow2_ceil((T + l.vec - 1) / l.vec);
        l.unroll = u.unroll ? u.unroll : 4;
        l.waves = u.waves ? u.waves : 4;
        const int64_t rows_per_wg = (int64_t)l.waves * l.unroll * (kWave / l.group);
        l.grid = (rows + rows_per_wg - 1) / rows_per_wg;
    } else if (l.mode == kModeRow) {
        l.unroll = u.unroll;
        l.waves = u.waves;
        l.wpr = u.waves_per_row;
        if (!l.unroll && !l.waves && !l.wpr) {
            // Element-aligned rows of 16-bit storage that take 3 or 9 chunks: waves of exactly 3 chunks instead of 4
            // with a quarter of their slots empty. These kernels issue the most instructions per byte, and the
            // empty slots cost them their share: bf16 [65000, 1025] 58 / 67 -> 72 / 74 % of peak, [16380, 4097]
            // (9 chunks, 3 waves) 59-65 / 62-68 -> 73 / 73 %. fp32 and rows of whole vectors gain nothing from it
            // (fp32 [87000, 769] 79 / 75 -> 76 / 72 %, bf16 [43000, 1536] 79 / 78 either way).
            const bool threes = l.ragged && esize == 2 && l.vec == full;
            if (threes && nch == 3) {
                l.unroll = 3;
                l.wpr = 1;
                l.waves = 4;
            } else if (threes && nch == 9) {
                l.unroll = 3;
                l.wpr = l.waves = 3;
            } else if (nch <= 4) {
                l.unroll = (l.vec == full) ? pow2_ceil(nch) : (nch == 1 ? 1 : 4);
                l.wpr = 1;
                l.waves = 4;
            } else if (nch <= 16) {
                // 4 waves per workgroup. 5-6 chunks: 2 chunks per wave; 7-8: 4 chunks per wave and two
                // rows per workgroup (fp32 [32768, 2048] 122 / 211 us against 124 / 215 with 2 chunks per
                // wave and one row, bf16 [16384, 4096] 63.2 / 109.5 against 65.0 / 111.3); 9-16: one row.
                l.unroll = (l.vec == full && nch <= 6) ? 2 : 4;
                l.wpr = (l.vec == full && (nch == 7 || nch == 8)) ? 2 : 4;
                l.waves = 4;
                // Element-aligned rows of 9-12 chunks: 3 waves (bf16 [16380, 4097]: 76 / 123 us, 96 / 149 with 4);
                // of 5-6 chunks: 3 waves x 2 chunks (bf16 [16376, 2049]: 45 / 66 us, 55 / 82 with 4 waves;
                // fp32 [32736, 1025]: 69 / 110 against 76 / 110).
                if (l.ragged && nch > 8 && nch <= 12) l.wpr = l.waves = 3;
                if (l.ragged && nch >= 5 && nch <= 6) l.wpr = l.waves = 3;
            } else {
                // Longer rows: a workgroup tile (waves x 4 chunks) that covers the row in one step, or
                // in as few as 16 waves allow -- each further step waits for the carry of the last --
                // with just the waves those steps need: a row of 36 chunks takes 9 waves, not 8 waves
                // twice or 16 waves of which 7 idle (fp32 [7456, 9000]: 138 / 250 us against 145 / 258).
                // Few rows as well: fewer steps count for more than more waves per row ([300, 16640]:
                // 15.5 / 23.9 us with 9 waves x 4 chunks x 2 steps, 18.8 / 27.1 with 16 waves x 4 x 2).
                l.unroll = 4;
                const int steps = (nch + 63) / 64;
                l.wpr = l.waves = (nch + steps * 4 - 1) / (steps * 4);
                // 16-bit storage, 17-24 chunks (to 28 when element-aligned): two steps of half as many waves with
                // 2 chunks each. These kernels are as much bound by their instructions as by memory (unpacking,
                // 8 elements per lane and chunk), and with 2 chunks per wave they need half the registers, so
                // twice the waves cover each other: bf16 [3883, 8640] 41.5 / 63.6 us -> 35.1 / 59.4 us, element-
                // aligned [3297, 10175] 46.1 / 69.3 -> 35.9 / 60.8 us. From 32 chunks on the single step wins back.
                if (esize == 2 && l.vec == full && nch <= (l.ragged ? 28 : 24)) {
                    l.unroll = 2;
                    l.wpr = l.waves = (nch + 3) / 4;
                }
            }
        } else {
            if (!l.unroll) l.unroll = 4;
            if (!l.waves) l.waves = l.wpr ? l.wpr : 4;
            if (!l.wpr) l.wpr = l.waves;
        }
        if (l.wpr < 1 || l.wpr > l.waves || l.waves % l.wpr != 0) return SCANSCAM_EPLAN;
        const int rows_per_wg = l.waves / l.wpr;
        l.grid = (rows + rows_per_wg - 1) / rows_per_wg;
    } else if (l.mode == kModeLookback) {
        // Tiles of 32 chunks (8192 fp32 elements): fewer, larger tiles keep the wait for the
        // carry short relative to the time a tile spends on its data. With very few rows the
        // tiles in flight are neighbours in one row, which publish almost together and so wait
        // longest for each other: 64 chunks there (up to 8 rows: forward +1 to +4 points of peak at
        // 2^26 fp32 elements; from 12 rows on the 32-chunk tile is 4 to 6 points faster).
        l.unroll = u.unroll ? u.unroll : 4;
        l.waves = u.waves ? u.waves : (rows <= 8 && l.unroll <= 4 ? 16 : 8);
        // Forward fp32 with up to 16 rows: the 64-chunk tile as 8 waves of 8 chunks (two workgroups per CU
        // instead of one of 16 waves): [1, 2^26] 61 -> 64 % of peak, [16, 2^22] 64 -> 66 %, [8, 2^21] 53 -> 57 %;
        // the backward pass gains nothing from it, 16-bit storage with 2 to 8 rows (bf16 [8, 2^22] 50 -> 43 us,
        // [4, 2^23] 48 -> 46 us, [2, 2^24] 49 -> 46 us; [1, 2^26] level, [16, 2^21] 47 -> 51 us).
        // (fp32 with 17 to 64 rows likewise while the whole problem is 8 M elements or less, i.e. up to 512 such tiles:
        // [32, 262144] forward 26.1 -> 20.0 us, [64, 131072] 25.4 -> 21.4 us; at 32 M elements the 32-chunk tile is level.)
        const bool few_tiles = esize == 4 && rows > 16 && rows <= 64 && rows * (int64_t)nch <= 32768;
        if (!u.waves && !u.unroll && !rev && l.vec == full && !l.ragged &&
            (esize == 4 ? (rows <= 16 || few_tiles) : (esize == 2 && rows >= 2 && rows <= 8))) {
            l.unroll = 8;
            l.waves = 8;
        }
        if (!u.waves && !u.unroll && rows > 8 && !(few_tiles && l.unroll == 8)) {
            // As many tiles as 8-wave tiles would take, but with only the waves they need: 75 chunks are 3
            // tiles of 7 waves (84 chunk slots), not of 8 (96).
            int tiles = (nch + kTileChunks - 1) / kTileChunks;
            // Element-aligned rows of 16-bit storage up to 96 chunks: tiles of up to 16 chunks (3-4 waves). Their
            // waves do more arithmetic per byte (components of partial vectors moved into place, masks per
            // element), and the smaller workgroups cover each other better: bf16 [2013, 33333] 55 / 58 -> 62 / 66 %
            // of peak, [3947, 17001] 59 / 63 -> 65 / 68 %, [1973, 34001] 61 / 62 -> 63 / 67 %; from 190 chunks on
            // the larger tile is 3-4 points faster, and rows of whole vectors keep it throughout.
            if (l.ragged && esize == 2 && nch <= 96) tiles = (nch + kTileChunks / 2 - 1) / (kTileChunks / 2);
            l.waves = (nch + tiles * l.unroll - 1) / (tiles * l.unroll);
        }
        const int tile_chunks = l.waves * l.unroll;
        out->tiles_per_row = (nch + tile_chunks - 1) / tile_chunks;
        // One ticket counter per row up to kMaxCounters; when rows do not divide
        // evenly every counter gets the grid share of the fullest one.
        out->counters = (int)(rows < kMaxCounters ? rows : kMaxCounters);
        // Row-major order: a few counters, so that their rows stay neighbours in memory.
        out->row_major = row_major_order(rows, out->tiles_per_row) ? 1 : 0;
        if (out->row_major) out->counters = kRowMajorCounters;
        const int64_t rows_per_counter = (rows + out->counters - 1) / out->counters;
        const int64_t tiles = rows * (int64_t)out->tiles_per_row;
        l.grid = (int64_t)out->counters * rows_per_counter * out->tiles_per_row;
        if (l.grid >= (int64_t(1) << 31)) return SCANSCAM_EINVAL;
        const int64_t supers = rows * (int64_t)((out->tiles_per_row + kSuper - 1) / kSuper);
        out->super_base = (int64_t)out->counters * kCounterStride + tiles * tile_words(dtype);
        out->ws_bytes = (size_t)(out->super_base + supers * super_words(dtype)) * sizeof(uint64_t);
    } else {
        return SCANSCAM_EPLAN;
    }

    if (l.ragged) {
        if (!u.unroll && l.unroll < 2) l.unroll = 2;  // instantiated for 2, 3 and 4 chunks per wave
        if (l.unroll != 2 && l.unroll != 3 && l.unroll != 4) return SCANSCAM_EPLAN;
    }
    if (!unroll_ok(l.vec, full, l.unroll)) return SCANSCAM_EPLAN;
    if (l.waves < 1 || l.waves > scanscam::kMaxWaves ||
        l.waves * kWave > scanscam::max_threads_for_unroll(l.unroll))
        return SCANSCAM_EPLAN;
    if (l.grid >= (int64_t(1) << 31)) return SCANSCAM_EINVAL;
    return SCANSCAM_OK;
}

bool aligned_to(const void *p, size_t n) { return (reinterpret_cast<uintptr_t>(p) % n) == 0; }

// Address of `scratch` on the current device: looked up once per device, with that device current
// (every GPU holds its own copy of the array at its own address), and kept.
constexpr int kMaxDevices = 64;
int noalloc_scratch(void **out)
{
    static std::mutex lock;
    static void *ptr[kMaxDevices];  // zero-initialised: not looked up yet
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return SCANSCAM_ELAUNCH;
    std::lock_guard<std::mutex> hold(lock);
    if (!ptr[dev]) {
        void *p = nullptr;
        if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) return SCANSCAM_ELAUNCH;
        ptr[dev] = p;
    }
    *out = ptr[dev];
    return SCANSCAM_OK;
}

const scanscam_strides *const kDense[5] = {nullptr, nullptr, nullptr, nullptr, nullptr};

// Tensor order everywhere below: a, x, h, y0, y1 (x = b forwards, gh backwards; y0 = h forwards,
// gb backwards; h and y1 = ga exist only backwards). st[k] == nullptr means dense.
int run(bool rev, const void *a, const void *x, const void *h, void *y0, void *y1,
        const scanscam_strides *const st[5], int64_t n0, int64_t n1, int64_t T, int dtype, void *workspace,
        size_t workspace_bytes, void *stream, const scanscam_plan *plan, void *start_event = nullptr,
        void *stop_event = nullptr, bool use_scratch = false, bool allow_flat = true)
{
    const int esize = elem_size(dtype);
    if (esize == 0) return SCANSCAM_EDTYPE;
    if (n0 < 0 || n1 < 0 || T < 0 || T >= kMaxT) return SCANSCAM_EINVAL;
    if (n0 == 0 || n1 == 0 || T == 0) return SCANSCAM_OK;
    if (n1 > INT64_MAX / n0) return SCANSCAM_EINVAL;
    const int64_t rows = n0 * n1;
    if (!a || !x || !y0 || (rev && (!h || !y1))) return SCANSCAM_EINVAL;

    const void *ptrs[5] = {a, x, rev ? h : a, y0, rev ? y1 : y0};
    const bool used[5] = {true, true, rev, true, rev};
    int64_t s0[5], s1[5];
    for (int k = 0; k < 5; k++) {
        const scanscam_strides *t = used[k] ? st[k] : nullptr;
        s0[k] = t ? t->outer : n1 * T;
        s1[k] = t ? t->row : T;
        if (s0[k] < 0 || s1[k] < 0) return SCANSCAM_EINVAL;
    }
    // Rows are independent, so the two levels may be merged or exchanged freely as long as every
    // tensor is walked the same way: one level when the groups follow each other at the row stride,
    // otherwise the longer level inside (the kernels spread the inner level over blockIdx.x).
    if (n1 == 1) {
        n1 = n0;
        n0 = 1;
        for (int k = 0; k < 5; k++) s1[k] = s0[k];
    }
    bool one_level = true;
    for (int k = 0; k < 5; k++) one_level = one_level && (!used[k] || s0[k] == n1 * s1[k]);
    if (n0 > 1 && one_level) {
        n1 = rows;
        n0 = 1;
    }
    if (n0 > n1) {
        for (int k = 0; k < 5; k++) {
            const int64_t t = s0[k];
            s0[k] = s1[k];
            s1[k] = t;
        }
        const int64_t t = n0;
        n0 = n1;
        n1 = t;
    }
    for (int k = 0; k < 5; k++) {
        if (n0 == 1) s0[k] = 0;
        if (n1 == 1) s1[k] = 0;
    }

    // 16-byte vectors need every row of every tensor to start on a 16-byte border.
    const int full = 16 / esize;
    bool aligned16 = true, aligned128 = true;
    const int line = 128 / esize;  // elements per 128-byte line
    for (int k = 0; k < 5; k++) {
        if (!used[k]) continue;
        if (!aligned_to(ptrs[k], (size_t)esize)) return SCANSCAM_EALIGN;
        aligned16 = aligned16 && aligned_to(ptrs[k], 16) && s0[k] % full == 0 && s1[k] % full == 0;
        aligned128 = aligned128 && aligned_to(ptrs[k], 128) && s0[k] % line == 0 && s1[k] % line == 0;
    }

    // The flat kernel takes dense [rows, T] tensors on 16-byte aligned bases (rows of any length).
    bool flat_ok = allow_flat && n0 == 1;
    for (int k = 0; k < 5; k++) flat_ok = flat_ok && (!used[k] || (aligned_to(ptrs[k], 16) && (n1 == 1 || s1[k] == T)));
    // The flat kernel's workgroups read a halo of their neighbours' spans (and a[e+1] / h[e-1] across span
    // borders backwards), so an output that shares bytes with an input -- an in-place call, which every other
    // kernel family allows because it reads only what it is about to write -- would race there.
    if (flat_ok) {
        const int64_t bytes = rows * T * esize;
        auto overlaps = [&](const void *p, const void *q) {
            const char *pc = static_cast<const char *>(p), *qc = static_cast<const char *>(q);
            return pc < qc + bytes && qc < pc + bytes;
        };
        for (int o = 3; o < 5; o++)
            for (int i = 0; i < 3; i++)
                if (used[o] && used[i] && overlaps(ptrs[o], ptrs[i])) flat_ok = false;
    }
    // One pair of events cannot bracket the flat launch and the launch for the rows it leaves over.
    if ((start_event || stop_event) && flat_rows(rows, T, full) != rows) flat_ok = false;

    Resolved r;
    const int rc = resolve(plan, rows, T, dtype, aligned16, aligned128, rev, &r, flat_ok);
    if (rc != SCANSCAM_OK) return rc;

    if (r.l.mode == kModeFlat) {
        const int64_t taken = flat_rows(rows, T, full);
        scanscam::FlatArgs fa;
        fa.a = a;
        fa.x = x;
        fa.h = h;
        fa.y0 = y0;
        fa.y1 = y1;
        fa.N = taken * T;
        fa.T = (int32_t)T;
        hipStream_t fs = static_cast<hipStream_t>(stream);
        hipEvent_t e0 = static_cast<hipEvent_t>(start_event), e1 = static_cast<hipEvent_t>(stop_event);
        hipError_t e = hipErrorInvalidValue;
        switch (dtype) {
        case SCANSCAM_F32: e = scanscam::launch_scan_flat<float>(fa, r.l.unroll, r.l.waves, rev, fs, e0, e1); break;
        case SCANSCAM_BF16: e = scanscam::launch_scan_flat<__bf16>(fa, r.l.unroll, r.l.waves, rev, fs, e0, e1); break;
        case SCANSCAM_F16: e = scanscam::launch_scan_flat<_Float16>(fa, r.l.unroll, r.l.waves, rev, fs, e0, e1); break;
        case SCANSCAM_F64: e = scanscam::launch_scan_flat<double>(fa, r.l.unroll, r.l.waves, rev, fs, e0, e1); break;
        }
        if (e != hipSuccess) return SCANSCAM_ELAUNCH;
        if (taken == rows) return SCANSCAM_OK;
        // The few rows left over (fewer than a vector has elements): the other kernels, on the tail of every tensor.
        const int64_t off = taken * T * esize;
        auto tail = [&](const void *q) { return q ? static_cast<const void *>(static_cast<const char *>(q) + off) : nullptr; };
        return run(rev, tail(a), tail(x), tail(h), const_cast<void *>(tail(y0)), const_cast<void *>(tail(y1)), kDense, 1,
                   rows - taken, T, dtype, workspace, workspace_bytes, stream, nullptr, nullptr, nullptr, use_scratch,
                   /*allow_flat=*/false);
    }

    ScanArgs args;
    args.a = a;
    args.x = x;
    args.h = h;
    args.y0 = y0;
    args.y1 = y1;
    for (int k = 0; k < 5; k++) {
        args.s0[k] = s0[k];
        args.s1[k] = s1[k];
    }
    args.rows = rows;
    args.n1 = n1;
    args.T = (int32_t)T;
    args.nch = r.nch;
    args.wpr = r.l.wpr;
    args.group = r.l.group;
    args.tiles_per_row = r.tiles_per_row;
    args.counters = r.counters;
    args.row_major = r.row_major;
    args.line_shift = r.line_shift;
    args.desc_base = r.counters * kCounterStride;
    args.super_base = r.super_base;
    args.spin_limit = (plan && plan->spin_limit > 0) ? plan->spin_limit : scanscam::kSpinLimit;
    args.ws = nullptr;

    hipStream_t s = static_cast<hipStream_t>(stream);
    // The caller's events, if any, are bound to the scan kernel itself (its start and end on the GPU).
    hipEvent_t ev0 = static_cast<hipEvent_t>(start_event), ev1 = static_cast<hipEvent_t>(stop_event);
    const bool timed = ev0 || ev1;
    auto launch = [&](const ScanArgs &la, const Launch &l) {
        switch (dtype) {
        case SCANSCAM_F32: return scanscam::launch_scan<float>(la, l, rev, s, ev0, ev1);
        case SCANSCAM_BF16: return scanscam::launch_scan<__bf16>(la, l, rev, s, ev0, ev1);
        case SCANSCAM_F16: return scanscam::launch_scan<_Float16>(la, l, rev, s, ev0, ev1);
        case SCANSCAM_F64: return scanscam::launch_scan<double>(la, l, rev, s, ev0, ev1);
        default: return hipErrorInvalidValue;
        }
    };

    if (r.l.mode == kModeLookback) {
        if (use_scratch) {
            // The library's own fixed array instead of a caller's workspace; every call clears the part
            // it uses (below), whatever the call before left there.
            if (r.ws_bytes > (size_t)SCANSCAM_NOALLOC_SCRATCH_BYTES) return SCANSCAM_ESCRATCH;
            const int src = noalloc_scratch(&workspace);
            if (src != SCANSCAM_OK) return src;
            workspace_bytes = SCANSCAM_NOALLOC_SCRATCH_BYTES;
        }
        if (!workspace || workspace_bytes < r.ws_bytes) return SCANSCAM_EWORKSPACE;
        if (!aligned_to(workspace, 8)) return SCANSCAM_EALIGN;
        args.ws = static_cast<uint64_t *>(workspace);
        const int64_t words = (int64_t)(r.ws_bytes / sizeof(uint64_t));
        if (clear_workspace(args.ws, words, args.desc_base, s) != hipSuccess) return SCANSCAM_ELAUNCH;
        // One launch over all rows; the kernel splits a row index into (group, row). Its grid is far
        // below every launch limit by construction.
        return launch(args, r.l) == hipSuccess ? SCANSCAM_OK : SCANSCAM_ELAUNCH;
    }

    // ROW and SMALL: blockIdx.x walks the n1 rows of a group, blockIdx.y the n0 groups. One launch
    // may hold at most 2^32 - 1 threads and 65535 groups; rows are independent, so a larger problem
    // is issued as several launches over consecutive slabs (only tensors of tens of GB get there).
    const int64_t threads = (int64_t)r.l.waves * kWave;
    const int64_t max_grid = ((int64_t(1) << 32) - 1) / threads;
    int64_t rows_per_wg = 1;
    if (r.l.mode == kModeRow) rows_per_wg = r.l.waves / r.l.wpr;
    if (r.l.mode == kModeSmall) rows_per_wg = (int64_t)r.l.waves * r.l.unroll * (kWave / r.l.group);
    const int64_t grid_x_all = (n1 + rows_per_wg - 1) / rows_per_wg;
    const int64_t slab_rows = grid_x_all <= max_grid ? n1 : max_grid * rows_per_wg;
    if (timed && (grid_x_all > max_grid || n0 > 65535 || n0 * grid_x_all > max_grid))
        return SCANSCAM_EINVAL;  // several launches: one pair of events cannot bracket them

    for (int64_t row0 = 0; row0 < n1; row0 += slab_rows) {
        const int64_t n = n1 - row0 < slab_rows ? n1 - row0 : slab_rows;
        const int64_t grid_x = (n + rows_per_wg - 1) / rows_per_wg;
        int64_t slab_groups = max_grid / grid_x;
        if (slab_groups > 65535) slab_groups = 65535;
        if (slab_groups < 1) slab_groups = 1;
        for (int64_t g0 = 0; g0 < n0; g0 += slab_groups) {
            ScanArgs slab = args;
            Launch l = r.l;
            const void **in[3] = {&slab.a, &slab.x, &slab.h};
            void **out[2] = {&slab.y0, &slab.y1};
            for (int k = 0; k < 5; k++) {
                const int64_t byte_off = (g0 * s0[k] + row0 * s1[k]) * esize;
                if (k < 3 && *in[k]) *in[k] = static_cast<const char *>(*in[k]) + byte_off;
                if (k >= 3 && *out[k - 3]) *out[k - 3] = static_cast<char *>(*out[k - 3]) + byte_off;
            }
            slab.rows = n;
            l.grid = grid_x;
            l.grid_y = (int)(n0 - g0 < slab_groups ? n0 - g0 : slab_groups);
            if (launch(slab, l) != hipSuccess) return SCANSCAM_ELAUNCH;
        }
    }
    return SCANSCAM_OK;
}

// Whether every tile of a time split takes the aggregates of all tiles before it instead of waiting for the chain of
// super-tiles. A tile then waits for nothing but its predecessors' folds, one memory round trip, where the chain takes one
// more per super-tile; each of its waves reads up to 8 aggregates of every channel. In calls of few rounds of workgroups
// that wait is most of the time (GPU time, us forward / backward, buffers in rotation): fp32 [1, 2541, 295] 12.7 / 13.9 -> 10.2 /
// 11.4, [10, 1083, 128] 12.8 / 14.7 -> 10.0 / 12.0, [3, 2000, 512] 14.5 / 18.7 -> 13.1 / 17.3, bf16 [2, 1643, 96] 12.4 / 13.9 ->
// 9.6 / 10.8, [6, 574, 256] 9.6 / 10.6 -> 8.3 / 8.6; 225 and 192 calls in fp32 and 16 bits 0.87 and 0.89 x in the mean, at most
// 1.04 and 1.06 (profiles/direct_lookback_random_shapes.txt), and larger ones gain little ([8, 4096, 512] 45.7 / 74.4 -> 44.0 /
// 73.0). It ends where
//   - more workgroups cover each other's waits, and the aggregates they read are what is left: [25, 1696, 384], 2100 workgroups,
//     0.97 / 0.99 x, [64, 1024, 333] backward, 3072 of them, 1.06 x, [24, 2048, 3072] backward, 18432, 543 -> 569, bf16 [90, 2048,
//     514] backward, 14400, 243 -> 256 us: 2048 at most, and 896 for 16 single 16-bit channels backwards (30 calls with fewer
//     0.78 to 1.03 x, 19 with more 0.98 to 1.10 x: [18, 1242, 151] 21.4 -> 23.4 us);
//   - a wave's aggregates span more than 1024 steps, or number more than 8: beyond what was measured;
//   - a lane holds 64 elements, one workgroup per CU (bf16 [8, 4096, 512] backward, 4 channels x 16 steps, 39.3 against 41.5);
//   - pairs are four words each: fp64 would lose as often as it gains ([4, 1489, 832] forward 45.1 against 57.1, [9, 599, 320] 17.0
//     / 21.2 against 18.1 / 23.1, [1, 2754, 250] 16.2 / 21.5 -> 13.5 / 19.2).
bool direct_lookback(const scanscam::ClLaunch &l, int esize, bool rev)
{
    const int per_wave = (l.segments + l.waves - 1) / l.waves;  // tiles
    const int most = esize == 2 && rev && l.vec == 1 && l.steps == 16 ? 896 : 2048;  // workgroups
    return scanscam::cl_direct_built(esize, l.vec, l.steps) && l.grid <= most && per_wave <= 8 &&
           per_wave * l.waves * l.steps <= 1024;
}

// Grid, LDS and workspace of a chosen launch; `virtual_steps`: steps before the first one that the tiles cover as well.
int size_cl(int64_t batch, int64_t T, int dtype, bool rev, int virtual_steps, scanscam::ClLaunch *l)
{
    const int64_t rowgroups = batch * l->groups;
    const int64_t tile_steps = (int64_t)l->waves * l->steps;
    const int64_t tiles = (T + virtual_steps + tile_steps - 1) / tile_steps;
    const int64_t vals = (int64_t)l->vec * kWave * value_words(dtype);  // words of one [vec][64] array of values
    l->ws_bytes = 0;
    l->segments = 1;
    if (l->kind == 2) {
        if (tiles >= (int64_t(1) << 31)) return SCANSCAM_EINVAL;
        l->segments = (int)tiles;  // the kernel's tiles per row-group
        const int64_t supers = (tiles + l->waves - 1) / l->waves;
        const int64_t pairs = (int64_t)l->vec * kWave * tile_words(dtype);  // words of one [vec][64] array of pairs
        l->ws_bytes = (size_t)(rowgroups * kCounterStride + rowgroups * tiles * pairs + rowgroups * supers * (pairs + vals)) *
                      sizeof(uint64_t);
    }
    if (l->segments <= 1) {  // a forced time split of a single tile: nothing to split after all
        l->kind = 0;
        l->ws_bytes = 0;
    }
    l->grid = rowgroups * l->segments;
    l->direct = l->kind == 2 && l->shift == 0 && direct_lookback(*l, elem_size(dtype), rev);
    const int arrays = l->kind == 2 ? scanscam::cl_lookback_arrays(l->direct) : 4;
    l->lds_bytes = (size_t)arrays * l->waves * l->vec * kWave * compute_size(dtype);
    if (l->grid >= (int64_t(1) << 31)) return SCANSCAM_EINVAL;
    return SCANSCAM_OK;
}

// Whether a walk's loads run a tile ahead, past the stores (scan_cl_kernel, PIPE). GPU time of random calls that take it, buffers in
// rotation, none of them used to find the rule (profiles/walk_loads_past_stores_random_shapes.txt): four fp32
// channels by 8 steps 0.95 x in the mean of 40 (0.85 to 1.01; [36, 702, 1472] 87.5 -> 79.4 us), two by 16 0.94 (0.87 to 1.0), two of fp64 by 8
// 0.92 forwards (0.83 to 1.0), 0.98 backwards (0.92 to 1.01), single ones of fp64 0.96 in the mean of 30 (0.89 to 1.02).
// Not taken
//   - below three tiles, which leave fewer than two that are whole (fp64 [27, 90, 800] 11.7 -> 12.1);
//   - where 8 waves of 32 or more words a lane leave one workgroup per CU with its registers and there are more: fp32 [930, 174, 160] 58.8 -> 62.6 ([201,
//     238, 160], one each, 22.3 -> 20.5);
//   - where a time step is two or four whole groups of channels, 2 or 4 KB in 16-byte lanes, from 220 workgroups on (memory's
//     order again, as far as the sizes tell: no counter was taken): fp32 [114, 578, 1024] 149 -> 171,
//     [234, 914, 512] 248 -> 271, [128, 2048, 512] 260 -> 271, [64, 2000, 1024] 263 -> 287, [224, 909, 512] 224 -> 233 (at 210 and 216, 0.94 and
//     0.96 x; 8 KB steps 0.89 to 0.97 x but [32, 2048, 2048] 278 -> 286); fp64 backwards at any number, [93, 772, 256] 133 -> 136,
//     [61, 1415, 512] 300 -> 320;
//   - single fp64 channels, two workgroups of 4 waves per CU: 1.0 to 1.07 x, [134, 777, 180] 101.5 -> 108.8;
//   - where nearly every CU has one workgroup and a time step's last group is not full, which memory's order bounds: fp32, 256 of
//     them, [64, 2048, 1016] 352 -> 368, [64, 2048, 1008] 287 -> 298, [64, 2048, 960] 298 -> 307, 245 of them,
//     [49, 925, 1132] 126 -> 128 (but 205, [41, 1355, 1216] 163 -> 151, and 714, [102, 591, 1680] 245 -> 235).
// `sT`: the tensors' time strides in elements; `cached`: the walk stores through the caches' normal policy, which these do not.
bool pipe_walk(const scanscam::ClLaunch &l, int64_t T, int64_t C, int esize, bool rev, const int64_t sT[5], bool cached)
{
    if (l.kind != 0 || l.group != kWave || l.ragged || l.shift != 0 || !scanscam::cl_pipe_built(esize, l.vec, l.steps, rev)) return false;
    // Two tiles whose accesses all exist, which the kernel takes for granted: a[t+1] of the first and h[t-1] of the last step do not.
    if (T < (int64_t)3 * l.waves * l.steps + (rev ? 1 : 0)) return false;
    if (l.waves > 4 && l.grid > kComputeUnits && l.vec * l.steps * esize >= 128) return false;
    // (Its resources end 2 GiB past a span's base, where lanes without channels store.)
    for (int k = 0; k < 5; k++)
        if ((uint64_t)sT[k] * (uint64_t)esize * 18u + (uint64_t)C * (uint64_t)esize >= (uint64_t(1) << 31)) return false;
    if (cached) return false;
    const int64_t group = (int64_t)kWave * l.vec;
    if (l.vec > 1 && (rev || l.grid >= 220) && (C == 2 * group || C == 4 * group)) return false;
    if (l.vec == 1 && l.waves <= 4 && l.grid > kComputeUnits && l.grid <= 2 * kComputeUnits) return false;
    return C % group == 0 || l.grid < kComputeUnits - 20 || l.grid > kComputeUnits;
}

// Bytes of LDS a backward walk asks for beyond its need, so that a CU holds half as many of its workgroups as its registers allow; 0
// where none. Once more of them run than fit at once, 16-bit spans of 4 x 16 (125 registers packed, 207 unpacked: 4 workgroups
// of 4 waves a CU or 2) and fp32 element-aligned ones of 2 x 16 (120, 136 before) lose by the better fit: bf16 [403, 120, 1360] 175 us as
// 4, 155 as 2 a CU, [937, 118, 372] 132 and 109, fp16 [672, 47, 1852] 141 and 126; where all fit at once they gain by it ([334, 107, 144] 17.5, 20.3).
// 44 random calls each against the unpacked form: bf16 0.96 -> 0.95 x (at most 1.23 -> 1.04), fp16 0.985 -> 0.975 (1.07 -> 1.01); fp32
// 1.015 -> 1.0, there not where the last eighth of a single tile's waves is idle ([420, 104, 839] 158, 171).
size_t idle_lds(const scanscam::ClLaunch &l, int64_t T, int esize, bool rev)
{
    if (!rev || l.kind != 0 || l.group != kWave || l.shift != 0 || l.steps != 16 || (l.waves != 4 && l.waves != 8)) return 0;
    const bool packed = esize == 2 && l.vec == 4 && !l.ragged;
    const bool aligned = esize == 4 && l.vec == 2 && l.ragged && T > (int64_t)l.waves * 14;
    const int fit = l.waves > 4 ? 2 : 4;
    if (!(packed || aligned) || l.grid <= (int64_t)fit * kComputeUnits) return 0;
    // A CU has 160 KB: one workgroup of 8 waves, two (fp32: three) of 4.
    const size_t share = l.waves > 4 ? 82 * 1024 : (packed ? 54 * 1024 : 41 * 1024);
    return share > l.lds_bytes ? share - l.lds_bytes : 0;
}

// Channels-last: the launch plan. `align`: the largest of 16, 8, 4 and the element size that every tensor's base
// and strides are multiples of (bytes). The choice itself is the cost model of scan_cl_plan.hpp: every field the
// caller's plan leaves at zero is chosen by the smallest estimated duration; this function turns the chosen
// candidate into launch parameters and sizes.
int resolve_cl(const scanscam_plan *user, int64_t batch, int64_t T, int64_t C, int dtype, int align, bool rev,
               scanscam::ClLaunch *l, double *predicted_us = nullptr)
{
    const int esize = elem_size(dtype);
    if (esize == 0) return SCANSCAM_EDTYPE;
    scanscam_plan u = {0, 0, 0, 0, 0, 0};
    if (user) u = *user;
    if (u.mode != SCANSCAM_MODE_AUTO && u.mode != kModeRow && u.mode != kModeLookback) return SCANSCAM_EPLAN;
    const scanscam::ClShape shape = {batch, T, C, esize, compute_size(dtype), align, rev};
    scanscam::ClCandidate c;
    // The choice is a pure function of (shape, caller's plan) and costs about a hundred microseconds (some forty
    // candidates through the cost model), so each thread remembers its last few dozen: a model calls the same shapes
    // over and over. Nothing but speed depends on it.
    struct Remembered {
        bool valid;
        int64_t batch, T, C;
        int dtype, align;
        bool rev;
        int32_t mode, vec, unroll, waves;
        scanscam::ClCandidate c;
        double us;
    };
    constexpr int kRemembered = 64;
    static thread_local Remembered remembered[kRemembered] = {};
    const uint64_t key = (uint64_t)batch * 0x9E3779B97F4A7C15ull ^ (uint64_t)T * 0xC2B2AE3D27D4EB4Full ^ (uint64_t)C * 0x165667B19E3779F9ull ^
                         (uint64_t)(dtype * 64 + align * 2 + (rev ? 1 : 0)) * 0x27D4EB2F165667C5ull ^
                         (uint64_t)(u.mode * 4096 + u.vec * 256 + u.unroll * 16 + u.waves);
    Remembered &slot = remembered[(key >> 32 ^ key) % kRemembered];
    if (slot.valid && slot.batch == batch && slot.T == T && slot.C == C && slot.dtype == dtype && slot.align == align &&
        slot.rev == rev && slot.mode == u.mode && slot.vec == u.vec && slot.unroll == u.unroll && slot.waves == u.waves) {
        c = slot.c;
        if (predicted_us) *predicted_us = slot.us;
    } else {
        double us = 0.0;
        if (!scanscam::cl_choose(shape, u, &c, &us)) return SCANSCAM_EPLAN;
        slot = Remembered{true, batch, T, C, dtype, align, rev, u.mode, u.vec, u.unroll, u.waves, c, us};
        if (predicted_us) *predicted_us = us;
    }

    l->vec = c.vec;
    l->steps = c.steps;
    l->waves = c.waves;
    l->kind = c.kind;
    l->group = c.group;
    l->ragged = c.ragged;
    l->shift = 0;
    l->groups = (int)scanscam::cl_groups(C, c.vec);
    l->vectors = kWave;
    return size_cl(batch, T, dtype, rev, 0, l);
}

// Channels-last tiles staged through LDS (scan_staged_kernels.hpp): whether that kernel can run the call, and its tile.
// Dense tensors on 16-byte borders, all channels of a batch element in one workgroup.
bool cl_dense(int64_t batch, int64_t T, int64_t C, const void *const ptrs[5], const int64_t sB[5], const int64_t sT[5])
{
    for (int k = 0; k < 5; k++)
        if (!aligned_to(ptrs[k], 16) || (T > 1 && sT[k] != C) || (batch > 1 && sB[k] != T * C)) return false;
    return true;
}

bool resolve_staged(int64_t batch, int64_t T, int64_t C, int esize, int64_t parts, scanscam::StagedArgs *out)
{
    if (C > scanscam::kStagedThreads || batch >= (int64_t(1) << 31)) return false;  // (the product below stays in range)
    // Steps per tile: what its vectors hold and what the threads' spans cover; then tiles of equal size, in spans of at
    // least half the steps a thread can take (every span costs every thread a read and an FMA for its carry).
    const int most_seg = scanscam::staged_steps(esize);
    const int64_t spans = scanscam::kStagedThreads / C;
    int64_t most = ((int64_t)scanscam::kStagedThreads * scanscam::kStagedVectors * 16 - 16) / (C * esize);
    if (most > spans * most_seg) most = spans * most_seg;
    const int64_t tiles = (T + most - 1) / most, rows = (T + tiles - 1) / tiles;
    int64_t seg = (rows + spans - 1) / spans;
    if (seg < (most_seg + 1) / 2) seg = (most_seg + 1) / 2;
    out->T = (int32_t)T;
    out->C = (int32_t)C;
    out->seg = (int32_t)seg;
    out->spans = (int32_t)((rows + seg - 1) / seg);
    const int64_t whole = out->spans * seg;  // (no span is cut short but those of the last tile)
    out->rows = (int32_t)(whole < most ? whole : most);
    // Parts of equal numbers of tiles.
    const int64_t all = (T + out->rows - 1) / out->rows;
    if (parts > all) parts = all;
    out->tiles = (int32_t)((all + parts - 1) / parts);
    out->parts = (int32_t)((all + out->tiles - 1) / out->tiles);
    out->ws = nullptr;
    return batch * out->parts <= ((int64_t(1) << 32) - 1) / scanscam::kStagedThreads;  // threads of one launch
}

size_t staged_bytes(int64_t batch, int64_t C, int esize, const scanscam::StagedArgs &st)
{
    if (st.parts <= 1) return 0;
    const size_t pair = esize == 8 ? sizeof(scanscam::PartPair<double>) : sizeof(scanscam::PartPair<float>);
    return scanscam::kStagedHeader * sizeof(uint64_t) + (size_t)(batch * st.parts * C) * pair;
}

// Into how many parts an automatic plan of that kernel cuts a batch element's time (1: one workgroup each, one launch);
// 0: the plan is one of scan_cl_plan.hpp. Measured against those (forward / backward, us of GPU time, buffers in rotation;
// random shapes with both sides: profiles/staged_route_random_shapes.txt).
// Whole batch elements, for few channels in lanes they do not fill: fp32 [1000, 1023, 17] 73.5 / 138 -> 41.0 / 74.5,
// [851, 467, 27] 41.2 / 69.2 -> 28.6 / 48.6, bf16 [1000, 1023, 17] 56.3 / 102 -> 22.8 / 41.8, [2048, 512, 40] 65.2 / 105 ->
// 46.2 / 80.0, fp64 [1000, 1023, 17] 115 / 209 -> 86.1 / 156. It ends where
//   - time steps are whole 128-byte lines (the walk streams them: fp32 [256, 1024, 128] 74.7 / 127 against 83.3 / 124) or
//     fill the lanes of the packed kernel: fp32 [512, 4096, 8] 39.5 / 68.9 against 45.8 / 63.0, bf16 [506, 4528, 2] 14.4 /
//     17.9 against 18.2 / 25.3, [338, 2002, 4] 10.3 / 11.5 against 13.6 / 19.7 (but [264, 119208, 4] 411 / 469 -> 273 / 376),
//     fp64 [463, 14524, 3] 124 / 223 against 223 / 255, and eight 16-bit channels below 12 M elements (a step 0.81 to 1.23 x
//     there, 0.78 to 0.92 x above);
//   - there are more channels, which fill the walk's lanes well (bf16 [1076, 490, 91] 79.1 / 138 against 85.8 / 147), but for
//     fp32 steps off the 16-byte border and fp64 (fp32 [1076, 490, 91] 131 / 217 -> 114 / 202, fp64 [1024, 90, 130] 72.4 /
//     129 -> 61.3 / 102);
//   - batch elements are too few workgroups (fp32, C = 33: 320 of them 44.8 / 64.5 -> 40.3 / 65.5, 192 of them 46.2 /
//     66.0 against 57.5 / 78.1; C = 130: 512 level, 320 37.4 / 60.7 against 51.9 / 87.8), more of them for the fewest
//     channels, whose tiles have the most spans (fp32 [435, 988, 3] 7.4 / 10.6 against 9.7 / 11.8, fp64 [343, 8902, 5] 131 /
//     211 against 171 / 205), or less than a tile each (fp32 [3000, 16, 24] 5.5 / 7.8 against 7.9 / 12.3; fp16 [5299, 101,
//     49], 10 KB each, 44.7 / 86.7 -> 40.0 / 61.4), below 512 of them also few time steps (bf16 [358, 246, 16] 6.2 / 7.5 against
//     7.2 / 9.6, fp32 [414, 345, 10] 10.3 / 13.0 -> 7.0 / 9.1).
// Parts, two launches that read gate and value twice but wait for nothing, for the fewer batch elements: fp32 [14, 13990,
// 24] 32.0 / 44.8 -> 21.5 / 29.9, [1, 250000, 8] 92 / 98 -> 20 / 26, bf16 [39, 11559, 30] 57 / 81 -> 34 / 45, fp64 [3, 200000, 24]
// 211 / 270 -> 107 / 158. 1280 workgroups, at most 256 parts (fp32 [1, 600000, 24] with 64 / 128 / 256 parts 309 / 159 / 86 us
// forwards; each workgroup folds the pairs before it). It ends where
//   - the one-pass tiles' chain is short: bf16 [11, 188, 53] 7.6 / 8.7 against 9.1 / 11.3, [8, 723, 23] 8.4 / 10.5 against 9.5 /
//     11.6, [15, 991, 47] 0.96 x, of 32 batch elements on [46, 255, 34] 8.8 / 9.4 against 9.8 / 11.9, [52, 799, 14] 10.9 / 14.6 ->
//     9.7 / 11.2; fp32 [12, 95, 61] 7.1 / 7.7 against 7.8 / 8.9, [22, 360, 19] 0.99 x, [6, 607, 51] 9.1 / 10.5 -> 8.1 / 9.2; fp64 [11, 49,
//     44] 0.97 x, [34, 74, 32] 9.3 / 9.3 -> 7.4 / 8.2; or short for the spans of a tile of very few channels, below 16 batch elements,
//     which the other kernels cut into tiles as well (fp32 [4, 5315, 2] 11.1 / 12.8 against 14.6 / 16.7, bf16 [1, 7948, 2] 11.4 /
//     14.8 against 13.2 / 16.2, [3, 26492, 2] 20.6 / 26.6 -> 14.0 / 16.3; [16, 19488, 2] 39.2 / 56.3 -> 14.8 / 18.7);
//   - more channels fill the lanes of the one-pass tiles, the sooner the more batch elements there are: fp32 [4, 100000, 40]
//     71 / 97 -> 65 / 100, [16, 25000, 40] 61 / 84 against 63 / 98, fp64 [14, 4134, 38] 24.4 / 33.9 against 28.6 / 36.8 ([13, 3223,
//     36] 0.84 x); bf16 [40, 32409, 51] 0.95 / 0.79 x, [100, 2500, 64] 31 / 47 against 37 / 52. Small calls up to 63 channels (fp32 [1,
//     3124, 61] 11.6 / 13.0 -> 10.0 / 11.1, fp64 [4, 222, 62] 9.8 / 11.3 -> 7.7 / 8.5). Above 64 a tile has no four spans (fp32 [1, 4032,
//     65] 12.0 / 13.7 against 14.0 / 15.5, fp64 [4, 2016, 65] 15.3 / 20.9 against 24.9 / 26.2); 64 itself would gain (fp32 [1, 4096,
//     64] 13.5 / 15.6 against 10.8 / 12.0) and has only kept the plan, and the bits, that it had.
//   - a walk of 128 batch elements or more keeps the memory busy: up to 320 only 16-bit calls of 8 M elements that the packed
//     kernel does not serve (bf16 [255, 54672, 2] 59 / 98 against 93 / 130, [242, 68888, 8] 244 / 325 against 255 / 373).
int staged_parts(int64_t batch, int64_t T, int64_t C, int esize)
{
    if (C > scanscam::kStagedThreads) return 0;
    const int64_t step = C * esize, elements = batch * T * C;
    // Steps that fill the packed kernel's lanes: 16-bit pairs, quads of few time steps, eights in small calls; fp32 and fp64
    // whose steps divide 64 bytes, and three fp64 channels (three of four lanes).
    const bool packed = esize == 2 ? C <= 2 || (C == 4 && T < 8192) || (C == 8 && elements < 12 << 20)
                                   : (step <= 64 && 64 % step == 0) || (esize == 8 && C == 3);
    int64_t most = 0;  // channels up to which time in parts is ahead
    if (batch < 128) {
        const int64_t steps = esize == 2 ? (batch < 32 ? 1024 : 512) : (esize == 4 ? 448 : 64);
        int64_t kib = 16;  // of a batch element
        if (batch < 32 && C < 8) kib = 24;
        if (batch < 16 && C < 5 && (C < 4 || esize == 2) && esize != 8) kib = C == 2 && esize == 4 ? 128 : 64;
        if (batch < 16 && C == 1) kib = 256;
        if (T >= steps && T * step >= kib * 1024) {
            if (elements <= (int64_t(1) << 19)) most = 63;
            else if (esize == 2) most = 52;
            else most = batch <= 8 ? 40 : (esize == 8 && batch <= 16 ? 36 : 28);
        }
    } else if (batch < 320 && esize == 2 && !packed && elements >= (int64_t(1) << 23) && (C != 8 || elements < 64 << 20)) {
        most = 40;
    }
    if (C <= most) {
        const int64_t parts = (1280 + batch - 1) / batch;
        return (int)(parts < 256 ? parts : 256);
    }
    if (step % 128 == 0 || packed) return 0;
    if (!(C <= 80 || esize == 8 || (esize == 4 && step % 16 != 0)) || T * step < 7680) return 0;
    if (batch < 512) return batch >= 320 && C <= 80 && T >= 256 && (esize == 2 || C >= (esize == 4 ? 4 : 8)) ? 1 : 0;
    return esize != 8 || C >= 8 || batch >= 768 ? 1 : 0;
}

// The parts in which a call with this plan takes the staged kernel, 0 for none: what a resolved plan says
// (scanscam_resolve_plan_cl writes it into waves_per_row), the automatic choice where the plan leaves everything open.
int staged_parts_of(const scanscam_plan *plan, int64_t batch, int64_t T, int64_t C, int esize)
{
    if (plan && plan->mode == kModeStaged) return plan->unroll > 0 ? plan->unroll : 1;
    if (plan && plan->waves_per_row > 0) return plan->waves_per_row;
    const bool free_plan = !plan || (plan->mode == SCANSCAM_MODE_AUTO && !plan->vec && !plan->unroll && !plan->waves);
    return free_plan ? staged_parts(batch, T, C, esize) : 0;
}

// Channels moved between neighbouring lanes (scan_cl_shift.hpp), for odd channel counts: which of its launches a call takes,
// as one number -- 64 * time steps per wave + 2 * waves + (1: tiles of time over workgroups, 0: a walk) --, 0 for none.
int shift_code(int steps, int waves, bool tiles) { return 64 * steps + 2 * waves + (tiles ? 1 : 0); }

int shift_vec(int esize) { return esize == 8 ? 2 : 4; }

// Fills a launch from that number; false where the kernels cannot run it.
bool resolve_shift(int64_t batch, int64_t T, int64_t C, int dtype, int code, scanscam::ClLaunch *l)
{
    const int esize = elem_size(dtype);
    l->vec = shift_vec(esize);
    l->steps = code / 64;
    l->waves = code / 2 % 32;
    l->kind = code % 2 == 1 ? 2 : 0;
    l->group = kWave;
    l->ragged = false;
    l->shift = (int)(C % l->vec);
    // The vector after a group's last one is loaded by a lane of its own; a time step's last group has at least one whole.
    const int64_t all = (C + l->vec - 1) / l->vec;
    l->groups = (int)((all + kWave - 2) / (kWave - 1));
    l->vectors = (int)((all + l->groups - 1) / l->groups);
    if (l->shift % 2 == 0 || T < 2 || C <= (int64_t)(kWave - 1) * l->vec || all - (int64_t)(l->groups - 1) * l->vectors < 2) return false;
    if (!scanscam::cl_shift_built(esize, l->vec, l->steps, l->kind) || l->waves < 1 ||
        l->waves > scanscam::cl_max_waves(l->vec, l->steps, l->kind, compute_size(dtype)))
        return false;
    return size_cl(batch, T, dtype, false, l->vec - 1, l) == SCANSCAM_OK && scanscam::cl_shift_built(esize, l->vec, l->steps, l->kind);  // (one tile: a walk)
}

// When an automatic call takes them. `reserve` is what it does without them, the cost model's plan: lanes of one channel, or
// wide ones that load and store at any element. Times of 1134 calls against that plan, buffers in rotation
// (profiles/moved_channels_random_shapes.txt): calls of 256 time steps or more that do not fit the last-level cache -- within it
// the two are level or up to 1.3 x behind --, by their (batch element, channel group) pairs:
//   A walk, a workgroup per pair, for 192 (16 bits backwards 144) to 512 of them (fp64 any number), whose groups fill 44 of 64
//   lanes. Up to 256, one per CU: 16 bits 0.76 to 0.98 forwards and 0.67 to 0.98 backwards, fp64 0.84 to 1.04 and 0.73 to 0.95,
//   fp32 backwards 0.79 to 1.05; forwards in fp32 only from 1 GiB of tensors on (0.87 to 1.03; below, where the reserve moves
//   up to 5.3 TB/s, 0.88 to 1.20, slower in three of four). From 257 to 320 a second round of workgroups is nearly empty
//   (16 bits up to 1.31 and 1.19, fp32 1.28 and 1.21, fp64 1.13; up to 384 16 bits forwards 0.76 to 1.12, fp32 0.87 to 1.04 and
//   0.85 to 1.11). Beyond, 16 bits 0.76 to 1.04 and 0.74 to 1.01, fp32 0.84 to 0.98 and 0.84 to 1.04, fp64 0.76 to 1.06 and
//   0.76 to 1.08.
//   fp32 [64, 2048, 1001] 346 / 573 -> 299 / 505 us, bf16 197 / 344 -> 158 / 263 us.
//   Tiles, for fewer. fp32 below 40 pairs, 8 steps x 8 waves: 0.70 to 1.05 forwards (with 24 pairs and more from 512 MiB on;
//   below up to 1.14), 0.68 to 1.02 backwards; up to 96 backwards, 4 x 8 where the reserve has 16 steps a wave 0.83 to 1.01 (8
//   steps, 0.88 to 1.08; forwards 0.89 to 1.29). 16 bits backwards, which is bound by its accesses more than by bytes, from 96
//   MiB on, 8 to 95 pairs: 0.57 to 1.06 (from 64 MiB on 0.71 to 1.16, with 97 to 143 pairs 0.65 to 1.23, below 8 0.74 to 1.29);
//   forwards they lose (0.92 to 1.4). fp64 has no fewer accesses per byte to gain (1.0 to 1.5).
//
// Tiles multiply the gates of their super-tiles together, waves^2 * steps of them, and a product that leaves fp32's range
// makes NaN of a scan value of zero (gates above one before the first value). They are taken only where the reserve
// multiplies as many together, in 16 bits with fewer steps where it multiplies 128 (0.70 to 1.00) and not at all where it is a
// walk, whose waves multiply 16 gates at most (tiles 0.68 to 1.25 there).
int shift_choice(int64_t batch, int64_t T, int64_t C, int esize, bool rev, const scanscam::ClLaunch &reserve)
{
    const int vec = shift_vec(esize);
    if (C % 2 == 0 || C <= (kWave - 1) * vec || T < 256) return 0;
    const int64_t bytes = batch * T * C * esize * (rev ? 5 : 3);
    const int64_t all = (C + vec - 1) / vec, groups = (all + kWave - 2) / (kWave - 1), pairs = batch * groups;
    const bool filled = all >= 44 * groups;
    const int product = reserve.kind == 2 ? reserve.waves * reserve.waves * reserve.steps : 0;
    const int64_t cache = kLastLevelCache;
    if (pairs >= (esize == 2 && rev ? 144 : 192)) {
        const int64_t least = pairs < 192 ? cache / 8 * 3 : (esize == 4 && !rev && pairs <= 256 ? 4 * cache : cache);
        const bool second_round = pairs > 256 && pairs <= (esize == 4 || (esize == 2 && !rev) ? 384 : 320);
        if (bytes <= least || !filled || second_round || (pairs > 512 && esize != 8)) return 0;
        return esize == 2 ? shift_code(rev ? 4 : 8, 8, false) : shift_code(8, 4, false);
    }
    if (esize == 2) {
        if (!rev || bytes <= cache / 8 * 3 || pairs < 8 || pairs >= 96 || (pairs >= 40 && !filled)) return 0;
        return product >= 256 ? shift_code(16, 4, true) : (product >= 128 ? shift_code(8, 4, true) : 0);
    }
    if (esize == 4 && filled && bytes > (rev ? cache / 4 * 5 : cache)) {
        if (pairs < (rev || bytes > 2 * cache ? 40 : 24)) return product >= 512 ? shift_code(8, 8, true) : 0;
        if (rev && pairs <= 96) return product >= 256 && reserve.steps >= 16 ? shift_code(4, 8, true) : 0;
    }
    return 0;
}

// The same for a call's plan: what a resolved plan says (scanscam_resolve_plan_cl writes the number's negative into
// waves_per_row), the automatic choice where the plan leaves everything open.
int shift_code_of(const scanscam_plan *plan, int64_t batch, int64_t T, int64_t C, int esize, bool rev, const scanscam::ClLaunch &reserve)
{
    if (plan && plan->waves_per_row < 0) return plan->waves_per_row > -4096 ? -plan->waves_per_row : 0;
    const bool free_plan = !plan || (plan->mode == SCANSCAM_MODE_AUTO && !plan->vec && !plan->unroll && !plan->waves && !plan->waves_per_row);
    return free_plan ? shift_choice(batch, T, C, esize, rev, reserve) : 0;
}

// The largest of 16, 8, 4 and the element size (bytes) that every base and stride of a call's tensors is a multiple of.
int cl_align(const void *const ptrs[5], const int64_t sB[5], const int64_t sT[5], int esize)
{
    int align = 16;
    for (int k = 0; k < 5; k++)
        while (align > esize && !(aligned_to(ptrs[k], (size_t)align) && (sB[k] * esize) % align == 0 && (sT[k] * esize) % align == 0))
            align >>= 1;
    return align;
}

// Whether every time step of every tensor is whole 128-byte lines.
bool cl_lines(const void *const ptrs[5], const int64_t sB[5], const int64_t sT[5], int esize)
{
    for (int k = 0; k < 5; k++)
        if ((sT[k] * esize) % 128 != 0 || !aligned_to(ptrs[k], 128) || (sB[k] * esize) % 128 != 0) return false;
    return true;
}

// Lanes of 8 bytes or less whose time steps are no whole lines write partial lines at both ends of every
// wave's store; non-temporal stores then cost 20 % of a plain copy's rate and stores left to the caches'
// normal policy nothing. Measured on the kernels: 16-bit storage 8 to 35 % faster in both directions (bf16
// [90, 2048, 514] 178 / 341 -> 139 / 298 us, [1000, 500, 130] 157 / 296 -> 120 / 202 us, [700, 300, 257] 112 / 217 ->
// 85 / 141 us; single channels backwards lose 10 %: [260, 4000, 48]), fp32 forwards and in tiles over workgroups
// 4 to 19 % ([8, 4096, 1000] 90 / 152 -> 83 / 128 us, [100, 3000, 300] forward 339 -> 276 us; a walk of all of T
// backwards loses up to 11 %); on whole lines they lose 6 to 14 %, and 16-byte lanes lose 6 to 11 % either way.
// (Element-aligned lanes of 8 bytes or less always store this way: the kernel's choice, not this flag's.)
bool cl_cached_stores(const scanscam::ClLaunch &l, bool lines, int esize, bool rev)
{
    const int lane_bytes = l.vec * esize;
    return !lines && lane_bytes <= 8 && esize <= 4 && (esize == 2 ? (lane_bytes > 2 || !rev) : (!rev || l.kind == 2));
}

int run_cl(bool rev, const void *a, const void *x, const void *h, void *y0, void *y1,
           const scanscam_strides *const st[5], int64_t batch, int64_t T, int64_t C, int dtype, void *workspace,
           size_t workspace_bytes, void *stream, const scanscam_plan *plan)
{
    const int esize = elem_size(dtype);
    if (esize == 0) return SCANSCAM_EDTYPE;
    if (batch < 0 || T < 0 || C < 0 || T >= kMaxT || C >= kMaxT) return SCANSCAM_EINVAL;
    if (batch == 0 || T == 0 || C == 0) return SCANSCAM_OK;
    if (!a || !x || !y0 || (rev && (!h || !y1))) return SCANSCAM_EINVAL;

    // Tensor order a, x, h, y0, y1; the forward pass has no h and no y1 (they alias a and y0).
    const void *ptrs[5] = {a, x, rev ? h : a, y0, rev ? y1 : y0};
    const int src[5] = {0, 1, rev ? 2 : 0, 3, rev ? 4 : 3};
    int64_t sB[5], sT[5];
    for (int k = 0; k < 5; k++) {
        const scanscam_strides *t = st[src[k]];
        sB[k] = batch == 1 ? 0 : (t ? t->outer : T * C);
        sT[k] = T == 1 ? 0 : (t ? t->row : C);
        if (sB[k] < 0 || sT[k] < 0 || sT[k] >= kMaxT) return SCANSCAM_EINVAL;
        if (!aligned_to(ptrs[k], (size_t)esize)) return SCANSCAM_EALIGN;
    }
    const int align = cl_align(ptrs, sB, sT, esize);
    const bool dense = cl_dense(batch, T, C, ptrs, sB, sT);
    auto run_staged = [&](scanscam::StagedArgs st) {
        st.a = a;
        st.x = x;
        st.h = rev ? h : a;  // never read in the forward pass
        st.y0 = y0;
        st.y1 = rev ? y1 : y0;
        // Any workspace with room for the flag word is one scanscam_workspace_timed_out may be asked about.
        if (workspace && workspace_bytes >= scanscam::kStagedHeader * sizeof(uint64_t) && aligned_to(workspace, 8))
            st.ws = static_cast<uint64_t *>(workspace);
        hipError_t e = hipErrorInvalidValue;
        hipStream_t s = static_cast<hipStream_t>(stream);
        switch (dtype) {
        case SCANSCAM_F32: e = scanscam::launch_scan_staged<float>(st, batch, rev, s); break;
        case SCANSCAM_BF16: e = scanscam::launch_scan_staged<__bf16>(st, batch, rev, s); break;
        case SCANSCAM_F16: e = scanscam::launch_scan_staged<_Float16>(st, batch, rev, s); break;
        case SCANSCAM_F64: e = scanscam::launch_scan_staged<double>(st, batch, rev, s); break;
        }
        return e == hipSuccess ? SCANSCAM_OK : SCANSCAM_ELAUNCH;
    };
    scanscam::StagedArgs staged;
    if (plan && plan->mode == kModeStaged) {
        if (plan->vec || plan->waves || plan->waves_per_row || plan->unroll < 0 || !dense ||
            !resolve_staged(batch, T, C, esize, staged_parts_of(plan, batch, T, C, esize), &staged))
            return SCANSCAM_EPLAN;
        const size_t need = staged_bytes(batch, C, esize, staged);
        if (need != 0 && (!workspace || workspace_bytes < need)) return SCANSCAM_EWORKSPACE;
        if (need != 0 && !aligned_to(workspace, 8)) return SCANSCAM_EALIGN;
        return run_staged(staged);
    }
    scanscam::ClLaunch l;
    const int rc = resolve_cl(plan, batch, T, C, dtype, align, rev, &l);
    if (rc != SCANSCAM_OK) return rc;
    // A wave addresses its steps (at most 16, and one neighbour on either side backwards) with 32-bit byte
    // offsets from its first one, the lane's channel included.
    for (int k = 0; k < 5; k++)
        if ((uint64_t)sT[k] * (uint64_t)esize * 18u + (uint64_t)C * (uint64_t)esize >= (uint64_t(1) << 32)) return SCANSCAM_EINVAL;

    const int parts = staged_parts_of(plan, batch, T, C, esize);
    const int code = parts > 0 ? 0 : shift_code_of(plan, batch, T, C, esize, rev, l);
    scanscam::ClLaunch shifted;
    if (code != 0 && dense && resolve_shift(batch, T, C, dtype, code, &shifted) &&
        (shifted.ws_bytes == 0 || (workspace && workspace_bytes >= shifted.ws_bytes && aligned_to(workspace, 8))))
        l = shifted;

    scanscam::ClArgs args;
    args.a = a;
    args.x = x;
    args.h = rev ? h : a;  // never read in the forward pass
    args.y0 = y0;
    args.y1 = rev ? y1 : y0;
    for (int k = 0; k < 5; k++) {
        args.sB[k] = sB[k];
        args.sT[k] = (int32_t)sT[k];
    }
    args.batch = batch;
    args.T = (int32_t)T;
    args.C = (int32_t)C;
    args.segments = l.segments;
    args.group = l.group;
    args.groups = l.groups;
    args.vectors = l.vectors;
    // Time steps that are not whole 128-byte lines: neighbouring channel groups on one XCD (see the kernel).
    const bool lines = cl_lines(ptrs, sB, sT, esize);
    args.xcd_order = (!lines && l.grid >= 64) ? 1 : 0;
    // Tiles over workgroups: a (batch element, channel group) pair keeps its XCD over all its tiles when their number
    // is a multiple of 8. Otherwise, from 128 pairs on, the XCDs take runs of n / 8 rounded up or down and the grid is
    // padded to 8 equal shares; the workgroups of a short run's last share return at once. (fp32 [9, 5318, 2059], 297
    // pairs dealt round-robin over the XCDs tile by tile: 401 / 706 us.)
    if (args.xcd_order && l.kind == 2) {
        const int64_t pairs = l.grid / l.segments;
        if (pairs % 8 != 0 && pairs >= 128) {
            args.xcd_order = 2;
            l.grid = 8 * ((pairs + 7) / 8) * l.segments;
            if (l.grid >= (int64_t(1) << 31)) return SCANSCAM_EINVAL;
        }
    }
    args.cached_stores = cl_cached_stores(l, lines, esize, rev) ? 1 : 0;
    // Loads through the caches' normal policy in element-aligned 8-byte lanes of fp32, once the call does not fit the
    // last-level cache. Against non-temporal ones, buffers in rotation (profiles/element_aligned_loads_random_shapes.txt): 64
    // calls beyond it 0.87 to 1.02 x, 0.94 x in the mean ([16, 4096, 1999] forwards 340 -> 298 us, [256, 500, 513] backwards
    // 296 -> 267 us), 97 calls within it 0.91 to 1.21 x, 1.03 x in the mean ([39, 32, 1823] 7.6 / 11.8 -> 9.2 / 13.8 us, [238,
    // 32, 733] 14.2 / 24.0 -> 16.1 / 26.3 us).
    args.cached_loads = (rev ? 5 : 3) * batch * T * C * esize > kLastLevelCache ? 1 : 0;
    args.ws = nullptr;
    args.spin_limit = (plan && plan->spin_limit > 0) ? plan->spin_limit : scanscam::kSpinLimit;

    hipStream_t s = static_cast<hipStream_t>(stream);
    if (l.kind != 0) {
        if (!workspace || workspace_bytes < l.ws_bytes) return SCANSCAM_EWORKSPACE;
        if (!aligned_to(workspace, 8)) return SCANSCAM_EALIGN;
    }
    if (parts > 0 && dense && resolve_staged(batch, T, C, esize, parts, &staged)) {
        const size_t need = staged_bytes(batch, C, esize, staged);
        if (need == 0 || (workspace && workspace_bytes >= need && aligned_to(workspace, 8))) {
                return run_staged(staged);
        }
    }
    if (l.kind != 0) {
        args.ws = static_cast<uint64_t *>(workspace);
        const int64_t words = (int64_t)(l.ws_bytes / sizeof(uint64_t));
        const int64_t rowgroups = batch * l.groups;
        if (clear_workspace(args.ws, words, rowgroups * kCounterStride, s) != hipSuccess) return SCANSCAM_ELAUNCH;
    }
    l.lds_bytes += idle_lds(l, T, esize, rev);
    l.pipe = pipe_walk(l, T, C, esize, rev, sT, args.cached_stores != 0);
    hipError_t e = hipErrorInvalidValue;
    switch (dtype) {
    case SCANSCAM_F32: e = scanscam::launch_scan_cl<float>(args, l, rev, s); break;
    case SCANSCAM_BF16: e = scanscam::launch_scan_cl<__bf16>(args, l, rev, s); break;
    case SCANSCAM_F16: e = scanscam::launch_scan_cl<_Float16>(args, l, rev, s); break;
    case SCANSCAM_F64: e = scanscam::launch_scan_cl<double>(args, l, rev, s); break;
    }
    return e == hipSuccess ? SCANSCAM_OK : SCANSCAM_ELAUNCH;
}

size_t workspace_for(int64_t rows, int64_t T, int dtype, int direction, const scanscam_plan *plan)
{
    // The caller's pointers are not known yet: cover both the 16-byte aligned
    // and the unaligned choice.
    size_t need = 0;
    for (int al = 0; al < 3; al++) {  // element-aligned, 16-byte aligned, 128-byte aligned rows
        Resolved r;
        if (resolve(plan, rows, T, dtype, al >= 1, al == 2, direction == SCANSCAM_BACKWARD, &r) == SCANSCAM_OK &&
            r.ws_bytes > need)
            need = r.ws_bytes;
    }
    return need;
}

}  // namespace

extern "C" {

int scanscam_scan_fwd(const void *a, const void *b, void *h, int64_t rows, int64_t T, int dtype,
                      void *workspace, size_t workspace_bytes, void *stream)
{
    return run(false, a, b, nullptr, h, nullptr, kDense, 1, rows, T, dtype, workspace, workspace_bytes, stream, nullptr);
}

int scanscam_scan_bwd(const void *a, const void *h, const void *gh, void *ga, void *gb, int64_t rows,
                      int64_t T, int dtype, void *workspace, size_t workspace_bytes, void *stream)
{
    return run(true, a, gh, h, gb, ga, kDense, 1, rows, T, dtype, workspace, workspace_bytes, stream, nullptr);
}

int scanscam_scan_fwd_noalloc(const void *a, const void *b, void *h, int64_t rows, int64_t T, int dtype, void *stream)
{
    return run(false, a, b, nullptr, h, nullptr, kDense, 1, rows, T, dtype, nullptr, 0, stream, nullptr, nullptr, nullptr,
               /*use_scratch=*/true);
}

size_t scanscam_workspace_bytes(int64_t rows, int64_t T, int dtype, int direction)
{
    return workspace_for(rows, T, dtype, direction, nullptr);
}

int scanscam_scan_fwd_plan(const void *a, const void *b, void *h, int64_t rows, int64_t T, int dtype,
                           void *workspace, size_t workspace_bytes, void *stream, const scanscam_plan *plan)
{
    return run(false, a, b, nullptr, h, nullptr, kDense, 1, rows, T, dtype, workspace, workspace_bytes, stream, plan);
}

int scanscam_scan_bwd_plan(const void *a, const void *h, const void *gh, void *ga, void *gb, int64_t rows,
                           int64_t T, int dtype, void *workspace, size_t workspace_bytes, void *stream,
                           const scanscam_plan *plan)
{
    return run(true, a, gh, h, gb, ga, kDense, 1, rows, T, dtype, workspace, workspace_bytes, stream, plan);
}

size_t scanscam_workspace_bytes_plan(int64_t rows, int64_t T, int dtype, int direction,
                                     const scanscam_plan *plan)
{
    return workspace_for(rows, T, dtype, direction, plan);
}

int scanscam_scan_fwd_timed(const void *a, const void *b, void *h, int64_t rows, int64_t T, int dtype,
                            void *workspace, size_t workspace_bytes, void *stream, const scanscam_plan *plan,
                            void *start_event, void *stop_event)
{
    return run(false, a, b, nullptr, h, nullptr, kDense, 1, rows, T, dtype, workspace, workspace_bytes, stream, plan,
               start_event, stop_event);
}

int scanscam_scan_bwd_timed(const void *a, const void *h, const void *gh, void *ga, void *gb, int64_t rows,
                            int64_t T, int dtype, void *workspace, size_t workspace_bytes, void *stream,
                            const scanscam_plan *plan, void *start_event, void *stop_event)
{
    return run(true, a, gh, h, gb, ga, kDense, 1, rows, T, dtype, workspace, workspace_bytes, stream, plan, start_event,
               stop_event);
}

int scanscam_scan_fwd_cl(const void *a, const void *b, void *h, int64_t batch, int64_t T, int64_t C, int dtype,
                         void *workspace, size_t workspace_bytes, void *stream, const scanscam_plan *plan)
{
    return run_cl(false, a, b, nullptr, h, nullptr, kDense, batch, T, C, dtype, workspace, workspace_bytes, stream, plan);
}

int scanscam_scan_bwd_cl(const void *a, const void *h, const void *gh, void *ga, void *gb, int64_t batch,
                         int64_t T, int64_t C, int dtype, void *workspace, size_t workspace_bytes, void *stream,
                         const scanscam_plan *plan)
{
    return run_cl(true, a, gh, h, gb, ga, kDense, batch, T, C, dtype, workspace, workspace_bytes, stream, plan);
}

size_t scanscam_workspace_bytes_cl(int64_t batch, int64_t T, int64_t C, int dtype, int direction,
                                   const scanscam_plan *plan)
{
    const int esize = elem_size(dtype);
    if (esize == 0 || batch <= 0 || T <= 0 || C <= 0 || T >= kMaxT || C >= kMaxT) return 0;
    size_t need = 0;
    const int parts = staged_parts_of(plan, batch, T, C, esize);
    scanscam::StagedArgs st;
    if (parts > 1 && resolve_staged(batch, T, C, esize, parts, &st)) need = staged_bytes(batch, C, esize, st);
    if (plan && plan->mode == kModeStaged) return need;
    // The caller's pointers are not known yet: every alignment the tensors may turn out to have.
    const bool rev = direction == SCANSCAM_BACKWARD;
    for (int align = 16; align >= esize; align >>= 1) {
        scanscam::ClLaunch l, shifted;
        if (resolve_cl(plan, batch, T, C, dtype, align, rev, &l) != SCANSCAM_OK) continue;
        if (l.ws_bytes > need) need = l.ws_bytes;
        const int code = align == esize && parts == 0 ? shift_code_of(plan, batch, T, C, esize, rev, l) : 0;  // (odd channel counts)
        if (code != 0 && resolve_shift(batch, T, C, dtype, code, &shifted) && shifted.ws_bytes > need) need = shifted.ws_bytes;
    }
    return need;
}

int scanscam_scan_fwd_strided(const void *a, const void *b, void *h, const scanscam_strides *sa,
                              const scanscam_strides *sb, const scanscam_strides *sh, int64_t n0, int64_t n1,
                              int64_t T, int dtype, void *workspace, size_t workspace_bytes, void *stream,
                              const scanscam_plan *plan)
{
    const scanscam_strides *const st[5] = {sa, sb, nullptr, sh, nullptr};
    return run(false, a, b, nullptr, h, nullptr, st, n0, n1, T, dtype, workspace, workspace_bytes, stream, plan);
}

int scanscam_scan_bwd_strided(const void *a, const void *h, const void *gh, void *ga, void *gb,
                              const scanscam_strides *sa, const scanscam_strides *sh, const scanscam_strides *sgh,
                              const scanscam_strides *sga, const scanscam_strides *sgb, int64_t n0, int64_t n1,
                              int64_t T, int dtype, void *workspace, size_t workspace_bytes, void *stream,
                              const scanscam_plan *plan)
{
    const scanscam_strides *const st[5] = {sa, sgh, sh, sgb, sga};
    return run(true, a, gh, h, gb, ga, st, n0, n1, T, dtype, workspace, workspace_bytes, stream, plan);
}

int scanscam_scan_fwd_cl_strided(const void *a, const void *b, void *h, const scanscam_strides *sa,
                                 const scanscam_strides *sb, const scanscam_strides *sh, int64_t batch, int64_t T,
                                 int64_t C, int dtype, void *workspace, size_t workspace_bytes, void *stream,
                                 const scanscam_plan *plan)
{
    const scanscam_strides *const st[5] = {sa, sb, nullptr, sh, nullptr};
    return run_cl(false, a, b, nullptr, h, nullptr, st, batch, T, C, dtype, workspace, workspace_bytes, stream, plan);
}

int scanscam_scan_bwd_cl_strided(const void *a, const void *h, const void *gh, void *ga, void *gb,
                                 const scanscam_strides *sa, const scanscam_strides *sh,
                                 const scanscam_strides *sgh, const scanscam_strides *sga,
                                 const scanscam_strides *sgb, int64_t batch, int64_t T, int64_t C, int dtype,
                                 void *workspace, size_t workspace_bytes, void *stream, const scanscam_plan *plan)
{
    const scanscam_strides *const st[5] = {sa, sgh, sh, sgb, sga};
    return run_cl(true, a, gh, h, gb, ga, st, batch, T, C, dtype, workspace, workspace_bytes, stream, plan);
}

int scanscam_workspace_timed_out(const void *workspace, void *stream, int *timed_out)
{
    if (!workspace || !timed_out) return SCANSCAM_EINVAL;
    if (!aligned_to(workspace, 8)) return SCANSCAM_EALIGN;
    uint64_t word = 0;
    if (hipStreamSynchronize(static_cast<hipStream_t>(stream)) != hipSuccess) return SCANSCAM_ELAUNCH;
    if (hipMemcpy(&word, static_cast<const uint64_t *>(workspace) + scanscam::kTimeoutWord, sizeof(word),
                  hipMemcpyDeviceToHost) != hipSuccess)
        return SCANSCAM_ELAUNCH;
    *timed_out = word != 0 ? 1 : 0;
    return SCANSCAM_OK;
}

int scanscam_noalloc_timed_out(void *stream, int *timed_out)
{
    if (!timed_out) return SCANSCAM_EINVAL;
    void *ws = nullptr;
    const int rc = noalloc_scratch(&ws);
    if (rc != SCANSCAM_OK) return rc;
    return scanscam_workspace_timed_out(ws, stream, timed_out);
}

int scanscam_resolve_plan(int64_t rows, int64_t T, int dtype, int direction, const scanscam_plan *plan,
                          scanscam_plan *out)
{
    if (!out) return SCANSCAM_EINVAL;
    Resolved r;
    // Dense tensors on allocation borders: rows start on line borders exactly when a row is whole lines.
    const int esize = elem_size(dtype);
    const bool lines = esize != 0 && (T * esize) % 128 == 0;
    const int rc = resolve(plan, rows, T, dtype, true, lines, direction == SCANSCAM_BACKWARD, &r, /*flat_ok=*/true);
    if (rc != SCANSCAM_OK) return rc;
    out->mode = r.l.mode;
    out->vec = r.l.vec;
    out->unroll = r.l.unroll;
    out->waves = r.l.waves;
    out->waves_per_row = r.l.mode == kModeRow ? r.l.wpr : 0;
    out->spin_limit = (plan && plan->spin_limit > 0) ? plan->spin_limit : scanscam::kSpinLimit;
    return SCANSCAM_OK;
}

int scanscam_resolve_plan_cl(int64_t batch, int64_t T, int64_t C, int dtype, int direction,
                             const scanscam_plan *plan, scanscam_plan *out)
{
    if (!out) return SCANSCAM_EINVAL;
    const int esize = elem_size(dtype);
    if (esize == 0) return SCANSCAM_EDTYPE;
    if (batch <= 0 || T <= 0 || C <= 0 || T >= kMaxT || C >= kMaxT) return SCANSCAM_EINVAL;
    // Dense tensors on allocation borders: every time step starts on the largest power of two that divides C elements.
    int align = 16;
    while (align > esize && !(batch == 1 && T == 1) && (C * esize) % align != 0) align >>= 1;
    scanscam::ClLaunch l;
    const int rc = resolve_cl(plan, batch, T, C, dtype, align, direction == SCANSCAM_BACKWARD, &l);
    if (rc != SCANSCAM_OK) return rc;
    const int parts = staged_parts_of(plan, batch, T, C, esize);  // (`out` may be the plan itself)
    const int code = parts > 0 ? 0 : shift_code_of(plan, batch, T, C, esize, direction == SCANSCAM_BACKWARD, l);
    scanscam::StagedArgs st;
    out->mode = l.kind == 2 ? kModeLookback : kModeRow;
    out->vec = l.vec;
    out->unroll = l.steps;
    out->waves = l.waves;
    out->waves_per_row = parts > 0 && resolve_staged(batch, T, C, esize, parts, &st) ? st.parts : 0;
    if (code != 0 && resolve_shift(batch, T, C, dtype, code, &l)) out->waves_per_row = -code;
    out->spin_limit = (plan && plan->spin_limit > 0) ? plan->spin_limit : scanscam::kSpinLimit;
    return SCANSCAM_OK;
}

int scanscam_predict_cl(int64_t batch, int64_t T, int64_t C, int dtype, int direction, const scanscam_plan *plan,
                        double *microseconds)
{
    if (!microseconds) return SCANSCAM_EINVAL;
    const int esize = elem_size(dtype);
    if (esize == 0) return SCANSCAM_EDTYPE;
    if (batch <= 0 || T <= 0 || C <= 0 || T >= kMaxT || C >= kMaxT) return SCANSCAM_EINVAL;
    int align = 16;
    while (align > esize && !(batch == 1 && T == 1) && (C * esize) % align != 0) align >>= 1;
    scanscam::ClLaunch l;
    return resolve_cl(plan, batch, T, C, dtype, align, direction == SCANSCAM_BACKWARD, &l, microseconds);
}

// For tests and measurements, not part of the interface in scanscam_hip.h: whether a call walks with its loads a tile ahead, past its
// stores (1 or 0; below zero: the negative of an error code). Tensors in the order a, x, h, y0, y1 (forwards h is a and y1 is y0),
// bases on 128-byte borders, `sB` and `sT` their strides in elements (NULL: dense). Launches nothing.
int scanscam_internal_walks_ahead(int64_t batch, int64_t T, int64_t C, int dtype, int direction, const int64_t *sB, const int64_t *sT,
                                  const scanscam_plan *plan)
{
    const int esize = elem_size(dtype);
    if (esize == 0) return -SCANSCAM_EDTYPE;
    if (batch <= 0 || T <= 0 || C <= 0 || T >= kMaxT || C >= kMaxT) return -SCANSCAM_EINVAL;
    const bool rev = direction == SCANSCAM_BACKWARD;
    const void *const ptrs[5] = {};
    int64_t b[5], t[5];
    for (int k = 0; k < 5; k++) {
        b[k] = batch == 1 ? 0 : (sB ? sB[k] : T * C);
        t[k] = T == 1 ? 0 : (sT ? sT[k] : C);
        if (b[k] < 0 || t[k] < 0 || t[k] >= kMaxT) return -SCANSCAM_EINVAL;
    }
    scanscam::ClLaunch l, shifted;
    const int rc = resolve_cl(plan, batch, T, C, dtype, cl_align(ptrs, b, t, esize), rev, &l);
    if (rc != SCANSCAM_OK) return -rc;
    const bool dense = cl_dense(batch, T, C, ptrs, b, t);
    const int parts = staged_parts_of(plan, batch, T, C, esize), code = parts > 0 ? 0 : shift_code_of(plan, batch, T, C, esize, rev, l);
    scanscam::StagedArgs staged;
    if (dense && ((code != 0 && resolve_shift(batch, T, C, dtype, code, &shifted)) ||
                  (parts > 0 && resolve_staged(batch, T, C, esize, parts, &staged))))
        return 0;
    return pipe_walk(l, T, C, esize, rev, t, cl_cached_stores(l, cl_lines(ptrs, b, t, esize), esize, rev)) ? 1 : 0;
}

const char *scanscam_strerror(int code)
{
    switch (code) {
    case SCANSCAM_OK: return "ok";
    case SCANSCAM_EINVAL: return "invalid argument (null pointer, negative or too large size)";
    case SCANSCAM_EDTYPE: return "unsupported storage type";
    case SCANSCAM_EALIGN: return "pointer not aligned to its element size (or workspace not to 8 bytes)";
    case SCANSCAM_EPLAN: return "launch plan not valid for this shape or alignment";
    case SCANSCAM_EWORKSPACE: return "workspace missing or smaller than scanscam_workspace_bytes()";
    case SCANSCAM_ELAUNCH: return "HIP runtime refused the kernel launch";
    case SCANSCAM_ESCRATCH:
        return "shape needs more look-back scratch than the library's fixed array (scanscam_scan_fwd_noalloc): "
               "use scanscam_scan_fwd with a workspace";
    default: return "unknown scanscam error code";
    }
}

int scanscam_abi_version(void) { return 3; }

}  // extern "C"
