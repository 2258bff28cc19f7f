// kg_internal.h -- arguments of the step kernels and the host-side launchers
// shared by kg_step.hip (device code) and kg_api.hip (the C ABI).
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include <vector>

namespace kg {

// Everything one explicit-Euler step needs, with the reference's scalar
// parameters pre-combined in the field's precision R the way the reference
// combines them (src/Kobayashi.cpp:139-215):
//   gx = (phiE - phiW) / dx            -> (phiE - phiW) * inv_dx
//   lap = (...) / (3 dx dx)            -> (...) * inv_3dx2
//   eps' = ((-eps_bar) j) delta sin()  -> neg_ebar_j_delta * sin()
//   m = alpha / pi * atan(...)         -> alpha_pi * atan(...)
//   phi' = phi + (...) dt / tau        -> phi + (...) * dt_tau
template <typename R>
struct StepArgs {
    const R *phi_in;
    const R *T_in;
    R *phi_out;
    R *T_out;
    R *theta;        // persistent angle, updated in place where a branch fires
    // old angles in another buffer, all of theta is then written: small tiles
    // (nullptr: in theta itself) and k_step_batch_direct
    const R *theta_in;
    int nx, ny;
    int boundary;    // 0 periodic, 1 zero-flux
    int ntiles;      // tiles of the grid
    R inv_dx, inv_dy, inv_3dx2, dt, dt_tau;
    R eps_bar, delta, aniso, theta0, neg_ebar_j_delta;
    R alpha_pi, gamma, teq, K, noise_a;
    uint32_t step, instance, key0, key1;
    // 1 when |aniso (theta - theta0)| may exceed the reduced sin/cos range
    // for some stored angle (the host tracks a bound on |theta|)
    int wide_angles;
    // 1: the step's output stores carry the non-temporal hint (set for
    // grids whose per-step working set exceeds the last-level cache: the
    // outputs are not read again within the launch, and without the hint
    // they evict the input lines neighbouring tiles still read as halos)
    int stream_out;
    // Tile status words of the fused kernel (one per 64 x 30 tile, bits in
    // kg_step.hip): stat_in describes the input buffers, stat_out the output
    // buffers; the word of the tile at (x0, y0) sits at tile_base +
    // (y0 / 30) * tiles_x + x0 / 64.  stat_in == nullptr: no status (every
    // tile loads and stores all of its fields).
    const uint32_t *stat_in;
    uint32_t *stat_out;
    int tile_base, tiles_x, tiles_y;
};

// Two-pass variant: pass-1 temporaries in global memory, as the reference's
// member arrays (src/Kobayashi.h:109-114).
template <typename R>
struct PassTemps {
    R *gx, *gy, *lap, *lapT, *eps, *epsd;
};

struct ReduceOut {
    double sum_phi, sum_T, sum_T_minus_K_phi, min_phi, max_phi, above_half;
    double nonfinite;
};

// The chunks of 2 x 4 tiles that one launch of the fused step works on,
// when not all: n chunk indices (row-major chunk order, c = cy * chunks_x +
// cx) in the order the launch deals them to the XCDs.  Every chunk left out
// holds phi = +0 and T = +0 on both buffers and keeps them over the launch,
// and its status words already say so (the host derives the list from
// a liveness request; kg_api.hip states the conditions).  Up to LIVE_MAX
// entries travel by value in the kernel arguments; a longer list is copied
// to device memory first and `dev` points at it (the same 16-bit entries).
// Either way the launch has only the listed chunks' blocks.
constexpr int LIVE_MAX = 1020;
struct LiveList {
    int n;
    int busy;                         // leading entries that are busy chunks (busy_chunk)
    const uint32_t *dev;              // n > LIVE_MAX: the entries, in device memory
    alignas(4) uint16_t c[LIVE_MAX];  // read by the kernel as 32-bit words
};
static_assert(LIVE_MAX % 2 == 0, "LiveList entries are read in pairs");
// A liveness request carried by a step launch: leading blocks of the launch
// write one flag byte per chunk to `flags` (pinned host memory, one byte per
// chunk, each written with a system-scope store):
//   tag << 5 | na << 1 | lv,
// lv = 1 if some tile within SKIP_MARGIN_X tile columns and SKIP_MARGIN_Y
// tile rows of the chunk (mapped by the boundary) has an input status word
// other than exactly "phi = +0, T = +0"; na = tiles of the chunk whose last
// step took the full path; tag in 1..LIVE_TAGS.  `blocks` is set by
// launch_step_fused.
struct LiveReq {
    uint8_t *flags;
    uint32_t tag;
    int blocks;
};
constexpr uint32_t LIVE_TAGS = 7;
// live == nullptr or live->n < 0: every chunk; req != nullptr (and the tile
// status on): the launch also answers a liveness request
template <typename R>
hipError_t launch_step_fused(const StepArgs<R> &a, hipStream_t s, const LiveList *live = nullptr,
                             const LiveReq *req = nullptr);
// Whether a chunk of `area` tiles, `na` of which took the full path when it
// was last asked about, is stepped as a busy one: its tiles load phi, T and
// theta at once, in one round trip, instead of asking their status words
// first, and claim nothing in the words they write.  All tiles of the chunk:
// 4096 x 4096 FP32 with 200 and 800 nuclei 75.7 -> 74.2 and 93.9 -> 90.5 us per
// step, 30 members of 128^2 .. 768^2 18.7 -> 18.3; from 3/4 of them the same
// within 0.5 %, from half of them the members 18.8.
__host__ __device__ inline int busy_chunk(int na, int area) { return na == area ? 1 : 0; }
// Append to out the chunks flagged live in flags[c] (one byte per chunk, as
// a LiveReq writes it), in the order a LiveList must hold them: by
// their count of active tiles, most first (a launch then ends on cheap
// tiles), the full launch's chunk order within one count.  False, with out
// incomplete, if some byte does not carry `tag` (not yet written by the
// request that tag names).
bool live_chunk_order(int nx, int ny, const uint8_t *flags, uint32_t tag,
                      std::vector<uint16_t> &out, int &busy);
// Liveness request over the chunks of a batch: flags[c] as a LiveReq writes
// them, for chunk c = (member, chunk column, chunk row) of chunks, from the
// status set stat_set (the input set of the next step).
// Chunks are cw x ch tiles, a shape of batch_chunk_shapes (else
// hipErrorInvalidValue).
template <typename R>
hipError_t launch_batch_live(const StepArgs<R> *members, const int4 *chunks, int nchunks,
                             const uint32_t *stat_set, uint32_t tag, uint8_t *flags, int cw,
                             int ch, hipStream_t s);
// Chunk grid of the fused step for an nx x ny grid (chunks_x * chunks_y chunks).
int fused_chunks_x(int nx);
int fused_chunks_y(int ny);
// Tile rows/columns of margin around a chunk that a liveness request checks,
// and the period (steps) of the host's requests.
constexpr int SKIP_MARGIN_X = 1, SKIP_MARGIN_Y = 1;  // tile columns, tile rows
constexpr int SKIP_PERIOD = 7;
// periods between a liveness request and the first launch that uses it
constexpr int SKIP_AGE = 1;
// grids with fewer chunks launch every chunk: a chunk list saves them at
// most about a microsecond per step, while its waits keep the host within
// two periods of the GPU, so handles stepped in turn would stop overlapping
// on the GPU (256 chunks of 2 x 4 tiles: about 2000 x 2000 cells)
constexpr int SKIP_MIN_CHUNKS = 256;
template <typename R>
hipError_t launch_step_two_pass(const StepArgs<R> &a, const PassTemps<R> &t, hipStream_t s);

// Bytes to allocate for a field of `bytes`: whole 16-byte words, so that
// fields can be cleared with 16-byte stores.
constexpr size_t padded_bytes(size_t bytes) { return (bytes + 15) / 16 * 16; }
// A disk of phi = 1 (the reference's 5-cell plus is the disk with r2 = 1); off:
// element offset of its grid in phi.
struct DiskEntry {
    size_t off;
    int nx, ny, cx, cy;
};
// Centres of disks that travel with a launch.
struct FewDisks {
    static constexpr int MAX = 8;
    int n;
    int cx[MAX], cy[MAX];
};
// All fields zero (n elements each, allocated with padded_bytes) but for phi on
// the disks of squared radius r2 in the nx x ny grid at phi.
template <typename R>
hipError_t launch_reset(R *phi, R *T, R *theta, size_t n, int nx, int ny, const FewDisks &disks,
                        double r2, hipStream_t s);
// phi = 1 on `count` disks of squared radius r2 (a list in device memory).
template <typename R>
hipError_t launch_disks(R *phi, const DiskEntry *disks, int count, double r2, hipStream_t s);

// Deterministic FP64 reduction; `partials` holds reduce_partials_size()
// doubles, `out` one ReduceOut (both device memory).
size_t reduce_partials_size();
template <typename R>
hipError_t launch_reduce(const R *phi, const R *T, size_t n, double K, double *partials,
                         ReduceOut *out, hipStream_t s);

// Largest |v| (NaN: infinity) of n values, 16-byte aligned, as MAX_ABS_BLOCKS
// partial maxima in out (device memory; not more than reduce_partials_size()).
constexpr int MAX_ABS_BLOCKS = 512;
template <typename R>
hipError_t launch_max_abs(const R *v, size_t n, double *out, hipStream_t s);

// phi -> colour ramp: 4 floats per cell (rgba8 false) or 4 bytes (true)
template <typename R>
hipError_t launch_colormap(const R *phi, int nx, int ny, int order, void *rgba, bool rgba8,
                           hipStream_t s);

// Front distances along n rays from (cx, cy) to phi = level (FP64 results,
// `radii` device memory of n doubles).
template <typename R>
hipError_t launch_front_profile(const R *phi, int nx, int ny, double cx, double cy, int n,
                                double level, double *radii, hipStream_t s);

// Tile of block b where STRIP tiles that follow one another go to one XCD
// (blocks go round-robin over the 8), so that neighbours' halos meet in its L2
// while a front's tiles still spread over all of them; strip_blocks(n) blocks
// cover n tiles (the last ones get none).  Against tiles dealt one by one, us
// per step, single grids with one nucleus per 60000 cells, strips of 8 / 16 / 32:
// FP32 300^2 2.7 -> 2.6 / 2.5 / 2.4, 448^2 4.4 -> 4.0 / 4.1 / 4.0, 600^2 6.0 ->
// 5.5 (16), FP64 420^2 7.3 -> 6.8 / 6.8 / 6.9, 800^2 12.8 -> 12.0 / 12.0 / 12.2,
// 1536 x 1200 24.8 -> 24.4 (16; 17.1 -> 14.7 with one nucleus); 32 loses on 384^2
// with many nuclei (4.0 -> 4.1 (16) / 4.5).  Rows of tiles or blocks of 4 x 4 and
// 2 x 8 tiles came out alike, wider ones slower.  The adjoint of 512^2 FP32,
// whose front sat in one or two contiguous eighths: 3346 -> 3173, of 24
// members 6990 -> 6732.
constexpr unsigned STRIP = 16, STRIP_XCDS = 8;
__host__ __device__ inline unsigned strip_tile(unsigned b)
{
    const unsigned i = b / STRIP_XCDS;
    return (i / STRIP * STRIP_XCDS + b % STRIP_XCDS) * STRIP + i % STRIP;
}
inline unsigned strip_blocks(size_t n)
{
    return (unsigned)((n + STRIP * STRIP_XCDS - 1) / (STRIP * STRIP_XCDS) * (STRIP * STRIP_XCDS));
}

// Shape of the small tiles a grid without tile status is stepped in, 0 = none
// (the 64 x 30 tiles; only those keep a status).
int small_shape(long long nx, long long ny, size_t esize);
// Launches of MULTI_STEPS steps on small grids: their shape (0: single steps
// only), and the launch -- phi and T from in to out, theta from theta_in to
// theta; with stride != 0 every step's state, stride elements apart.
constexpr int MULTI_STEPS = 3;
// Their shape from the cells and the number of tiles blocks(rows) of 32 x rows
// cells: 8 = 32 x 8 on 768 threads; 12 .. 32 = 32 x that on 1024 threads;
// MULTI_HALF + rows = on 512 threads; (batches) MULTI_ONE + rows = one step,
// MULTI_768 + rows = on 768 threads.
// Tall tiles have less halo (2.1 pass-1 cells per cell and step at 8 rows, 1.4
// at 32) but few blocks, so: the least tile of which two per CU, all that 1024
// threads leave room for, hold the whole grid, and where none does, 512 threads,
// four per CU.  us per step of FP32 grids, one nucleus per 30000 cells, 8 rows /
// 16 on 768 threads / the rows of this rule: 360^2 3.24 / - / -, 400^2 4.2 / 4.2
// / 3.6 (12), 512^2 5.4 / 4.35 / 4.26 (16), 570^2 5.8 / 5.0 / 4.7 (20), 600^2 6.9
// / 6.3 / 5.3 (24), 660^2 8.1 / 7.0 / 5.8 (28), 720^2 9.1 / 7.5 / 6.4 (32), 800^2
// 10.8 / 9.0 / 8.2 (20 on 512), 1030 x 771 - / - / 8.0 (8 rows on 256 threads
// 8.4), 1449 x 1447 - / 16.8 / 14.9 (32 on 512; 20 on 512 15.5).  A few tiles over
// two per CU cost little (532 at 448^2: 3.7 against 4.1 with 16 rows), 540 at
// 630^2 do (24 rows 6.8, 28 rows 5.7).  FP64 cells cost more, so there only
// where a single step does not fill the chip: 12 rows up to two tiles per CU
// (384^2 6.7 -> 5.6, 448^2 7.0 -> 6.4; 600^2 with 16 rows 8.4 -> 9.4).
// Two steps a launch gave 3.1 at 250^2 where three gave 2.4, four 2.6.
constexpr int MULTI_HALF = 100, MULTI_768 = 200, MULTI_ONE = 300;
template <typename B>
inline int multi_pick(size_t cells, size_t esize, B blocks)
{
    constexpr long long CUS = 256, PAIRS = 2 * CUS + CUS / 10;
    if (cells <= (size_t)1 << 17)
        return 8;
    for (int rows = 12; rows <= (esize == 8 ? 12 : 32); rows += 4)
        if (blocks(rows) <= PAIRS)
            return rows;
    if (esize == 8)
        return 0;
    return MULTI_HALF + (cells <= (size_t)3 << 19 ? 20 : 32);
}
int multi_shape(long long nx, long long ny, size_t esize);
template <typename R>
hipError_t launch_step_multi(const StepArgs<R> &a, size_t stride, hipStream_t s);
// The same over a batch's members, in tiles of multi_tile_x x multi_tile_y(shape)
// cells (tiles[b] = member, x0, y0; member < 0: padding), between fields whose
// members start at off[m].
template <typename R>
struct MultiIO {
    const R *phi_in, *T_in, *theta_in;
    R *phi_out, *T_out, *theta_out;
};
int multi_tile_x();
int multi_tile_y(int shape);
int multi_shape_steps(int shape);  // steps a launch of that shape takes
template <typename R>
hipError_t launch_batch_multi(int shape, const StepArgs<R> *members, const size_t *off,
                              const int4 *tiles, int ntiles, const MultiIO<R> &io, uint32_t step,
                              size_t stride, hipStream_t s);
// Number of 64 x 30 tiles of the fused kernel on an nx x ny grid.
int fused_tiles(int nx, int ny);
// Tile status can be kept for an nx x ny grid with this boundary (every halo
// of a tile lies in its 3 x 3 tile neighbourhood); fill `n` words with v.
bool fused_status_ok(int nx, int ny, int boundary);
hipError_t launch_fill_u32(uint32_t *p, size_t n, uint32_t v, hipStream_t s);
// Output tile size of the fused kernel (members of a batch are cut into it).
int fused_tile_x();
int fused_tile_y();
// Chunk shape of the fused step's chunk lists (tiles) and the rotation of
// successive chunk rows; a batch cuts its members into chunks of one of the
// batch_chunk_shapes (writes up to cap (width, height) pairs, returns how
// many there are), batch_chunk_w x batch_chunk_h unless it chooses another,
// and its liveness requests check the same chunks.
int fused_chunk_w();
int fused_chunk_h();
int fused_chunk_skew();
int batch_chunk_w();
int batch_chunk_h();
int batch_chunk_shapes(int (*out)[2], int cap);

// A batch's chunk lists kept on the device: its chunks (member, chunk
// column, chunk row) of cw x ch tiles, two flag buffers of nchunks bytes,
// the listed table (listed_cap entries), its length (-1: the full table),
// a count of the lists made, and the tile status sets (stat_tiles words
// each).
struct DeviceLists {
    const int4 *chunks;
    int nchunks, cw, ch;
    uint8_t *flags2;
    int4 *listed;
    int listed_cap;
    int *count;
    uint32_t *periods;
    const uint32_t *stat;
    int stat_tiles;
};
// Batched step over a tile table (member, x0, y0); the step counter is
// *step_base + step_add and its parity picks the ping-pong direction.  bcm:
// the boundary every member has (0, 1), or 2 when they differ.  With dl,
// the launch is preceded by the device lists' list and request kernels
// (both return at once except at multiples of SKIP_PERIOD) and uses the
// listed table when there is one.
template <typename R>
hipError_t launch_step_batch(const StepArgs<R> *members, const int4 *tiles, int ntiles,
                             const uint32_t *step_base, uint32_t step_add, int bcm, hipStream_t s,
                             const DeviceLists *dl = nullptr);
// One grid of a (possibly batched) adjoint: its step parameters and the
// element offset of its fields in every buffer.
template <typename R>
struct AdjMember {
    StepArgs<R> a;
    size_t off;
};
// Batched step between given buffers (theta too: theta_in to theta) at an
// absolute step count.
template <typename R>
hipError_t launch_step_batch_direct(const AdjMember<R> *members, const int4 *tiles, int ntiles,
                                    const R *phi_in, const R *T_in, const R *theta_in, R *phi_out,
                                    R *T_out, R *theta, uint32_t step, hipStream_t s);
hipError_t launch_advance(uint32_t *step_base, uint32_t n, hipStream_t s);

}  // namespace kg
