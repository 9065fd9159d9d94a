// The projections on either side of the absorbed MLA decode, completing the
// decode step of an MLA attention block (reference README.md:76-85, 104-110):
//
//   before:  Q*[b, h, :512] = q_nope[b, h, :] W_UK[h]        (absorbed key up-projection)
//            Q*[b, h, 512:] = q_rope[b, h, :]
//   decode:  O*[b, h, :]    = softmax(Q* C^T / sqrt(192)) C[:, :512]   (mla_decode_*)
//   after:   o[b, h, :]     = O*[b, h, :] W_UV[h]^T           (value up-projection)
//            out[b, :]      = o[b, :, :] (flattened) W_O^T    (output projection)
//
// with W_UK, W_UV [n_h][128][512] (the per-head key / value halves of the
// latent up-projection, torch Linear layout: out_features x in_features) and
// W_O [d_model][n_h * 128]. The softmax scale stays in the decode kernel, so
// Q* carries no scale. Batched over the B decode tokens.
//
// These are weight-streaming GEMMs with M = B rows, all MFMA kernels of this
// file: the two per-head ones (W_UK, W_UV: 128 KB of weights per head) one
// workgroup per (head, column slice, row group), with the rope columns of Q*
// copied by the absorption kernel; the output projection (one [B x n_h*128] x
// [n_h*128 x d_model] product, bound by streaming W_O) stream-K over units of
// 64 columns x 32 rows, or 128 columns x up to 256 rows. fp16 / bf16
// inputs, fp32 accumulation. No reference code exists for this part (the
// reference stops at the decode kernel).
#include <algorithm>
#include <cstdint>
#include <type_traits>

#include "mla_device.hpp"
#include "mla_internal.hpp"
#include "mla_mi355x.h"
#include "mla_ring.hpp"

namespace mla {
namespace {

constexpr int kNope = 128;  // per-head query / value width before absorption
constexpr int kRope = 64;
constexpr int kLatent = 512;
constexpr int kDK = kLatent + kRope;

bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

// Absorption, one workgroup (4 waves) per (head h, 128-column slice cs, row
// group):
//   Q*[b, h, 128 cs + n] = sum_k q_nope[b, h, k] W_UK[h][k][128 cs + n],
// computed as its transpose D[n][b] on 16x16x32 MFMAs. The W_UK slice (128 x
// 128) and the q_nope rows, kAbsorbTiles tiles of 16 at a time, come into LDS by
// direct loads that are all in flight before one wait: rows are 256 bytes, with
// 16-byte chunk c of row r at c ^ (r mod 16). W_UK is read as the A operand (n
// x k) with the LDS transpose read, q_nope as the B operand.
// Wave w owns columns 32 w .. +31 (two 16-column tiles) for all rows. It is
// bound by the bytes (16.8 MB of W_UK and 196 KB a row at 128 heads) and one
// memory round trip: against rows loaded by every wave for itself and 8-byte
// stores, B = 32, 128 heads 6.3 -> 5.9 us, B = 256 23.9 -> 16.4 (the 16-byte
// stores 2.5 us of it).
// The slice cs = 0 also copies the 64 rope columns of each row.
constexpr int kAbsorbTiles = 4;

template <typename E>
__global__ __launch_bounds__(256) void absorb_kernel(const E *__restrict__ q_nope, const E *__restrict__ q_rope,
                                                     const E *__restrict__ w_uk, E *__restrict__ q_star,
                                                     int batch, int num_heads, int group_rows)
{
    using E8 = typename Vec<E>::v8;
    using E4 = typename Vec<E>::v4;
    __shared__ __attribute__((aligned(1024))) E s_w[kNope * 128];
    __shared__ __attribute__((aligned(1024))) E s_q[kAbsorbTiles * 16 * kNope];
    const int h = blockIdx.x >> 2, cs = blockIdx.x & 3;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l16 = lane & 15, g = lane >> 4;
    const int row0 = blockIdx.y * group_rows, row1 = min(row0 + group_rows, batch);  // the group's rows
    // load units of 4 rows: lane -> row lane / 16, stored chunk lane mod 16
    auto load_tiles = [&](int r) {
        const E *base = q_nope + ((size_t)row0 * num_heads + h) * kNope;
        const int ru = 4 * wave + g;  // row within a tile (rows past the group re-read its last one)
#pragma unroll
        for (int t = 0; t < kAbsorbTiles; ++t)
            if (r + 16 * t < row1 - row0)
                global_to_lds16(base, min(r + 16 * t + ru, row1 - 1 - row0) * num_heads * (kNope * 2) + 16 * (l16 ^ ru),
                                s_q + (16 * t + 4 * wave) * kNope);
    };
    const E *wsrc = w_uk + (size_t)h * kNope * kLatent + 128 * cs;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int k = 32 * wave + 4 * i + g;
        global_to_lds16(wsrc, k * (kLatent * 2) + 16 * (l16 ^ (k & 15)), s_w + (32 * wave + 4 * i) * 128);
    }
    load_tiles(0);
    if (cs == 0) {  // the rope columns, 8 chunks of 16 bytes per row
        for (int i = tid; i < (row1 - row0) * 8; i += 256) {
            const int b = row0 + (i >> 3), c = i & 7;
            *(uint4 *)(q_star + ((size_t)b * num_heads + h) * kDK + kLatent + 8 * c) =
                *(const uint4 *)(q_rope + ((size_t)b * num_heads + h) * kRope + 8 * c);
        }
    }
    MLA_WAIT_VMCNT(0);
    lds_barrier();
    // A operands (n x k): row i of tile nt is column 8 (i / 4) + 4 nt + i mod 4
    // of the wave's 32, so that a lane ends up with 8 adjacent columns; lane
    // (g, i) holds W[32 kk + 8 g .. +7] of it, from two transpose reads of 4 rows
    E8 a[2][kNope / 32];
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) {
#pragma unroll
        for (int kk = 0; kk < kNope / 32; ++kk) {
            E4 part[2];
#pragma unroll
            for (int hf = 0; hf < 2; ++hf) {
                const int row = 32 * kk + 8 * g + 4 * hf + (l16 >> 2);
                const int col = 32 * wave + 8 * (l16 & 3) + 4 * nt;  // 4 columns, 8 bytes
                part[hf] = lds_read_tr16<E>(s_w + row * 128 + 8 * ((col >> 3) ^ (row & 15)) + (col & 7));
            }
            a[nt][kk] = E8{part[0][0], part[0][1], part[0][2], part[0][3], part[1][0], part[1][1], part[1][2], part[1][3]};
        }
    }
    for (int r = 0; r < row1 - row0; r += 16 * kAbsorbTiles) {
        if (r > 0) {
            lds_barrier();  // every wave has read the tiles before
            load_tiles(r);
            MLA_WAIT_VMCNT(0);
            lds_barrier();
        }
        const int tiles = min((row1 - row0 - r + 15) / 16, kAbsorbTiles);
        for (int t = 0; t < tiles; ++t) {
            floatx4 acc[2] = {floatx4{0.f, 0.f, 0.f, 0.f}, floatx4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
            for (int kk = 0; kk < kNope / 32; ++kk) {
                const E8 qv = *(const E8 *)(s_q + (16 * t + l16) * kNope + 8 * ((4 * kk + g) ^ l16));
#pragma unroll
                for (int nt = 0; nt < 2; ++nt)
                    acc[nt] = mfma16x16x32(a[nt][kk], qv, acc[nt]);
            }
            // lane (g, b) holds columns 8 g + 4 nt .. +3 of row b
            const int b = row0 + r + 16 * t + l16;
            if (b < row1) {
                const E8 v = {(E)acc[0][0], (E)acc[0][1], (E)acc[0][2], (E)acc[0][3],
                              (E)acc[1][0], (E)acc[1][1], (E)acc[1][2], (E)acc[1][3]};
                *(E8 *)(q_star + ((size_t)b * num_heads + h) * kDK + 128 * cs + 32 * wave + 8 * g) = v;
            }
        }
    }
}

// Value up-projection:
//   o[b, h * 128 + j] = sum_k O*[b, h, k] W_UV[h][j][k],
// as its transpose D[j][b] on 16x16x32 MFMAs: W_UV rows (k contiguous) are the
// A operand, 32 of them per wave, held in registers; O* rows the B operand.
// One workgroup per (head, column group of NW waves, row group of up to TP
// 16-row tiles). The rows (1 KB each) come into LDS by direct loads, 16-byte
// chunk c of row r at c ^ (r mod 16), so that each crosses L2 once per column
// group, and every load of the workgroup is in flight before the one wait for
// them all: it is bound by the bytes and one memory round trip (B = 160, 128
// heads, 43 MB: 46 -> 12 us against one-wave workgroups that loaded each
// 16-row tile when they came to it; B = 32, 22 MB: 6.8 -> 5.9).
template <typename E, int NW, int TP>
__global__ __launch_bounds__(64 * NW) void value_proj_kernel(const E *__restrict__ o_star, const E *__restrict__ w_uv,
                                                                E *__restrict__ o, int batch, int num_heads, int groups)
{
    using E8 = typename Vec<E>::v8;
    constexpr int kSlices = 4 / NW;  // column groups per head
    __shared__ __attribute__((aligned(1024))) E s_o[TP * 16 * kLatent];
    // heads innermost, so that the workgroups of a head sit on one XCD (when n_h mod 8 = 0)
    const int h = blockIdx.x % num_heads, rest = blockIdx.x / num_heads;
    const int cs = rest % kSlices, rg = rest / kSlices;
    const int lane = threadIdx.x & 63, l16 = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int j0 = 32 * (NW * cs + wave);
    const int tiles = (batch + 15) / 16;
    // tiles / groups tiles each, and one more in the first tiles mod groups
    // (rg * tiles passes 2^31 from 2.1 M rows of one head on)
    const int per = tiles / groups, extra = tiles - per * groups;
    const int b0 = 16 * (rg * per + min(rg, extra));
    const int lim = min(b0 + 16 * (per + (rg < extra)), batch) - 1;  // this group's last row
    // row i of A tile jt is column 8 (i / 4) + 4 jt + i mod 4 of the wave's 32,
    // so that a lane ends up with 8 adjacent columns
    E8 a[2][kLatent / 32];
#pragma unroll
    for (int jt = 0; jt < 2; ++jt) {
        const E *wrow = w_uv + ((size_t)h * kNope + j0 + 8 * (l16 >> 2) + 4 * jt + (l16 & 3)) * kLatent + 8 * g;
#pragma unroll
        for (int kk = 0; kk < kLatent / 32; ++kk)
            a[jt][kk] = *(const E8 *)(wrow + 32 * kk);
    }
#pragma unroll
    for (int i = 0; i < 16 * TP / NW; ++i) {
        const int r = wave + NW * i;  // rows past the group's last stay as they are: theirs is not stored
        if (b0 + r <= lim)
            global_to_lds16(o_star + ((size_t)(b0 + r) * num_heads + h) * kLatent, 16 * (lane ^ (r & 15)), s_o + r * kLatent);
    }
    MLA_WAIT_VMCNT(0);
    lds_barrier();
    floatx4 acc[2][TP];
#pragma unroll
    for (int jt = 0; jt < 2; ++jt)
#pragma unroll
        for (int t = 0; t < TP; ++t)
            acc[jt][t] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kk = 0; kk < kLatent / 32; ++kk) {
#pragma unroll
        for (int t = 0; t < TP; ++t) {
            const E8 ov = *(const E8 *)(s_o + (16 * t + l16) * kLatent + 8 * ((4 * kk + g) ^ l16));
#pragma unroll
            for (int jt = 0; jt < 2; ++jt)
                acc[jt][t] = mfma16x16x32(a[jt][kk], ov, acc[jt][t]);
        }
    }
    // lane (g, b) holds columns j0 + 8 g + 4 jt .. +3 of row b0 + 16 t + b
#pragma unroll
    for (int t = 0; t < TP; ++t) {
        const int b = b0 + 16 * t + l16;
        if (b > lim)
            continue;
        const floatx4 v = acc[0][t], u = acc[1][t];
        *(E8 *)(o + (size_t)b * num_heads * kNope + (size_t)h * kNope + j0 + 8 * g) =
            E8{(E)v[0], (E)v[1], (E)v[2], (E)v[3], (E)u[0], (E)u[1], (E)u[2], (E)u[3]};
    }
}

// v to columns n .. n + 3 of row b of out [batch][N], those in range
template <typename E>
__device__ __forceinline__ void store4(E *__restrict__ out, floatx4 v, int b, int n, int batch, int N)
{
    using E4 = typename Vec<E>::v4;
    if (b >= batch)
        return;
    E *o = out + (size_t)b * N + n;
    if (n + 3 < N && (N & 3) == 0) {
        *(E4 *)o = E4{(E)v[0], (E)v[1], (E)v[2], (E)v[3]};
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (n + i < N)
                o[i] = (E)v[i];
    }
}

// Output projection:
//   out[b, n] = sum_k x[b, k] W_O[n, k]      (x = the value projection, [B x K], K = n_h * 128)
// as its transpose D[n][b] on 16x16x32 MFMAs, W_O rows the A operand and x
// rows the B operand. W_O (168 MB at n_h = 128, d_model 5120) is the one
// large operand and is streamed from HBM once.
//  * Work: a unit is 64 output columns (64 rows of W_O) x 32 rows of x over
//    all K, in kChunk-column chunks; the (unit, chunk) steps, units
//    outermost, are cut into equal contiguous ranges, one per workgroup of a
//    grid of at most one workgroup per CU (stream-K). Every CU thus streams
//    the same share of W_O whatever d_model / 64 is (160 column blocks of 32
//    on 256 CUs would leave 96 idle). A unit that one workgroup covers whole
//    is stored directly; the pieces of a unit split between workgroups (at
//    most a first and a last one per workgroup) are stored as fp32 partial
//    tiles that reduce_units_kernel adds in a fixed order. Plain stores and
//    loads: against nontemporal ones the call (value projection, W_O and the
//    reduce, cold weights) read 41.2-41.4 against 41.6 us at B = 32, d_model
//    5120, and 0.4-1.9% less at four other shapes. (Adding the pieces up in
//    the kernel instead, by the last workgroup to finish a piece of the unit
//    on agent-scope completion counters, measured slower: 40.3 us against
//    32.4 + 4.8 us for the two kernels, from the release / acquire cache
//    maintenance.)
//  * Within a workgroup the chunks run through one kStages-deep LDS ring
//    with no break at unit boundaries: 64 rows of W_O and 32 rows of x per
//    stage, filled by direct global->LDS loads of 512 contiguous bytes of two
//    rows each. Every load is one of these, so the waits are explicit counts
//    that leave the later stages in flight. 16-byte chunk c of a 512-byte row
//    sits at c ^ (row mod 16), which spreads the operand reads (16 rows, one
//    chunk each) over the LDS banks.
//  * Wave w owns the 16 columns 16w .. +15 of the unit for both 16-row tiles
//    of x over every K-step, so no sums cross waves. x (1 MB for B = 32 at
//    n_h = 128) is re-read from L2 by every workgroup, half a byte per byte
//    of W_O; measured, these x loads were the largest cost beside W_O itself.
//  * K is a multiple of 128: a last chunk of 128 columns re-reads each row's
//    last 16 valid bytes in place of the missing ones and skips its K-steps
//    past K. Columns past N and rows past B read clamped addresses and are
//    not stored.
constexpr int kChunk = 256;        // K per ring stage (512 bytes of a row)
constexpr int kStages = 3;         // ring stages (48 KB each: 32 KB of W_O, 16 KB of x)
constexpr int kCols = 64;          // output columns (W_O rows) per unit
constexpr int kUnitsPerWave = 12;  // load units per wave and stage (8 of W_O, 4 of x)
constexpr int kMaxGrid = 512;      // workgroups of the output projection (partial slots: 2 each)
constexpr int kPartTile = kCols * 32;  // floats of one partial tile [32 rows][64 columns]

// the (unit, chunk) steps [g P, min(T, (g + 1) P)) of workgroup g
struct OutProjGeom {
    int n_blocks;  // column blocks of kCols
    int chunks;    // K chunks per unit
    int steps;     // T = units x chunks
    int per_wg;    // P
    int grid;
};

template <typename E>
__global__ __launch_bounds__(256) void out_proj_kernel(const E *__restrict__ x, const E *__restrict__ w,
                                                       E *__restrict__ out, float *__restrict__ part,
                                                       int batch, int K, int N, OutProjGeom geo)
{
    using E8 = typename Vec<E>::v8;
    constexpr int kRowHalves = kChunk;           // one row of a stage
    constexpr int kXOff = kCols * kRowHalves;     // halves: x rows follow the W_O rows
    constexpr int kStage = kXOff + 32 * kRowHalves;
    __shared__ __attribute__((aligned(1024))) E s_ring[kStages][kStage];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // uniform: the load bases are scalars
    const int l16 = lane & 15, g = lane >> 4;
    const int s_first = (int)blockIdx.x * geo.per_wg;
    const int n_steps = min(geo.steps - s_first, geo.per_wg);

    struct Step {
        int unit, c, n0, b0;
    };
    auto step_at = [&](int j) -> Step {
        Step st;
        const int gs = s_first + j;
        st.unit = __builtin_amdgcn_readfirstlane(gs / geo.chunks);
        st.c = __builtin_amdgcn_readfirstlane(gs - st.unit * geo.chunks);
        st.n0 = __builtin_amdgcn_readfirstlane((st.unit % geo.n_blocks) * kCols);
        st.b0 = __builtin_amdgcn_readfirstlane((st.unit / geo.n_blocks) * 32);
        return st;
    };
    // load unit u of a stage: rows 2u, 2u + 1 (lanes 0-31, 32-63) of the
    // W_O part (u < 32) or of the x part; lane: stored chunk position,
    // fetching logical chunk (lane & 31) ^ (row mod 16), at most the chunk's
    // last valid one
    auto unit = [&](const E *rows_base, int row_lim, int c, int st, int off, int u) {
        int ln = lane;
        asm volatile("" : "+v"(ln));
        const int r = 2 * u + (ln >> 5);
        const int valid = min(kChunk, K - c * kChunk) / 8;  // 16-byte chunks of this K-chunk (16 or 32)
        const E *src = rows_base + (size_t)min(2 * u, row_lim) * K + (size_t)c * kChunk;
        // rows 2u and 2u + 1 are K apart; a row past row_lim re-reads row_lim
        const int dr = min(2 * u + 1, row_lim) - min(2 * u, row_lim);
        global_to_lds16(src, (ln >> 5) * dr * K * 2 + 16 * min((ln & 31) ^ (r & 15), valid - 1),
                        &s_ring[st][off + 2 * u * kRowHalves]);
    };
    auto issue = [&](int j, int st) {
        const Step sp = step_at(j);
#pragma unroll
        for (int i = 0; i < 8; ++i)
            unit(w + (size_t)sp.n0 * K, N - 1 - sp.n0, sp.c, st, 0, 8 * wave + i);
#pragma unroll
        for (int i = 0; i < 4; ++i)
            unit(x + (size_t)sp.b0 * K, batch - 1 - sp.b0, sp.c, st, kXOff, 4 * wave + i);
    };
    // operand of K-step kk of row `row` of the part at `off` of stage st
    auto op = [&](int st, int off, int row, int kk) -> E8 {
        return *(const E8 *)(&s_ring[st][off + row * kRowHalves + 8 * ((4 * kk + g) ^ (row & 15))]);
    };
    floatx4 acc[2] = {floatx4{0.f, 0.f, 0.f, 0.f}, floatx4{0.f, 0.f, 0.f, 0.f}};
    bool first_piece = true;  // the unit in progress is this workgroup's first
    int piece_c0 = step_at(0).c;
#pragma unroll
    for (int j = 0; j < kStages; ++j)
        if (j < n_steps)
            issue(j, j);
    for (int j = 0; j < n_steps; ++j) {
        const int st = j % kStages;
        const Step sp = step_at(j);
        // this wave's units of chunk j have landed (later stages may still be
        // in flight; tile stores issued since are younger than them), then
        // every wave's
        const int after = min(kStages - 1, n_steps - 1 - j);
        if (after >= 2)
            MLA_WAIT_VMCNT(2 * kUnitsPerWave);
        else if (after == 1)
            MLA_WAIT_VMCNT(kUnitsPerWave);
        else
            MLA_WAIT_VMCNT(0);
        lds_barrier();
        auto ksteps = [&](auto n) {  // n K-steps of 32: 8, or 4 in a 128-column last chunk
#pragma unroll
            for (int kk = 0; kk < decltype(n)::value; ++kk) {
                const E8 a = op(st, 0, 16 * wave + l16, kk);
                const E8 x0 = op(st, kXOff, l16, kk), x1 = op(st, kXOff, 16 + l16, kk);
                acc[0] = mfma16x16x32(a, x0, acc[0]);
                acc[1] = mfma16x16x32(a, x1, acc[1]);
            }
        };
        if (K - sp.c * kChunk >= kChunk)
            ksteps(std::integral_constant<int, kChunk / 32>{});
        else
            ksteps(std::integral_constant<int, kChunk / 64>{});
        lds_barrier();  // every wave has read stage st
        if (j + kStages < n_steps)
            issue(j + kStages, st);
        const bool unit_end = sp.c == geo.chunks - 1;
        if (!unit_end && j != n_steps - 1)
            continue;
        // ---- end of this workgroup's piece of a unit: lane (g, b) of tile bt
        // holds D[n0 + 16 wave + 4 g .. +3][b0 + 16 bt + b]
        const bool whole = piece_c0 == 0 && unit_end;
        const int slot = 2 * (int)blockIdx.x + (first_piece ? 0 : 1);
#pragma unroll
        for (int bt = 0; bt < 2; ++bt) {
            const floatx4 v = acc[bt];
            acc[bt] = floatx4{0.f, 0.f, 0.f, 0.f};
            const int bl = 16 * bt + l16;        // row within the unit
            const int cl = 16 * wave + 4 * g;    // column within the unit
            const int b = sp.b0 + bl, n = sp.n0 + cl;
            if (!whole) {
                // every row and column of the tile, so the sums stay in bounds
                *(floatx4 *)(part + (size_t)slot * kPartTile + bl * kCols + cl) = v;
            } else {
                store4(out, v, b, n, batch, N);
            }
        }
        first_piece = false;
        piece_c0 = 0;
    }

}

// out of the units split between workgroups: the sum of their pieces,
// workgroup by workgroup (one thread per 4 columns of a row)
template <typename E>
__global__ __launch_bounds__(256) void reduce_units_kernel(const float *__restrict__ part, E *__restrict__ out,
                                                           int batch, int N, OutProjGeom geo)
{
    const int quads = (N + 3) / 4;
    const int t = blockIdx.x * 256 + threadIdx.x;
    if (t >= batch * quads)
        return;
    const int b = t / quads, n = 4 * (t - b * quads);
    const int u = (b / 32) * geo.n_blocks + n / kCols;
    const int g_lo = u * geo.chunks / geo.per_wg, g_hi = (u * geo.chunks + geo.chunks - 1) / geo.per_wg;
    if (g_lo == g_hi)  // one workgroup covered the unit and stored it
        return;
    // the pieces in batches of 8 whose loads are all in flight before the
    // sums (in workgroup order)
    floatx4 v = {0.f, 0.f, 0.f, 0.f};
    const float *tile0 = part + (b % 32) * kCols + n % kCols;
    for (int g0 = g_lo; g0 <= g_hi; g0 += 8) {
        floatx4 p[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int g = g0 + i;
            const int slot = 2 * g + (u == g * geo.per_wg / geo.chunks ? 0 : 1);
            p[i] = g <= g_hi ? *(const floatx4 *)(tile0 + (size_t)slot * kPartTile)
                             : floatx4{0.f, 0.f, 0.f, 0.f};
        }
#pragma unroll
        for (int i = 0; i < 8; ++i)
            v += p[i];
    }
    store4(out, v, b, n, batch, N);
}

// Output projection of more than 32 rows (use_wide). The 32-row units above stream W_O
// once per 32 rows; here a unit is 128 output columns x every row (32 RT of
// them, at most 256), so that W_O crosses once per row block and x is re-read
// half as often per byte of it.
//  * Same stream-K split: the (unit, 64-column K chunk) steps, units
//    outermost, in equal contiguous ranges, one per workgroup, at most one
//    workgroup per CU.
//  * 512 threads: wave w computes columns 32 (w mod 4) .. +31 of rows
//    16 RT (w / 4) .. + 16 RT - 1 over every K-step, on 16x16x32 MFMAs with
//    W_O rows the A operand and x rows the B operand.
//  * A ring stage is the chunk's 128 rows of W_O, then 32 RT rows of x, 128
//    bytes each, filled by direct global->LDS loads of 8 rows; 16-byte chunk
//    c of row r sits at c ^ (r / 2 mod 8), which puts the 16 rows of an
//    operand read on 16 different 16-byte positions of a 256-byte LDS bank
//    period. The ring is as deep as the LDS allows (6 stages at 64 rows, 3 at
//    256), one barrier per step: after it every wave has read stage j - 1,
//    whose slot takes chunk j - 1 + kStages.
//  * The pieces of a unit shared by workgroups go to fp32 tiles in the
//    workspace, tile (workgroup g, unit u) at slot g + u, in MFMA accumulator
//    order (every store and load 1 KB contiguous); reduce_wide_kernel adds
//    them in workgroup order.
//  * K (a multiple of 128) has no partial chunk; rows past N or past the
//    batch re-read the last one and are not stored.
template <int RT>
struct Wide {
    static constexpr int kCols = 128;
    static constexpr int kRows = 32 * RT;
    static constexpr int kK = 64;                                     // K per stage
    static constexpr int kStageBytes = (kCols + kRows) * kK * 2;
    static constexpr int kFit = 160 * 1024 / kStageBytes;
    static constexpr int kStages = kFit > 6 ? 6 : kFit;
    static constexpr int kTile = kCols * kRows;                       // floats of a partial tile
    static constexpr int kWUnits = 2;                                 // W_O load units per wave and stage
};

template <int N>
__device__ __forceinline__ void wait_vmcnt_at_most()
{
    MLA_WAIT_VMCNT(N);
}

// waits until at most `stages` (0 .. S) younger stages of U load units are in flight
template <int U, int S>
__device__ __forceinline__ void wait_younger(int stages)
{
    if constexpr (S > 0) {
        if (stages >= S) {
            wait_vmcnt_at_most<U * S>();
            return;
        }
        wait_younger<U, S - 1>(stages);
    } else {
        wait_vmcnt_at_most<0>();
    }
}

template <typename E, int RT>
__global__ __launch_bounds__(512) void out_proj_wide_kernel(const E *__restrict__ x, const E *__restrict__ w,
                                                            E *__restrict__ out, float *__restrict__ part,
                                                            int batch, int K, int N, OutProjGeom geo)
{
    using T = Wide<RT>;
    using E8 = typename Vec<E>::v8;
    constexpr int kXUnits = (RT + 1) / 2;  // x load units of waves 0..3; waves 4..7 have RT / 2
    __shared__ __attribute__((aligned(1024))) char s_ring[T::kStages * T::kStageBytes];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l16 = lane & 15, g = lane >> 4;
    const int wc = wave & 3, wr = wave >> 2;
    const int s_first = (int)blockIdx.x * geo.per_wg;
    const int n_steps = min(geo.steps - s_first, geo.per_wg);
    const unsigned ring_lds = (unsigned)(uintptr_t)(const __attribute__((address_space(3))) char *)s_ring;

    // ---- loads: unit u of a stage's W_O (x) part is its rows 8u .. 8u + 7;
    // lane -> row 8u + lane / 8, stored position lane mod 8. Wave w issues
    // units w, w + 8, ...
    const int lrow = 8 * wave + (lane >> 3);                    // row of the wave's first unit
    const int lchunk = 16 * ((lane & 7) ^ ((lrow >> 1) & 7));    // (the same for rows 64 further)
    int i_unit = s_first / geo.chunks, i_c = s_first - i_unit * geo.chunks;  // next (unit, chunk) to issue
    int off_w[T::kWUnits], off_x[kXUnits];
    const E *w_base = nullptr, *x_base = nullptr;
    auto set_unit = [&](int unit) {
        const int n0 = (unit % geo.n_blocks) * T::kCols, b0 = (unit / geo.n_blocks) * T::kRows;
        w_base = w + (size_t)n0 * K;
        x_base = x + (size_t)b0 * K;
#pragma unroll
        for (int i = 0; i < T::kWUnits; ++i)
            off_w[i] = min(lrow + 64 * i, N - 1 - n0) * K * 2 + lchunk;
#pragma unroll
        for (int i = 0; i < kXUnits; ++i)
            off_x[i] = min(lrow + 64 * i, batch - 1 - b0) * K * 2 + lchunk;
    };
    set_unit(i_unit);
    auto issue = [&](int slot) {
        const unsigned dst = ring_lds + slot * T::kStageBytes + 1024 * wave;
        const E *wb = w_base + (size_t)i_c * T::kK, *xb = x_base + (size_t)i_c * T::kK;
#pragma unroll
        for (int i = 0; i < T::kWUnits; ++i)
            global_to_lds16_at(wb, off_w[i], dst + 8192 * i);
#pragma unroll
        for (int i = 0; i < kXUnits; ++i)
            if (RT % 2 == 0 || i < kXUnits - 1 || wave < 4)
                global_to_lds16_at(xb, off_x[i], dst + T::kCols * T::kK * 2 + 8192 * i);
        if (++i_c == geo.chunks) {
            i_c = 0;
            ++i_unit;
            if (i_unit * geo.chunks < geo.steps)
                set_unit(i_unit);
        }
    };
    // ---- operands: lane (g, i) reads K 32 kk + 8 g .. +7 of row i of a 16-row group
    const char *a_lane = s_ring + (32 * wc + l16) * (T::kK * 2);
    const char *x_lane = s_ring + (T::kCols + 16 * RT * wr + l16) * (T::kK * 2);
    const int sw = (l16 >> 1) & 7;

    floatx4 acc[2][RT];
    auto clear = [&]() {
#pragma unroll
        for (int nt = 0; nt < 2; ++nt)
#pragma unroll
            for (int r = 0; r < RT; ++r)
                acc[nt][r] = floatx4{0.f, 0.f, 0.f, 0.f};
    };
    clear();
    int unit = i_unit, c = i_c, piece_c0 = i_c, slot = 0, i_slot = 0;
    auto next = [](int s) { return s + 1 == T::kStages ? 0 : s + 1; };
#pragma unroll
    for (int j = 0; j < T::kStages - 1; ++j)
        if (j < n_steps) {
            issue(i_slot);
            i_slot = next(i_slot);
        }
    for (int j = 0; j < n_steps; ++j) {
        // this wave's units of chunk j have landed (younger chunks stay in
        // flight; tile stores issued since are younger than them), then every wave's
        const int younger = min(T::kStages - 2, n_steps - 1 - j);
        if (RT % 2 == 0 || wave < 4)
            wait_younger<T::kWUnits + kXUnits, T::kStages - 2>(younger);
        else
            wait_younger<T::kWUnits + RT / 2, T::kStages - 2>(younger);
        lds_barrier();
        if (j + T::kStages - 1 < n_steps) {
            issue(i_slot);
            i_slot = next(i_slot);
        }
        const char *as = a_lane + slot * T::kStageBytes, *xs = x_lane + slot * T::kStageBytes;
#pragma unroll
        for (int kk = 0; kk < T::kK / 32; ++kk) {
            const int ch = 16 * ((4 * kk + g) ^ sw);
            E8 a[2], xv[RT];
#pragma unroll
            for (int nt = 0; nt < 2; ++nt)
                a[nt] = *(const E8 *)(as + 16 * nt * (T::kK * 2) + ch);
#pragma unroll
            for (int r = 0; r < RT; ++r)
                xv[r] = *(const E8 *)(xs + 16 * r * (T::kK * 2) + ch);
#pragma unroll
            for (int r = 0; r < RT; ++r)
#pragma unroll
                for (int nt = 0; nt < 2; ++nt)
                    acc[nt][r] = mfma16x16x32(a[nt], xv[r], acc[nt][r]);
        }
        slot = next(slot);
        const bool unit_end = c == geo.chunks - 1;
        if (unit_end || j == n_steps - 1) {
            // ---- end of this workgroup's piece of a unit: lane (g, b) of acc[nt][r]
            // holds D[n0 + 32 wc + 16 nt + 4 g .. +3][b0 + 16 RT wr + 16 r + b]
            const bool whole = piece_c0 == 0 && unit_end;
            if (!whole) {
                float *tile = part + (size_t)((int)blockIdx.x + unit) * T::kTile + (size_t)wave * (2 * RT * 256) + 4 * lane;
#pragma unroll
                for (int nt = 0; nt < 2; ++nt)
#pragma unroll
                    for (int r = 0; r < RT; ++r)
                        *(floatx4 *)(tile + (nt * RT + r) * 256) = acc[nt][r];
            } else {
                const int n0 = (unit % geo.n_blocks) * T::kCols + 32 * wc + 4 * g;
                const int b0 = (unit / geo.n_blocks) * T::kRows + 16 * RT * wr + l16;
#pragma unroll
                for (int nt = 0; nt < 2; ++nt)
#pragma unroll
                    for (int r = 0; r < RT; ++r)
                        store4(out, acc[nt][r], b0 + 16 * r, n0 + 16 * nt, batch, N);
            }
            clear();
            piece_c0 = 0;
        }
        if (unit_end) {
            c = 0;
            ++unit;
        } else {
            ++c;
        }
    }
}

// out of the units of out_proj_wide_kernel split between workgroups: the sum
// of their pieces, workgroup by workgroup (one wave per 16 x 16 tile)
template <typename E, int RT>
__global__ __launch_bounds__(256) void reduce_wide_kernel(const float *__restrict__ part, E *__restrict__ out,
                                                          int batch, int N, OutProjGeom geo)
{
    using T = Wide<RT>;
    const int lane = threadIdx.x & 63, l16 = lane & 15, g = lane >> 4;
    const int t = (int)blockIdx.x * 4 + (int)(threadIdx.x >> 6);  // (unit, wave, nt, r)
    const int u = t / (16 * RT), ti = t - u * (16 * RT);
    const int g_lo = u * geo.chunks / geo.per_wg, g_hi = (u * geo.chunks + geo.chunks - 1) / geo.per_wg;
    if (g_lo == g_hi)  // one workgroup covered the unit and stored it
        return;
    const int wave = ti / (2 * RT), nt = ti / RT & 1, r = ti % RT;
    const int b = (u / geo.n_blocks) * T::kRows + 16 * RT * (wave >> 2) + 16 * r + l16;
    const int n = (u % geo.n_blocks) * T::kCols + 32 * (wave & 3) + 16 * nt + 4 * g;
    const float *tile = part + (size_t)(g_lo + u) * T::kTile + (size_t)ti * 256 + 4 * lane;
    floatx4 v = {0.f, 0.f, 0.f, 0.f};
    // batches of 8 pieces whose loads are all in flight before the sums
    for (int p0 = 0; p0 <= g_hi - g_lo; p0 += 8) {
        floatx4 p[8];
#pragma unroll
        for (int i = 0; i < 8; ++i)
            p[i] = p0 + i <= g_hi - g_lo ? *(const floatx4 *)(tile + (size_t)(p0 + i) * T::kTile)
                                         : floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < 8; ++i)
            v += p[i];
    }
    store4(out, v, b, n, batch, N);
}

OutProjGeom out_proj_geom(int n_blocks, int row_blocks, int chunks, int max_grid)
{
    OutProjGeom geo;
    geo.n_blocks = n_blocks;
    geo.chunks = chunks;
    geo.steps = n_blocks * row_blocks * chunks;
    geo.per_wg = (geo.steps + max_grid - 1) / max_grid;
    geo.grid = (geo.steps + geo.per_wg - 1) / geo.per_wg;
    return geo;
}

// out_proj_kernel's units
OutProjGeom narrow_geom(int batch, int K, int N, int max_grid)
{
    return out_proj_geom((N + kCols - 1) / kCols, (batch + 31) / 32, (K + kChunk - 1) / kChunk,
                         std::min(max_grid, kMaxGrid));
}

// out_proj_wide_kernel's, in equal row blocks of at most 256 rows
constexpr int kWideMaxGrid = 256;  // the partial slots are sized for this many on any device
// 32-row steps of a row block
int wide_rt(int batch)
{
    const int blocks = (batch + 255) / 256;
    return ((batch + blocks - 1) / blocks + 31) / 32;
}

OutProjGeom wide_geom(int batch, int K, int N, int max_grid)
{
    const int rows = 32 * wide_rt(batch);
    return out_proj_geom((N + 127) / 128, (batch + rows - 1) / rows, K / 64, std::min(max_grid, kWideMaxGrid));
}

// Whether a call takes the wide units. Up to 32 rows both forms stream W_O
// once, and the narrow one's shorter prologue wins. Past that they win once
// W_O holds kWideMinTotalSteps of their steps (32 MB); below that its
// re-reads hit the caches and the wide units' partial tiles weigh more (whole
// projection, bf16, narrow / wide: 256 steps, n_h 16, d_model 1000: B = 64
// 9.7 / 10.0 us, B = 256 16.7 / 18.6; 512 steps, d_model 2048: B = 64 11.1 /
// 11.3, B = 256 19.1 / 23.3; 1024 steps, n_h 32: B = 40 13.8 / 15.4; 2048
// steps, n_h 128, d_model 1000: B = 33 21.5 / 20.0, B = 64 22.6 / 21.6;
// d_model 5120: B = 40 64.6 / 44.4, B = 64 66.1 / 46.1, B = 160 152 / 61.7,
// B = 256 231 / 78.5).
constexpr int kWideMinTotalSteps = 2048;

bool use_wide(int batch, int K, int N)
{
    return batch > 32 && (int64_t)((N + 127) / 128) * (K / 64) >= kWideMinTotalSteps;
}

// Bytes of the partial tiles of the calls of up to `batch` rows, whatever the
// device: never fewer for more rows, so that a buffer sized for the most rows of
// a serving loop serves all its steps. A single call's need falls where its
// row blocks get shorter: 128 heads, d_model 5120, 256 rows in one block 38.8 MB,
// 257 rows in two blocks of 160 27.5 MB.
size_t out_proj_part_bytes(int batch, int K, int N)
{
    // out_proj_kernel: two tiles for each workgroup
    auto narrow = [&](int rows) {
        const int64_t steps = (int64_t)((N + kCols - 1) / kCols) * ((rows + 31) / 32) * ((K + kChunk - 1) / kChunk);
        return (size_t)2 * std::min<int64_t>(steps, kMaxGrid) * kPartTile * 4;
    };
    if (!use_wide(batch, K, N))
        return narrow(batch);
    // out_proj_wide_kernel: one for each workgroup and unit (tile g + u), of 32 rt rows
    auto wide = [&](int64_t row_blocks, int rt) {
        return (size_t)(kWideMaxGrid + (N + 127) / 128 * row_blocks) * 128 * 32 * rt * 4;
    };
    const int blocks = (batch + 255) / 256;
    const size_t fewer = blocks > 1 ? wide(blocks - 1, 8) : narrow(32);
    return std::max(fewer, wide(blocks, wide_rt(batch)));
}

template <typename E, int RT>
void launch_wide(const E *x, const E *w, E *out, float *part, int batch, int K, int N, hipStream_t s)
{
    const OutProjGeom geo = wide_geom(batch, K, N, current_cu_count());
    hipLaunchKernelGGL((out_proj_wide_kernel<E, RT>), dim3(geo.grid), dim3(512), 0, s, x, w, out, part, batch, K, N, geo);
    if (geo.per_wg % geo.chunks != 0 && geo.grid > 1)  // some unit is shared
        hipLaunchKernelGGL((reduce_wide_kernel<E, RT>), dim3(geo.steps / geo.chunks * 4 * RT), dim3(256), 0, s, part, out,
                           batch, N, geo);
}

template <typename E>
void launch_out_proj(const E *x, const E *w, E *out, float *part, int batch, int K, int N, hipStream_t s)
{
    if (use_wide(batch, K, N)) {
        switch (wide_rt(batch)) {
        case 2: return launch_wide<E, 2>(x, w, out, part, batch, K, N, s);
        case 3: return launch_wide<E, 3>(x, w, out, part, batch, K, N, s);
        case 4: return launch_wide<E, 4>(x, w, out, part, batch, K, N, s);
        case 5: return launch_wide<E, 5>(x, w, out, part, batch, K, N, s);
        case 6: return launch_wide<E, 6>(x, w, out, part, batch, K, N, s);
        case 7: return launch_wide<E, 7>(x, w, out, part, batch, K, N, s);
        default: return launch_wide<E, 8>(x, w, out, part, batch, K, N, s);
        }
    }
    const OutProjGeom geo = narrow_geom(batch, K, N, current_cu_count());
    hipLaunchKernelGGL(out_proj_kernel<E>, dim3(geo.grid), dim3(256), 0, s, x, w, out, part, batch, K, N, geo);
    const int quads = batch * ((N + 3) / 4);
    if (geo.per_wg % geo.chunks != 0 && geo.grid > 1)
        hipLaunchKernelGGL(reduce_units_kernel<E>, dim3((quads + 255) / 256), dim3(256), 0, s, part, out, batch, N, geo);
}

size_t align256(size_t n) { return (n + 255) / 256 * 256; }

// Row groups (multiples of 16 rows): so many that few heads still give 512
// workgroups (n_h 16, B = 256: 13.8 us in one group with rows loaded per wave,
// 4.3 in eight; n_h 32 15.4 and 6.4 in four). 128 heads keep one, as each group
// brings W_UK into LDS again (B = 256, four groups of four tiles: 27.8 us
// against 23.9 in one, both with rows loaded per wave).
template <typename E>
void launch_absorb(const E *q_nope, const E *q_rope, const E *w_uk, E *q_star, int batch, int num_heads, hipStream_t s)
{
    const int tiles = (batch + 15) / 16;
    const int most = std::min(tiles, (128 + num_heads - 1) / num_heads);
    const int rows = 16 * ((tiles + most - 1) / most);
    hipLaunchKernelGGL(absorb_kernel<E>, dim3(num_heads * 4, (batch + rows - 1) / rows), dim3(256), 0, s, q_nope, q_rope,
                       w_uk, q_star, batch, num_heads, rows);
}

int absorb(bool bf16, const void *q_nope, const void *q_rope, const void *w_uk, void *q_star,
           int batch, int num_heads, void *stream)
{
    if (!q_nope || !q_rope || !w_uk || !q_star || batch < 1 || num_heads < 1 || num_heads > 4096 ||
        (int64_t)batch * num_heads * kDK > INT32_MAX)
        return MLA_STATUS_INVALID_VALUE;
    if (!aligned16(q_nope) || !aligned16(q_rope) || !aligned16(w_uk) || !aligned16(q_star))
        return MLA_STATUS_MISALIGNED;
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (bf16)
        launch_absorb(static_cast<const __bf16 *>(q_nope), static_cast<const __bf16 *>(q_rope),
                      static_cast<const __bf16 *>(w_uk), static_cast<__bf16 *>(q_star), batch, num_heads, s);
    else
        launch_absorb(static_cast<const _Float16 *>(q_nope), static_cast<const _Float16 *>(q_rope),
                      static_cast<const _Float16 *>(w_uk), static_cast<_Float16 *>(q_star), batch, num_heads, s);
    const hipError_t e = hipPeekAtLastError();
    return e == hipSuccess ? MLA_STATUS_SUCCESS : record_hip_error(e);
}

template <typename E, int NW>
auto value_proj_for(int tp)
{
    switch (tp) {
    case 1: return value_proj_kernel<E, NW, 1>;
    case 2: return value_proj_kernel<E, NW, 2>;
    case 3: return value_proj_kernel<E, NW, 3>;
    case 4: return value_proj_kernel<E, NW, 4>;
    case 5: return value_proj_kernel<E, NW, 5>;
    case 6: return value_proj_kernel<E, NW, 6>;
    case 7: return value_proj_kernel<E, NW, 7>;
    default: return value_proj_kernel<E, NW, 8>;
    }
}

// Row groups: as few as 8 tiles a workgroup allow, since each reads all of
// W_UV again (at most 4 tiles, B = 160, 128 heads: 15.1 us against 12.3; 256:
// 16.2 against 14.8), but 256 workgroups where the heads give fewer (n_h 16,
// B = 256: 6.2 us with four groups, 10.6 with two; B = 32 3.6 with two, 4.1
// with one). Then the widest column group that leaves 256 workgroups (two
// column groups, 32 rows, 128 heads: 5.9 us against 6.4 with two row groups).
template <typename E>
void launch_value_proj(const E *o_star, const E *w_uv, E *o, int batch, int num_heads, hipStream_t s)
{
    const int tiles = (batch + 15) / 16;
    const int groups = std::max((tiles + 7) / 8, std::min(tiles, (64 + num_heads - 1) / num_heads));
    const int tp = (tiles + groups - 1) / groups;
    const int nw = num_heads * groups >= 256 ? 4 : num_heads * groups >= 128 ? 2 : 1;
    auto k = nw == 4 ? value_proj_for<E, 4>(tp) : nw == 2 ? value_proj_for<E, 2>(tp) : value_proj_for<E, 1>(tp);
    hipLaunchKernelGGL(k, dim3(num_heads * (4 / nw) * groups), dim3(64 * nw), 0, s, o_star, w_uv, o, batch, num_heads,
                       groups);
}

// o[b, h*128 + j] = O*[b, h, :] . W_UV[h][j][:], then out [B x d_model] = o W_O^T
template <typename E>
void project_typed(const E *o_star, const E *w_uv, const E *w_o, E *out, E *o, float *part, int batch, int num_heads,
                   int d_model, hipStream_t s)
{
    launch_value_proj(o_star, w_uv, o, batch, num_heads, s);
    launch_out_proj(o, w_o, out, part, batch, num_heads * kNope, d_model, s);
}

int project(bool bf16, const void *o_star, const void *w_uv, const void *w_o, void *out,
            void *workspace, size_t workspace_bytes, int batch, int num_heads, int d_model, void *stream)
{
    if (!o_star || !w_uv || !w_o || !out || !workspace || batch < 1 || num_heads < 1 || num_heads > 4096 ||
        d_model < 1 || (int64_t)batch * num_heads * kLatent > INT32_MAX || (int64_t)batch * d_model > INT32_MAX)
        return MLA_STATUS_INVALID_VALUE;
    if (!aligned16(o_star) || !aligned16(w_uv) || !aligned16(w_o) || !aligned16(out) || !aligned16(workspace))
        return MLA_STATUS_MISALIGNED;
    if (workspace_bytes < mla_project_output_workspace_size(batch, num_heads, d_model))
        return MLA_STATUS_WORKSPACE_TOO_SMALL;
    hipStream_t s = static_cast<hipStream_t>(stream);
    // workspace: o [B x n_h*128] (16-bit), then the W_O kernel's partial tiles
    char *ws = static_cast<char *>(workspace);
    float *part = reinterpret_cast<float *>(ws + align256((size_t)batch * num_heads * kNope * 2));
    if (bf16)
        project_typed(static_cast<const __bf16 *>(o_star), static_cast<const __bf16 *>(w_uv),
                      static_cast<const __bf16 *>(w_o), static_cast<__bf16 *>(out), reinterpret_cast<__bf16 *>(ws), part,
                      batch, num_heads, d_model, s);
    else
        project_typed(static_cast<const _Float16 *>(o_star), static_cast<const _Float16 *>(w_uv),
                      static_cast<const _Float16 *>(w_o), static_cast<_Float16 *>(out), reinterpret_cast<_Float16 *>(ws),
                      part, batch, num_heads, d_model, s);
    const hipError_t e = hipPeekAtLastError();
    return e == hipSuccess ? MLA_STATUS_SUCCESS : record_hip_error(e);
}

}  // namespace
}  // namespace mla

extern "C" {

size_t mla_project_output_workspace_size(int batch, int num_heads, int d_model)
{
    if (batch < 1 || num_heads < 1 || num_heads > 4096 || d_model < 1)
        return 0;
    // the value projection [B x n_h*128] (16-bit), then the output
    // projection's fp32 partial tiles
    const int hv = num_heads * mla::kNope;
    return mla::align256((size_t)batch * hv * 2) + mla::out_proj_part_bytes(batch, hv, d_model);
}

int mla_absorb_query_fp16(const void *q_nope, const void *q_rope, const void *w_uk, void *q_star, int batch,
                          int num_heads, void *stream)
{
    return mla::absorb(false, q_nope, q_rope, w_uk, q_star, batch, num_heads, stream);
}

int mla_absorb_query_bf16(const void *q_nope, const void *q_rope, const void *w_uk, void *q_star, int batch,
                          int num_heads, void *stream)
{
    return mla::absorb(true, q_nope, q_rope, w_uk, q_star, batch, num_heads, stream);
}

int mla_project_output_fp16(const void *o_star, const void *w_uv, const void *w_o, void *out, void *workspace,
                            size_t workspace_bytes, int batch, int num_heads, int d_model, void *stream)
{
    return mla::project(false, o_star, w_uv, w_o, out, workspace, workspace_bytes, batch,
                        num_heads, d_model, stream);
}

int mla_project_output_bf16(const void *o_star, const void *w_uv, const void *w_o, void *out, void *workspace,
                            size_t workspace_bytes, int batch, int num_heads, int d_model, void *stream)
{
    return mla::project(true, o_star, w_uv, w_o, out, workspace, workspace_bytes, batch,
                        num_heads, d_model, stream);
}

}  // extern "C"
