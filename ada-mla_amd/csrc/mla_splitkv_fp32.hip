// fp32 split-KV MLA decode for gfx950 (the --fp32 path): same math and the
// same partial tile layout as the fp16 kernel, with O kept unnormalised in
// fp32, on fp32 MFMAs (16x16x4f32) or on bf16 ones over operands split in three
// ("Products" below), so that the result keeps fp32 precision end to end.
//
// Replaces mla_decode_fused (reference csrc/mla_decode_fused_fwd.cuh:50-352,
// launcher csrc/mla_decode_fused_fwd_sm89.cu:6-60), which ran one CTA per 16
// heads over the whole sequence (8 CTAs at 128 heads). Here the sequence is
// split so the grid fills the GPU, and the splits are merged by
// mla_combine.hip.
//
// Workgroup = 8 wave64s (two per SIMD), 16 or 32 heads (one or two 16-head
// sub-tiles carried by every wave), blocks of 16 tokens, in two roles
// pipelined one block apart: at step t the S waves form the logits and the
// softmax of block t while the O waves add block t - 1 into O, so one wave's
// softmax and LDS traffic overlap the other's MFMAs on each SIMD. The roles
// run separate loops with the same two barriers per step.
//  * S waves 0..3: S^T = C Q*^T, wave w owning K-quarter [144w, 144w + 144)
//    of each 16x16 tile (its Q* slices stay in VGPRs); the four partial tiles
//    are summed through LDS (barrier X), and every S wave of a sub-tile
//    redoes its (tiny) softmax, so all of them hold the running max and sum;
//    one publishes P and the rescale factor of each head for the O waves.
//    Each lane reads 4 consecutive K of both operands with one 16-byte LDS
//    read and feeds them to 4 MFMAs per sub-tile (the same K permutation on A
//    and B).
//  * O waves 4..7: O^T = C_N^T P^T, wave 4 + w owning 128 output columns,
//    read from LDS as 16-byte runs: MFMA tile t (0..3) of half h takes as its
//    row i the value dim 128w + 64h + 4i + t, so one ds_read_b128 of dims
//    128w + 64h + 4i .. +3 feeds four MFMAs and the 16 lanes of a token row
//    read 256 contiguous bytes. The store undoes the permutation: lane
//    (head j, g) of the four tiles holds the 16 dims of natural tile
//    8w + 4h + g. An O wave runs one of its block's four token quads (two at
//    32 heads) before barrier X and the rest after it, so that its MFMAs fill
//    the S wave's softmax on the same SIMD.
//  * C blocks go HBM -> LDS by the direct global->LDS load (36 loads of 1 KB
//    per block: 20 issued by the O waves before their MFMAs, 16 by the S
//    waves after their softmax) into a 4-slot ring, two blocks ahead of the
//    S waves; Q* comes through ring slots 2 (and 3) the same way at the
//    start of a piece. Rows are 2304 bytes with 16-byte chunk c of row r at
//    c ^ (r mod 16), so the S waves' row reads (16 rows, one chunk) and the
//    O waves' token-row reads (16 chunks of one row) both touch 16 distinct
//    chunk positions of a 256-byte bank period.
//
// Products (kSplit, calls whose chunks hold 64 tokens or more): fp32 MFMAs issue
// one 16x16x4 per 32 cycles and SIMD, which bound the step (2176 cycles of them
// at 16 heads, 4352 at 32). Both operands of both products are instead split
// into three bf16 parts after their LDS read (all 24 bits, split_bf16), and six
// of the nine partial products run on 16x16x32 bf16 MFMAs with fp32 sums: 816
// cycles of them at 16 heads, 1632 at 32. A step then takes 2650 cycles at 16
// heads (3250 on fp32 MFMAs) and 4070 at 32 (5690): before barrier X the S
// waves' chain of LDS reads, splits and MFMAs (2050 of them at 32 heads), after
// it the O waves' second half and their wait for the next block's loads. Error against
// float64 for N(0, 1) inputs, fp32 MFMAs -> split: 4.8e-7 -> 2.9e-7 (N = 4096,
// relative 2-norm), 3.2e-7 -> 2.2e-7 (N = 20011), 2.5e-7 -> 2.0e-7 (N = 65536); in
// any single value column, however small, at most 1e-6. us per call at 128
// heads, same box: N = 4096 22.5 -> 20.8, N = 8192 35.4 -> 29.9, N = 20011
// 61.1 -> 47.1, N = 65536 168.5 -> 126.6. (Two fp16 parts and three products were
// faster, 20.4, 27.3, 40.0 and 101.0, but hold 22 bits of an entry and nothing
// below 2^-36, whatever the size of its column.)
#include <type_traits>

#include "mla_device.hpp"
#include "mla_internal.hpp"
#include "mla_ring.hpp"

namespace mla {

#ifdef MLA_TIMELINE
// Timeline build only (see mla_splitkv_fp16.hip): per workgroup of the fp32
// kernel, wave 0 (an S wave) records s_memrealtime at entry (slot 0), at the
// first step (1), at the end of the step loop (2) and after its stores
// complete (3), the block count (11), and s_memtime sums over the steps: to
// barrier X (6), from X to the wait before barrier Y (7), that wait and Y
// (8), and its own work before X (4) and after it (5); wave 4 (an O wave)
// records its own work before X (9) and after it (10).
constexpr int kTimelineWorkgroupsF32 = 8192;
__device__ unsigned long long mla_timeline_stamps_f32[kTimelineWorkgroupsF32 * 16];
#define MLA_STAMP32W(w, e, v)                                                              \
    do {                                                                                   \
        if (wave == (w) && lane == 0 && blockIdx.x < kTimelineWorkgroupsF32)               \
            mla_timeline_stamps_f32[blockIdx.x * 16 + (e)] = (unsigned long long)(v);      \
    } while (0)
#define MLA_STAMP32(e, v) MLA_STAMP32W(0, e, v)
#define MLA_MT32() __builtin_amdgcn_s_memtime()
#else
#define MLA_STAMP32(e, v) \
    do {                  \
    } while (0)
#define MLA_STAMP32W(w, e, v) \
    do {                      \
    } while (0)
#endif

namespace {

constexpr int kBT = 16;                  // tokens per block
constexpr int kRing = 4;                 // C ring slots
constexpr int kRowChunks = kDK / 4;      // 16-byte chunks per row (144)
constexpr int kSlot = kBT * kDK;         // floats per ring slot (36 KB)
constexpr int kLoads = kSlot * 4 / 1024; // 1 KB direct loads per block (36)
// O wave 4 + w issues units w, w + 4, ... (kLoadsO of them) before its first
// MFMAs of a step, S wave w units 4 kLoadsO + w, + 4, ... (kLoadsS) after its
// softmax: such a load holds its wave until it is accepted, so each role
// issues its share where it has slack
constexpr int kLoadsO = 5;
constexpr int kLoadsS = 4;
static_assert(4 * (kLoadsO + kLoadsS) == kLoads, "load split");
constexpr int kWaves = 8;
constexpr int kKQ = kDK / 4;             // K per S wave (144)
// The small tiles exchanged through LDS at every step -- the partial S^T
// tiles [wave][head][token] and P [head][token] -- have rows of 16 floats,
// four 16-byte chunks, chunk k of row r stored at k ^ ((r >> 1) & 3). The
// 16-byte accesses of lanes (row j, chunk g) are then free of bank
// conflicts (measured on gfx950 with SQ_LDS_BANK_CONFLICT in probe kernels;
// rows of 20 floats conflicted on the reads, 0.33 of LDS-active cycles).
// P is stored quad-transposed: token 4 ks + g of head j is element ks of
// chunk g of row j, so lane (j, g) of an O wave reads its tokens g, g + 4,
// g + 8, g + 12 as one 16-byte chunk.
constexpr int kTRow = 16;
__device__ __forceinline__ int tile_at(int row, int chunk)
{
    return row * kTRow + 4 * (chunk ^ ((row >> 1) & 3));
}
static_assert(kRowChunks % 16 == 0, "the row swizzle stays within a row");
static_assert(kLoads == 36, "block loads");

// ---- products on bf16 MFMAs (the kernel's kSplit path): a number is the sum of
// three bf16 parts of 8 bits, which hold all 24 (below 2^-110, where the third
// is subnormal, what is above 2^-133), and a product the six of its nine
// partial products that exceed 2^-24 of it, summed in fp32. This is the
// splitting that Henry, Tang and Heinecke ("Leveraging the bfloat16 Artificial
// Intelligence Datatype For Higher-Precision Computations", 2019) describe. bf16
// has the exponents of fp32, so nothing depends on the values' range, and
// subnormal operands and products are kept (both measured on gfx950).
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float floatx2 __attribute__((ext_vector_type(2)));
struct Parts4 {
    bf16x4 p[3];
};
// upper 16 bits of two floats
__device__ __forceinline__ unsigned upper_halves(float x0, float x1)
{
    return __builtin_amdgcn_perm(__float_as_uint(x1), __float_as_uint(x0), 0x07060302u);
}
__device__ __forceinline__ bf16x4 parts_of(unsigned lo, unsigned hi)
{
    return __builtin_bit_cast(bf16x4, uint2{lo, hi});
}
// x less the lower (upper) of two bf16 numbers, exact where the difference is:
// one v_dot2c_f32_bf16 with (-1, 0) or (0, -1). The factors are in registers
// the compiler cannot see into: as the inline constant -1.0, which it makes of
// the lower one, the instruction took it for the upper number (gfx950).
// Checked there to be exact for 2^21 random fp32 numbers of all exponents,
// subnormal ones among them.
struct MinusOne {
    unsigned lower = 0x0000bf80u, upper = 0xbf800000u;
    __device__ __forceinline__ MinusOne() { asm("" : "+s"(lower), "+s"(upper)); }
};
__device__ __forceinline__ float less_bf16(float x, unsigned pair, unsigned factors)
{
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, pair), __builtin_bit_cast(bf16x2, factors), x,
                                           false);
}
// The first part is x rounded or truncated, the second the rest rounded and the
// third, exactly, what is left. The entries of C are truncated, so that those
// up to the largest fp32 number stay finite, Q* and P rounded: the three
// products left out are then below 2^-24 of the whole. Rounding would take the
// largest fp32 numbers to infinity: Q*'s first parts stop at the largest bf16
// number (kRoundFinite), P, at most 1, has none.
constexpr float kMaxBf16 = 0x1.fep127f;
enum FirstPart { kTruncate, kRound, kRoundFinite };
template <FirstPart kFirst>
__device__ __forceinline__ Parts4 split_bf16(floatx4 x, const MinusOne &m)
{
    unsigned w[3][2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const floatx2 v = {x[2 * i], x[2 * i + 1]};
        if constexpr (kFirst == kTruncate) {
            w[0][i] = upper_halves(v[0], v[1]);
        } else {
            floatx2 f = v;
            if constexpr (kFirst == kRoundFinite)
                f = {__builtin_amdgcn_fmed3f(v[0], -kMaxBf16, kMaxBf16),
                     __builtin_amdgcn_fmed3f(v[1], -kMaxBf16, kMaxBf16)};
            w[0][i] = __builtin_bit_cast(unsigned, __builtin_convertvector(f, bf16x2));
        }
        const floatx2 r = {less_bf16(v[0], w[0][i], m.lower), less_bf16(v[1], w[0][i], m.upper)};
        w[1][i] = __builtin_bit_cast(unsigned, __builtin_convertvector(r, bf16x2));
        w[2][i] = upper_halves(less_bf16(r[0], w[1][i], m.lower), less_bf16(r[1], w[1][i], m.upper));
    }
    return {parts_of(w[0][0], w[0][1]), parts_of(w[1][0], w[1][1]), parts_of(w[2][0], w[2][1])};
}
__device__ __forceinline__ bf16x8 join(bf16x4 a, bf16x4 b)
{
    return __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7);
}
// kSplit: the token of row i of an S^T tile, bits 1 and 2 of i exchanged. Lane
// group g then holds P of tokens split_token(4g .. 4g + 3), and neither the S
// waves' reads of rows split_token(0 .. 15) nor the O waves' of rows
// split_token(4g + r) conflict: a 16-byte read serves lanes 0-3 and 12-15 of one
// 16-lane group with 4-11 of the next, whose stored chunks have to differ. (In
// order the O waves' reads conflicted, with 4g + r and g + 4r exchanged the S
// waves': 0.23 and 0.25 of the LDS-active cycles at N = 4096.)
__device__ __forceinline__ int split_token(int i)
{
    return (i & 9) | (i & 2) << 1 | (i & 4) >> 1;
}
// kSplit: a new reference max is set this far above the block's (log2 units), so
// that P stays at most 1 and most later blocks rescale nothing.
constexpr float kAbove = 4.f;

// HT: heads per workgroup (16 or 32), as HT / 16 sub-tiles of 16 heads that
// every wave carries side by side: the S waves' C rows and the O waves' C_N
// columns are read from LDS once for all of them, so a 32-head workgroup
// fills each C block once for twice the heads.
template <int HT, bool kSplit>
__global__ __attribute__((amdgpu_flat_work_group_size(64 * kWaves, 64 * kWaves), amdgpu_waves_per_eu(2, 2)))
void splitkv_fp32_kernel(const float *__restrict__ q,
                         const float *__restrict__ c,
                         const int *__restrict__ cu_seqlens,
                         float *__restrict__ o_part,
                         float *__restrict__ m_part,
                         float *__restrict__ l_part,
                         int num_heads, int batch, int total_tokens, int chunk,
                         int n_head_tiles, int xcd_remap, float scale_log2)
{
    constexpr int kNS = HT / 16;          // 16-head sub-tiles
    // O waves' token quads before barrier X (the rest after it, beside the
    // S waves' softmax). A SIMD's S and O waves share one MFMA pipe (one
    // fp32 16x16x4 per 32 cycles), so quads moved before X only lengthen that
    // phase; after X they hide the softmax. 32-head tiles run all four after
    // X; 16-head tiles measure the same with one quad before it.
    constexpr int kQuadsA = kNS == 1 ? 1 : 0;
    // kSplit: one of two 64-dim halves before X (N = 20011, 128 heads, with 0 / 1 /
    // 2 of them there: 49.2 / 47.4 / 48.1 us; N = 4096 22.5 / 21.6 / 22.6)
    constexpr int kHalvesA = 1;
    __shared__ __attribute__((aligned(1024))) float s_c[kRing * kSlot];
    __shared__ __attribute__((aligned(16))) float s_s[4 * HT * kTRow];
    // P of two blocks: fp32 [head][token] tiles, or (kSplit) per sub-tile the
    // lanes' bf16 parts (64 x 16 bytes [first, second], then 64 x 8 [third])
    constexpr int kPBytes = kSplit ? kNS * 1536 : HT * kTRow * 4;
    __shared__ __attribute__((aligned(16))) char s_p_mem[2 * kPBytes];
    float *s_p = reinterpret_cast<float *>(s_p_mem);
    __shared__ float s_alpha[2 * HT];

    const MinusOne minus;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const bool s_role = wave < 4;
    const int w4 = wave & 3;  // K quarter (S waves) or 128-column group (O waves)
    // S waves: the sub-tile whose softmax this wave runs (S waves w4 < kNS
    // publish its P and rescale factors and store its m and l)
    const int my_sh = w4 % kNS;
    const int l16 = lane & 15;
    const int g = lane >> 4;
    MLA_STAMP32(0, __builtin_amdgcn_s_memrealtime());
#ifdef MLA_TIMELINE
    unsigned long long ph_a = 0, ph_b = 0, ph_o = 0, tm = 0, wk_a = 0, wk_b = 0;
#endif

    int split, ht;
    {
        const int bid = blockIdx.x;
        if (xcd_remap) {
            const int x = bid & 7, li = bid >> 3;
            split = (li / n_head_tiles) * 8 + x;
            ht = li % n_head_tiles;
        } else {
            split = bid / n_head_tiles;
            ht = bid - split * n_head_tiles;
        }
    }
    if ((long long)split * chunk >= total_tokens)  // a padding workgroup of the grid
        return;
    const int lo = split * chunk;
    const int hi = min(lo + chunk, total_tokens);
    const int head0 = ht * HT;

    int b = 0;
    const int nseq = cu_seqlens ? batch : 1;
    if (cu_seqlens) {
        int l = 0, r = batch;
        while (r - l > 1) {
            const int mid = (l + r) >> 1;
            if (cu_seqlens[mid] <= lo) l = mid; else r = mid;
        }
        b = l;
    }

    // LDS float offset of (row, logical 16-byte chunk) in a slot
    auto slot_at = [](int row, int ch) { return row * kDK + 4 * (ch ^ (row & 15)); };

    for (; b < nseq; ++b) {
        int seq_lo = 0, seq_hi = total_tokens;
        if (cu_seqlens) {
            seq_lo = min(max(cu_seqlens[b], 0), total_tokens);
            seq_hi = min(max(cu_seqlens[b + 1], seq_lo), total_tokens);
        }
        if (seq_lo >= hi)
            break;
        const int p_lo = max(seq_lo, lo);
        const int p_hi = min(seq_hi, hi);
        if (p_lo >= p_hi)
            continue;
        const int slot = split + b;
        const int nblk = (p_hi - p_lo + kBT - 1) / kBT;

        // block j's direct loads of this wave into ring slot j % kRing: unit
        // u covers the slot's physical chunks [64u, 64u + 64); lane i's chunk
        // p = 64u + i is row p / 144, stored chunk p % 144, i.e. logical
        // chunk (p % 144) ^ (row mod 16). Rows past the piece repeat its last
        // token (their logits are masked).
        // 16 rows of 576 floats from base (rows past `last` repeat row
        // `last`) into the ring slot at dst
        auto issue_rows = [&](const float *base, int last, const float *dst) {
#pragma unroll
            for (int k = 0; k < (s_role ? kLoadsS : kLoadsO); ++k) {
                const int u = (s_role ? 4 * kLoadsO : 0) + w4 + 4 * k;
                const int pch = 64 * u + lane;
                const int row = pch / kRowChunks;
                const int sch = pch - row * kRowChunks;
                const int lch = sch ^ (row & 15);
                const int src_row = min(row, last);
                global_to_lds16(base, (src_row * kRowChunks + lch) * 16, dst + 256 * u);
            }
        };
        auto issue_block = [&](int j) {
            const int t0 = p_lo + j * kBT;
            issue_rows(c + (size_t)t0 * kDK, p_hi - 1 - t0, s_c + (j % kRing) * kSlot);
        };

        // the ring and the P / alpha buffers of a previous piece are free
        __syncthreads();
        // Prologue: Q* of the head tile (16 heads per sub-tile, swizzled
        // like C rows) into ring slots 2 .. 2 + kNS - 1, blocks 0 and 1
        // into slots 0 and 1, all by direct loads. The S waves take Q*
        // into registers (and split it) as soon as it has landed, while
        // block 0 still may not have. Q* does not pass through the
        // compiler's own loads: it would count them, and not the direct
        // loads issued after them, and then wait for them inside the
        // block loop, where its vmcnt waits would drain the ring loads of
        // block t + 2 at every step.
#pragma unroll
        for (int sh = 0; sh < kNS; ++sh)
            issue_rows(q + ((size_t)b * num_heads + head0 + 16 * sh) * kDK, 15, s_c + (2 + sh) * kSlot);
        issue_block(0);
        if (nblk > 1)
            issue_block(1);
        if (nblk > 1) {
            if (s_role) MLA_WAIT_VMCNT(2 * kLoadsS); else MLA_WAIT_VMCNT(2 * kLoadsO);
        } else {
            if (s_role) MLA_WAIT_VMCNT(kLoadsS); else MLA_WAIT_VMCNT(kLoadsO);
        }
        __syncthreads();
        auto wait_block0 = [&]() {
            if (nblk > 1) {
                if (s_role) MLA_WAIT_VMCNT(kLoadsS); else MLA_WAIT_VMCNT(kLoadsO);
            } else {
                MLA_WAIT_VMCNT(0);
            }
            __syncthreads();  // block 0 has landed; Q* read: slots 2 .. take blocks 2 .. from step 0 on
        };
        // The two roles run separate loops with the same barriers (two per
        // step), so that the S waves' Q* and the O waves' accumulators share
        // registers.
        if (s_role) {
            // Q* slices, head head0 + 16 sh + l16, dims kKQ*w4 + 16*kq + 4*g .. +3
            floatx4 qf[kNS][kSplit ? 1 : kKQ / 16];
            // kSplit: the slice's bf16 parts; pairs of kq are one K = 32 operand,
            // and the ninth, with two parts of C in the K of its operand, is
            // [first, first], [second, second] and [third, first]
            bf16x8 qp[kNS][3][kSplit ? 5 : 1];
#pragma unroll
            for (int sh = 0; sh < kNS; ++sh) {
                const float *qs = s_c + (2 + sh) * kSlot;
                floatx4 v[kKQ / 16];
#pragma unroll
                for (int kq = 0; kq < kKQ / 16; ++kq)
                    v[kq] = *(const floatx4 *)(qs + slot_at(l16, 36 * w4 + 4 * kq + g));
                if constexpr (kSplit) {
#pragma unroll
                    for (int pr = 0; pr < 4; ++pr) {
                        const Parts4 a = split_bf16<kRoundFinite>(v[2 * pr], minus);
                        const Parts4 a4 = split_bf16<kRoundFinite>(v[2 * pr + 1], minus);
#pragma unroll
                        for (int e = 0; e < 3; ++e)
                            qp[sh][e][pr] = join(a.p[e], a4.p[e]);
                    }
                    const Parts4 a = split_bf16<kRoundFinite>(v[8], minus);
                    qp[sh][0][4] = join(a.p[0], a.p[0]);
                    qp[sh][1][4] = join(a.p[1], a.p[1]);
                    qp[sh][2][4] = join(a.p[2], a.p[0]);
                } else {
#pragma unroll
                    for (int kq = 0; kq < kKQ / 16; ++kq)
                        qf[sh][kq] = v[kq];
                }
            }
            wait_block0();
            MLA_STAMP32(1, __builtin_amdgcn_s_memrealtime());
            MLA_STAMP32(11, nblk);

            const int s_row = kSplit ? split_token(l16) : l16;
            float m_run = -INFINITY, l_run = 0.f;  // sub-tile my_sh; kSplit: the reference m
            for (int t = 0; t <= nblk; ++t) {
#ifdef MLA_TIMELINE
                tm = MLA_MT32();
#endif
                if (t < nblk) {
                    // ---- partial S^T of block t over this wave's K-quarter
                    const float *cs = s_c + (t % kRing) * kSlot;
                    floatx4 acc[kNS];
                    auto row = [&](int kq) { return *(const floatx4 *)(cs + slot_at(s_row, 36 * w4 + 4 * kq + g)); };
#pragma unroll
                    for (int sh = 0; sh < kNS; ++sh)
                        acc[sh] = floatx4{0.f, 0.f, 0.f, 0.f};
                    if constexpr (kSplit) {
                        // the products of the first parts in acc, those 2^-8
                        // and 2^-16 as large in sums of their own
                        floatx4 acc1[kNS], acc2[kNS];
#pragma unroll
                        for (int sh = 0; sh < kNS; ++sh)
                            acc1[sh] = acc2[sh] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                        for (int pr = 0; pr < 4; ++pr) {
                            const Parts4 a = split_bf16<kTruncate>(row(2 * pr), minus);
                            const Parts4 a4 = split_bf16<kTruncate>(row(2 * pr + 1), minus);
                            bf16x8 cp[3];
#pragma unroll
                            for (int e = 0; e < 3; ++e)
                                cp[e] = join(a.p[e], a4.p[e]);
#pragma unroll
                            for (int sh = 0; sh < kNS; ++sh) {
                                acc[sh] = mfma16x16x32(cp[0], qp[sh][0][pr], acc[sh]);
                                acc1[sh] = mfma16x16x32(cp[0], qp[sh][1][pr], acc1[sh]);
                                acc2[sh] = mfma16x16x32(cp[0], qp[sh][2][pr], acc2[sh]);
                            }
#pragma unroll
                            for (int sh = 0; sh < kNS; ++sh) {
                                acc1[sh] = mfma16x16x32(cp[1], qp[sh][0][pr], acc1[sh]);
                                acc2[sh] = mfma16x16x32(cp[1], qp[sh][1][pr], acc2[sh]);
                            }
#pragma unroll
                            for (int sh = 0; sh < kNS; ++sh)
                                acc2[sh] = mfma16x16x32(cp[2], qp[sh][0][pr], acc2[sh]);
                        }
                        const Parts4 a = split_bf16<kTruncate>(row(8), minus);
                        const bf16x8 c01 = join(a.p[0], a.p[1]), c02 = join(a.p[0], a.p[2]);
                        float total = 0.f;
#pragma unroll
                        for (int sh = 0; sh < kNS; ++sh) {
                            acc[sh] = mfma16x16x32(c01, qp[sh][0][4], acc[sh]);
                            acc1[sh] = mfma16x16x32(c01, qp[sh][1][4], acc1[sh]);
                            acc2[sh] = mfma16x16x32(c02, qp[sh][2][4], acc2[sh]);
                        }
#pragma unroll
                        for (int sh = 0; sh < kNS; ++sh) {
                            acc[sh] += acc1[sh] + acc2[sh];
                            total += (acc[sh][0] + acc[sh][1]) + (acc[sh][2] + acc[sh][3]);
                        }
                        const bool lost = !(fabsf(total) < INFINITY);
                        // the parts of an infinity make every product NaN, and
                        // a first part's product may pass the largest number
                        // before the others come off it. The logit itself may be
                        // -inf, a token of no weight: the block again, on
                        // fp32 MFMAs over Q* added up from its parts
                        if (__builtin_expect(__builtin_amdgcn_ballot_w64(lost) != 0, 0)) {
#pragma unroll
                            for (int sh = 0; sh < kNS; ++sh)
                                acc[sh] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                            for (int kq = 0; kq < kKQ / 16; ++kq) {
                                const floatx4 x = row(kq);
#pragma unroll
                                for (int sh = 0; sh < kNS; ++sh) {
                                    bf16x8 e[3] = {qp[sh][0][kq / 2], qp[sh][1][kq / 2], qp[sh][2][kq / 2]};
                                    // (keeps the sums out of the block loop's registers)
                                    asm volatile("" : "+v"(e[0]), "+v"(e[1]), "+v"(e[2]));
#pragma unroll
                                    for (int jj = 0; jj < 4; ++jj) {
                                        const int i = 4 * (kq & 1) + jj;
                                        acc[sh] = mfma16x16x4f32(
                                            x[jj], ((float)e[2][i] + (float)e[1][i]) + (float)e[0][i], acc[sh]);
                                    }
                                }
                            }
                        }
                    } else {
#pragma unroll
                        for (int kq = 0; kq < kKQ / 16; ++kq) {
                            const floatx4 a = row(kq);
#pragma unroll
                            for (int jj = 0; jj < 4; ++jj)
#pragma unroll
                                for (int sh = 0; sh < kNS; ++sh)
                                    acc[sh] = mfma16x16x4f32(a[jj], qf[sh][kq][jj], acc[sh]);
                        }
                    }
#pragma unroll
                    for (int sh = 0; sh < kNS; ++sh)
                        *(floatx4 *)(s_s + tile_at(w4 * HT + 16 * sh + l16, g)) = acc[sh];
                }
#ifdef MLA_TIMELINE
                wk_a += MLA_MT32() - tm;
#endif
                __syncthreads();  // barrier X: the four partial S^T tiles are in LDS
#ifdef MLA_TIMELINE
                { const unsigned long long t2 = MLA_MT32(); ph_a += t2 - tm; tm = t2; }
#endif
                if (t < nblk) {
                    // ---- full tile and softmax of sub-tile my_sh (every S
                    // wave of the sub-tile, identical results)
                    const int t0 = p_lo + t * kBT;
                    const float *sp = s_s + tile_at(16 * my_sh + l16, g);  // (the swizzle repeats every 16 rows)
                    const floatx4 sdot = ((*(const floatx4 *)sp + *(const floatx4 *)(sp + HT * kTRow)) +
                                          *(const floatx4 *)(sp + 2 * HT * kTRow)) +
                                         *(const floatx4 *)(sp + 3 * HT * kTRow);
                    float sv[4];
                    float mx = -INFINITY;
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        sv[i] = t0 + (kSplit ? split_token(4 * g + i) : 4 * g + i) < p_hi ? sdot[i] * scale_log2 : -INFINITY;
                        mx = fmaxf(mx, sv[i]);
                    }
                    mx = max_over_lane_groups(mx);
                    const float mn = !kSplit ? fmaxf(m_run, mx) : mx > m_run ? mx + kAbove : m_run;
                    const float alpha = kSplit && mn == m_run ? 1.f : fast_exp2(m_run - mn);
                    m_run = mn;
                    floatx4 pv;
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        pv[i] = fast_exp2(sv[i] - mn);
                    l_run = l_run * alpha + ((pv[0] + pv[1]) + (pv[2] + pv[3]));
                    if (w4 < kNS) {
                        if constexpr (kSplit) {
                            // P's parts of this lane's tokens, as lane (l16, g) of
                            // an O wave takes them
                            const Parts4 pp = split_bf16<kRound>(pv, minus);
                            char *pw = s_p_mem + (t & 1) * kPBytes + my_sh * 1536;
                            *(bf16x8 *)(pw + 16 * lane) = join(pp.p[0], pp.p[1]);
                            *(bf16x4 *)(pw + 1024 + 8 * lane) = pp.p[2];
                        } else {
                            // token 4g + i is element g of chunk i (quad-transposed)
                            float *pw = s_p + (t & 1) * HT * kTRow;
#pragma unroll
                            for (int i = 0; i < 4; ++i)
                                pw[tile_at(16 * my_sh + l16, i) + g] = pv[i];
                        }
                        if (g == 0)
                            s_alpha[(t & 1) * HT + 16 * my_sh + l16] = alpha;
                    }
                }
                // the S waves' share of block t + 2; block t + 1 landed before
                // the barrier (block t + 2's loads stay in flight)
                if (t + 2 < nblk) {
                    issue_block(t + 2);
                    MLA_WAIT_VMCNT(kLoadsS);
                } else {
                    MLA_WAIT_VMCNT(0);
                }
#ifdef MLA_TIMELINE
                { const unsigned long long t2 = MLA_MT32(); ph_b += t2 - tm; wk_b += t2 - tm; tm = t2; }
#endif
                __syncthreads();  // barrier Y: P and alpha of block t, block t + 1 are in LDS
#ifdef MLA_TIMELINE
                { const unsigned long long t2 = MLA_MT32(); ph_o += t2 - tm; }
#endif
            }
            MLA_STAMP32(2, __builtin_amdgcn_s_memrealtime());
#ifdef MLA_TIMELINE
            MLA_STAMP32(6, ph_a);
            MLA_STAMP32(7, ph_b);
            MLA_STAMP32(8, ph_o);
            MLA_STAMP32W(0, 4, wk_a);
            MLA_STAMP32W(0, 5, wk_b);
#endif
            const float lsum = sum_over_lane_groups(l_run);
            if (w4 < kNS && lane < 16) {
                const size_t mi = (size_t)slot * num_heads + head0 + 16 * my_sh + lane;
                __builtin_nontemporal_store(m_run, m_part + mi);
                __builtin_nontemporal_store(lsum, l_part + mi);
            }
        } else {
            wait_block0();

            floatx4 o[kNS][8];
#pragma unroll
            for (int sh = 0; sh < kNS; ++sh)
#pragma unroll
                for (int dt = 0; dt < 8; ++dt)
                    o[sh][dt] = floatx4{0.f, 0.f, 0.f, 0.f};
            // P of block j: this lane's tokens g, g + 4, g + 8, g + 12, or
            // (kSplit) [first, first], [second, second] and [third, first] of its
            // four (split_token), which meet [first, second] (twice) and [first,
            // third] of their C: 16 tokens fill the K = 32 operands
            floatx4 pq[kNS];
            bf16x8 pp[kNS][3];
            // parts [k0, k1) of block j's second product: four token quads, or
            // (kSplit) two 64-dim halves over all 16 tokens
            constexpr int kParts = kSplit ? 2 : 4, kPartsA = kSplit ? kHalvesA : kQuadsA;
            auto o_parts = [&](int j, auto k0, auto k1) {
                const float *cs = s_c + (j % kRing) * kSlot;
                if constexpr (kSplit) {
#pragma unroll
                    for (int h = decltype(k0)::value; h < decltype(k1)::value; ++h) {
                        floatx4 x[4];
#pragma unroll
                        for (int r = 0; r < 4; ++r)
                            x[r] = *(const floatx4 *)(cs + slot_at(split_token(4 * g + r), 32 * w4 + 16 * h + l16));
#pragma unroll
                        for (int tt = 0; tt < 4; ++tt) {
                            const floatx4 xt = {x[0][tt], x[1][tt], x[2][tt], x[3][tt]};
                            const Parts4 a = split_bf16<kTruncate>(xt, minus);
                            const bf16x8 c01 = join(a.p[0], a.p[1]), c02 = join(a.p[0], a.p[2]);
#pragma unroll
                            for (int sh = 0; sh < kNS; ++sh)
                                o[sh][4 * h + tt] = mfma16x16x32(c02, pp[sh][2], o[sh][4 * h + tt]);
#pragma unroll
                            for (int sh = 0; sh < kNS; ++sh)
                                o[sh][4 * h + tt] = mfma16x16x32(c01, pp[sh][1], o[sh][4 * h + tt]);
#pragma unroll
                            for (int sh = 0; sh < kNS; ++sh)
                                o[sh][4 * h + tt] = mfma16x16x32(c01, pp[sh][0], o[sh][4 * h + tt]);
                        }
                    }
                } else {
#pragma unroll
                    for (int ks = decltype(k0)::value; ks < decltype(k1)::value; ++ks) {
                        const int row = 4 * ks + g;
#pragma unroll
                        for (int h = 0; h < 2; ++h) {
                            const floatx4 a = *(const floatx4 *)(cs + slot_at(row, 32 * w4 + 16 * h + l16));
#pragma unroll
                            for (int tt = 0; tt < 4; ++tt)
#pragma unroll
                                for (int sh = 0; sh < kNS; ++sh)
                                    o[sh][4 * h + tt] = mfma16x16x4f32(a[tt], pq[sh][ks], o[sh][4 * h + tt]);
                        }
                    }
                }
            };
            for (int t = 0; t <= nblk; ++t) {
#ifdef MLA_TIMELINE
                tm = MLA_MT32();
#endif
                // block t + 2 into the slot that block t - 2 left at the end
                // of the previous step (the O waves' share)
                if (t + 2 < nblk)
                    issue_block(t + 2);
                if (t >= 1) {
                    // ---- O^T += C_N^T P^T of block t - 1 (rescaled by its alpha first)
#pragma unroll
                    for (int sh = 0; sh < kNS; ++sh) {
                        if constexpr (kSplit) {
                            const char *pr = s_p_mem + ((t - 1) & 1) * kPBytes + sh * 1536;
                            const bf16x8 p01 = *(const bf16x8 *)(pr + 16 * lane);
                            const bf16x4 p2 = *(const bf16x4 *)(pr + 1024 + 8 * lane);
                            const bf16x4 p0 = __builtin_shufflevector(p01, p01, 0, 1, 2, 3);
                            const bf16x4 p1 = __builtin_shufflevector(p01, p01, 4, 5, 6, 7);
                            pp[sh][0] = join(p0, p0);
                            pp[sh][1] = join(p1, p1);
                            pp[sh][2] = join(p2, p0);
                        } else {
                            pq[sh] = *(const floatx4 *)(s_p + ((t - 1) & 1) * HT * kTRow + tile_at(16 * sh + l16, g));
                        }
                        const float alpha = s_alpha[((t - 1) & 1) * HT + 16 * sh + l16];
                        if (!kSplit || __builtin_amdgcn_ballot_w64(alpha != 1.f) != 0) {
#pragma unroll
                            for (int dt = 0; dt < 8; ++dt)
                                o[sh][dt] *= alpha;
                        }
                    }
                    o_parts(t - 1, std::integral_constant<int, 0>{}, std::integral_constant<int, kPartsA>{});
                }
#ifdef MLA_TIMELINE
                wk_a += MLA_MT32() - tm;
                tm = MLA_MT32();
#endif
                __syncthreads();  // barrier X
                if (t >= 1)
                    o_parts(t - 1, std::integral_constant<int, kPartsA>{}, std::integral_constant<int, kParts>{});
                if (t + 2 < nblk)
                    MLA_WAIT_VMCNT(kLoadsO);
                else
                    MLA_WAIT_VMCNT(0);
#ifdef MLA_TIMELINE
                wk_b += MLA_MT32() - tm;
#endif
                __syncthreads();  // barrier Y
            }
#ifdef MLA_TIMELINE
            MLA_STAMP32W(4, 9, wk_a);
            MLA_STAMP32W(4, 10, wk_b);
#endif
            // in the MFMA accumulator order of natural 16 x 16 tiles (frag_offset):
            // lane (head j, g) holds, over o[sh][4h .. 4h+3], dims 16g .. 16g+15 of
            // tile 8*w4 + 4h + g of sub-tile sh, element r of o[sh][4h + t]
            // being dim 4r + t of it; each store writes 4 runs of 256
            // contiguous bytes. Nontemporal, as the partials are read once,
            // by the combine (see mla_splitkv_fp16.hip)
            float *obase = o_part + (size_t)slot * num_heads * kDV;
#pragma unroll
            for (int sh = 0; sh < kNS; ++sh)
#pragma unroll
                for (int h = 0; h < 2; ++h)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const floatx4 v = {o[sh][4 * h][r], o[sh][4 * h + 1][r], o[sh][4 * h + 2][r],
                                           o[sh][4 * h + 3][r]};
                        __builtin_nontemporal_store(
                            v, (floatx4 *)(obase + frag_offset(head0 + 16 * sh + l16,
                                                               128 * w4 + 64 * h + 16 * g + 4 * r)));
                    }
        }
#ifdef MLA_TIMELINE
        MLA_WAIT_VMCNT(0);
#endif
        MLA_STAMP32(3, __builtin_amdgcn_s_memrealtime());
    }
}

}  // namespace

hipError_t launch_splitkv_fp32(const Problem &pb, const Plan &p, const Partials &w, hipStream_t s)
{
    if (p.n_chunks == 0)
        return hipSuccess;
    if (p.head_tile != 16 && p.head_tile != 32)
        return hipErrorInvalidValue;
    const dim3 grid(grid_chunks(p) * p.n_head_tiles), block(64 * kWaves);
    // split products from chunks of 64 tokens on, where splitting Q* begins to pay
    // (us per call, fp32 MFMAs / split: N = 1024, 32-token chunks 13.5 / 13.9, N =
    // 2048, 64-token ones 16.3 / 16.1, N = 3000, 96 19.3 / 18.9; 16 heads, N =
    // 16384, 64 17.3 / 16.9)
    const bool split = p.chunk >= 64;
    auto k = p.head_tile == 32 ? (split ? splitkv_fp32_kernel<32, true> : splitkv_fp32_kernel<32, false>)
                               : (split ? splitkv_fp32_kernel<16, true> : splitkv_fp32_kernel<16, false>);
    hipLaunchKernelGGL(k, grid, block, 0, s,
                       (const float *)pb.q, (const float *)pb.c, pb.cu_seqlens,
                       static_cast<float *>(w.o), w.m, w.l, pb.num_heads, pb.batch, pb.total_tokens,
                       p.chunk, p.n_head_tiles, p.xcd_remap, pb.scale_log2);
    // the launch's own error; hipPeekAtLastError leaves a sticky error from
    // the caller's earlier work in place for the caller to see
    return hipPeekAtLastError();
}

}  // namespace mla

#ifdef MLA_TIMELINE
extern "C" int mla_timeline_read_f32(void *dst, size_t bytes)
{
    const size_t n = bytes < sizeof(mla::mla_timeline_stamps_f32) ? bytes : sizeof(mla::mla_timeline_stamps_f32);
    return (int)hipMemcpyFromSymbol(dst, HIP_SYMBOL(mla::mla_timeline_stamps_f32), n, 0, hipMemcpyDeviceToHost);
}
#endif
