// `flash_attn_sparse_128`: flash attention over the sparse selector's pass lists, head_dim 128, bf16 in and out.
// Reference semantics: the mako-common kernel of this name, described in docs/architecture.md:123-130 and
// docs/performance.md:162-181. The queries of cube i (head h) attend the tokens of the cubes idx[h][i][0 .. cnt) and
// every dense row (text, keyframe, audio); a dense row's query attends every token; padding slots of cubes at the
// grid's edge are neither keys nor outputs.
//
// Design (gfx950, v_mfma_f32_32x32x16_bf16):
// - The reference gathers each head's rows into cube order (heads_partial with the cube map), attends, and writes the
//   outputs back to the model's rows. Here the kernel reads q, k, v where they lie, in the model's order (the grid
//   layout) or already gathered, through the same cube arithmetic as the selector, and writes the output rows in
//   place: no gather or scatter pass.
// - A workgroup is one (head, 64-row query tile): two waves of 32 queries. Tiles are numbered dense runs of 64 first,
//   then one per cube; the dense query tiles of every head come first in the grid (they attend every token, ten
//   times a cube tile's work), then the cube tiles head by head (share_of: a few heads at a time), so their K and V stay
//   hot in the MALL.
// - Scores are computed transposed, S^T = K Q^T (keys as the MFMA's M, queries as N): the accumulator puts all of
//   a query's keys in one lane and its lane + 32 twin, so the softmax's row maximum and sum are in-lane plus one
//   cross-half exchange, and the rescale of a query's output is one factor per lane.
// - The output is also transposed, O^T += V^T P^T. P^T is the B operand as the score accumulator leaves it in
//   registers; the contraction order over keys is free, so the V^T fragment's key positions follow it: position p of
//   16-key chunk c is key 32 (c / 2) + 16 (c % 2) + 8 (p % 8 / 4) + 4 (p / 8) + p % 4.
// - K and V tiles (64 rows each, 32 KB) go from global memory straight into LDS (buffer_load ... lds), one stage: four
//   workgroups share a CU, and one's loads arrive while the others compute. (Two stages, and the next tile's K during
//   P V with its V during the scores, measured slower.) Each lane fetches whichever source chunk its LDS slot holds,
//   so the layouts are free, with one constraint from the address unit: the four lanes of a quad must fetch one
//   aligned 64-byte piece (a quad spread over four rows is four accesses, and held the K/V stream to about 16 bytes a
//   clock a CU). K is 256-byte rows whose 16-byte chunks are XOR-swizzled by the row (operand reads of 16 rows hit distinct
//   banks); V is 1 KB blocks of 4 keys whose 64-byte pieces are interleaved, read with ds_read_b64_tr_b16. That
//   instruction hands lane i of a 16-lane group element i & 3 of the 8-byte rows named by lanes (i >> 2) + 4 j,
//   j = 0..3: with lane L naming key (L >> 2)'s columns d0 + 4 (L & 3) .. + 3, lane i receives column d0 + i of four
//   keys, a V^T fragment, with no transpose in registers. Padding slots are fetched from past the buffer's end, which
//   reads zeros.
// - Each cube tile walks its pass list from a rotated start (position rank mod S of S, S the cube workgroups an XCD
//   holds at once, rank the tile's place in its XCD's sequence), wrapping round. The XCD's resident tiles then sweep
//   the key cubes together, so a K/V tile one of them fetches is still in L2 when the others that selected it reach
//   it: the L2 hit rate at 768p went from 11-15% to 29-35% and the L2 misses fell by a fifth, for 2.4% less time.
//   The first 4 S tiles of an XCD walk from the start of their lists instead: they start in step (the whole first round
//   at once, and the next rounds nearly so), and tiles in step share their K/V tiles by walking together. 5 heads at
//   768p: 7.37-7.40 ms against 7.96-7.98 rotated from the first tile and 7.73-7.75 never rotated; 40 heads: 54.0-54.4
//   against 54.2-54.6 (68.1 never rotated).
// - A grid that is not a multiple of 4 in every direction leaves cubes at its edge with few tokens (16 of 64 slots in a
//   one-frame image, 32 or less in 37% of the cubes of 37 x 17 x 30). The PACK kernel walks a list's whole cubes first
//   and then its other cubes' tokens in groups of 16, four groups of any cubes to a key tile, so key tiles are full but
//   for the last; queries are numbered by token too, so a wave that none falls to only loads. 37 x 17 x 30, 56 heads,
//   ratio 0.1: 3.35 -> 2.22 ms, every cube selected 22.3 -> 16.3 (together with the loads' addresses worked out without
//   branches); 1 x 43 x 84, 40 heads, ratio 0.5: 3.64 -> 1.05. Fragment reads ahead and the exponentials between the
//   P V MFMAs then took these to 2.07, 15.5 and 0.93.
// - Softmax in base 2 with the scale folded into the exponent. A query's running maximum moves only when a tile
//   raises it by more than 8 (in log2 units): P stays below 2^8, and most tiles skip the rescale of O.
#include "mh3_common.hpp"

#include <algorithm>
#include <type_traits>

namespace mh3 {
namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));

constexpr uint32_t kAttnThreads = 128;
constexpr bool kAttnSweep = true; // rotate each cube tile's pass list so an XCD's resident tiles sweep the keys together
constexpr uint32_t kAttnInStep = 4; // rounds of an XCD's cube tiles that walk their lists unrotated (1, 2, 8: slower;
                                    // 3, 5, 6: within 1%)
constexpr uint32_t kSegEntries = 512;             // pass-list entries a segment holds (PACK)
constexpr uint32_t kSegWords = 3u * kSegEntries;  // a whole cube takes one word, another at most 3 groups
constexpr uint32_t kNoTile = 0xffffffffu;

struct AttnParams {
    const uint16_t* q;
    const uint16_t* k;
    const uint16_t* v;
    uint16_t* out;
    const int32_t* idx;
    const int32_t* cnt;
    uint64_t row0, dense_row0, head_stride, row_stride;
    uint32_t gt, gh, gw, ch, cw, plane; // plane = ch * cw cubes a frame group
    uint32_t cubes, heads, n_dense, nd; // nd: dense tiles of 64 rows
    uint32_t layout, out_stride;
    // The workgroup-to-tile map: `share` XCDs take a head's cube tiles in contiguous parts of `per`, and `groups` =
    // 8 / share heads run at once; XCD x takes the dense tiles x dense_per .. of all heads' in turn.
    uint32_t share, groups, per, dense_per;
    uint32_t sweep; // cube workgroups an XCD runs at once (0: pass lists in plain order)
    uint32_t slots; // workgroups the chip runs at once
    uint32_t eager_from; // list length from which a PACED call's cube tile reads eight ahead (eager_list)
    FastDiv div_plane, div_cw; // c / plane and c / cw by multiply-high: a key tile's cube coordinates cost a few
                               // scalar instructions instead of integer divisions
    float scale_log2;    // score scale times log2(e): softmax in base 2
    const int32_t* order; // or null: head h's j-th cube tile takes query cube order[h cubes + j] (clamped)
};

// A tile of 64 slots. kind 0: dense run (slot l is row base + l, a token while l < lim_t); 1: cube in the grid layout
// (slot (dt, dy, dx) is row base + (dt gh + dy) gw + dx); 2: cube gathered (row base + l); a cube slot is a token while
// dt < lim_t, dy < lim_y, dx < lim_x. kind 3: no tile (an index outside the cubes): no tokens.
struct Tile {
    uint64_t base;
    uint32_t kind, lim_t, lim_y, lim_x;
};

__device__ __forceinline__ Tile make_tile(const AttnParams& p, uint32_t t)
{
    Tile r{0, 3u, 0, 0, 0};
    if (t == kNoTile)
        return r;
    if (t < p.nd) {
        r.kind = 0;
        r.base = p.dense_row0 + 64ull * t;
        r.lim_t = min(64u, p.n_dense - 64u * t);
        return r;
    }
    const uint32_t c = t - p.nd;
    const uint32_t ct = p.div_plane.div(c), rem = c - ct * p.plane, cy = p.div_cw.div(rem), cx = rem - cy * p.cw;
    r.lim_t = min(4u, p.gt - 4u * ct);
    r.lim_y = min(4u, p.gh - 4u * cy);
    r.lim_x = min(4u, p.gw - 4u * cx);
    if (p.layout == MH3_CUBES_GRID) {
        r.kind = 1;
        r.base = p.row0 + (uint64_t(4u * ct) * p.gh + 4u * cy) * p.gw + 4u * cx;
    } else {
        r.kind = 2;
        r.base = p.row0 + 64ull * c;
    }
    return r;
}

__device__ __forceinline__ bool slot_token(const Tile& r, uint32_t l)
{
    if (r.kind == 0)
        return l < r.lim_t;
    if (r.kind == 3)
        return false;
    return (l >> 4) < r.lim_t && ((l >> 2) & 3u) < r.lim_y && (l & 3u) < r.lim_x;
}

// The slot's grid-layout offset (dt gh + dy) gw + dx; below 2^32 (the host checks 4 gh gw < 2^32).
__device__ __forceinline__ uint32_t grid_offset(const AttnParams& p, uint32_t l)
{
    return ((l >> 4) * p.gh + ((l >> 2) & 3u)) * p.gw + (l & 3u);
}

__device__ __forceinline__ uint64_t slot_row(const AttnParams& p, const Tile& r, uint32_t l)
{
    return r.base + (r.kind == 1 ? uint64_t(grid_offset(p, l)) : uint64_t(l));
}

// The tokens of a cube tile (none of another), and the row, from the tile's base, of its i-th token counted without the
// padding (i < 64). A division by 1 .. 4 is a multiplication by 128 / d rounded up and a shift (exact for i < 64).
__device__ __forceinline__ uint32_t tile_tokens(const Tile& r) { return r.lim_t * r.lim_y * r.lim_x; }
__device__ __forceinline__ uint32_t small_recip(uint32_t d)
{
    return d == 1u ? 128u : d == 2u ? 64u : d == 3u ? 43u : 32u;
}
struct TokenRows {
    uint32_t mx, nx, my, ny, sy, st; // reciprocals and limits of x and y; rows a step in y and t takes
    __device__ __forceinline__ TokenRows(const AttnParams& p, const Tile& r)
        : mx(small_recip(r.lim_x)), nx(r.lim_x), my(small_recip(r.lim_y)), ny(r.lim_y), sy(r.kind == 1 ? p.gw : 4u),
          st(r.kind == 1 ? p.gh * p.gw : 16u)
    {
    }
    __device__ __forceinline__ uint32_t operator()(uint32_t i) const
    {
        const uint32_t a = (i * mx) >> 7, dt = (a * my) >> 7;
        return dt * st + (a - dt * ny) * sy + (i - a * nx);
    }
};

__device__ __forceinline__ uint4 load16(const uint16_t* p)
{
    return *reinterpret_cast<const uint4*>(p);
}

typedef __attribute__((address_space(3))) void* lds_ptr_t;
typedef short v4i16 __attribute__((ext_vector_type(4)));

// s_waitcnt that waits for vmcnt == 0 only (gfx9 encoding: vmcnt bits 3:0 and 15:14, expcnt 6:4, lgkmcnt 11:8),
// between scheduling barriers so the compiler moves no memory access across it.
__device__ __forceinline__ void wait_vm0()
{
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0x0070 | 0x0F00);
    __builtin_amdgcn_sched_barrier(0);
}

__device__ __forceinline__ void lds_barrier()
{
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xC07F); // lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

constexpr uint32_t kStageBytes = 32768; // K 16 KB, then V 16 KB
constexpr uint32_t kSegBytes = 4u * (kSegWords + 2u * kSegEntries / 64u);
constexpr uint32_t kPastEnd = 0x80000000u; // a buffer offset past num_records: the load reads zeros
constexpr uint32_t kRecords = 0x7fffffffu;

__device__ __forceinline__ bool tile_full(const Tile& r)
{
    return r.kind == 0 ? r.lim_t == 64u : (r.kind != 3 && r.lim_t == 4u && r.lim_y == 4u && r.lim_x == 4u);
}

// PACED: a call of heads so large that its tiles may be bound by the K/V stream past L2 (stream_bound); those then read
// a fragment right before its MFMA, all others eight ahead.
template <bool PACK, bool PACED>
__global__ __launch_bounds__(kAttnThreads, 2) void attn_sparse_kernel(AttnParams p)
{
    extern __shared__ __attribute__((aligned(16))) char lds[]; // K, V; with PACK the segment's entries (kSegWords)

    const uint32_t tid = threadIdx.x, lane = tid & 63u, n = lane & 31u, hh = lane >> 5;
    // The wave index is uniform: held in a scalar register, the DMA's per-instruction row offsets (soffset) are
    // scalar arithmetic and take no vector registers (which otherwise spill).
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);

    // This workgroup's head and query tile: the dense query tiles of every head first, then the cube tiles. Blocks
    // go to the 8 XCDs round-robin (block b to XCD b % 8). An XCD takes a contiguous part of a head's cubes in raster
    // order (or in p.order's), so the workgroups resident on it are query cubes whose pass lists overlap and meet in
    // its L2; how many XCDs share a head is the host's choice (share_of).
    uint32_t h, qt, rank = 0; // rank: the workgroup's place in its XCD's sequence of cube tiles
    {
        const uint32_t b = blockIdx.x, x = b % 8u, dense_blocks = 8u * p.dense_per;
        if (b < dense_blocks) {
            const uint32_t l = x * p.dense_per + b / 8u;
            // A head's dense tiles, which walk the same keys in the same order, share each K/V tile in one L2 (5
            // heads at 768p: 7.29-7.32 ms against 7.47-7.48 with a head's tiles dealt over the 8 XCDs).
            if (l >= p.nd * p.heads)
                return;
            h = l / p.nd;
            qt = l - h * p.nd;
        } else {
            const uint32_t k = (b - dense_blocks) / 8u, round = k / p.per;
            h = round * p.groups + x / p.share;
            const uint32_t j = (x % p.share) * p.per + (k - round * p.per); // the cube tile's place among its head's
            if (h >= p.heads || j >= p.cubes)
                return;
            rank = k;
            qt = p.nd + (p.order ? min(uint32_t(p.order[uint64_t(h) * p.cubes + j]), p.cubes - 1u) : j);
        }
    }
    const uint64_t hoff = uint64_t(h) * p.head_stride;
    const uint16_t* qh = p.q + hoff;
    const uint16_t* kh = p.k + hoff;
    const uint16_t* vh = p.v + hoff;

    // The key tiles: a dense query tile takes every cube then the dense runs; cube i its pass list then the dense runs.
    const bool dense_q = qt < p.nd;
    uint32_t n_sel = p.cubes;
    const int32_t* list = nullptr;
    if (!dense_q) {
        const uint64_t item = uint64_t(h) * p.cubes + (qt - p.nd);
        list = p.idx + item * p.out_stride;
        n_sel = uint32_t(min(max(p.cnt[item], 0), int32_t(p.out_stride)));
    }
    // The pass list is walked from position rot, wrapping round: a workgroup that starts when the XCD's resident ones
    // are a fraction f into their lists starts a fraction f into its own, so the resident tiles sweep the key cubes
    // together and a K/V tile fetched for one is still in that XCD's L2 when the others that selected it reach it.
    // The first kAttnInStep rounds of an XCD's sequence start (nearly) together and walk from position 0 in step.
    // The order only changes the softmax's summation order.
    const bool rotated = !dense_q && p.sweep && rank >= kAttnInStep * p.sweep;
    const uint32_t rot = rotated ? uint32_t(uint64_t(rank % p.sweep) * n_sel / p.sweep) : 0u;
    auto key_cube = [&](uint32_t e) -> uint32_t { // entry e < n_sel: its key cube, or kNoTile
        if (dense_q)
            return e;
        const uint32_t ee = e + rot < n_sel ? e + rot : e + rot - n_sel;
        const int32_t j = list[ee];
        return j >= 0 && uint32_t(j) < p.cubes ? uint32_t(j) : kNoTile;
    };

    // DMA source offsets of this wave's 8 K and 8 V instructions. Instruction i = 8 wave + u of the workgroup's 16
    // fills the LDS kilobyte 1024 i with slots 4 i .. 4 i + 3 (K rows, and V's keys); the hardware puts lane L's
    // 16 bytes at position 16 L of it, and each lane fetches whichever source chunk that position holds:
    //   K: position L holds chunk (L % 16) ^ (r % 16) of tile row r = 4 i + L / 16 (256-byte rows whose 16-byte
    //      chunks are XOR-swizzled by the row, so that the MFMA operand reads of 16 rows hit distinct banks);
    //   V: position L holds chunk 4 (L / 16) + L % 4 of key 4 i + (L / 4) % 4 (the four keys' 64-byte pieces
    //      interleaved, so that a transposed read of four keys' 8-byte rows hits distinct banks).
    // Either way every four consecutive lanes fetch one aligned 64-byte piece of one row, which the address unit
    // takes as one access. (Lanes of a quad on four different rows, the layout this replaced, cost four accesses and
    // capped the K/V stream at about 16 bytes a clock a CU.) Slots 4 i .. 4 i + 3 are four consecutive rows in both
    // layouts (in the grid dt = i / 4, dy = i % 4, dx = 0 .. 3), so each offset is a lane constant (voffset) plus a
    // term of i alone (soffset).
    const uint32_t rs2 = uint32_t(p.row_stride) * 2u, gw_rs2 = p.gw * rs2;
    const uint32_t k_row = lane >> 4, k_pos = lane & 15u, v_key = (lane >> 2) & 3u;
    const uint32_t v_chunk = 16u * (4u * (lane >> 4) + (lane & 3u)), v_off = v_key * rs2 + v_chunk;
    uint32_t k_chunk[4]; // K chunk (L % 16) ^ (r % 16), r % 16 = 4 (i % 4) + L / 16
#pragma unroll
    for (uint32_t u = 0; u < 4; ++u)
        k_chunk[u] = 16u * (k_pos ^ (4u * u + k_row));
    auto rsrc_of = [&](const uint16_t* head, uint64_t row) {
        return __builtin_amdgcn_make_buffer_rsrc(
            reinterpret_cast<char*>(const_cast<uint16_t*>(head)) + row * p.row_stride * 2ull, 0, int(kRecords),
            kRsrcFlags);
    };
    // Starts tile t's loads; returns its key mask (bit l: slot l is a token). A cube here is whole (a call whose grid
    // has padding takes the kernel with PACK, which gives it only whole cubes); a dense run may end early.
    auto dma_tile = [&](uint32_t t) -> uint64_t {
        const Tile tl = make_tile(p, t);
        const uint32_t live = tl.kind == 0 ? tl.lim_t : tl.kind == 3 ? 0u : 64u;
        const __amdgpu_buffer_rsrc_t rk = rsrc_of(kh, tl.base), rv = rsrc_of(vh, tl.base);
        // Slot 4 i's row, i = 8 wave + u, from the tile's base, in bytes.
        const uint32_t st = tl.kind == 1 ? p.gh * gw_rs2 : 16u * rs2, sy = tl.kind == 1 ? gw_rs2 : 4u * rs2;
        const uint32_t s0 = 2u * wave * st;
        char* const dst = lds + 8192u * wave;
        if (live == 64u) {
#pragma unroll
            for (uint32_t u = 0; u < 8; ++u) {
                const int so = int(s0 + (u >> 2) * st + (u & 3u) * sy);
                __builtin_amdgcn_raw_ptr_buffer_load_lds(rk, (lds_ptr_t)(dst + 1024u * u), 16,
                                                         k_row * rs2 + k_chunk[u & 3u], so, 0, 0);
                __builtin_amdgcn_raw_ptr_buffer_load_lds(rv, (lds_ptr_t)(dst + 16384u + 1024u * u), 16, v_off, so, 0, 0);
            }
            return ~0ull;
        }
#pragma unroll
        for (uint32_t u = 0; u < 8; ++u) {
            const uint32_t slot = 32u * wave + 4u * u, ko = k_row * rs2 + k_chunk[u & 3u];
            const int so = int(s0 + (u >> 2) * st + (u & 3u) * sy);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rk, (lds_ptr_t)(dst + 1024u * u), 16,
                                                     slot + k_row < live ? ko : kPastEnd, so, 0, 0);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rv, (lds_ptr_t)(dst + 16384u + 1024u * u), 16,
                                                     slot + v_key < live ? v_off : kPastEnd, so, 0, 0);
        }
        return (1ull << live) - 1ull;
    };
    // PACK: a tile of `groups` (up to four) groups of 16 tokens, each of some cube at the grid's edge: lane g (of each
    // four) holds group g's word, the cube in its low 30 bits and the group's number in it above. Each wave loads two of
    // the groups; a lane works out its own key's row.
    auto dma_packed = [&](uint32_t word, uint32_t groups) -> uint64_t {
#pragma unroll
        for (uint32_t gg = 0; gg < 2; ++gg) {
            const uint32_t g = 2u * wave + gg, w = __builtin_amdgcn_readlane(word, gg + 2u * wave);
            const Tile tl = make_tile(p, p.nd + (w & 0x3fffffffu));
            const uint32_t first = 16u * (w >> 30), tokens = g < groups ? tile_tokens(tl) : 0u;
            const TokenRows row(p, tl);
            const __amdgpu_buffer_rsrc_t rk = rsrc_of(kh, tl.base), rv = rsrc_of(vh, tl.base);
            char* const dst = lds + 4096u * g;
#pragma unroll
            for (uint32_t u = 0; u < 4; ++u) {
                const uint32_t kk = first + 4u * u + k_row, vk = first + 4u * u + v_key;
                const uint32_t ko = row(kk) * rs2 + k_chunk[u], vo = row(vk) * rs2 + v_chunk;
                __builtin_amdgcn_raw_ptr_buffer_load_lds(rk, (lds_ptr_t)(dst + 1024u * u), 16,
                                                         kk < tokens ? ko : kPastEnd, 0, 0, 0);
                __builtin_amdgcn_raw_ptr_buffer_load_lds(rv, (lds_ptr_t)(dst + 16384u + 1024u * u), 16,
                                                         vk < tokens ? vo : kPastEnd, 0, 0, 0);
            }
        }
        // Slot l is token l % 16 of group l / 16.
        const uint32_t w = uint32_t(__builtin_amdgcn_ds_bpermute(int(lane >> 4) * 4, int(word)));
        const Tile tl = make_tile(p, p.nd + (w & 0x3fffffffu));
        return __ballot((lane >> 4) < groups && 16u * (w >> 30) + (lane & 15u) < tile_tokens(tl));
    };

    // This wave's 32 queries as the B operand of S^T = K Q^T: lane (n, hh) holds d 16 dc + 8 hh .. + 7 of query n.
    const Tile qtile = make_tile(p, qt);
    // Query i of a tile is its slot i; with PACK the i-th token of a cube tile, so that a wave none of them falls to
    // (a cube of up to 32 tokens) only loads.
    const uint32_t qslot = 32u * wave + n;
    const bool by_token = PACK && (qtile.kind == 1 || qtile.kind == 2);
    const bool q_token = by_token ? qslot < tile_tokens(qtile) : slot_token(qtile, qslot);
    const uint64_t qrow = by_token ? qtile.base + TokenRows(p, qtile)(qslot) : slot_row(p, qtile, qslot);
    const bool idle = by_token && 32u * wave >= tile_tokens(qtile);
    bf16x8_t qf[8];
#pragma unroll
    for (int dc = 0; dc < 8; ++dc) {
        const uint4 t = q_token ? load16(qh + qrow * p.row_stride + 16u * dc + 8u * hh) : uint4{0u, 0u, 0u, 0u};
        qf[dc] = __builtin_bit_cast(bf16x8_t, t);
    }

    floatx16 o[4];
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int e = 0; e < 16; ++e)
            o[b][e] = 0.0f;
    float m_run = -__builtin_inff(), l_run = 0.0f;
    // Fragment addresses: lane constants, and immediates or (K's swizzle) an XOR with 32 dc.
    //   K: row 32 b + n, chunk 2 dc + hh at 8192 b + 256 n + 16 ((2 dc + hh) ^ (n % 16)) = 8192 b + (k_lane ^ 32 dc).
    //   V: key k, column d of a 4-key block at 256 (d / 32) + 64 k + 2 (d % 32); lane L of 16-lane group grp names
    //      key L / 4's columns d0 + 4 (L % 4) .. + 3, d0 = 32 db + 16 (grp % 2), of the block 2 (8 b + 4 g) + grp / 2.
    const uint32_t k_lane = 256u * n + 16u * (hh ^ (n & 15u));
    const uint32_t L = lane & 15u, grp = lane >> 4;
    const uint32_t v_lane = 1024u * (grp >> 1) + 32u * (grp & 1u) + 64u * (L >> 2) + 8u * (L & 3u);

    // One tile: its scores, their softmax, and its part of the output; ahead: how many fragments are read ahead of their
    // MFMAs.
    auto attend = [&](uint64_t mask, auto ahead) {
        constexpr int kAhead = decltype(ahead)::value;
        const char* ks = lds;
        const char* vs = lds + 16384u + v_lane;
        auto read_k = [&](int j) { // key block j % 2, d chunk j / 2
            return *reinterpret_cast<const bf16x8_t*>(ks + 8192u * (j & 1) + (k_lane ^ (32u * (j >> 1))));
        };
        auto read_v = [&](int j) { // 16-key chunk j / 4, d block j % 4: two transposed reads (positions 0-3, 4-7)
            const uint32_t off = 4096u * (j >> 2) + 256u * (j & 3);
            const v4i16 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                (v4i16 __attribute__((address_space(3)))*)(const_cast<char*>(vs) + off));
            const v4i16 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                (v4i16 __attribute__((address_space(3)))*)(const_cast<char*>(vs) + off + 2048u));
            return __builtin_bit_cast(bf16x8_t, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
        };

        // S^T: lane (n, hh), element i of block b is key 32 b + 8 (i / 4) + 4 hh + i % 4 of query n. The fragment reads
        // go kAhead MFMAs ahead, held in that order (left to itself the compiler reads each right before its MFMA).
        floatx16 s[2];
        bf16x8_t frag[kAhead];
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int i = 0; i < 16; ++i)
                s[b][i] = 0.0f;
#pragma unroll
        for (int j = 0; j < kAhead; ++j)
            frag[j] = read_k(j);
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            __builtin_amdgcn_sched_barrier(0);
            s[j & 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(frag[j % kAhead], qf[j >> 1], s[j & 1], 0, 0, 0);
            if (j + kAhead < 16)
                frag[j % kAhead] = read_k(j + kAhead);
        }
        __builtin_amdgcn_sched_barrier(0);
        // Online softmax in base 2: padding keys score -inf; the maximum moves only when it rises by more than 8.
        float mt = -__builtin_inff();
        if (mask != ~0ull) {
            // Kept a branch: left to itself the compiler computes all 32 selects for every tile (100 instructions
            // beside the softmax's 130).
            asm volatile("" ::: "memory");
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                const uint32_t live = uint32_t(mask >> (32 * b)) >> (4u * hh); // bit 8 (i / 4) + i % 4: element i
#pragma unroll
                for (int i = 0; i < 16; ++i)
                    s[b][i] = live & (1u << (8 * (i >> 2) + (i & 3))) ? s[b][i] : -__builtin_inff();
            }
        }
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int i = 0; i < 16; ++i)
                mt = fmaxf(mt, s[b][i]);
        mt = fmaxf(mt, __shfl_xor(mt, 32, kWave)) * p.scale_log2;
        if (__ballot(mt > m_run + 8.0f)) {
            const float m_new = fmaxf(m_run, mt);
            const float alpha = m_run == -__builtin_inff() ? 0.0f : __builtin_amdgcn_exp2f(m_run - m_new);
            m_run = m_new;
            l_run *= alpha;
#pragma unroll
            for (int b = 0; b < 4; ++b)
#pragma unroll
                for (int i = 0; i < 16; ++i)
                    o[b][i] *= alpha;
        }
        const float m_ref = m_run == -__builtin_inff() ? 0.0f : m_run;
        // O^T (d 32 db + 8 (i / 4) + 4 hh + i % 4 of query n) += V^T P^T; P^T chunk c is elements 8 (c % 2) .. + 7 of
        // block c / 2. V's first fragments arrive during the first chunk's exponentials, and each later chunk's
        // exponentials go between the MFMAs of the chunk before it.
#pragma unroll
        for (int j = 0; j < kAhead; ++j)
            frag[j] = read_v(j);
        __builtin_amdgcn_sched_barrier(0);
        float ps = 0.0f;
        uint32_t pw[2][4];
        auto exp_pair = [&](int c, int e) { // elements 2 e and 2 e + 1 of chunk c
            const int b = c >> 1, i = 8 * (c & 1) + 2 * e;
            const float p0 = __builtin_amdgcn_exp2f(fmaf(s[b][i], p.scale_log2, -m_ref));
            const float p1 = __builtin_amdgcn_exp2f(fmaf(s[b][i + 1], p.scale_log2, -m_ref));
            ps += p0 + p1;
            pw[c & 1][e] = pack_bf16(p0, p1);
        };
#pragma unroll
        for (int e = 0; e < 4; ++e)
            exp_pair(0, e);
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const uint32_t* w = pw[c & 1];
            const bf16x8_t pf = __builtin_bit_cast(bf16x8_t, uint4{w[0], w[1], w[2], w[3]});
#pragma unroll
            for (int db = 0; db < 4; ++db) {
                const int j = 4 * c + db;
                __builtin_amdgcn_sched_barrier(0);
                o[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(frag[j % kAhead], pf, o[db], 0, 0, 0);
                if (j + kAhead < 16)
                    frag[j % kAhead] = read_v(j + kAhead);
                if (c < 3)
                    exp_pair(c + 1, db);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        l_run += ps;
    };
    // `count` tiles: entry(v) names tile v, fetched while the tile before it is in flight; load(v, entry) starts its
    // loads and returns its key mask.
    auto walk = [&](uint32_t count, auto entry, auto load, auto ahead) {
        uint32_t next = count ? entry(0u) : 0u;
        for (uint32_t v = 0; v < count; ++v) {
            const uint64_t mask = load(v, next);
            if (v + 1u < count)
                next = entry(v + 1u);
            wait_vm0();
            lds_barrier(); // tile v is in LDS for every wave
            if (!PACK || !idle)
                attend(mask, ahead);
            lds_barrier(); // every wave is done with it before it is overwritten
        }
    };
    // Every key tile of this workgroup's walk, at one pace.
    auto run = [&](auto ahead) {
        if constexpr (!PACK) {
            walk(
                n_sel + p.nd,
                [&](uint32_t e) {
                    const uint32_t c = e < n_sel ? key_cube(e) : 0u;
                    return e >= n_sel ? e - n_sel : c == kNoTile ? kNoTile : p.nd + c;
                },
                [&](uint32_t, uint32_t tile) { return dma_tile(tile); }, ahead);
        } else {
            // The entries a segment at a time: its whole cubes from the front of seg[], and the groups of 16 tokens of the
            // others from the back, each in list order.
            uint32_t* const seg = reinterpret_cast<uint32_t*>(lds + kStageBytes);
            uint32_t* const counts = seg + kSegWords; // per 64 entries: whole cubes, groups
            for (uint32_t s0 = 0;; s0 += kSegEntries) {
                const uint32_t n_seg = min(kSegEntries, n_sel - min(s0, n_sel)), runs = (n_seg + 63u) / 64u;
                const bool last = s0 + kSegEntries >= n_sel;
                uint32_t word[kSegEntries / kAttnThreads], n_groups[kSegEntries / kAttnThreads];
                bool whole[kSegEntries / kAttnThreads];
    #pragma unroll
                for (uint32_t k = 0; k < kSegEntries / kAttnThreads; ++k) {
                    const uint32_t e = kAttnThreads * k + tid;
                    word[k] = e < n_seg ? key_cube(s0 + e) : kNoTile;
                    const Tile tl = make_tile(p, word[k] == kNoTile ? kNoTile : p.nd + word[k]);
                    whole[k] = tile_full(tl);
                    n_groups[k] = whole[k] ? 0u : (tile_tokens(tl) + 15u) / 16u; // 0 .. 3
                    const uint32_t nw = uint32_t(__popcll(__ballot(whole[k])));
                    const uint32_t ng = uint32_t(__popcll(__ballot(n_groups[k] & 1u)) +
                                                 2 * __popcll(__ballot(n_groups[k] & 2u)));
                    if (lane == 0 && 2u * k + wave < runs) {
                        counts[2u * (2u * k + wave)] = nw;
                        counts[2u * (2u * k + wave) + 1u] = ng;
                    }
                }
                lds_barrier();
                uint32_t n_whole = 0, n_group = 0;
    #pragma unroll
                for (uint32_t k = 0; k < kSegEntries / kAttnThreads; ++k) {
                    const uint64_t below = lanes_below(int(lane));
                    uint32_t at_w = n_whole, at_g = n_group;
    #pragma unroll
                    for (uint32_t w = 0; w < 2; ++w) {
                        if (2u * k + w >= runs)
                            continue;
                        const uint32_t nw = counts[2u * (2u * k + w)], ng = counts[2u * (2u * k + w) + 1u];
                        at_w += w < wave ? nw : 0u;
                        at_g += w < wave ? ng : 0u;
                        n_whole += nw;
                        n_group += ng;
                    }
                    at_w += uint32_t(__popcll(__ballot(whole[k]) & below));
                    at_g += uint32_t(__popcll(__ballot(n_groups[k] & 1u) & below) +
                                     2 * __popcll(__ballot(n_groups[k] & 2u) & below));
                    if (whole[k])
                        seg[at_w] = word[k];
                    for (uint32_t g = 0; g < n_groups[k]; ++g)
                        seg[kSegWords - 1u - (at_g + g)] = word[k] | g << 30;
                }
                lds_barrier();
                n_whole = __builtin_amdgcn_readfirstlane(n_whole);
                n_group = __builtin_amdgcn_readfirstlane(n_group);
                const uint32_t packed = (n_group + 3u) / 4u;
                walk(
                    n_whole + packed + (last ? p.nd : 0u),
                    [&](uint32_t v) -> uint32_t {
                        const uint32_t g0 = 4u * (v - n_whole); // of a packed tile: its first group
                        return seg[v < n_whole              ? v
                                   : v - n_whole < packed ? kSegWords - 1u - min(g0 + (lane & 3u), n_group - 1u)
                                                          : 0u];
                    },
                    [&](uint32_t v, uint32_t word) {
                        if (v - n_whole < packed)
                            return dma_packed(word, min(n_group - 4u * (v - n_whole), 4u));
                        return dma_tile(v < n_whole ? p.nd + __builtin_amdgcn_readfirstlane(word) : v - n_whole - packed);
                    },
                    ahead);
                if (last)
                    break;
            }
        }
    };
    using Ahead1 = std::integral_constant<int, 1>;
    using Ahead8 = std::integral_constant<int, 8>;
    if constexpr (!PACED) {
        run(Ahead8{});
    } else {
        // A dense tile walks every key tile, and in a call of few heads that chain can take as long as all of the cube
        // tiles: it then reads eight ahead too. That is where it is longer than a workgroup's share of all the call's
        // walks (the lists' mean from 64 of the head's counts; 5 heads of 2016 cubes, 512 dense rows: ratio 0.02 4.80 ->
        // 4.22 ms, 0.05 5.35 -> 4.75, 0.1 7.36 and 7.48; 1440 cubes at 0.1 3.87 -> 3.69, 1760 5.43 and 5.44), and where
        // the cube tiles do (40 heads of 1440 with every cube selected: 224 ms all ahead, 247 but for the dense tiles).
        bool eager = n_sel >= p.eager_from;
        if (dense_q) {
            const int32_t n = p.cnt[uint64_t(h) * p.cubes + (uint64_t(lane) * p.cubes >> 6)];
            const float mean = wave_sum(float(min(max(n, 0), int32_t(p.out_stride)))) * (1.0f / 64.0f);
            const float chain = float(p.cubes) + float(p.nd), dense = float(p.nd);
            const float walks = float(p.heads) * (float(p.cubes) * (mean + dense) + dense * chain);
            eager = __builtin_amdgcn_readfirstlane(chain * float(p.slots) > walks || mean >= float(p.eager_from));
        }
        if (eager)
            run(Ahead8{});
        else
            run(Ahead1{});
    }

    // Normalize and write the query rows (a gathered cube's padding slots get zeros; other non-tokens nothing).
    const float l_tot = l_run + __shfl_xor(l_run, 32, kWave);
    const float inv = q_token && l_tot > 0.0f ? 1.0f / l_tot : 0.0f;
    if (PACK && qtile.kind == 2 && !slot_token(qtile, qslot)) {
        uint16_t* orow = p.out + hoff + slot_row(p, qtile, qslot) * p.row_stride;
#pragma unroll
        for (int j = 0; j < 8; ++j)
            *reinterpret_cast<uint4*>(orow + 16 * j + 8u * hh) = uint4{0u, 0u, 0u, 0u};
    }
    if (q_token) {
        uint16_t* orow = p.out + hoff + qrow * p.row_stride;
#pragma unroll
        for (int db = 0; db < 4; ++db)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const uint32_t d0 = 32u * db + 8u * g + 4u * hh;
                *reinterpret_cast<uint2*>(orow + d0) = uint2{pack_bf16(o[db][4 * g] * inv, o[db][4 * g + 1] * inv),
                                                             pack_bf16(o[db][4 * g + 2] * inv, o[db][4 * g + 3] * inv)};
            }
    }
}

} // namespace
} // namespace mh3

namespace {

// How many XCDs share one head's cube tiles (8, 4, 2 or 1), `bytes` being a head's K and V. Fewer XCDs a head mean more
// of its query cubes on each L2 at once, over the same keys (56 heads, 33 x 15 x 35, 9 MB a head: 3.90 ms at 8, 3.72 at
// 2 and 1; the dense 37 x 17 x 30: 23.2 and 22.5), but 8 / share heads' K and V in flight at once, which costs as they
// fill the 256 MB MALL (40 heads of 66 MB, independent and overlapping lists: 53.0 and 49.4 ms at 8, 50.2 and 48.8 at 4,
// 49.0 and 50.2 at 2, 49.1 and 51.9 at 1). The limit of 144 MB lies just above two such heads, the most that was better
// for both. The heads must also divide over the groups (5 heads of 66 MB: 6.7 ms at 8, 7.9 at 4, 9.4 at 1).
uint32_t share_of(uint32_t heads, uint64_t bytes)
{
    uint32_t share = 1;
    while (share < 8u && (heads % (8u / share) != 0 || 8u / share * bytes > (144ull << 20)))
        share *= 2u;
    return share;
}

// Whether an XCD's resident cube workgroups (four a CU) are through the call's cube tiles in under 16 rounds.
bool few_rounds(const mh3::AttnParams& p)
{
    return uint64_t(p.per) * ((p.heads + p.groups - 1u) / p.groups) < 8u * uint64_t(mh3::host::cu_count());
}

// Whether the call's cube tiles may wait for the K/V stream past L2 rather than for their own work: a head's K and V
// (`bytes`) many times an XCD's 4 MB of L2. The time is then the bytes past L2 over some 7.4 TB/s, whatever a tile's own
// work takes, and a steadier pace, which keeps the tiles' sweeps together, beats a faster one: reading each fragment
// right before its MFMA, the hit rate is 41% against 30% (2016 cubes, 40 heads, ratio 0.1: 348 and 418 GB past L2; 48.2
// against 54.0 ms, overlapping lists 47.2 and 52.0; 1440 cubes, independent lists 25.1 and 27.1). In smaller heads eight
// ahead are faster (1024 cubes 12.9 and 12.6; 37 x 17 x 30 dense 16.3 and 15.5). Grids with cubes at their edges too: 5
// heads of 31 x 48 x 84 7.42 and 7.10 ms, 32 x 45 x 80 5.78 and 5.62, 40 heads of 33 x 48 x 84 60.0 and 59.0, at ratio 0.3
// 180 and 168. In calls of few rounds the line lies lower (5 heads, ratio 0.1: 768 cubes 1.52 and 1.44 ms, 1024 2.25 and
// 2.11; 576 equal), 40 heads of 1024 cubes 12.6 and 12.9.
bool stream_bound(uint64_t bytes, bool few) { return bytes > (uint64_t(few ? 20 : 40) << 20); }

// The list length from which a tile of a stream-bound call reads eight ahead all the same (a tile sees its own list's
// length; idx's width says nothing): every cube, which the tiles then walk together at either pace, unless the heads are
// larger still and of whole cubes (40 heads of 2016 cubes: ratio 0.25 134 ms eight ahead and 119 paced, 0.3 177 and 140,
// overlapping lists 170 and 138, 0.6 319 and 272, 1 495 and 460; 20 heads of 1440 at 0.3 37 and 36, 1 113 and 119; 40 of
// 31 x 48 x 84 at 1 454 and 475). In a call of few rounds, of which the unrotated first ones are much, it is a fifth of
// the cubes (8 heads of 2016: 0.3 31.0 and 31.9, 0.5 51.3 and 53.4), or, where all XCDs share each head, a third of the
// key tiles, the dense ones among them (5 heads of 768 cubes: 0.2 1.85 and 1.77, 0.3 2.70 and 2.56; of 128 cubes and
// 60,000 dense rows 14.2 and 14.5).
uint32_t eager_list(const mh3::AttnParams& p, uint64_t bytes, bool pack)
{
    if (few_rounds(p)) {
        const uint32_t third = (p.cubes + p.nd + 2u) / 3u;
        return p.share == 8u ? third - std::min(third, p.nd) : (p.cubes + 4u) / 5u;
    }
    return pack || bytes < (56ull << 20) ? p.cubes : ~0u;
}

// order: null for the plain entry point; `ordered`: the ordered one, which needs it.
int launch_attn(const MH3AttnArgs* args, const uint16_t* q, const uint16_t* k, const uint16_t* v, const int32_t* idx,
                const int32_t* cnt, const int32_t* order, bool ordered, uint16_t* out, mh3_stream_t stream)
{
    using namespace mh3;
    if (!args)
        return MH3_ERR_POINTER;
    const MH3CubeArgs& c = args->cubes;
    if (c.layout != MH3_CUBES_GRID && c.layout != MH3_CUBES_GATHERED)
        return MH3_ERR_PARAM;
    if (c.heads == 0 || c.grid_t == 0 || c.grid_h == 0 || c.grid_w == 0 || c.head_dim == 0 || c.out_stride == 0)
        return MH3_ERR_SHAPE;
    if (c.head_dim != 128)
        return MH3_ERR_UNSUPPORTED;
    if (!(args->scale >= 0.0f) || args->scale == __builtin_inff())
        return MH3_ERR_PARAM;
    if (!q || !k || !v || !idx || !cnt || !out || (ordered && !order))
        return MH3_ERR_POINTER;
    if (out == q || out == k || out == v)
        return MH3_ERR_PARAM;
    if (c.row_stride % 8 != 0 || c.head_stride % 8 != 0 || c.row_stride < 128 || !host::aligned16(q) ||
        !host::aligned16(k) || !host::aligned16(v) || !host::aligned16(out) ||
        reinterpret_cast<uintptr_t>(order) % 4u != 0u)
        return MH3_ERR_ALIGN;
    AttnParams p{};
    p.gt = c.grid_t, p.gh = c.grid_h, p.gw = c.grid_w;
    p.ch = (p.gh + 3u) / 4u, p.cw = (p.gw + 3u) / 4u;
    const uint64_t cth = (p.gt + 3u) / 4u, plane = uint64_t(p.ch) * p.cw, cubes = cth * plane;
    const uint64_t nd = (uint64_t(args->n_dense) + 63u) / 64u;
    // Row offsets within a tile, in bytes, stay below 2^31 (the DMA's 32-bit buffer offsets).
    const uint64_t tile_rows = c.layout == MH3_CUBES_GRID ? (3ull * p.gh + 4u) * p.gw : 64u;
    if (cubes * c.heads >= (1ull << 31) || (cubes + nd) * c.heads >= (1ull << 31) ||
        std::max<uint64_t>(tile_rows, 64u) * c.row_stride * 2u >= (1ull << 31))
        return MH3_ERR_SHAPE;
    // The dense rows may not overlap the video rows.
    const uint64_t video = c.layout == MH3_CUBES_GRID ? uint64_t(p.gt) * p.gh * p.gw : 64ull * cubes;
    if (args->n_dense && args->dense_row0 < c.row0 + video && c.row0 < args->dense_row0 + args->n_dense)
        return MH3_ERR_PARAM;
    // Nor may out overlap q, k, v or the pass lists, which other workgroups are still reading (each starts by reading
    // its own query tile and list): q, k, v and out each span from the array's start to the last head's last row
    // (video or dense) that the call reads or writes.
    const uint64_t last_row =
        std::max<uint64_t>(c.row0 + video, args->n_dense ? args->dense_row0 + args->n_dense : 0u) - 1u;
    const uint64_t span = ((uint64_t(c.heads) - 1u) * c.head_stride + last_row * c.row_stride + 128u) * 2u;
    {
        const host::Span in[] = {{q, span},
                                 {k, span},
                                 {v, span},
                                 {idx, uint64_t(c.heads) * cubes * c.out_stride * 4u},
                                 {cnt, uint64_t(c.heads) * cubes * 4u},
                                 {order, uint64_t(c.heads) * cubes * 4u}};
        const host::Span o[] = {{out, span}};
        if (host::any_overlap(in, o))
            return MH3_ERR_PARAM;
    }
    p.q = q, p.k = k, p.v = v, p.out = out, p.idx = idx, p.cnt = cnt, p.order = order;
    p.row0 = c.row0, p.dense_row0 = args->dense_row0, p.head_stride = c.head_stride, p.row_stride = c.row_stride;
    p.plane = uint32_t(plane), p.cubes = uint32_t(cubes), p.heads = c.heads, p.n_dense = args->n_dense;
    p.div_plane = FastDiv::make(p.plane);
    p.div_cw = FastDiv::make(p.cw);
    p.nd = uint32_t(nd), p.layout = c.layout, p.out_stride = c.out_stride;
    const uint64_t bytes = (video + args->n_dense) * 512ull; // a head's K and V
    // Workgroups of a launch with `share` XCDs a head. A launch holds under 2^32 threads: shares that do not divide the
    // cubes round up to up to 7 more workgroups a head, which millions of heads of one cube each do not have to spare.
    const auto blocks_of = [&](uint32_t share) {
        const uint64_t per = (cubes + share - 1u) / share, groups = 8u / share;
        return 8u * ((nd * c.heads + 7u) / 8u + per * ((c.heads + groups - 1u) / groups));
    };
    p.share = share_of(c.heads, bytes);
    if (blocks_of(p.share) * kAttnThreads >= (1ull << 32))
        p.share = 1u;
    const uint64_t blocks = blocks_of(p.share);
    if (blocks * kAttnThreads >= (1ull << 32))
        return MH3_ERR_SHAPE;
    p.groups = 8u / p.share, p.per = (p.cubes + p.share - 1u) / p.share, p.dense_per = (p.nd * p.heads + 7u) / 8u;
    const float scale = args->scale > 0.0f ? args->scale : 0.08838834764831845f; // 1 / sqrt(128)
    p.scale_log2 = scale * 1.4426950408889634f;
    const bool pack = p.gt % 4u != 0 || p.gh % 4u != 0 || p.gw % 4u != 0, paced = stream_bound(bytes, few_rounds(p));
    p.eager_from = eager_list(p, bytes, pack);
    const auto kernel = pack    ? paced ? &attn_sparse_kernel<true, true> : &attn_sparse_kernel<true, false>
                        : paced ? &attn_sparse_kernel<false, true> : &attn_sparse_kernel<false, false>;
    const void* kern = reinterpret_cast<const void*>(kernel);
    const size_t lds = kStageBytes + (pack ? kSegBytes : 0u);
    if (const hipError_t e = host::allow_dynamic_lds(kern, lds); e != hipSuccess)
        return host::hip_error(e);
    if (kAttnSweep) {
        int per_cu = 0;
        if (const hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kern, int(kAttnThreads), lds);
            e != hipSuccess)
            return host::hip_error(e);
        // The sweep period: the cube workgroups an XCD holds at once (half or twice that measured slower), and a
        // sixteenth more in stream-bound calls of few rounds, whose tiles then start a little behind those before them
        // (5 heads of 2016 cubes: independent lists 7.35 -> 7.21 ms, overlapping 6.73 -> 6.56, ratio 0.15 10.9 -> 10.7;
        // 40 heads 48.9 -> 50.3).
        p.slots = uint32_t(std::max(per_cu, 1)) * uint32_t(host::cu_count());
        p.sweep = p.slots / 8u + (paced && few_rounds(p) ? p.slots / 128u : 0u);
    }
    hipLaunchKernelGGL(kernel, dim3(uint32_t(blocks)), dim3(kAttnThreads), lds, static_cast<hipStream_t>(stream), p);
    return host::check_launch();
}

} // namespace

extern "C" int mh3_flash_attn_sparse_128(const MH3AttnArgs* args, const uint16_t* q, const uint16_t* k,
                                         const uint16_t* v, const int32_t* idx, const int32_t* cnt, uint16_t* out,
                                         mh3_stream_t stream)
{
    return launch_attn(args, q, k, v, idx, cnt, nullptr, false, out, stream);
}

extern "C" int mh3_flash_attn_sparse_128_ordered(const MH3AttnArgs* args, const uint16_t* q, const uint16_t* k,
                                                 const uint16_t* v, const int32_t* idx, const int32_t* cnt,
                                                 const int32_t* order, uint16_t* out, mh3_stream_t stream)
{
    return launch_attn(args, q, k, v, idx, cnt, order, true, out, stream);
}
