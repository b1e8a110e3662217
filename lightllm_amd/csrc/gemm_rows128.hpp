// Block-scaled FP8 GEMM on gfx950, a weight stream with the activation block in LDS: at most 384 activation rows as one block, or
// tiled over M for up to 4096 rows and more.
//
// With so few rows of X every weight byte is used once (TN = 2) per launch, so the launch is a stream over W, and
// the square tiles spend it badly: a 128x128 tile keeps 16 KiB of W per K step in flight and one round of such tiles
// is bound by the latency of its steps, not by the memory.  This kernel is the 64-row tile of the grouped GEMM
// (gemm_small.hpp) with more rows and a dense epilogue:
//
//   16*MT activation rows (MT MFMA row blocks) x 128*TN weight rows, K step 128.
//     TN = 2: up to 128 rows (MT <= 8; 16 on two ring slots) against 256 weight rows; TN = 1: up to 384 rows
//     (MT <= 24) against 128.
//   WV waves (8; fewer for some unsplit launches, see below), wave w owns 16*TN weight rows and all activation rows:
//   MT x TN MFMA blocks per K step.
//   A ring of two or three slots of W (128*TN x 128 B) and one of X (16*MT x 128 B), three where they fit.  A wave fetches
//   its own W rows (2*TN requests of 1 KiB per step) into its own part of a slot and is the only one to read them, so the
//   W stream needs no barrier.  The X block is shared: one barrier per step, before the products of its last row blocks,
//   makes the next step visible and frees the slot for step + slots.
//   The K loop is a software pipeline over groups of two to four row blocks: behind every product stand the LDS reads of
//   operands of the next group (of the next step's first group and W rows at the end of a step) and the scale fold of the
//   product two before it.  Left to itself the compiler read each operand right before its product, and the step waited
//   for the LDS a dozen times.  What bounds it now: the vector instructions beside the products (4 per MFMA) on two waves
//   a SIMD, and for a step's first and last products what all waves do at the same time; without any LDS reads it is as
//   fast, without any loads 13 % faster.  us, before / now: 333 x 27648 x 5120 69 / 57 (1.4 / 1.2 us a step), 2047 x 2112 x
//   7168 52.8 / 45.9, 960 x 6144 x 4096 40.5 / 32.8, 160 x 36864 x 7168 80.3 / 68.6, 384 x 4096 x 14336 51.4 / 45.2, 80 x
//   28672 x 4096 32.4 / 29.4; level where the memory is the bound (48 x 36864 x 7168 52.3 / 52.7, 32 x 18432 x 7168 30.9).
//   X scales come in [rows][8 steps] chunks by 4-byte requests (any scale layout); the W scales of the tile's
//   128-wide n blocks are requested to LDS once, behind the rows of the first step.
//   A compute unit pulls 35 to 40 GB/s from HBM through this tile, so the launch wants a workgroup on every unit:
//   when the tiles are too few for that the K range is shared between workgroups.  Their partial sums are
//   16*MT x 128*TN floats each, too many for the last workgroup of a tile to add alone (one compute unit reads
//   about 40 GB/s): they go to the workspace and a second, device-wide launch adds them in split order.
//
//   What a unit pulls is X and W together - the X block comes from L2, but through the same requests - so a launch
//   whose 256-row tiles leave units idle and whose K cannot be shared usefully runs narrower workgroups instead
//   (WV = 5 or 6: 160 or 192 weight rows), as many as there are units: every unit then loads less per K step.
//   The same holds for 129..208 rows on a wide N, whose 128-row tiles need a second round and whose 256x256 tiles
//   leave units idle: workgroups of 4..7 waves at TN = 1 (64..112 weight rows) or, on a wider N still, 5..8 waves at
//   TN = 2 with up to 13 row blocks (160..256 weight rows), whichever makes one round.  Every wave reads the whole X
//   block from LDS, so the time of such a launch grows with M: from 209 rows on the same tile runs over several m tiles (up to 13
//   row blocks each, in one to four rounds), wherever that is estimated ahead of the square tiles and of a shared K.
//
//   (Half-width tiles of four waves on two slots, two workgroups to a unit, were tried for shapes whose 256-row
//   tiles leave units idle and cannot share K usefully - N = 36864: 144 tiles on 256 units - and were slower: 85 us
//   against 69 at M = 128.)
//
// Arithmetic, operand layouts in LDS and the epilogue are those of the other tiled kernels (gemm_tile.hpp).
#pragma once
#include "gemm_tile.hpp"

namespace mi355 {

// XS: ring slots of X, 0 for as many as there is room for.
template <int MT, int TN_ = 2, int WV = 8, int XS = 0>
struct Rows128Cfg {
    static_assert(WV >= 4 && WV <= 8 && MT >= 1 && MT <= (TN_ == 2 ? 16 : 24) && (TN_ == 1 || TN_ == 2), "");
    static constexpr int TN = TN_, WNS = 16 * TN, kWaves = WV, kThreads = 64 * WV, BN = WNS * WV;
    static constexpr int NBLK = (BN + 2 * kBlockN - 2) / kBlockN;  // 128-wide n blocks a tile can touch (two or three)
    static constexpr int NWW = 2 * TN;                         // W requests per wave and step (8 rows each)
    static constexpr int XG = 2 * MT;                          // 8-row request groups of the X block
    static constexpr int NXW = (XG + kWaves - 1) / kWaves;     // X requests per wave (groups repeat if XG % 8 != 0)
    static constexpr int kXBytes = 16 * MT * 128, kWBytes = BN * 128;
    // one chunk of X scales: [rows][8 steps] (odd groups of eight rows have the halves of the steps swapped, so that the 16 rows of a
    // block lie on different banks).  Eight lanes request the 32 bytes of a row together; with a row per lane and the steps apart
    // the 64 requests met no neighbour, and ahead of the first step they held up the W rows: 253 x 1920 x 20352, 9 steps a
    // workgroup, 33.2 us / 31.8, 187 x 3584 x 7936 24.5 / 23.7, over 159 shapes of 209..384 rows 2 %.
    static constexpr int kChunkBytes = 2 * MT * 256;
    // ring slots of W and of X: three where they fit beside the scales of a long K
    static constexpr int NSW = MT <= 8 ? 3 : 2;
    static constexpr int NSX = XS ? XS : 3 * kXBytes + NSW * kWBytes + 2 * kChunkBytes <= 157 * 1024 ? 3 : 2;
    // (the counts of requests in flight hold where an X slot is requested as far ahead as a W slot, or farther)
    static_assert(NSX >= NSW, "");
    // X row blocks are read from LDS in groups of at most this many; one group's reads run beside another's products
    static constexpr int kGroup = TN == 1 ? 4 : MT == 7 || MT == 8 ? 4 : 3;
    static constexpr int NG = 2 * ((MT + 2 * kGroup - 1) / (2 * kGroup)), G = (MT + NG - 1) / NG;  // (even: two buffers in turn)
    static constexpr int group_at(int g) { return g * MT / NG; }
    static constexpr int group_of(int block) {
        int g = 0;
        while (group_at(g + 1) <= block) ++g;
        return g;
    }
    static constexpr int kWOff = NSX * kXBytes;                // the W ring
    static constexpr int kWsOff = kWOff + NSW * kWBytes;       // W scales [NBLK][steps]
    static constexpr int kTileElems = 16 * MT * BN;
    static constexpr int chunk_off(int steps) { return (kWsOff + NBLK * steps * 4 + 127) & ~127; }
    static constexpr int lds_bytes(int steps) { return chunk_off(steps) + 2 * kChunkBytes; }
};

// f(integral_constant<int, 0>) ... f(integral_constant<int, N - 1>)
template <int I, int N, typename F>
__device__ __forceinline__ void static_for_from(const F &f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        static_for_from<I + 1, N>(f);
    }
}
template <int N, typename F>
__device__ __forceinline__ void static_for(const F &f) {
    static_for_from<0, N>(f);
}

// One lane's 4*TN consecutive outputs of row `row`: columns nbase + 4*TN*g4 + [0, 4*TN).
template <int TN>
__device__ __forceinline__ void rows128_store(const GemmArgs &p, int row, int nbase, int g4, const float *o) {
    uint16_t *cp = p.C + (int64_t)row * p.ldc + nbase + lane_col<TN>(g4, 0);
    if (p.vec_store && nbase + 16 * TN <= p.N) {
        if constexpr (TN == 2) {
            *(v4i *)cp = v4i{(int)pack_out2(o[0], o[1], p.out_f16), (int)pack_out2(o[2], o[3], p.out_f16),
                             (int)pack_out2(o[4], o[5], p.out_f16), (int)pack_out2(o[6], o[7], p.out_f16)};
        } else {
            *(v2i *)cp = v2i{(int)pack_out2(o[0], o[1], p.out_f16), (int)pack_out2(o[2], o[3], p.out_f16)};
        }
    } else {
#pragma unroll
        for (int e = 0; e < 4 * TN; ++e)
            if (nbase + lane_col<TN>(g4, 0) + e < p.N) cp[e] = (uint16_t)out_bits(o[e], p.out_f16);
    }
}

// TURN: the tiles start at different K steps (GemmArgs::turn_mask).
template <int MT, int TN, int WV, bool SPLIT, bool TURN = false, int XS = 0>
__global__ __launch_bounds__(64 * WV) void block_fp8_gemm_rows128_kernel(const GemmArgs p) {
    using Cfg = Rows128Cfg<MT, TN, WV, XS>;
    // a few rows wait for the memory, not for the matrix cores: the W rows of a slot are requested again as soon as they are read
    constexpr bool kWFirst = SPLIT && MT <= 4;
    constexpr int WNS = Cfg::WNS, NXW = Cfg::NXW, XG = Cfg::XG, NWW = Cfg::NWW, NSX = Cfg::NSX, NSW = Cfg::NSW;
    extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r16 = lane & 15, g4 = lane >> 4, sub = lane >> 3;
    const uint32_t pch = (uint32_t)(lane & 7);

    uint32_t tile_n, tile_m = 0, split = 0;
    if constexpr (SPLIT) {
        tile_n = blockIdx.x / (uint32_t)p.splits;
        split = blockIdx.x - tile_n * (uint32_t)p.splits;
    } else if (p.tiles_m > 1) {
        // more rows than one block holds: tiles_m x tiles_n tiles, one contiguous run per XCD (workgroup ids go round-robin
        // over the 8 XCDs), m fastest inside groups of group_m m tiles: a run is a compact block of tiles, and the L2 fetches
        // the fewest distinct rows of X and W for it (rowsm_group)
        const uint32_t per_xcd = gridDim.x >> 3;  // the grid is a multiple of 8
        const uint32_t logical = (blockIdx.x & 7u) * per_xcd + (blockIdx.x >> 3);
        if (logical >= (uint32_t)p.total_tiles) return;
        const uint32_t width = (uint32_t)(p.group_m * p.tiles_n), first = logical / width * (uint32_t)p.group_m;
        const uint32_t in_group = logical % width, group = min((uint32_t)p.tiles_m - first, (uint32_t)p.group_m);
        tile_n = in_group / group;
        tile_m = first + in_group - tile_n * group;
    } else {
        tile_n = blockIdx.x;
    }
    const int n0 = (int)tile_n * Cfg::BN;
    const int m0 = (int)tile_m * (16 * MT);
    const int KB = p.K / kBlockK;
    int kb_begin = 0, kb_end = KB;
    if constexpr (SPLIT) {
        const int per = KB / p.splits, rem = KB % p.splits;
        kb_begin = (int)split * per + min((int)split, rem);
        kb_end = kb_begin + per + ((int)split < rem ? 1 : 0);
    }
    const int steps = kb_end - kb_begin;
    const uint32_t lds0 = lds_addr(lds);

    // ---- request offsets (rows past the matrices are clamped; their results are never stored)
    uint32_t xoff[NXW], xdst[NXW], sc_row[NXW], sdst[NXW];
    int sodd[NXW];
#pragma unroll
    for (int i = 0; i < NXW; ++i) {
        const int g = (wave + Cfg::kWaves * i) % XG;  // waves beyond the block repeat a group (same bytes)
        const int row = 8 * g + sub;
        const uint32_t src = (uint32_t)min(m0 + row, p.M - 1);
        xoff[i] = src * (uint32_t)p.ldx + (pch ^ swz((uint32_t)row)) * 16u;
        xdst[i] = (uint32_t)g * 1024u;
        sc_row[i] = src * (uint32_t)p.xs_m;
        sdst[i] = (uint32_t)g * 256u;
        sodd[i] = (g & 1) * 4;
    }
    uint32_t woff[NWW];
#pragma unroll
    for (int i = 0; i < NWW; ++i) {
        const int w = 8 * i + sub;  // LDS row inside the wave's span of 16*TN rows
        const int tn = w >> 4, gg = (w >> 2) & 3, vv = w & 3;
        const int nl = wave * WNS + lane_col<TN>(gg, tn) + vv;
        const int nc = min(n0 + nl, p.N - 1) - n0;
        woff[i] = (uint32_t)nc * (uint32_t)p.ldw + (pch ^ swz((uint32_t)w)) * 16u;
    }
    const uint8_t *wg = p.W + (int64_t)n0 * p.ldw + (int64_t)kb_begin * kBlockK;
    const uint8_t *xg = p.X + (int64_t)kb_begin * kBlockK;
    const uint32_t wdst = (uint32_t)Cfg::kWOff + (uint32_t)wave * (WNS * 128u);
    const uint32_t chunk_off = (uint32_t)Cfg::chunk_off(steps);

    // step `it` in K order, counted from where this tile starts (GemmArgs::turn_mask: 0, or the range is a multiple of 16
    // steps - the scale chunks alternate between their two buffers across the end of the range, too)
    const int rot = TURN ? (int)((5u * tile_n) & (uint32_t)p.turn_mask) : 0;
    auto turn = [&](int it) -> int { return TURN && it + rot >= steps ? it + rot - steps : it + rot; };
    auto issue_w = [&](int slot, int it) {
        const uint32_t sb = lds0 + (uint32_t)slot * Cfg::kWBytes + wdst;
        const uint8_t *wk = wg + (int64_t)turn(it) * kBlockK;
#pragma unroll
        for (int i = 0; i < NWW; ++i) dma_g2l_b128(sb + (uint32_t)i * 1024u, wk, woff[i]);
    };
    auto issue_x = [&](int slot, int it) {
        const uint32_t sb = lds0 + (uint32_t)slot * Cfg::kXBytes;
        const uint8_t *xk = xg + (int64_t)turn(it) * kBlockK;
#pragma unroll
        for (int i = 0; i < NXW; ++i) dma_g2l_b128(sb + xdst[i], xk, xoff[i]);
    };
    auto issue_scales = [&](int chunk) {
        const float *base = p.Xs + (int64_t)(kb_begin + 8 * chunk) * p.xs_k;
#pragma unroll
        for (int i = 0; i < NXW; ++i) {
            const uint32_t st = (uint32_t)min((lane & 7) ^ sodd[i], steps - 1 - 8 * chunk) * (uint32_t)p.xs_k;
            dma_g2l_b32(lds0 + chunk_off + (uint32_t)(chunk & 1) * Cfg::kChunkBytes + sdst[i], base, (sc_row[i] + st) * 4u);
        }
    };

    // ---- per-lane LDS read offsets
    const uint32_t fr = swz((uint32_t)r16);
    const uint32_t c0 = ((uint32_t)(2 * g4)) ^ fr, c1 = c0 ^ 1u;
    const uint32_t xr0 = (uint32_t)r16 * 128u + c0 * 16u, xr1 = (uint32_t)r16 * 128u + c1 * 16u;
    const uint32_t wr0 = wdst + xr0, wr1 = wdst + xr1;
    const uint32_t sr8 = chunk_off + (uint32_t)r16 * 32u;

    // ---- the W scales of the tile's n blocks go to LDS once
    auto issue_w_scales = [&]() {
        const int nb0 = n0 / kBlockN, last = (p.N + kBlockN - 1) / kBlockN - 1 - nb0, count = Cfg::NBLK * steps;
        const float *base = p.Ws + (int64_t)nb0 * p.ws_n + (int64_t)kb_begin * p.ws_k;
        const bool near = p.ws_n >= 0 && p.ws_k >= 0 && p.ws_n < (1 << 27) && p.ws_k < (1 << 27) / steps;  // 32-bit byte offsets
        for (int i0 = 64 * wave; i0 < count; i0 += Cfg::kThreads) {
            const int i = i0 + lane, b = (i >= steps ? 1 : 0) + (Cfg::NBLK > 2 && i >= 2 * steps ? 1 : 0), it = i - b * steps;
            if (i < count) {
                if (near) dma_g2l_b32(lds0 + (uint32_t)(Cfg::kWsOff + i0 * 4), base, (uint32_t)(min(b, last) * (int)p.ws_n + it * (int)p.ws_k) * 4u);
                else ((float *)(lds + Cfg::kWsOff))[i] = base[min(b, last) * p.ws_n + it * p.ws_k];
            }
        }
    };
    // ---- first requests, in the order of the steady state: step j issues W(j+NSW), then X(j+NSX) (kWFirst: X(j+NSX), then
    // W(j+NSW+1)).  A scale chunk is requested by the step behind the one that requests its first X block, or earlier: it has to
    // be older than the W rows that may be in flight when that block is waited for.  The W scales stand behind what step 0
    // multiplies and ahead of what may be in flight when step 0 is waited for (ahead of everything else they cost a short K 0.3 to
    // 0.5 us: 30 x 52776 x 256 6.8 / 6.4 us, 76 x 58128 x 256 8.7 / 8.2, 20 x 52336 x 640 10.0 / 9.7).
    constexpr int kAhead = kWFirst ? 1 : 0;
#pragma unroll
    for (int j = -3; j < 0; ++j) {
        const int wi = j + NSW, xi = j + NSX;
        if (wi >= 0 && wi < steps) issue_w(wi, wi);
        if (wi == 0 && NSX > NSW) issue_w_scales();
        if (xi >= 0 && xi < steps) {
            issue_x(xi, xi);
            if (xi == 0 || (xi < NSX - 1 + kAhead && (turn(xi) & 7) == 0)) issue_scales(turn(xi) >> 3);
        }
        if (wi == 0 && NSX == NSW) issue_w_scales();
    }
    const float *wsl = (const float *)(lds + Cfg::kWsOff) + ((n0 + wave * WNS) / kBlockN - n0 / kBlockN) * steps;

    v4f acc[MT][TN];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};

    // ---- the K loop: while the products of one group of row blocks run, the operands of the next are read from LDS, a read or
    // two behind every product (in one burst all waves would wait for the LDS at the same time)
    v8i wf[2][TN], xf[2][Cfg::G];
    float xs[2][Cfg::G];
    // the k-th operand of a wave's W rows / of a group of X row blocks
    auto operand = [&](const uint8_t *at, uint32_t r0, uint32_t r1) {
        const v4i lo = *(const v4i *)(at + r0), hi = *(const v4i *)(at + r1);
        return v8i{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    };
    auto read_w = [&](auto k, v8i(&f)[TN], const uint8_t *st) { f[k.value] = operand(st + k.value * 2048, wr0, wr1); };
    auto read_x = [&](auto k, auto buf, auto group, const uint8_t *st, const float *sp) {
        constexpr int block = Cfg::group_at(group.value) + k.value;
        xf[buf.value][k.value] = operand(st + block * 2048, xr0, xr1);
        xs[buf.value][k.value] = sp[block * 128];
    };
    auto x_scales = [&](int kb) { return (const float *)(lds + sr8 + ((kb >> 3) & 1) * Cfg::kChunkBytes + ((kb & 7) ^ (r16 >> 3) * 4) * 4); };
    int xslot = 0, wslot = 0;
    // before the products of group g
    auto enter_group = [&](auto g, auto left, int it) {
        constexpr int L = left.value;
        if constexpr (L > 0 && g.value == Cfg::NG - 2) {
            // this wave's W rows and X groups of step it + 1 have landed; X(it+2), W(it+2) and W(it+3) may be in flight
            wait_vmcnt<(L >= 2 && NSX == 3 ? NXW : 0) + (L >= 2 ? NWW : 0) + (L >= 3 && NSW == 3 ? NWW : 0)>();
        } else if constexpr (L > 0 && g.value == Cfg::NG - 1) {
            // step it + 1 is visible to all; everyone has read all of X(it) (the reads behind those of X are of the wave's own W rows)
            lds_barrier<kWFirst ? 0 : 2 * TN>();
            if constexpr (L >= NSX) issue_x(xslot, it + NSX);
            if constexpr (kWFirst && L > NSW) issue_w(wslot + 1 == NSW ? 0 : wslot + 1, it + 1 + NSW);
        }
    };
    // One step with `left` (kLeft: as many or more) steps behind it.  It has no branch: with one between the products the compiler
    // moves the folds behind it and keeps every product in registers until then.
    auto step = [&](auto left, int it, const v8i(&w)[TN], v8i(&wn)[TN]) {
        constexpr int NG = Cfg::NG, L = left.value;
        const int xnext = xslot + 1 == NSX ? 0 : xslot + 1, wnext = wslot + 1 == NSW ? 0 : wslot + 1;
        const uint8_t *st = lds + xslot * Cfg::kXBytes;
        const int kb = turn(it);
        if constexpr (!kWFirst && L >= NSW) {
            wait_lgkm<0>();  // the rows of W(it) have been read
            issue_w(wslot, it + NSW);
        }
        const float ws_cur = wsl[kb];
        const float *sp = x_scales(kb), *sp_next = x_scales(L > 0 ? turn(it + 1) : 0);
        // what is read during group g: the row blocks of the next group, behind the last one those of the next step, and during
        // the last but one also the W rows of the next step
        auto reads = [](int g) {
            return g + 1 < NG ? Cfg::group_at(g + 2) - Cfg::group_at(g + 1) + (L > 0 && g == NG - 2 ? TN : 0) : L > 0 ? Cfg::group_at(1) : 0;
        };
        auto read = [&](auto k, auto g) {
            using Buf = std::integral_constant<int, (g.value & 1) ^ 1>;
            if constexpr (g.value + 1 < NG) {
                constexpr int n = Cfg::group_at(g.value + 2) - Cfg::group_at(g.value + 1);
                if constexpr (k.value == n) __builtin_amdgcn_sched_barrier(0);
                if constexpr (k.value < n) read_x(k, Buf{}, std::integral_constant<int, g.value + 1>{}, st, sp);
                else read_w(std::integral_constant<int, k.value - n>{}, wn, lds + wnext * Cfg::kWBytes);
            } else {
                read_x(k, Buf{}, std::integral_constant<int, 0>{}, lds + xnext * Cfg::kXBytes, sp_next);
            }
        };
        constexpr int E = MT * TN, kLag = 2;
        v4f parts[kLag + 1];
        float sc[3];  // of the row blocks whose products are on their way
        static_for<E + kLag>([&](auto at) {
            constexpr int e = at.value, ge = e < E ? Cfg::group_of(e / TN) : NG - 1;
            constexpr int e0 = Cfg::group_at(ge) * TN, n = (Cfg::group_at(ge + 1) - Cfg::group_at(ge)) * TN;
            if constexpr (e < E && e == e0) {
                if constexpr (ge == NG - 1 && Cfg::group_at(ge) == 0)  // (one row block: the first group is empty)
                    enter_group(std::integral_constant<int, 0>{}, left, it);
                if constexpr (ge == NG - 1 && Cfg::group_at(ge) == 0) static_for<reads(0)>([&](auto k) { read(k, std::integral_constant<int, 0>{}); });
                enter_group(std::integral_constant<int, ge>{}, left, it);
            }
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (e < E) {
                parts[e % (kLag + 1)] = mfma_16x16x128_fp8(w[e % TN], xf[ge & 1][e / TN - Cfg::group_at(ge)], v4f{0.f, 0.f, 0.f, 0.f});
                if constexpr (e % TN == 0) sc[e / TN % 3] = xs[ge & 1][e / TN - Cfg::group_at(ge)] * ws_cur;
                constexpr int R = reads(ge), r0 = (e - e0) * R / n, r1 = (e - e0 + 1) * R / n;
                static_for_from<r0, r1>([&](auto k) { read(k, std::integral_constant<int, ge>{}); });
            }
            if constexpr (e >= kLag) {
                constexpr int f = e - kLag;
                acc[f / TN][f % TN] += parts[f % (kLag + 1)] * sc[f / TN % 3];
            }
            if constexpr (e < E && e >= kLag) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // the MFMA first,
                __builtin_amdgcn_sched_group_barrier(0x100, 6, 0);  // the reads,
                __builtin_amdgcn_sched_group_barrier(0x002, 5, 0);  // an older product's fold behind it
            }
        });
        __builtin_amdgcn_sched_barrier(0);
        xslot = xnext;
        wslot = wnext;
    };
    // step 0 has landed (what follows it in the order of the first requests may be in flight)
    if (steps >= 3) wait_vmcnt<(NSX - 1) * NXW + (NSW - 1) * NWW>();
    else if (steps == 2) wait_vmcnt<NXW + NWW>();
    else wait_vmcnt<0>();
    lds_barrier();
    static_for<TN>([&](auto k) { read_w(k, wf[0], lds); });
    static_for<Cfg::group_at(1)>(
        [&](auto k) { read_x(k, std::integral_constant<int, 0>{}, std::integral_constant<int, 0>{}, lds, x_scales(turn(0))); });
    // the scale chunks that start with one of the X blocks [a, b]
    auto scales_from = [&](int a, int b) {
        for (int xi = a; xi <= b; ++xi)
            if ((turn(xi) & 7) == 0) issue_scales(turn(xi) >> 3);
    };
    if (kWFirst && steps > NSW) {
        wait_lgkm<0>();
        issue_w(0, NSW);
    }
    constexpr int kLeft = kWFirst ? 4 : 3;
    int it = 0;
    for (; it + kLeft + 1 < steps; it += 2) {
        scales_from(it + NSX - 1 + kAhead, it + NSX + kAhead);
        step(std::integral_constant<int, kLeft>{}, it, wf[0], wf[1]);
        step(std::integral_constant<int, kLeft>{}, it + 1, wf[1], wf[0]);
    }
    // the last steps, each an instantiation of its own: the last one on wf[0], the one before on wf[1] and so on
    scales_from(it + NSX - 1 + kAhead, steps - 1);
    if ((steps - it) % 2 == 0) {
#pragma unroll
        for (int j = 0; j < TN; ++j) wf[1][j] = wf[0][j];
    }
    static_for<kLeft>([&](auto i) {
        constexpr int left = kLeft - i.value;
        if (steps - it > left) step(std::integral_constant<int, left>{}, steps - 1 - left, wf[left & 1], wf[(left & 1) ^ 1]);
    });
    step(std::integral_constant<int, 0>{}, steps - 1, wf[0], wf[1]);

    // ---- shared K range: the partial sums go to the workspace in register order ([wave][block][lane] float4);
    // rows128_reduce_kernel adds them in split order and writes C
    if constexpr (SPLIT) {
        constexpr int F = MT * TN;
        float *part = p.partials + ((int64_t)tile_n * p.splits + split) * Cfg::kTileElems + (wave * F * 64 + lane) * 4;
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) *(v4f *)(part + (i * TN + j) * 256) = acc[i][j];
        return;
    }

    // ---- epilogue: lane (r16, g4) holds row 16*i + r16 and the 4*TN columns n0 + 16*TN*wave + 4*TN*g4 + [0, 4*TN)
    const int nbase = n0 + wave * WNS;
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        const int rl = m0 + 16 * i + r16;
        if (rl >= p.M) continue;
        float o[4 * TN];
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int vv = 0; vv < 4; ++vv) o[4 * j + vv] = acc[i][j][vv];
        rows128_store<TN>(p, rl, nbase, g4, o);
    }
}

// Second launch of a shared-K GEMM: thread (tile, wave, row block i, lane) adds its TN accumulator blocks over the
// splits in split order and stores 4*TN consecutive outputs of row 16*i + lane % 16.
template <int MT, int TN>
__global__ __launch_bounds__(256) void rows128_reduce_kernel(const GemmArgs p) {
    using Cfg = Rows128Cfg<MT, TN, 8>;  // K is shared between 8-wave workgroups only
    constexpr int WNS = Cfg::WNS, F = MT * TN;
    const int lane = threadIdx.x & 63;
    const int item = blockIdx.x * 4 + (threadIdx.x >> 6);  // (tile, wave, i)
    const int tiles = (p.N + Cfg::BN - 1) / Cfg::BN;
    if (item >= tiles * Cfg::kWaves * MT) return;
    const int i = item % MT, wave = (item / MT) % Cfg::kWaves, tile_n = item / (MT * Cfg::kWaves);
    const int r16 = lane & 15, g4 = lane >> 4;
    const float *src = p.partials + (int64_t)tile_n * p.splits * Cfg::kTileElems + (wave * F * 64 + lane) * 4 + (i * TN) * 256;
    v4f a[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j) a[j] = *(const v4f *)(src + j * 256);
    int sp = 1;
    for (; sp + 4 <= p.splits; sp += 4) {
        v4f b[4][TN];
#pragma unroll
        for (int d = 0; d < 4; ++d)
#pragma unroll
            for (int j = 0; j < TN; ++j) b[d][j] = *(const v4f *)(src + (int64_t)(sp + d) * Cfg::kTileElems + j * 256);
#pragma unroll
        for (int d = 0; d < 4; ++d)
#pragma unroll
            for (int j = 0; j < TN; ++j) a[j] += b[d][j];
    }
    for (; sp < p.splits; ++sp)
#pragma unroll
        for (int j = 0; j < TN; ++j) a[j] += *(const v4f *)(src + (int64_t)sp * Cfg::kTileElems + j * 256);
    const int rl = 16 * i + r16;
    if (rl >= p.M) return;
    float o[4 * TN];
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int vv = 0; vv < 4; ++vv) o[4 * j + vv] = a[j][vv];
    rows128_store<TN>(p, rl, tile_n * Cfg::BN + wave * WNS, g4, o);
}

}  // namespace mi355
