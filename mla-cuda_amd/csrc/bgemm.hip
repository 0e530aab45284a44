// Large-tile GEMM for the 16-bit (bf16 / fp16) products of many activation rows (a prefill
// chunk, a verify batch of hundreds of tokens): 2a1, 2a2 with 2b in its epilogue, 2c, 3d, the
// KV projection and the output projection.  plan_gemm (gemm.hip) says where it takes over
// from the weight-streaming engine (wgemm.hip), which is built around one 128-row tile, and
// which products are too small for its tiles and stay on the tiled engine.
//
// What bounds it: the 16-bit matrix cores, if the operands arrive in time.  Per 16-deep K
// step a wave of the 256 x 256 tile reads 6 fragments (6 KB) for 8 MFMAs (256 cycles), so
// eight waves draw 96 bytes a clock from LDS and stage 32 more, within what two waves per
// SIMD reach (203); a 128 x 128 tile of four waves needs half as much again and, with one
// wave per SIMD, waits for each step's reads.
//
// Workgroup = 8 wave64s, 2 x 4 over a BM x BN tile (256 x 256, 256 x 128, 128 x 128), each
// wave BM/2 x BN/4 in 32x32 blocks.  K is walked in 32-deep slices through an LDS ring of NS
// stages, both operands global -> LDS with direct-to-LDS loads:
//   A (and W when NT): rows of 64 bytes, 16-byte chunk c of row r at c ^ ((r >> 2) & 3): the
//     16 lanes of a ds_read_b128 cycle (8 rows of one chunk and 8 of the other, or 16 rows of
//     one) touch 16 different 16-byte slots of 256 bytes;
//   W (NN): rows of 2 BN bytes, N-contiguous as in memory, chunk c of row r at c ^ 4(r & 3),
//     read back K-contiguous with the transposing ds_read_b64_tr_b16 (wgemm.hip's layout).
// The fragments are double-buffered in registers a K step ahead.  Slice s + 1 is waited for,
// and the workgroup's one barrier per slice stands, before the last K step of slice s, whose
// fragments are already in registers: the barrier is passed under MFMAs, and after it slice
// s + NS may overwrite slice s.  So NS - 1 slices are in flight at any time.
//
// The grid is what runs at once (one workgroup per CU, two of 128 x 128); a workgroup walks its
// tiles with one unbroken stream of slices, so that the next tile's first ones load while a
// tile's results are written.  16-bit results go through LDS beside the ring (each wave its own
// part, 32 rows at a time) to whole 16-byte stores.
//
// Measured (bf16, tiled engine against this one): o_proj at M = 4096 1,320 -> 796 us (1,210
// TFLOP/s, a large library product of this card 1,163); 2a2 at M = 2048 249 -> 157 us with an
// fp32 result, 254 + 29 (2b) -> 170-183 us with 2b in its epilogue; 2a1 at M = 2048 144 -> 60 us
// in 5 splits, whose sum makes 2a-n 7.8 -> 15.7 us (as a product with its reduction launch
// 148 -> 67); 2c at M = 2048 214 -> 93-95 us (with a workgroup per tile 107-116),
// 3d at M = 4096 195 -> 155 us (188).
#include <algorithm>

#include "kernels.h"
#include "mma.h"
#include "stage.h"

namespace mla {

namespace {

typedef float v2f __attribute__((ext_vector_type(2)));

constexpr int kBThreads = 512;
constexpr int kBKS = 32;          // K per slice
constexpr int kBGroupM = 8;       // M tiles walked before the next N tile

struct BArgs {
    const uint16_t* A; int64_t lda, sAg;
    const uint16_t* B; int64_t ldb, sBg;
    float* C; uint16_t* C16; int64_t ldc, sCg;   // split == 1: one of them
    float* ws; int64_t ws_split;                 // split > 1: partials [split][G][M][N]
    int M, N, K, G, split, k_chunk, tiles_m, tiles_n;
    QUpEpilogue q;                               // QUP kernels: 2a2 with 2b
};

template <typename TL, int BM, int BN, int NS, int MINB, bool NT, bool QUP>
__global__ void __launch_bounds__(kBThreads, MINB) bgemm_kernel(BArgs a) {
    static_assert(!NT || !QUP, "2a2 reads N-contiguous W");
    constexpr int RB = BM / 64, CB = BN / 128;         // 32x32 blocks per wave
    constexpr int kAStage = BM * 2 * kBKS, kBStage = BN * 2 * kBKS;
    constexpr int kStage = kAStage + kBStage;
    constexpr int kLoadsA = kAStage / 8192, kLoadsB = kBStage / 8192;   // 1 KB loads per wave
    constexpr int kLoads = kLoadsA + kLoadsB;
    constexpr int kBRow = 2 * BN;                      // NN: bytes per W row of a slice
    constexpr int kCols = BN / 4, kRowB = 2 * kCols;   // a wave's columns, 16-bit result row
    constexpr int kOutWave = 32 * kRowB;               // 16-bit results of one block row
    constexpr int kOutLanes = kRowB / 16, kOutRows = 64 / kOutLanes;    // per 16-byte store
    constexpr int kStores = BM / 2 / kOutRows;         // 16-bit stores of a wave and tile
    // QUP: slices of a tile that hold its rows' cos / sin table (rope = 64: 32 pairs a row)
    constexpr int kTabRow = 32 * 8;
    constexpr int kTab = QUP ? (BM * kTabRow + kStage - 1) / kStage : 0;
    static_assert(kStage % (32 * kTabRow) == 0, "a block row's table rows lie in one stage");
    static_assert(kTab < NS, "the table fits the ring");
    __shared__ __attribute__((aligned(1024))) uint8_t smem[NS * kStage + 8 * kOutWave];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t lds0 = lds_addr(smem);

    // ---- tiles.  XCD x (workgroups b with b % 8 = x) owns a contiguous run of the tile order and
    // its workgroups interleave over it.  One group: within a K split kBGroupM M tiles per N tile,
    // so the workgroups an XCD runs together share A and W panels in L2.  Groups (a head's columns
    // of a row of all heads each): M tiles outermost, every eighth of them starting an eighth of
    // the groups further on, so that what runs at one time covers whole stretches of the rows at
    // different offsets (3d at M = 4096: 169 us against 188 with the groups outermost, which
    // touches 2 KB in every 16 at a pitch of 128 KB).
    const int total = a.tiles_m * a.tiles_n * a.split * a.G;
    const int x = blockIdx.x % kNumXCDs, per = gridDim.x / kNumXCDs;
    const int first = x * (total / kNumXCDs) + min(x, total % kNumXCDs);
    const int t_end = first + total / kNumXCDs + (x < total % kNumXCDs ? 1 : 0);
    const int t_begin = first + blockIdx.x / kNumXCDs;
    if (t_begin >= t_end) return;
    struct Job {
        uint64_t a_base, b_base;    // of the tile's first K slice
        uint32_t a_bytes, b_bytes;  // of a slice: rows (NT: columns) past the matrix lie past them
        int m0, n0, sp, g, nsl;
    };
    auto job_at = [&](int t) __attribute__((always_inline)) {
        int tm, tn;
        Job j;
        if (a.G > 1) {   // split == 1
            tn = t % a.tiles_n;
            const int tg = t / a.tiles_n;
            tm = tg / a.G;
            j.g = (tg % a.G + tm * kNumXCDs / a.tiles_m * (a.G / kNumXCDs)) % a.G;
            j.sp = 0;
        } else {
            const int plane = a.tiles_m * a.tiles_n;
            j.sp = t / plane;
            const int p = t - j.sp * plane;
            const int grp = p / (kBGroupM * a.tiles_n);
            const int gm = min(kBGroupM, a.tiles_m - grp * kBGroupM);
            const int q = p - grp * kBGroupM * a.tiles_n;
            tm = grp * kBGroupM + q % gm;
            tn = q / gm;
            j.g = 0;
        }
        j.m0 = tm * BM;
        j.n0 = tn * BN;
        const int k0 = j.sp * a.k_chunk;
        j.nsl = (min(a.K, k0 + a.k_chunk) - k0) / kBKS;   // whole slices
        j.a_base = reinterpret_cast<uint64_t>(a.A + j.g * a.sAg + (int64_t)j.m0 * a.lda + k0);
        j.b_base = reinterpret_cast<uint64_t>(
            a.B + j.g * a.sBg + (NT ? (int64_t)j.n0 * a.ldb + k0 : (int64_t)k0 * a.ldb + j.n0));
        const int rows = min(BM, a.M - j.m0), cols = min(BN, a.N - j.n0);
        j.a_bytes = (uint32_t)(rows - 1) * (uint32_t)a.lda * 2u + 2u * kBKS;
        j.b_bytes = NT ? (uint32_t)(cols - 1) * (uint32_t)a.ldb * 2u + 2u * kBKS
                       : (uint32_t)(kBKS - 1) * (uint32_t)a.ldb * 2u + 2u * (uint32_t)cols;
        return j;
    };

    // ---- staging: one stream of slices, a tile's K slices (and its table slices) after the
    // other's, NS of them ahead of the MFMAs; past the last tile they load zeros (the same wait
    // counts)
    // rows of 64 bytes: a load covers 16 of them, lane l chunk position l % 4 of row l / 4
    auto krow_off = [&](int row, int64_t ld) __attribute__((always_inline)) {
        return (uint32_t)row * (uint32_t)ld * 2u + 16u * ((lane & 3) ^ ((row >> 2) & 3));
    };
    uint32_t a_voff[kLoadsA], b_voff[kLoadsB];
    #pragma unroll
    for (int q = 0; q < kLoadsA; ++q)
        a_voff[q] = krow_off((BM / 8) * wave + 16 * q + (lane >> 2), a.lda);
    auto set_b_voff = [&](int n0) __attribute__((always_inline)) {
        #pragma unroll
        for (int q = 0; q < kLoadsB; ++q) {
            if constexpr (NT) {
                b_voff[q] = krow_off((BN / 8) * wave + 16 * q + (lane >> 2), a.ldb);
            } else {
                constexpr int kChunks = kBRow / 16, kRows = 1024 / kBRow;
                const int r = (wave * kLoadsB + q) * kRows + lane / kChunks;
                const int c = (lane % kChunks) ^ (4 * (r & 3));
                // columns past N read zeros (N is a multiple of 8: a chunk is inside or outside)
                b_voff[q] = ((uint32_t)r * (uint32_t)a.ldb * 2u + 16u * c) | oob_mask(8 * c, a.N - n0);
            }
        }
    };
    int it = t_begin, is = 0;   // next slice of the stream: tile, slice
    uint32_t ist = 0;           // and its ring stage
    Job ij = job_at(it);
    set_b_voff(ij.n0);
    struct Slice { v4i ra, rb; uint32_t st, tab, tab_mask; };
    auto next_slice = [&]() __attribute__((always_inline)) {
        if (is == ij.nsl + kTab) {   // (here, not after the last slice: its loads still use b_voff)
            is = 0;
            it += per;
            if (it < t_end) {
                ij = job_at(it);
                set_b_voff(ij.n0);
            } else {
                ij.a_bytes = ij.b_bytes = 0;
                ij.a_base = ij.b_base = reinterpret_cast<uint64_t>(a.A);
                ij.nsl = 0x40000000;   // never a table slice
            }
        }
        Slice d;
        d.st = __builtin_amdgcn_readfirstlane(lds0 + ist * kStage);
        ist = ist + 1 == NS ? 0 : ist + 1;
        d.tab = 0;
        d.tab_mask = 0;
        if (!QUP || is < ij.nsl) {
            d.ra = rsrc_span(ij.a_base + 2ull * kBKS * (uint64_t)is, 0, ij.a_bytes);
            d.rb = rsrc_span(ij.b_base + 2ull * kBKS * (uint64_t)is * (NT ? 1ull : (uint64_t)a.ldb), 0,
                             ij.b_bytes);
        } else {
            // the rows' cos / sin table (2a-n wrote it; rope / 2 pairs a row), linear in the stages
            const int rows = min(BM, a.M - ij.m0);
            d.ra = rsrc_span(reinterpret_cast<uint64_t>(a.q.cos_sin + (int64_t)ij.m0 * a.q.rope), 0,
                             (uint32_t)rows * (uint32_t)a.q.rope * 4u);
            d.rb = d.ra;
            d.tab = (uint32_t)(is - ij.nsl) * kStage;
            d.tab_mask = ~0u;
        }
        ++is;
        return d;
    };
    auto issue = [&](const Slice& d, int q) __attribute__((always_inline)) {
        const uint32_t off = q < kLoadsA ? (uint32_t)(wave * kLoadsA + q) * 1024u
                                         : kAStage + (uint32_t)(wave * kLoadsB + q - kLoadsA) * 1024u;
        uint32_t v = q < kLoadsA ? a_voff[q < kLoadsA ? q : 0] : b_voff[q < kLoadsA ? 0 : q - kLoadsA];
        if constexpr (QUP) v ^= (v ^ (d.tab + off + 16u * lane)) & d.tab_mask;
        dma16(q < kLoadsA ? d.ra : d.rb, d.st + off, v);
    };

    // ---- fragments: wave (wm, wn) covers rows (BM/2) wm .. and columns (BN/4) wn ..
    const int wm = wave >> 2, wn = wave & 3;
    uint32_t a_rd[RB], b_rd[CB];
    #pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
        const int row = (BM / 2) * wm + 32 * rb + (lane & 31);
        a_rd[rb] = (uint32_t)row * 64u + 16u * ((lane >> 5) ^ ((row >> 2) & 3));
    }
    const int G4 = lane >> 4, q4 = (lane >> 2) & 3, i4 = lane & 3;
    #pragma unroll
    for (int cb = 0; cb < CB; ++cb) {
        if constexpr (NT) {
            const int n = (BN / 4) * wn + 32 * cb + (lane & 31);
            b_rd[cb] = kAStage + (uint32_t)n * 64u + 16u * ((lane >> 5) ^ ((n >> 2) & 3));
        } else {
            const int chunk = ((BN / 4) * wn + 32 * cb + 16 * (G4 & 1) + 4 * i4) / 8;
            b_rd[cb] = kAStage + (uint32_t)(8 * (G4 >> 1) + q4) * kBRow +
                       16u * (chunk ^ (4 * q4)) + 8u * (i4 & 1);
        }
    }
    typedef short v4s __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) v4s lds_v4s;
    auto a_frag = [&](uint32_t st, int kt, int rb) __attribute__((always_inline)) {
        return *reinterpret_cast<const v4u*>(smem + st + (a_rd[rb] ^ (32u * kt)));
    };
    auto b_frag = [&](uint32_t st, int kt, int cb) __attribute__((always_inline)) {
        if constexpr (NT) {
            return *reinterpret_cast<const v4u*>(smem + st + (b_rd[cb] ^ (32u * kt)));
        } else {
            const uint32_t o = st + b_rd[cb] + (uint32_t)(16 * kt) * kBRow;
            const v4s lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s*)(smem + o));
            const v4s hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s*)(smem + o + 4 * kBRow));
            return __builtin_bit_cast(v4u, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
        }
    };

    v4u af[2][RB], bf[2][CB];
    v16f acc[RB][CB];
    // One K step: the MFMAs of buffer `cur` with the next step's fragment reads (from stage
    // `st`, step kt, into the other buffer) and, after the barrier, a slice's loads between them.
    auto step = [&](int cur, bool read, uint32_t st, int kt, const Slice* d) __attribute__((always_inline)) {
        #pragma unroll
        for (int rb = 0; rb < RB; ++rb) {
            if (read) {
                if (rb == 0) {
                    #pragma unroll
                    for (int cb = 0; cb < CB; ++cb) bf[cur ^ 1][cb] = b_frag(st, kt, cb);
                }
                af[cur ^ 1][rb] = a_frag(st, kt, rb);
            }
            #pragma unroll
            for (int cb = 0; cb < CB; ++cb)
                acc[rb][cb] = Mma<TL>::sub(af[cur][rb], bf[cur][cb], 0, acc[rb][cb]);
            if (d) {
                constexpr int n = (kLoads + RB - 1) / RB;
                #pragma unroll
                for (int q = rb * n; q < (rb + 1) * n && q < kLoads; ++q) issue(*d, q);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };

    #pragma unroll
    for (int s = 0; s < NS; ++s) {
        const Slice d = next_slice();
        #pragma unroll
        for (int q = 0; q < kLoads; ++q) issue(d, q);
    }
    uint32_t u = 0;   // ring stage of the slice the MFMAs take next
    auto after = [&](uint32_t v) __attribute__((always_inline)) { return v + 1 == NS ? 0u : v + 1; };
    const bool out16 = QUP || a.C16;
    #pragma unroll 1
    for (int t = t_begin; t < t_end; t += per) {
        const Job job = job_at(t);
        // The tile's first slice has landed.  The loads still allowed are older than the tile
        // before's stores, so those need not have completed (their number is fixed for 16-bit C:
        // buffer stores, issued whether in range or not).
        if (!QUP && a.C16 && t != t_begin) wait_vm<(NS - 1) * kLoads + kStores>();
        else wait_vm<(NS - 1) * kLoads>();
        lds_barrier();
        #pragma unroll
        for (int cb = 0; cb < CB; ++cb) bf[0][cb] = b_frag(u * kStage, 0, cb);
        #pragma unroll
        for (int rb = 0; rb < RB; ++rb) af[0][rb] = a_frag(u * kStage, 0, rb);
        #pragma unroll
        for (int rb = 0; rb < RB; ++rb)
            #pragma unroll
            for (int cb = 0; cb < CB; ++cb) acc[rb][cb] = v16f{};
        #pragma unroll 1
        for (int s = 1; s < job.nsl; ++s) {
            const uint32_t st = u * kStage;
            u = after(u);
            step(0, true, st, 1, nullptr);
            const Slice d = next_slice();
            wait_vm<(NS - 2) * kLoads>();      // slice s has landed
            lds_barrier();                     // every wave's part of it; slice s - 1 is in registers
            step(1, true, u * kStage, 0, &d);  // the slice NS further into the stage of slice s - 1
        }
        {
            const uint32_t st = u * kStage;
            u = after(u);
            step(0, true, st, 1, nullptr);
            const Slice d = next_slice();
            lds_barrier();                     // the last slice is in registers
            step(1, false, 0, 0, &d);
        }

        const int64_t row0 = job.m0 + (BM / 2) * wm;
        const int col0 = job.n0 + (BN / 4) * wn;
        const int qk = a.q.nope + a.q.rope;
        // the epilogue's lane-dependent offsets stay inside the tile loop (hoisted out of it they
        // would hold registers through the main loop)
        int lane_e = lane;
        asm volatile("" : "+v"(lane_e));
        const int lane = lane_e;
        const bool odd = lane & 1;
        if constexpr (QUP) {
            // 2b on the rope columns.  A 32-column block lies inside one head's nope or rope part;
            // the pair partner of column c is column c ^ 1, the neighbouring lane.  (Read from
            // global memory here, block by block, the table cost 2a2 104 us of 264 at M = 2048.)
            wait_vm<(NS - kTab) * kLoads>();   // the table has landed
            lds_barrier();
            #pragma unroll
            for (int cb = 0; cb < CB; ++cb) {
                const int j0 = (col0 + 32 * cb) % qk;
                if (j0 < a.q.nope) continue;
                // 32 table rows (8 KB) lie in one stage: a uniform base, this lane's row and pair,
                // and a constant per accumulator element
                const uint32_t mine = (uint32_t)(4 * (lane >> 5)) * kTabRow +
                                      4u * (uint32_t)((j0 - a.q.nope + (lane & 31)) & ~1);
                #pragma unroll
                for (int rb = 0; rb < RB; ++rb) {
                    const uint32_t o = (uint32_t)((BM / 2) * wm + 32 * rb) * kTabRow;
                    const uint8_t* const tab = smem + (u + o / kStage) % NS * kStage + o % kStage + mine;
                    #pragma unroll
                    for (int e = 0; e < 16; ++e) {
                        const v2f cs = *reinterpret_cast<const v2f*>(tab + (8 * (e >> 2) + (e & 3)) * kTabRow);
                        const float own = acc[rb][cb][e], other = dpp_move<0xB1>(own);
                        acc[rb][cb][e] = odd ? rope_odd(other, own, cs[0], cs[1])
                                             : rope_even(own, other, cs[0], cs[1]);
                    }
                }
            }
            lds_barrier();   // every wave is done with the table: its stages take the next slices
            #pragma unroll
            for (int i = 0; i < kTab; ++i) {
                const Slice d = next_slice();
                #pragma unroll
                for (int q = 0; q < kLoads; ++q) issue(d, q);
                u = after(u);
            }
        }
        if (out16) {
            // ---- 16-bit results, a block row (32 rows) at a time through this wave's part of LDS:
            // 16-byte chunk c of row r at c ^ (r & 7) (64 columns) or c ^ (r & 3) (32 columns)
            constexpr int kSw = kCols == 64 ? 7 : 3;
            uint8_t* const mine = smem + NS * kStage + wave * kOutWave;
            const int c = lane % kOutLanes, col = col0 + 8 * c;
            uint16_t* dst = nullptr;
            int64_t ld = 0;
            if constexpr (QUP) {
                const int h = col / qk, j = col - h * qk;
                const bool rope = j >= a.q.nope;
                ld = (int64_t)a.q.H * (rope ? a.q.rope : a.q.nope);
                dst = rope ? static_cast<uint16_t*>(a.q.q_rope) + (int64_t)h * a.q.rope + j - a.q.nope
                           : static_cast<uint16_t*>(a.q.q_nope) + (int64_t)h * a.q.nope + j;
            }
            const __amdgpu_buffer_rsrc_t rc = make_rsrc(a.C16 + (int64_t)job.g * a.sCg + (int64_t)job.m0 * a.ldc);
            const uint32_t cmask = oob_mask(col, a.N);
            #pragma unroll
            for (int rb = 0; rb < RB; ++rb) {
                #pragma unroll
                for (int cb = 0; cb < CB; ++cb) {
                    const int c2 = 32 * cb + ((lane & 31) & ~1);
                    #pragma unroll
                    for (int e = 0; e < 16; e += 2) {
                        const float x0 = acc[rb][cb][e], x1 = acc[rb][cb][e + 1];
                        const float p0 = dpp_move<0xB1>(x0), p1 = dpp_move<0xB1>(x1);
                        const int row = acc_row(odd ? e + 1 : e, lane);
                        const uint32_t w = odd ? Half<TL>::pack2(p1, x1) : Half<TL>::pack2(x0, p0);
                        *reinterpret_cast<uint32_t*>(mine + row * kRowB + 16 * ((c2 >> 3) ^ (row & kSw)) +
                                                     2 * (c2 & 7)) = w;
                    }
                }
                __builtin_amdgcn_wave_barrier();
                #pragma unroll
                for (int i = 0; i < 32 / kOutRows; ++i) {
                    const int r = i * kOutRows + lane / kOutLanes;
                    const v4u v = *reinterpret_cast<const v4u*>(mine + r * kRowB + 16 * (c ^ (r & kSw)));
                    const int64_t row = row0 + 32 * rb + r;
                    if constexpr (QUP) {
                        if (row < a.M && col < a.N) *reinterpret_cast<v4u*>(dst + row * ld) = v;
                    } else {
                        const uint32_t off = (uint32_t)((BM / 2) * wm + 32 * rb + r) * (uint32_t)a.ldc * 2u +
                                             2u * (uint32_t)col;
                        __builtin_amdgcn_raw_buffer_store_b128(v, rc, (int)(off | cmask | oob_mask((int)row, a.M)), 0, 0);
                    }
                }
                __builtin_amdgcn_wave_barrier();
            }
        } else {
            float* out;
            int64_t ld;
            if (a.split > 1) {
                out = a.ws + (int64_t)job.sp * a.ws_split + (int64_t)job.g * a.M * a.N;
                ld = a.N;
            } else {
                out = a.C + (int64_t)job.g * a.sCg;
                ld = a.ldc;
            }
            #pragma unroll
            for (int rb = 0; rb < RB; ++rb)
                #pragma unroll
                for (int cb = 0; cb < CB; ++cb) {
                    const int col = col0 + 32 * cb + (lane & 31);
                    #pragma unroll
                    for (int e = 0; e < 16; ++e) {
                        const int64_t row = row0 + 32 * rb + acc_row(e, lane);
                        if (row < a.M && col < a.N) out[row * ld + col] = acc[rb][cb][e];
                    }
                }
        }
    }
    wait_vm<0>();    // the loads past the last tile have landed: none may outlive the workgroup's LDS
}

template <typename TL, bool NT, bool QUP>
hipError_t launch_bgemm_t(const BArgs& a, const GemmPlan& plan, dim3 grid, hipStream_t stream) {
    const dim3 block(kBThreads);
    if (plan.bm == 256 && plan.bn == 256)
        hipLaunchKernelGGL((bgemm_kernel<TL, 256, 256, 4, 2, NT, QUP>), grid, block, 0, stream, a);
    else if (plan.bm == 256 && plan.bn == 128)
        hipLaunchKernelGGL((bgemm_kernel<TL, 256, 128, 6, 2, NT, QUP>), grid, block, 0, stream, a);
    else if (plan.bm == 128 && plan.bn == 128)
        hipLaunchKernelGGL((bgemm_kernel<TL, 128, 128, 4, 4, NT, QUP>), grid, block, 0, stream, a);
    else
        return hipErrorInvalidValue;
    return hipGetLastError();
}

}  // namespace

bool bgemm_tile(int bm, int bn) {
    return (bm == 256 && (bn == 256 || bn == 128)) || (bm == 128 && bn == 128);
}

bool bgemm_supported(const GemmProblem& p, int bm, int bn, int split) {
    const OutType own16 = p.f16 ? kOutF16 : kOutBF16;
    return p.half && !p.a_f32 && p.amode == kAPlain && split >= 1 && bgemm_tile(bm, bn) &&
           (p.out_type == kOutF32 || split > 1 || p.out_type == own16) && !p.k_len && !p.b_pages &&
           p.M > 0 && p.G >= 1 && (p.G == 1 || split == 1) &&   // job_at's order of groups has no splits
           p.N % 8 == 0 && p.K % kBKS == 0 && p.lda >= kBKS &&
           (p.b_nt ? p.ldb >= p.K : p.ldb >= p.N) &&
           // 16-byte aligned rows and groups, of the operands and of a 16-bit C
           p.lda % 8 == 0 && p.ldb % 8 == 0 && p.sAg % 8 == 0 && p.sBg % 8 == 0 &&
           (p.out_type == kOutF32 || split > 1 || (p.ldc % 8 == 0 && p.sCg % 8 == 0)) &&
           // 32-bit buffer offsets within a tile, a 16-bit C's too (its columns among them)
           (p.out_type == kOutF32 || split > 1 || ((int64_t)bm * p.ldc + p.N) * 2 < kRsrcRange) &&
           (int64_t)bm * p.lda * 2 < kRsrcRange &&
           (int64_t)(p.b_nt ? bn : kBKS) * p.ldb * 2 < kRsrcRange;
}

bool bgemm_aligned(const GemmProblem& p) {
    auto low = [](const void* x) { return reinterpret_cast<uintptr_t>(x) & 15; };
    if (low(p.A) || low(p.B)) return false;
    if (p.qup) return !low(p.qup->q_nope) && !low(p.qup->q_rope) && !(reinterpret_cast<uintptr_t>(p.qup->cos_sin) & 7);
    return !low(p.C);
}

hipError_t launch_bgemm(const GemmProblem& p, const GemmPlan& plan, float* partials,
                        hipStream_t stream) {
    if (!bgemm_supported(p, plan.bm, plan.bn, plan.split) || !bgemm_aligned(p) ||
        plan.k_chunk <= 0 || plan.k_chunk % kBKS != 0 || (int64_t)plan.k_chunk * plan.split < p.K ||
        (int64_t)plan.k_chunk * (plan.split - 1) >= p.K || (plan.split > 1 && !partials))
        return hipErrorInvalidValue;
    BArgs a;
    a.A = static_cast<const uint16_t*>(p.A); a.lda = p.lda; a.sAg = p.sAg;
    a.B = static_cast<const uint16_t*>(p.B); a.ldb = p.ldb; a.sBg = p.sBg;
    const bool c16 = p.out_type != kOutF32 && plan.split == 1;
    a.C = c16 ? nullptr : static_cast<float*>(p.C); a.ldc = p.ldc; a.sCg = p.sCg;
    a.C16 = c16 ? static_cast<uint16_t*>(p.C) : nullptr;
    a.ws = partials; a.ws_split = (int64_t)p.G * p.M * p.N;
    a.M = p.M; a.N = p.N; a.K = p.K; a.G = p.G;
    a.split = plan.split; a.k_chunk = plan.k_chunk;
    a.tiles_m = (p.M + plan.bm - 1) / plan.bm;
    a.tiles_n = (p.N + plan.bn - 1) / plan.bn;
    const int64_t tiles = (int64_t)a.tiles_m * a.tiles_n * a.split * a.G;
    if (tiles <= 0 || tiles > 0x3fffffff || (int64_t)a.tiles_m * kNumXCDs > 0x7fffffff) return hipErrorInvalidValue;
    // as many workgroups as run at once, a multiple of the XCDs; each walks its XCD's tiles
    const int64_t resident = (int64_t)kNumCUs * (plan.bm == 128 ? 2 : 1);
    const dim3 grid((unsigned)(std::min(tiles, resident) + kNumXCDs - 1) / kNumXCDs * kNumXCDs);
    if (p.qup) {
        // the rope epilogue alone (rope = 64): 2c is its own launch on this engine
        if (plan.split != 1 || p.qup->w_uk || p.qup->rope != 64 || !qup_supported(p, *p.qup, plan)) return hipErrorInvalidValue;
        a.q = *p.qup;
        return p.f16 ? launch_bgemm_t<f16_t, false, true>(a, plan, grid, stream)
                     : launch_bgemm_t<bf16_t, false, true>(a, plan, grid, stream);
    }
    if (p.b_nt)
        return p.f16 ? launch_bgemm_t<f16_t, true, false>(a, plan, grid, stream)
                     : launch_bgemm_t<bf16_t, true, false>(a, plan, grid, stream);
    return p.f16 ? launch_bgemm_t<f16_t, false, false>(a, plan, grid, stream)
                 : launch_bgemm_t<bf16_t, false, false>(a, plan, grid, stream);
}

}  // namespace mla
