// Large-tile GEMM for the 16-bit (bf16 / fp16) products of many activation rows (a prefill
// chunk, a verify batch of hundreds of tokens): 2a1, 2a2 with 2b in its epilogue, 2c, 3d, the
// KV projection and the output projection.  plan_gemm (gemm.hip) says where it takes over
// from the weight-streaming engine (wgemm.hip), which is built around one 128-row tile.
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
// 16-bit results go through LDS (each wave its own part) to whole 16-byte stores.
//
// Measured (bf16, tiled engine against this one): o_proj at M = 4096 1,320 -> 808 us (1,190
// TFLOP/s, a large library product of this card 1,163), at M = 1332 634 -> 336 us; 2a2 at
// M = 2048 251 -> 160 us with an fp32 result, 254 + 29 (2b) -> 181-188 us with 2b in its
// epilogue; 2a1 at M = 2048 125 -> 62 us with the sum of its splits.
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
    constexpr int kWaveOut = (BM / 2) * (BN / 4) * 2;  // 16-bit results of a wave
    static_assert(8 * kWaveOut <= NS * kStage, "the results fit the ring");
    __shared__ __attribute__((aligned(1024))) uint8_t smem[NS * kStage];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // Tile order: an XCD walks a contiguous run; within a (group, split) plane kBGroupM M
    // tiles per N tile, so the workgroups an XCD runs together share A and W panels in L2.
    const int t = xcd_logical_block(blockIdx.x, gridDim.x);
    const int plane_tiles = a.tiles_m * a.tiles_n;
    const int plane = t / plane_tiles, in_plane = t - plane * plane_tiles;
    const int grp = in_plane / (kBGroupM * a.tiles_n);
    const int gm = min(kBGroupM, a.tiles_m - grp * kBGroupM);
    const int in_grp = in_plane - grp * kBGroupM * a.tiles_n;
    const int tm = grp * kBGroupM + in_grp % gm, tn = in_grp / gm;
    const int sp = plane % a.split, g = plane / a.split;
    const int m0 = tm * BM, n0 = tn * BN;
    const int k_begin = sp * a.k_chunk;
    const int nsl = (min(a.K, k_begin + a.k_chunk) - k_begin) / kBKS;   // whole slices
    const int rows_a = min(BM, a.M - m0), cols_b = min(BN, a.N - n0);

    // ---- staging
    const uint32_t lds0 = lds_addr(smem);
    const uint64_t a_base = reinterpret_cast<uint64_t>(a.A + g * a.sAg + (int64_t)m0 * a.lda);
    const uint64_t b_base = reinterpret_cast<uint64_t>(
        a.B + g * a.sBg + (NT ? (int64_t)n0 * a.ldb : (int64_t)n0));
    // rows of 64 bytes: a load covers 16 of them, lane l chunk position l % 4 of row l / 4
    auto krow_off = [&](int row, int64_t ld) __attribute__((always_inline)) {
        return (uint32_t)row * (uint32_t)ld * 2u + 16u * ((lane & 3) ^ ((row >> 2) & 3));
    };
    uint32_t a_voff[kLoadsA], b_voff[kLoadsB];
    #pragma unroll
    for (int q = 0; q < kLoadsA; ++q)
        a_voff[q] = krow_off((BM / 8) * wave + 16 * q + (lane >> 2), a.lda);
    #pragma unroll
    for (int q = 0; q < kLoadsB; ++q) {
        if constexpr (NT) {
            b_voff[q] = krow_off((BN / 8) * wave + 16 * q + (lane >> 2), a.ldb);
        } else {
            constexpr int kChunks = kBRow / 16, kRows = 1024 / kBRow;
            const int r = (wave * kLoadsB + q) * kRows + lane / kChunks;
            const int c = (lane % kChunks) ^ (4 * (r & 3));
            // columns past N read zeros (N is a multiple of 8: a chunk is inside or outside)
            b_voff[q] = ((uint32_t)r * (uint32_t)a.ldb * 2u + 16u * c) | oob_mask(8 * c, cols_b);
        }
    }
    // bytes of a slice: rows past rows_a (NT: cols_b) lie past them
    const uint32_t a_bytes = (uint32_t)(rows_a - 1) * (uint32_t)a.lda * 2u + 2u * kBKS;
    const uint32_t b_bytes = NT ? (uint32_t)(cols_b - 1) * (uint32_t)a.ldb * 2u + 2u * kBKS
                                : (uint32_t)(kBKS - 1) * (uint32_t)a.ldb * 2u + 2u * (uint32_t)cols_b;
    const uint32_t tab_bytes = QUP ? (uint32_t)rows_a * (uint32_t)a.q.rope * 4u : 0u;
    struct Slice { v4i ra, rb; uint32_t st; int tab; };   // tab: table part, or -1
    auto slice_of = [&](int s) __attribute__((always_inline)) {
        const int k = k_begin + s * kBKS;
        const bool live = s < nsl;   // slices past the range load zeros (the same wait counts)
        Slice d;
        d.st = __builtin_amdgcn_readfirstlane(lds0 + (uint32_t)(s % NS) * kStage);
        d.ra = rsrc_span(a_base + 2ull * (uint64_t)k, 0, live ? a_bytes : 0u);
        d.rb = rsrc_span(b_base + 2ull * (uint64_t)k * (NT ? 1ull : (uint64_t)a.ldb), 0,
                         live ? b_bytes : 0u);
        d.tab = -1;
        if constexpr (QUP) {
            if (!live) {
                d.tab = s - nsl;
                d.ra = rsrc_span(reinterpret_cast<uint64_t>(a.q.cos_sin + (int64_t)m0 * a.q.rope), 0,
                                 tab_bytes);
            }
        }
        return d;
    };
    // QUP: the tile rows' cos / sin table (2a-n wrote it; rope / 2 pairs a row, at most 64 KB)
    // takes the place of the first slices past the K range, byte i kStage + j of it at byte j
    // of slice nsl + i's stage: the loads the loop issues there anyway, waited for after it.
    // (Read from global memory in the epilogue, block by block, it cost 2a2 104 us of 264 at
    // M = 2048.)
    static_assert(!QUP || NS * kStage >= BM * 256 + kStage, "the table fits the free stages");
    auto issue = [&](const Slice& d, int q, bool table) __attribute__((always_inline)) {
        if (table) {
            const uint32_t off = (uint32_t)(wave * kLoads + q) * 1024u;
            dma16(d.ra, d.st + off, (uint32_t)d.tab * kStage + off + 16u * lane, 0);
            return;
        }
        if (q < kLoadsA)
            dma16(d.ra, d.st + (uint32_t)(wave * kLoadsA + q) * 1024u, a_voff[q], 0);
        else
            dma16(d.rb, d.st + kAStage + (uint32_t)(wave * kLoadsB + q - kLoadsA) * 1024u,
                  b_voff[q - kLoadsA], 0);
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

    v16f acc[RB][CB];
    #pragma unroll
    for (int rb = 0; rb < RB; ++rb)
        #pragma unroll
        for (int cb = 0; cb < CB; ++cb) acc[rb][cb] = v16f{};

    #pragma unroll
    for (int s = 0; s < NS; ++s) {
        const Slice d = slice_of(s);
        #pragma unroll
        for (int q = 0; q < kLoads; ++q) issue(d, q, QUP && s >= nsl);
    }
    wait_vm<(NS - 1) * kLoads>();   // slice 0 has landed
    lds_barrier();
    v4u af[2][RB], bf[2][CB];
    #pragma unroll
    for (int cb = 0; cb < CB; ++cb) bf[0][cb] = b_frag(0, 0, cb);
    #pragma unroll
    for (int rb = 0; rb < RB; ++rb) af[0][rb] = a_frag(0, 0, rb);

    // One K step: the MFMAs of buffer `cur` with the next step's fragment reads (from stage
    // `st`, step kt, into the other buffer) and, after the barrier, a slice's loads between them.
    auto step = [&](int cur, uint32_t st, int kt, const Slice* d, bool table) __attribute__((always_inline)) {
        #pragma unroll
        for (int rb = 0; rb < RB; ++rb) {
            if (rb == 0)
                #pragma unroll
                for (int cb = 0; cb < CB; ++cb) bf[cur ^ 1][cb] = b_frag(st, kt, cb);
            af[cur ^ 1][rb] = a_frag(st, kt, rb);
            #pragma unroll
            for (int cb = 0; cb < CB; ++cb)
                acc[rb][cb] = Mma<TL>::sub(af[cur][rb], bf[cur][cb], 0, acc[rb][cb]);
            if (d) {
                constexpr int per = (kLoads + RB - 1) / RB;
                #pragma unroll
                for (int q = rb * per; q < (rb + 1) * per && q < kLoads; ++q) issue(*d, q, table);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    auto slice = [&](int s, bool table) __attribute__((always_inline)) {
        const uint32_t st = (uint32_t)(s % NS) * kStage, st1 = (uint32_t)((s + 1) % NS) * kStage;
        step(0, st, 1, nullptr, false);
        const Slice d = slice_of(s + NS);
        wait_vm<(NS - 2) * kLoads>();   // slice s + 1 has landed
        lds_barrier();                  // every wave's part of it; slice s is in registers
        step(1, st1, 0, &d, table);     // slice s + NS into the stage of slice s
    };
    int s = 0;
    if constexpr (QUP) {
        #pragma unroll 1
        for (; s < nsl - NS; ++s) slice(s, false);
    }
    #pragma unroll 1
    for (; s < nsl; ++s) slice(s, QUP);
    wait_vm<0>();    // the loads past the range have landed
    lds_barrier();   // every wave's, and every wave is done with the ring

    const int64_t row0 = m0 + (BM / 2) * wm;
    const int col0 = (BN / 4) * wn;
    if (QUP || a.C16) {
        // ---- 16-bit results (2a2: the rope columns rotated), through this wave's part of LDS:
        // rows of BN/4 columns, 16-byte chunk c of row r at c ^ (r & 7) (BN/4 = 32: c ^ (r & 3))
        constexpr int kCols = BN / 4, kRowB = 2 * kCols, kSw = kCols == 64 ? 7 : 3;
        uint8_t* const mine = smem + wave * kWaveOut;
        const bool odd = lane & 1;
        const int qk = a.q.nope + a.q.rope;
        if constexpr (QUP) {
            // a 32-column block lies inside one head's nope or rope part; the pair partner of
            // column c is column c ^ 1, the neighbouring lane
            #pragma unroll
            for (int cb = 0; cb < CB; ++cb) {
                const int j0 = (n0 + col0 + 32 * cb) % qk;
                if (j0 < a.q.nope) continue;
                const int i = (j0 - a.q.nope + (lane & 31)) >> 1;
                #pragma unroll
                for (int rb = 0; rb < RB; ++rb)
                    #pragma unroll
                    for (int e = 0; e < 16; ++e) {
                        const int row = (BM / 2) * wm + 32 * rb + acc_row(e, lane);
                        const uint32_t o = (uint32_t)row * (uint32_t)a.q.rope * 4u + 8u * i;
                        const uint32_t part = o / kStage;
                        const v2f cs = *reinterpret_cast<const v2f*>(
                            smem + ((uint32_t)nsl + part) % NS * kStage + (o - part * kStage));
                        const float own = acc[rb][cb][e], other = dpp_move<0xB1>(own);
                        acc[rb][cb][e] = odd ? rope_odd(other, own, cs[0], cs[1])
                                             : rope_even(own, other, cs[0], cs[1]);
                    }
            }
            lds_barrier();   // every wave is done with the table
        }
        #pragma unroll
        for (int rb = 0; rb < RB; ++rb)
            #pragma unroll
            for (int cb = 0; cb < CB; ++cb) {
                const int c2 = 32 * cb + ((lane & 31) & ~1);
                #pragma unroll
                for (int e = 0; e < 16; e += 2) {
                    const float x0 = acc[rb][cb][e], x1 = acc[rb][cb][e + 1];
                    const float p0 = dpp_move<0xB1>(x0), p1 = dpp_move<0xB1>(x1);
                    const int row = 32 * rb + acc_row(odd ? e + 1 : e, lane);
                    const uint32_t w = odd ? Half<TL>::pack2(p1, x1) : Half<TL>::pack2(x0, p0);
                    *reinterpret_cast<uint32_t*>(mine + row * kRowB + 16 * ((c2 >> 3) ^ (row & kSw)) +
                                                 2 * (c2 & 7)) = w;
                }
            }
        __builtin_amdgcn_wave_barrier();
        // 16 bytes per lane, kRowB / 16 lanes a row; only this wave's own values are read
        constexpr int kLanes = kRowB / 16, kPer = 64 / kLanes;
        const int c = lane % kLanes, col = n0 + col0 + 8 * c;
        uint16_t* dst;
        int64_t ld;
        if constexpr (QUP) {
            const int h = col / qk, j = col - h * qk;
            const bool rope = j >= a.q.nope;
            ld = (int64_t)a.q.H * (rope ? a.q.rope : a.q.nope);
            dst = rope ? static_cast<uint16_t*>(a.q.q_rope) + (int64_t)h * a.q.rope + j - a.q.nope
                       : static_cast<uint16_t*>(a.q.q_nope) + (int64_t)h * a.q.nope + j;
        } else {
            ld = a.ldc;
            dst = a.C16 + (int64_t)g * a.sCg + col;
        }
        #pragma unroll
        for (int i = 0; i < BM / 2 / kPer; ++i) {
            const int r = i * kPer + lane / kLanes;
            const v4u v = *reinterpret_cast<const v4u*>(mine + r * kRowB + 16 * (c ^ (r & kSw)));
            if (row0 + r < a.M && col < a.N) *reinterpret_cast<v4u*>(dst + (row0 + r) * ld) = v;
        }
        return;
    }
    float* out;
    int64_t ld;
    if (a.split > 1) {
        out = a.ws + (int64_t)sp * a.ws_split + (int64_t)g * a.M * a.N;
        ld = a.N;
    } else {
        out = a.C + (int64_t)g * a.sCg;
        ld = a.ldc;
    }
    #pragma unroll
    for (int rb = 0; rb < RB; ++rb)
        #pragma unroll
        for (int cb = 0; cb < CB; ++cb) {
            const int col = n0 + col0 + 32 * cb + (lane & 31);
            #pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int64_t row = row0 + 32 * rb + acc_row(e, lane);
                if (row < a.M && col < a.N) out[row * ld + col] = acc[rb][cb][e];
            }
        }
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
           p.M > 0 && p.G >= 1 && p.N % 8 == 0 && p.K % kBKS == 0 && p.lda >= kBKS &&
           (p.b_nt ? p.ldb >= p.K : p.ldb >= p.N) &&
           // 16-byte aligned rows and groups, of the operands and of a 16-bit C
           p.lda % 8 == 0 && p.ldb % 8 == 0 && p.sAg % 8 == 0 && p.sBg % 8 == 0 &&
           (p.out_type == kOutF32 || split > 1 || (p.ldc % 8 == 0 && p.sCg % 8 == 0)) &&
           // 32-bit buffer offsets within a tile
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
    const int64_t blocks = (int64_t)a.tiles_m * a.tiles_n * a.split * a.G;
    if (blocks <= 0 || blocks > 0x7fffffff) return hipErrorInvalidValue;
    const dim3 grid((unsigned)blocks);
    if (p.qup) {
        // the rope epilogue alone: 2c is its own launch on this engine
        if (plan.split != 1 || p.qup->w_uk || !qup_supported(p, *p.qup, plan)) return hipErrorInvalidValue;
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
