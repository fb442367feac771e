// W4A8: fp8 (e4m3) activations x int4 weights on the CDNA4 fp8 matrix core.
//
// Semantics of the reference's W4A8 path (fpA_intB runner instantiated for __nv_fp8_e4m3 x uint4
// with half scales, cpp/tensorrt_llm/kernels/cutlass_kernels/fpA_intB_gemm/fpA_intB_gemm_template.h,
// selected by weightOnlyGroupwiseQuantMatmulPlugin.cpp:203-276): the int4 weight is dequantized
// with fp16 scales/zeros and rounded to e4m3, the MMA accumulates fp8 x fp8 products in float32,
// and the epilogue applies alpha and the bias: out = T(alpha * acc + bias).  Group sizes: 128 and its
// multiples (the reference's pre-Hopper launcher takes 128 only, fpA_intB_gemm_template.h:136-142; its
// Hopper launcher any multiple of the K tile, launchers/fpA_intB_launcher_sm90.inl:190-198).
//
// Output tile 16*RT rows x 256 columns, 8 wavefronts side by side along N with 32 columns each (two a SIMD: one issues
// under the other's waits); packed weights go global -> registers and are dequantized once per workgroup, between the
// MFMAs; the activation tile is DMA-ed global -> LDS; skinny problems split K through the float32 partial buffer.
// Requests run three steps of 128 rows of K ahead, into four LDS buffers and register stages: a wavefront waits for
// nothing it requested less than two steps ago, and reads the next step's first operands before the barrier.
// The matrix instruction is the CDNA4 v_mfma_f32_32x32x64_f8f6f4 (e4m3 x e4m3): twice the work of a 16x16x128 one for an
// issue slot.  A lane supplies 32 k-values of its row / column; which 32 is free as long as A
// and B agree: lane (kh, row) takes the 16 values 32 j + 16 kh ... of two slabs j, two neighbouring chunks of the weight
// layout and one 16-byte read of the activations each.
// An fp8 activation fragment is half the size of a 16-bit one, so LDS holds fragment PAIRS: 16
// rows x 64 k = 1 KiB, written by one DMA instruction (lane 4r+q fetches row r's 16-byte chunk
// q ^ (r>>2): quads read 64 contiguous bytes, the XOR spreads the reads of a block's rows over the banks).
// Measured (bf16 output, group 128, no zero-points, us; before: four wavefronts of 64 columns, 16x16x128 instructions,
// two buffers, arithmetic conversion): 4096 x 28672 at 64 / 1990 / 8192 rows 55.9 -> 26.8 / 234 -> 198 / 851 -> 737 (2.61
// PFLOP/s), 8192 x 57344 at 128 / 256 rows 119 -> 69.6 / 116 -> 107, 4096 x 4096 at 1990 rows 54.3 -> 36.2 (128-row tiles).
// With zero-points, on another box: 4096 x 28672 at 1990 / 8192 rows 255 -> 200 / 908 -> 753, 8192 x 57344 at 1024 rows 475 -> 393.
// By step, 8192 x 57344 at 128 rows: 32x32x64 109, eight wavefronts 88, three steps ahead 75, look-up conversion 70.
// What bounds it (profiles/gemm_w4a8_gate_up_m4096.md): 128-row tiles the conversions (8192 x 57344 at 128 rows: the vector unit
// issues for 68 % of the cycles, the matrix core is busy for 53 %, and half of the vector work runs under matrix
// instructions); 256-row ones the matrix core (4096 x 28672 at 4096 rows: busy for 76 %; vector unit 54 %, LDS 38 %) and the clock
// that it brings down to 1.54 GHz.
#include "gemm_common.h"
#include "w4a8_common.h"

namespace woq
{

// PERSIST (256-row tiles, whole K, bf16 output, no bias): one workgroup per CU walks tiles b, b + grid, ...
// as the 16-bit prefill kernel does (gemm_kernel.h): the last steps of a tile already request the
// first weights and A tiles of the next one, and a finished tile's outputs are read out of
// the accumulators, scaled, packed and stored right before the matrix instruction that starts each
// block's new sum.  The 8 us or so that a tile spends outside its main loop (first loads, the
// conversion of the first operand set, 128 KiB of stores, the relaunch) weigh twice as much here as
// there: a tile's main loop is half as long.
constexpr int kW4a8Waves = 8;
constexpr int kOneTile = 0, kPersistPairs = 1, kPersist = 2; // persistent forms: steps in pairs (any even K), in fours

constexpr uint32_t kLdsReach = 0x10000; // of an LDS instruction's immediate offset
template <bool UPPER>
struct W4a8Buf // one activation tile in LDS
{
    static constexpr bool upper = UPPER;
    u32x4* data;
};

template <int ODT, bool ZERO, int RT, bool SPLITK, int LOOP = kOneTile>
__global__ void __launch_bounds__(kW4a8Waves * 64) __attribute__((amdgpu_waves_per_eu(2, 2))) gemm_w4a8_kernel(GemmParams p)
{
    constexpr bool PERSIST = LOOP != kOneTile, DEEP = LOOP != kPersistPairs;
    constexpr int NW = kW4a8Waves;
    static_assert(!PERSIST || (RT == 16 && !SPLITK && ODT == WOQ_BF16), "persistent form: 256-row tiles, whole K, bf16 out");
    using EO = Elem<ODT>;
    constexpr int TK = 128, NS = 16 / NW;
    constexpr int BM = RT * 16;
    constexpr int BLK = 32, RB = BM / BLK, CB = NS * 16 / BLK; // 32 x 32 blocks of a wavefront along M and N
    constexpr int KI = TK / 64;                                // matrix instructions along a tile row
    constexpr int PAIRS = RT * 2;      // fragment pairs (1 KiB) of one A tile
    constexpr int A_BYTES = BM * TK;   // e4m3: one byte per element
    static_assert(PAIRS % NW == 0 && CB == 1, "one column block a wavefront; fragment pairs spread evenly over the wavefronts");

    __shared__ u32x4 a_lds0[A_BYTES / 16];
    __shared__ u32x4 a_lds1[A_BYTES / 16];
    __shared__ u32x4 a_lds2[A_BYTES / 16];
    __shared__ u32x4 a_lds3[A_BYTES / 16];
    constexpr bool UPPER = 4 * A_BYTES > (int) kLdsReach; // buffers 2 and 3 lie beyond what an LDS read's immediate offset reaches
    W4a8Buf<false> const a_buf0{a_lds0}, a_buf1{a_lds1};
    W4a8Buf<UPPER> const a_buf2{a_lds2}, a_buf3{a_lds3};

    // Tile of virtual block vb (the block index, or with PERSIST the block index plus a multiple of the
    // grid size, which is a multiple of 8): XCD-contiguous chunks of the tile order, m fastest inside
    // groups of 4 m-tiles - the 32 workgroups of an XCD then cover about 4 x 8 tiles and share 4
    // activation panels and 8 weight panels in its L2 instead of all 16 activation panels and 2
    int const total = p.tiles_m * p.tiles_n;
    int const per_xcd = (total + 7) / 8;
    auto tile_of = [&](int vb, int& tm_, int& tn_) -> bool
    {
        int t = (vb & 7) * per_xcd + (vb >> 3);
        bool const exists = (vb >> 3) < per_xcd && t < total;
        t = exists ? t : 0; // (no branch: the persistent loop's registers do not survive one between its steps)
        constexpr int kGroupM = 4;
        int const in_group = kGroupM * p.tiles_n;
        int const first_m = (t / in_group) * kGroupM;
        int const gsz = p.tiles_m - first_m < kGroupM ? p.tiles_m - first_m : kGroupM;
        tm_ = first_m + (t % in_group) % gsz;
        tn_ = (t % in_group) / gsz;
        return exists;
    };
    int vb = (int) blockIdx.x;
    int tm, tn;
    if (!tile_of(vb, tm, tn))
        return;

    int const lane = threadIdx.x & 63;
    int const wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int const row_in = lane & 31, kh = lane >> 5; // row of a block, half of K that the lane feeds
    int const K = p.k;
    int const kt_begin = SPLITK ? (int) blockIdx.y * p.tiles_per_split : 0;
    int const KT = SPLITK ? (kt_begin + p.tiles_per_split < p.k_tiles ? kt_begin + p.tiles_per_split : p.k_tiles)
                          : p.k_tiles;
    int m0 = tm * BM;
    int strip0 = tn * (kGemmBN / 16) + wave * NS;

    constexpr uint32_t kOob = 0x80000000u;
    auto const act_rsrc = make_rsrc(p.act, (uint32_t) p.m * (uint32_t) K);
    uint32_t const sz_bytes = (uint32_t) p.scale_rows * (uint32_t) p.n * 2u;
    // table row of tile row kt (w4a8_scale_row) without its case distinction, which becomes a branch in the persistent
    // loop: kt itself for groups of 128, else kt / (group / 128), as the upper half of 2 kt * ceil(2^31 / (group / 128))
    uint32_t const magic = p.group_magic ? (p.group_magic >> 1) + (p.group_magic & 1u) : 0x80000000u;
    auto const sc_rsrc = make_rsrc(p.scales, sz_bytes);
    auto const zr_rsrc = make_rsrc(ZERO ? p.zeros : p.scales, sz_bytes);
    auto const w_rsrc = make_rsrc(p.weight, (uint32_t) p.strips * (uint32_t) p.k_tiles * 1024u);

    // per-lane request addresses of one tile (PERSIST keeps those of the next tile beside them)
    struct TileCtx
    {
        uint32_t wlane[CB], sc_lane[CB]; // column blocks of two strips; chunks 2 kh and 2 kh + 1 of the lane's column
        uint32_t dma_lane_base;
        uint32_t oob; // kOob: there is no such tile, every request reads zeros
    };
    // Which weight column a lane feeds to row row_in of its block is free.  A block's sums come back with lane
    // (kh, row_in) holding operand rows 8 g + 4 kh + e, g, e = 0 ... 3 (register 4 g + e): dealt out so that these are
    // the 16 consecutive columns of strip kh of the pair (two 16-byte accesses per output row), or, for the split-K form,
    // whose blocks are not transposed, operand row = column (a store covers 128 consecutive bytes)
    int const lane_slot = SPLITK ? row_in >> 4 : (row_in >> 2) & 1;
    int const lane_col = SPLITK ? row_in & 15 : (row_in >> 3) * 4 + (row_in & 3);
    auto make_ctx = [&](int tm_, int tn_, bool valid) -> TileCtx
    {
        TileCtx x;
        int const first = tn_ * (kGemmBN / 16) + wave * NS;
#pragma unroll
        for (int cb = 0; cb < CB; ++cb)
        {
            int const want = first + 2 * cb + lane_slot, strip = want < p.strips ? want : p.strips - 1;
            x.wlane[cb] = ((uint32_t) strip * (uint32_t) p.k_tiles * 64u + (uint32_t) (kh * 32 + lane_col)) * 16u;
            x.sc_lane[cb] = (uint32_t) (strip * 16 + lane_col) * 2u;
        }
        // A tile -> LDS: wavefront w moves pairs w, w+8, ...: piece i is pair f = w + 8i = half w % 2 of
        // row tile 4i + w / 2
        x.dma_lane_base = (uint32_t) (tm_ * BM + (wave / 2) * 16 + (lane >> 2)) * (uint32_t) K
            + (uint32_t) ((wave % 2) * 64 + (((lane & 3) ^ ((lane >> 4) & 3)) * 16));
        x.oob = valid ? 0u : 0x80000000u;
        return x;
    };
    TileCtx cur = make_ctx(tm, tn, true);

    f32x16 acc[RB][CB];
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int cb = 0; cb < CB; ++cb)
            acc[rb][cb] = f32x16{};

    // ---- A tile -> LDS; K is a multiple of 128, so only kt >= KT falls out of range (rows past M fall
    // outside the descriptor by themselves).
    constexpr int DMA_OPS = PAIRS / NW;
    uint32_t const dma_piece_stride = (uint32_t) NW * 8u * (uint32_t) K;
    auto dma_base = [&](int kt, TileCtx const& x) -> uint32_t
    { return (x.dma_lane_base + (uint32_t) kt * (uint32_t) TK) | ((uint32_t) (KT - 1 - kt) & kOob) | x.oob; };
    auto dma_piece = [&](auto buf, uint32_t base, int i)
    {
        int const f = wave + i * NW;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(act_rsrc,
            (__attribute__((address_space(3))) void*) (reinterpret_cast<char*>(buf.data) + f * 1024), 16,
            (int) (base + (uint32_t) i * dma_piece_stride), 0, 0, 0);
    };
    // Matrix instruction ki of a tile row covers slabs 2 ki and 2 ki + 1; lane (kh, row_in) supplies the 16 values
    // 32 j + 16 kh ... of each - two consecutive chunks of 8 of the weight layout, one 16-byte read of the activations:
    // chunk (j & 1) * 2 + kh of row row_in % 16 in fragment pair ki, stored at position chunk ^ swizzle (the phases of a
    // 128-bit LDS read take rows 0-3, 12-15 of one fragment and rows 4-11 of the other: all banks, no conflict)
    uint32_t a_lane_off[2];
#pragma unroll
    for (int jj = 0; jj < 2; ++jj)
        a_lane_off[jj] = (uint32_t) ((row_in >> 4) * 2048 + ((row_in & 15) * 4 + ((jj * 2 + kh) ^ ((row_in >> 2) & 3))) * 16);

    // The immediate offset of an LDS read reaches 64 KiB.  With 256-row tiles the buffers 2 and 3 lie beyond it, and the compiler,
    // which does not split an offset, kept an address register for each of their 32 reads: 14 of them (with zero-points; ten
    // without) in scratch memory, whose reloads waited for every request in flight.  These are the same offsets as seen
    // from 64 KiB on, which it is not told (4096 x 28672 at 1990 / 8192 rows with zero-points 210 -> 200 / 788 -> 753 us, without
    // 202 -> 198 / 763 -> 745)
    uint32_t a_lane_upper[2];
#pragma unroll
    for (int jj = 0; jj < 2; ++jj)
    {
        a_lane_upper[jj] = a_lane_off[jj] + kLdsReach;
        if constexpr (UPPER)
            asm volatile("" : "+v"(a_lane_upper[jj]));
    }

    struct BStage
    {
        u32x4 w[NS]; // [column block][chunk 2 kh, 2 kh + 1]
        uint32_t s[CB]; // (32 bits: a 16-bit loop variable is merged into its register by an instruction that waits for the load)
        uint32_t z[CB];
    };
    constexpr int FETCH_OPS = NS + CB * (ZERO ? 2 : 1);
    auto fetch_piece = [&](BStage& st, int kt, int i, TileCtx const& x)
    {
        uint32_t const past = ((uint32_t) (KT - 1 - kt) & kOob) | x.oob; // kt >= KT: every load of the step reads zeros
        if (i < NS)
            st.w[i] = buffer_load_x4(w_rsrc, x.wlane[i / 2] + (((uint32_t) kt * 1024u | past) + (uint32_t) (i % 2 * 256)));
        else
        {
            int const s = (i - NS) % CB;
            uint32_t const off = (__umulhi((uint32_t) kt * 2u, magic) * (uint32_t) p.n * 2u + x.sc_lane[s]) | past;
            if (i < NS + CB)
                st.s[s] = buffer_load_u16(sc_rsrc, off);
            else
                st.z[s] = buffer_load_u16(zr_rsrc, off);
        }
    };

    // ---- one step = one tile row of K = KI * RB iterations of one MFMA.  Iteration (ki, rb)
    // issues the activation reads of the operand A_AHEAD ahead, its share of the memory requests
    // and of the conversions, then the MFMA of the row block.
    // The operands of one instruction along K (8 registers) are all there is of converted weights: while the row blocks
    // are multiplied with those of ki = 0, ki = 1 of the same step is converted, meanwhile ki = 0 of the next step.
    // Conversion is a look-up (w4a8_common.h): a (group, column) has sixteen possible e4m3 results; the two lanes that feed
    // a column each compute eight of them - the same FMA and saturating conversion as dequant4_fp8, so the bytes are
    // identical, with zero-points or without - and exchange them.  15 instructions per eight weights against 21 issue slots
    // of the arithmetic form (the conversion instruction takes two).
    constexpr int A_AHEAD = 2;
    // Two row blocks: the conversions end right in front of the next matrix instruction, which reads them
    constexpr bool B_JUST_WRITTEN = RB <= 2;
    Fp8LookupConsts const lut = fp8_lookup_consts();
    f16x2 qv[4]; // the lane's eight signed values 8 kh - 8 ... 8 kh - 1, as halves for mixed-precision FMAs
#pragma unroll
    for (int i = 0; i < 4; ++i)
        qv[i] = f16x2{(_Float16) (8 * kh - 8 + 2 * i), (_Float16) (8 * kh - 7 + 2 * i)};
    constexpr int TABLE_PARTS = 6; // of a table's construction: four pairs of entries, two exchanges
    auto table_part = [&](Fp8Table& T, BStage const& st, int part)
    {
        if (part < 4)
        {
            _Float16 const sh = bit_cast<_Float16>((uint16_t) st.s[0]);
            _Float16 const zh = bit_cast<_Float16>((uint16_t) (ZERO ? st.z[0] : 0u));
            float const v0 = __builtin_fmaf((float) qv[part][0], (float) sh, (float) zh);
            float const v1 = __builtin_fmaf((float) qv[part][1], (float) sh, (float) zh);
            uint32_t& d = T.t[part / 2];
            d = part % 2 == 0 ? (uint32_t) __builtin_amdgcn_cvt_pk_fp8_f32(v0, v1, 0, false)
                              : (uint32_t) __builtin_amdgcn_cvt_pk_fp8_f32(v0, v1, (int) d, true);
        }
        else // lanes below 32 have entries 0 ... 7, the others 8 ... 15
        {
            uint32_t const own = T.t[part - 4];
            auto const both = __builtin_amdgcn_permlane32_swap(own, own, false, false);
            T.t[part - 4] = both[0];
            T.t[part - 2] = both[1];
        }
    };
    // look-up unit u = (slab parity, load) of instruction ki: eight weights -> two registers of its operand
    constexpr int UNITS = 4;
    auto unit_word = [&](BStage const& st, int ki, int u) { return st.w[u & 1][2 * ki + (u >> 1)]; };
    auto unit_begin = [&](uint32_t (&part)[4], Fp8Table const& T, BStage const& st, int ki, int u)
    { fp8_lookup8_begin(unit_word(st, ki, u), T, lut, part); };
    auto unit_end = [&](uint32_t const (&part)[4], u32x8& b, BStage const& st, int ki, int u)
    {
        uint32_t lo, hi;
        fp8_lookup8_end(unit_word(st, ki, u), lut, part, lo, hi);
        b[u * 2] = lo;
        b[u * 2 + 1] = hi;
    };

    // PERSIST: where the finished tile's outputs go: byte offset of (row m0 + row_in, column strip0 * 16 + kh * 16)
    // of the tile to store (N is a multiple of the tile width: every strip exists; rows past M fall
    // outside the descriptor); kOob: no finished tile yet
    [[maybe_unused]] auto const out_rsrc = make_rsrc(p.out, (uint32_t) p.m * (uint32_t) p.n * 2u);
    [[maybe_unused]] uint32_t prev_off = kOob;
    [[maybe_unused]] uint32_t const rb_stride = (uint32_t) BLK * (uint32_t) p.n * 2u;
    auto store_block = [&](int rb, int cb)
    {
        // explicit AGPR-source moves: a plain VALU use of the block would pull every accumulator into the
        // VGPR half of the file for the whole loop.  The pack to bf16 does not depend on the conversion
        // mode the main loop runs in (that concerns fp16 and fp8 results only).
#pragma unroll
        for (int h = 0; h < 2; ++h)
        {
            float v[8];
#pragma unroll
            for (int x = 0; x < 8; ++x)
                asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(v[x]) : "a"(acc[rb][cb][h * 8 + x]));
            u32x4 o;
#pragma unroll
            for (int x = 0; x < 8; x += 2)
                o[x / 2] = EO::pack(p.alpha * v[x], p.alpha * v[x + 1]);
            __builtin_amdgcn_raw_buffer_store_b128(
                o, out_rsrc, (int) (prev_off + (uint32_t) rb * rb_stride + (uint32_t) (cb * 64 + h * 16)), 0, 0);
        }
    };

    // One step.  buf / buf_after: the A tiles of this step and (DEEP) of the next one, both landed; the last iterations
    // already read the next step's first operands.  The A tile of tile row kt_a of tile xa goes to buf_req, the packed
    // weights of tile row kt_w of tile xw to st_req - three steps ahead (not DEEP: one and two): the same tile's, or with
    // PERSIST the next tile's first ones.  first_tag: the first step of a tile in the persistent loop.
    constexpr int ITERS = RB * KI;
    constexpr int A_RING = 4; // slots; A_AHEAD + 1 are in use
    static_assert(ITERS % A_RING == 0, "a step starts on slot 0");
    u32x8 a_ring[A_RING];
    auto a_read = [&](auto buf, int it) -> u32x8 // row block it % RB, instruction it / RB of a tile row
    {
        typedef __attribute__((address_space(3))) char const lds_char;
        typedef __attribute__((address_space(3))) u32x4 const lds_u32x4;
        auto const at = [&](int jj) -> u32x4
        {
            uint32_t const c = (uint32_t) ((it % RB) * 4096 + (it / RB) * 1024);
            return *(lds_u32x4*) ((lds_char*) buf.data + (buf.upper ? a_lane_upper[jj] + (c - kLdsReach) : a_lane_off[jj] + c));
        };
        return __builtin_shufflevector(at(0), at(1), 0, 1, 2, 3, 4, 5, 6, 7);
    };
    u32x8 b[KI]; // converted weights, by instruction along K
    auto compute = [&](auto first_tag, auto buf, auto buf_after, Fp8Table const& T, Fp8Table& T_next,
                       BStage const& st, BStage const& st_next, auto buf_req, int kt_a, TileCtx const& xa, BStage& st_req,
                       int kt_w, TileCtx const& xw) __attribute__((always_inline))
    {
        constexpr bool FIRST = decltype(first_tag)::value;
        uint32_t const next_base = dma_base(kt_a, xa);
        if constexpr (!DEEP)
        {
#pragma unroll
            for (int i = 0; i < A_AHEAD; ++i)
                a_ring[i] = a_read(buf, i);
        }
        __builtin_amdgcn_sched_barrier(0);
        uint32_t part[4];
#pragma unroll
        for (int it = 0; it < ITERS; ++it)
        {
            // the A-tile DMAs first, the weight-side requests after them: with kPersistPairs the barrier
            // that ends the step then waits for the DMAs only (vector-memory operations retire in
            // order) and leaves the weight loads, which travel from HBM, a whole further step
            constexpr int DMA_WINDOW = ITERS / 2 > 0 ? ITERS / 2 : 1;
#pragma unroll
            for (int q = 0; q < DMA_OPS; ++q)
                if (q * DMA_WINDOW / DMA_OPS == it)
                    dma_piece(buf_req, next_base, q);
            constexpr int FETCH_FIRST = ITERS / 2, FETCH_WINDOW = ITERS - ITERS / 2 - 1 > 0 ? ITERS - ITERS / 2 - 1 : 1;
#pragma unroll
            for (int q = 0; q < FETCH_OPS; ++q)
                if (FETCH_FIRST + q * FETCH_WINDOW / FETCH_OPS == it)
                    fetch_piece(st_req, kt_w, q, xw);
            if (DEEP || it + A_AHEAD < ITERS)
                a_ring[(it + A_AHEAD) % A_RING]
                    = it + A_AHEAD < ITERS ? a_read(buf, it + A_AHEAD) : a_read(buf_after, it + A_AHEAD - ITERS);
            u32x8 const a_cur = a_ring[it % A_RING];
            int const rb = it % RB, ki = it / RB;
            // weights as the first operand: the accumulator holds the TRANSPOSED block, a lane 16
            // consecutive columns of one output row (16-byte epilogue accesses)
            // (the split-K variant keeps the plain orientation: its float32 stores cover 128 consecutive
            // bytes per row and instruction)
            if constexpr (SPLITK)
                mma_fp8_acc<RT == 16, B_JUST_WRITTEN>(a_cur, b[ki], acc[rb][0]);
            else if (FIRST && ki == 0)
            {
                store_block(rb, 0); // the previous tile's sums leave right before the block starts the new tile's
                mma_fp8_first<RT == 16>(b[ki], a_cur, acc[rb][0]);
            }
            else
                mma_fp8_acc<RT == 16, B_JUST_WRITTEN>(b[ki], a_cur, acc[rb][0]);
            // behind the MFMA its share of the conversions, half units at a time: a wavefront issues in order, so the
            // VALU work has to sit between the matrix instructions to run under them
            BStage const& src = ki == 0 ? st : st_next;
            Fp8Table const& table = ki == 0 ? T : T_next;
#pragma unroll
            for (int half = 0; half < 2 * UNITS; ++half)
                if (half * RB / (2 * UNITS) == rb)
                {
                    if (half % 2 == 0)
                        unit_begin(part, table, src, 1 - ki, half / 2);
                    else
                        unit_end(part, b[1 - ki], src, 1 - ki, half / 2);
                }
            if (ki == 0)
            {
#pragma unroll
                for (int i = 0; i < TABLE_PARTS; ++i)
                    if (i * RB / TABLE_PARTS == rb)
                        table_part(T_next, st_next, i);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };

    // ---- main loop: four steps per iteration so that LDS buffers and weight stages
    // are distinct objects.  Step kt converts ki = 1 of its own weights (stage kt % 4) and ki = 0 of the next step's and
    // requests A tile and weights of step kt+3.  (kPersistPairs: two steps per iteration, two buffers and stages; A tile
    // of step kt+1, weights of step kt+2.)
    BStage st0, st1, st2, st3;
    Fp8Table t0, t1;
    fp8_saturation_on(); // the conversions rely on it; off again before the epilogue
    auto request_a = [&](auto buf, int kt)
    {
        uint32_t const base = dma_base(kt, cur);
#pragma unroll
        for (int i = 0; i < DMA_OPS; ++i)
            dma_piece(buf, base, i);
    };
    auto request_w = [&](BStage& st, int kt)
    {
#pragma unroll
        for (int i = 0; i < FETCH_OPS; ++i)
            fetch_piece(st, kt, i, cur);
    };
    request_a(a_buf0, kt_begin);
    request_w(st0, kt_begin);
    if constexpr (DEEP)
        request_a(a_buf1, kt_begin + 1);
    request_w(st1, kt_begin + 1);
    if constexpr (DEEP)
    {
        request_a(a_buf2, kt_begin + 2);
        request_w(st2, kt_begin + 2);
    }
#pragma unroll
    for (int i = 0; i < TABLE_PARTS; ++i)
        table_part(t0, st0, i);
#pragma unroll
    for (int u = 0; u < UNITS; ++u)
    {
        uint32_t part[4];
        unit_begin(part, t0, st0, 0, u);
        unit_end(part, b[0], st0, 0, u);
    }
    // DEEP: A(kt) and A(kt+1) have landed for every wavefront (the requests of the step before, DMA_OPS + FETCH_OPS loads,
    // may still be out: loads return in order, whatever stores the persistent loop has issued between them); everyone is
    // done reading A(kt-1), whose buffer this step's requests go to.  Else: A(kt) has landed (FETCH_OPS weight-side
    // loads were requested after it).
    auto step_barrier = [&]()
    { asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(DEEP ? DMA_OPS + FETCH_OPS : FETCH_OPS) : "memory"); };
    std::false_type const plain{};
    auto deep_step = [&](auto tag, auto buf, auto buf_after, Fp8Table const& T, Fp8Table& T_next, BStage const& st,
                         BStage const& st_next, auto buf_req, BStage& st_req, int kt, TileCtx const& x) __attribute__((always_inline))
    {
        compute(tag, buf, buf_after, T, T_next, st, st_next, buf_req, kt, x, st_req, kt, x);
        step_barrier();
    };
    // tile rows kt ... kt+3 (past the end of K both operands read as zeros); the last three requests may be another tile's
    auto four_steps = [&](auto tag, int kt, TileCtx const& x, int kt_x) __attribute__((always_inline))
    {
        deep_step(tag, a_buf0, a_buf1, t0, t1, st0, st1, a_buf3, st3, kt + 3, cur);
        deep_step(plain, a_buf1, a_buf2, t1, t0, st1, st2, a_buf0, st0, kt_x, x);
        deep_step(plain, a_buf2, a_buf3, t0, t1, st2, st3, a_buf1, st1, kt_x + 1, x);
        compute(plain, a_buf3, a_buf0, t1, t0, st3, st0, a_buf2, kt_x + 2, x, st2, kt_x + 2, x);
        mma_settle(); // the compiler may move accumulators behind the loop and does not see that they are still being written
        step_barrier();
    };
    if constexpr (DEEP)
    {
        step_barrier();
#pragma unroll
        for (int i = 0; i < A_AHEAD; ++i)
            a_ring[i] = a_read(a_buf0, i);
    }
    if constexpr (!PERSIST)
    {
        int kt = kt_begin;
        for (; kt + 2 < KT; kt += 4)
            four_steps(plain, kt, cur, kt + 4);
        if (kt < KT) // one or two left (leaving the loop from its middle would cost a second copy of the accumulators)
        {
            deep_step(plain, a_buf0, a_buf1, t0, t1, st0, st1, a_buf3, st3, kt + 3, cur);
            compute(plain, a_buf1, a_buf2, t1, t0, st1, st2, a_buf0, kt + 4, cur, st0, kt + 4, cur);
        }
    }
    else
    {
        // Straight-line first and last steps around a plain inner loop (KT a multiple of 4, >= 8; in pairs: even, >= 4; the
        // shape the 16-bit kernel's persistent loop has, for the same reason: every AGPR is an
        // accumulator, and a branch between first-step and ordinary code inside a loop makes the
        // allocator keep second copies of them).  In a tile's last three (two) steps the requests are the next tile's
        // first ones.
        bool has_next;
        do
        {
            int tmn = 0, tnn = 0;
            has_next = tile_of(vb + (int) gridDim.x, tmn, tnn);
            TileCtx const nxt = make_ctx(tmn, tnn, has_next);
            if constexpr (DEEP)
            {
                four_steps(std::true_type{}, 0, cur, 4);
                for (int kt = 4; kt < KT - 4; kt += 4)
                    four_steps(plain, kt, cur, kt + 4);
                four_steps(plain, KT - 4, nxt, 0);
            }
            else
            {
                auto pair = [&](auto tag, int kt, TileCtx const& x, int kt_x) __attribute__((always_inline))
                {
                    step_barrier();
                    compute(tag, a_buf0, a_buf0, t0, t1, st0, st1, a_buf1, kt + 1, cur, st0, kt_x, x);
                    step_barrier();
                    compute(plain, a_buf1, a_buf1, t1, t0, st1, st0, a_buf0, kt_x, x, st1, kt_x + 1, x);
                    mma_settle();
                };
                pair(std::true_type{}, 0, cur, 2);
                for (int kt = 2; kt < KT - 2; kt += 2)
                    pair(plain, kt, cur, kt + 2);
                pair(plain, KT - 2, nxt, 0);
            }
            // this tile's outputs: stored during the next tile's first step (or below)
            prev_off = ((uint32_t) (m0 + row_in) * (uint32_t) p.n + (uint32_t) (strip0 * 16 + kh * 16)) * 2u;
            vb += (int) gridDim.x;
            m0 = tmn * BM;
            strip0 = tnn * (kGemmBN / 16) + wave * NS;
            cur = nxt;
        } while (has_next);
        mma_drain();
        fp8_saturation_off();
#pragma unroll
        for (int rb = 0; rb < RB; ++rb)
#pragma unroll
            for (int cb = 0; cb < CB; ++cb)
                store_block(rb, cb);
        return;
    }

    // ---- epilogue: out = T(alpha * acc + bias), or partial sums into the float32 buffer --------
    mma_drain();
    fp8_saturation_off();
    if constexpr (SPLITK)
    {
        // plain orientation: register 4 g + e is (row rb * 32 + 8 g + 4 kh + e, the lane's own column);
        // this K slice's own slab of the partial buffer (a slice past the end of K stores zeros)
        float* const slab = p.partial + (size_t) blockIdx.y * ((size_t) p.m * p.n);
#pragma unroll
        for (int cb = 0; cb < CB; ++cb)
        {
            int const strip = strip0 + 2 * cb + lane_slot;
#pragma unroll
            for (int rb = 0; rb < RB; ++rb)
#pragma unroll
                for (int r = 0; r < 16; ++r)
                {
                    int const row = m0 + rb * BLK + (r >> 2) * 8 + kh * 4 + (r & 3);
                    if (strip < p.strips && row < p.m)
                        slab[(size_t) row * p.n + strip * 16 + lane_col] = acc[rb][cb][r];
                }
        }
        return;
    }
    uint16_t* out16 = static_cast<uint16_t*>(p.out);
    // a lane holds 16 consecutive columns of output row m0 + rb * 32 + row_in: two 16-byte stores
    typedef __attribute__((address_space(1))) u32x4 global_u32x4;
#pragma unroll
    for (int cb = 0; cb < CB; ++cb)
    {
        int const strip = strip0 + 2 * cb + kh;
        if (strip >= p.strips)
            continue;
#pragma unroll
        for (int h = 0; h < 2; ++h)
        {
            int const col = strip * 16 + h * 8;
            float bias[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
            if (!SPLITK && p.bias)
            {
#pragma unroll
                for (int x = 0; x < 8; ++x)
                    bias[x] = EO::load(p.bias, col + x);
            }
#pragma unroll
            for (int rb = 0; rb < RB; ++rb)
            {
                int const row = m0 + rb * BLK + row_in;
                if (row >= p.m)
                    continue;
                float v[8];
#pragma unroll
                for (int x = 0; x < 8; ++x)
                    v[x] = after_mode_change(__builtin_fmaf(p.alpha, acc[rb][cb][h * 8 + x], bias[x]));
                u32x4 const o = {EO::pack(v[0], v[1]), EO::pack(v[2], v[3]), EO::pack(v[4], v[5]), EO::pack(v[6], v[7])};
                *(global_u32x4*) (out16 + (size_t) row * p.n + col) = o;
            }
        }
    }
}

template <int ODT, bool ZERO, int RT>
int launch_w4a8_variant(GemmParams const& gp, hipStream_t stream)
{
    int const total = gp.tiles_m * gp.tiles_n;
    dim3 grid(((total + 7) / 8) * 8, gp.k_splits), block(kW4a8Waves * 64);
    note_launch("gemm w4a8 rt=%d splits=%d", RT, gp.k_splits);
    if (gp.k_splits > 1)
    {
        size_t const count = (size_t) gp.m * gp.n;
        hipLaunchKernelGGL((gemm_w4a8_kernel<ODT, ZERO, RT, true>), grid, block, 0, stream, gp);
        hipLaunchKernelGGL((gemm_finish_partial<ODT>), dim3((unsigned) ((count / 4 + 255) / 256)), dim3(256), 0, stream,
            gp.out, gp.partial, gp.bias, gp.alpha, gp.m, gp.n, gp.k_splits);
    }
    else
    {
        // 256-row tiles, bf16 out: one persistent workgroup per CU when that means at least two tiles each
        int const cus = gemm_persistent_workgroups();
        bool persist = false;
        if constexpr (RT == 16 && ODT == WOQ_BF16)
            persist = cus > 0 && total > cus && gp.k_tiles % 2 == 0 && gp.k_tiles >= 4 && gp.n % kGemmBN == 0 && !gp.bias
                && (uint64_t) gp.m * (uint64_t) gp.n * 2 < ((uint64_t) 1 << 31)
                // byte offsets of the padded last row tile, and of the rejected offset plus 15 row tiles, stay below 2^32
                && (uint64_t) gp.tiles_m * 256 * (uint64_t) gp.n * 2 < ((uint64_t) 1 << 32) && gp.n < (1 << 22);
        note_launch("gemm w4a8 rt=%d splits=1 persistent=%d", RT, (int) persist);
        if (persist)
        {
            if constexpr (RT == 16 && ODT == WOQ_BF16)
            {
                if (gp.k_tiles % 4 == 0 && gp.k_tiles >= 8)
                    hipLaunchKernelGGL((gemm_w4a8_kernel<ODT, ZERO, RT, false, kPersist>), dim3(cus), block, 0, stream, gp);
                else
                    hipLaunchKernelGGL((gemm_w4a8_kernel<ODT, ZERO, RT, false, kPersistPairs>), dim3(cus), block, 0, stream, gp);
            }
        }
        else
            hipLaunchKernelGGL((gemm_w4a8_kernel<ODT, ZERO, RT, false>), grid, block, 0, stream, gp);
    }
    hipError_t err = hipGetLastError();
    if (err != hipSuccess)
        return fail(WOQ_ERR_RUNTIME, "W4A8 gemm kernel launch failed: %s", hipGetErrorString(err));
    return WOQ_OK;
}

template <int ODT, bool ZERO>
int launch_w4a8_rt(GemmParams const& gp, int rt, hipStream_t s)
{
    switch (rt)
    {
    case 4: return launch_w4a8_variant<ODT, ZERO, 4>(gp, s);
    case 8: return launch_w4a8_variant<ODT, ZERO, 8>(gp, s);
    default: return launch_w4a8_variant<ODT, ZERO, 16>(gp, s);
    }
}

int launch_gemm_w4a8(MatmulProblem const& p, GemmPlan const& plan, void* stream)
{
    GemmParams gp;
    gp.act = p.act;
    gp.weight = p.weight;
    gp.scales = p.scales;
    gp.zeros = p.zeros;
    gp.bias = p.bias;
    gp.out = p.out;
    gp.alpha = p.alpha;
    gp.m = p.m;
    gp.n = p.n;
    gp.k = p.k;
    gp.k_tiles = (p.k + 127) / 128;
    gp.strips = p.n / kTileN;
    gp.scale_rows = (p.k + p.group_size - 1) / p.group_size;
    gp.group_magic = w4a8_scale_row_magic(p.group_size);
    gp.tiles_m = (p.m + plan.rt * 16 - 1) / (plan.rt * 16);
    gp.tiles_n = (p.n + kGemmBN - 1) / kGemmBN;
    gp.k_splits = plan.k_splits;
    gp.tiles_per_split = (gp.k_tiles + plan.k_splits - 1) / plan.k_splits;
    gp.tiles_per_split += gp.tiles_per_split & 1; // the main loop walks tile rows in pairs
    gp.partial = static_cast<float*>(p.workspace);
    if (plan.k_splits > 1 && (!p.workspace || p.workspace_bytes < plan.ws_bytes))
        return fail(WOQ_ERR_WORKSPACE, "split-K needs %zu workspace bytes", plan.ws_bytes);
    auto s = static_cast<hipStream_t>(stream);
    bool const zero = p.zeros != nullptr;
    if (p.out_dtype == WOQ_BF16)
        return zero ? launch_w4a8_rt<WOQ_BF16, true>(gp, plan.rt, s) : launch_w4a8_rt<WOQ_BF16, false>(gp, plan.rt, s);
    return zero ? launch_w4a8_rt<WOQ_FP16, true>(gp, plan.rt, s) : launch_w4a8_rt<WOQ_FP16, false>(gp, plan.rt, s);
}

} // namespace woq
