// 8 to 512 rows without a barrier in the main loop: the rows between the decode kernels and the tall prefill tiles
// (the reference covers them with CUTLASS tiles of 16 ... 64 rows and split-K,
// cpp/tensorrt_llm/kernels/cutlass_kernels/cutlass_heuristic.cpp:59-140).
//
// On narrow matrices the tiled kernels spend most of such a launch outside its arithmetic: a barrier every 128 rows of K
// with one to three steps' requests in flight, and a K split across workgroups whose float32 slabs need a second launch
// (4096 x 4096 at 48 rows: 12 us + 4 us for 0.8 us of matrix instructions and 1.4 us of weights).  Here
//   * a workgroup owns NS neighbouring strips of 16 columns x RT row tiles of 16 rows and its wavefronts split K
//     (wavefront w takes tile rows w, w + WAVES, ...): whole-K workgroups fill the chip without a second launch, and the
//     wavefronts never wait for each other before the sums are added, so that one wavefront's expansion and scale
//     arithmetic runs under another's matrix instructions;
//   * every wavefront moves its own activation fragments by DMA into its own part of LDS, 64 rows of K at a time and a
//     unit (four with two row tiles) ahead, and reads each once for all NS strips: loading them straight into registers
//     would make quads of lanes read four different rows, which the L1 serves at a quarter of its rate (measured: 48 rows
//     on 4096 x 28672 30.1 us that way, 25.4 this way);
//   * packed weights go straight to the registers that feed the matrix core, two tile rows ahead; lane (kg, c) fetches
//     the scales and zeros of tile row kg of four, column c, and a lane permute hands them out;
//   * the arithmetic is that of the other streaming kernels: P = A x (q + OFFSET) per group and strip,
//     S = A x ones per group, out += s * P + (z - OFFSET * s) * S in float32 (per-channel scales: once, at the end);
//   * the wavefronts are added through LDS in a fixed order (bit-reproducible); on long K a split across workgroups
//     stays possible (float32 slabs in the workspace, the tiled kernels' finish pass).
// What bounds it: the issue rate - a 16x16x32 matrix instruction takes 9 issue cycles and a vector instruction 4, i.e.
// about 390 cycles per strip and tile row at four row tiles against 256 of the matrix core - and the launch itself; on
// wide matrices also the activations, which every workgroup of 64 columns fetches again (without those requests 48 rows
// on 4096 x 28672 take 19 instead of 24 us), where the tiled kernels' 256 columns win from 64 rows on.
// Measured (bf16, group 128, zeros; before -> now, us): 4096 x 4096 at 32 / 48 / 64 / 160 rows 10.5 -> 7.9 / 14.2 -> 9.6 /
// 15.7 -> 10.2 / 20.8 -> 13.6; 4096 x 6144 at 48 rows 16.0 -> 10.7; 8192 x 8192 at 48 rows 19.2 -> 17.2; 4096 x 28672 at
// 48 rows 27.5 -> 23.7 (2.6 TB/s of weights); group 64, 8192 x 10240 at 16 rows 17.3 -> 14.2.
// Needs k to be a multiple of the weight tile's rows (128 for int4, 64 for int8).
#pragma once

#include "gemm_common.h"

namespace woq
{

struct MidTail
{
    void const* bias;
    void* out;
    float* partial; // [slices, m, n] float32 when K is split across workgroups, else NULL
    float alpha;
    int m;
    int tiles_per_split; // tile rows of K per workgroup
};

constexpr int kMidChunk = 8; // strip groups that all row tiles visit before the next ones (their weights stay in the L2)

template <int DT, int BITS, int GROUP, bool ZERO, int RT, int NS, int WAVES>
__global__ void __launch_bounds__(WAVES * 64) __attribute__((amdgpu_waves_per_eu(2)))
mid_kernel(void const* weight, void const* act, void const* scales, void const* zeros, int k_tiles, int strips,
    int groups_per_xcd, int n, int k, int tiles_m, MidTail tail)
{
    using E = Elem<DT>;
    constexpr int TK = BITS == 4 ? 128 : 64; // rows of K in a 1 KiB tile
    constexpr int SLABS = TK / 32;
    constexpr bool PER_CHANNEL = GROUP == 0;
    constexpr int SEGS = (!PER_CHANNEL && GROUP < TK) ? TK / GROUP : 1; // scale groups inside a tile row
    constexpr int SEG_SLABS = SLABS / SEGS;
    constexpr float OFF = BITS == 4 ? Fine4<DT>::kOffset : Offset<DT, BITS>::value;
    constexpr uint32_t kOob = 0x80000000u;
    constexpr int UNITS = SLABS / 2;            // units of 64 rows of K in a tile row
    constexpr int UNIT_BYTES = 2 * RT * 1024;   // activation fragments of one unit
    constexpr int STAGES = RT <= 2 ? 4 : 2;     // units in flight or in use per wavefront
    static_assert((4 * UNITS) % STAGES == 0, "a stage is a compile-time choice in the unrolled loop");
    // one object per stage: the compiler's waits for LDS-DMA are per object; the sums meet in stages 0 and 1 afterwards
    constexpr int STAGE_VECS = WAVES * UNIT_BYTES / 16, RED_VECS = 2 * NS * RT * 64;
    __shared__ u32x4 stage0[STAGE_VECS > RED_VECS ? STAGE_VECS : RED_VECS];
    __shared__ u32x4 stage1[STAGE_VECS > RED_VECS ? STAGE_VECS : RED_VECS];
    __shared__ u32x4 stage2[STAGES > 2 ? STAGE_VECS : 1];
    __shared__ u32x4 stage3[STAGES > 2 ? STAGE_VECS : 1];
    static_assert(GROUP == 0 || GROUP == 64 || GROUP == 128, "per-channel scales or group scales of 64 or 128 rows");
    static_assert(GROUP == 0 || GROUP <= TK || BITS == 8, "a group covers at most one int4 tile row");
    static_assert(!(PER_CHANNEL && ZERO), "per-channel scales come without zeros");

    // ---- which strips, rows and slice of K ----
    int const groups = (strips + NS - 1) / NS;
    int idx = (int) (blockIdx.x >> 3), tm = 0;
    if (tiles_m > 1) // within an XCD: chunks of strip groups, all row tiles of a chunk, the groups of the chunk
    {
        int const chunk = idx / (kMidChunk * tiles_m), rem = idx - chunk * (kMidChunk * tiles_m);
        int const left = groups_per_xcd - chunk * kMidChunk, size = left < kMidChunk ? left : kMidChunk;
        tm = rem / size;
        idx = chunk * kMidChunk + (rem - tm * size);
    }
    int const group = (int) (blockIdx.x & 7) * groups_per_xcd + idx;
    if (group >= groups)
        return; // whole workgroup leaves together
    int const m = tail.m;
    int const m0 = tm * (RT * 16);
    int const kt_begin = (int) blockIdx.y * tail.tiles_per_split;
    int const kt_end = kt_begin + tail.tiles_per_split < k_tiles ? kt_begin + tail.tiles_per_split : k_tiles;

    int const lane = threadIdx.x & 63;
    int const wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int const c = lane & 15, kg = lane >> 4;
    int const first = kt_begin + wave; // this wavefront's tile rows: first, first + WAVES, ...
    int const iters = kt_end > first ? (kt_end - first + WAVES - 1) / WAVES : 0;

    auto const w_rsrc = make_rsrc(weight, (uint32_t) strips * (uint32_t) k_tiles * 1024u);
    auto const act_rsrc = make_rsrc(act, (uint32_t) m * (uint32_t) k * 2u);
    uint32_t const sz_bytes = (PER_CHANNEL ? 1u : (uint32_t) k / (uint32_t) (GROUP ? GROUP : 1)) * (uint32_t) n * 2u;
    auto const sc_rsrc = make_rsrc(scales, sz_bytes);
    auto const zr_rsrc = make_rsrc(ZERO ? zeros : scales, sz_bytes);
    uint32_t a_lane[RT], wlane[NS], sc_lane[NS];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
    {
        // lane 4 r + q moves a 16-byte chunk of row r, so that quads read 64 contiguous bytes (see frag_swizzle);
        // rows past m cost no traffic and read as zeros
        int const row = m0 + rt * 16 + (lane >> 2);
        a_lane[rt] = row < m ? ((uint32_t) row * (uint32_t) k + (uint32_t) (((lane & 3) ^ frag_swizzle(lane >> 4)) * 8)) * 2u
                             : kOob;
    }
#pragma unroll
    for (int s = 0; s < NS; ++s)
    {
        int const strip = group * NS + s;
        wlane[s] = strip < strips ? ((uint32_t) strip * (uint32_t) k_tiles * 64u + (uint32_t) lane) * 16u : kOob;
        sc_lane[s] = strip < strips ? (uint32_t) (strip * 16 + c) * 2u : kOob;
    }

    u32x4 w[2][NS];
    uint32_t sz[NS][SEGS], sz_next[NS][SEGS]; // scale (low half) and zero (high half) of the lane's tile row
    // requests of the wavefront's tile row i; past its last one they fall outside the descriptors
    auto past = [&](int i) -> uint32_t { return (uint32_t) (iters - 1 - i) & kOob; };
    auto fetch_w = [&](u32x4(&dst)[NS], int i)
    {
        uint32_t const out = past(i), off = (uint32_t) (first + i * WAVES) * 1024u;
#pragma unroll
        for (int s = 0; s < NS; ++s)
        {
            if constexpr (RT <= 3) // one workgroup reads these weights up to 48 rows (from 65 on several of three row tiles do)
                dst[s] = buffer_load_x4_once(w_rsrc, (wlane[s] + off) | out);
            else
                dst[s] = buffer_load_x4(w_rsrc, (wlane[s] + off) | out);
        }
    };
    // activation fragments of one unit (64 rows of K) of tile row i -> this wavefront's part of a stage
    auto dma_a = [&](u32x4* stage, int i, int unit)
    {
        uint32_t const out = past(i), off = (uint32_t) (first + i * WAVES) * (uint32_t) (TK * 2) + (uint32_t) (unit * 128);
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
#pragma unroll
            for (int j = 0; j < 2; ++j)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(act_rsrc,
                    (__attribute__((address_space(3))) void*) (reinterpret_cast<char*>(stage)
                        + wave * (UNIT_BYTES) + (j * RT + rt) * 1024),
                    16, (int) (((a_lane[rt] + off) | out) + (uint32_t) j * 64u), 0, 0, 0);
    };
    auto fetch_sz = [&](uint32_t(&dst)[NS][SEGS], int i0)
    {
        if constexpr (!PER_CHANNEL)
        {
            uint32_t const kt = (uint32_t) (first + (i0 + kg) * WAVES);
#pragma unroll
            for (int seg = 0; seg < SEGS; ++seg)
            {
                uint32_t const g = (kt * (uint32_t) TK + (uint32_t) (seg * (TK / SEGS))) / (uint32_t) (GROUP ? GROUP : 1);
                uint32_t const off = g * (uint32_t) n * 2u;
#pragma unroll
                for (int s = 0; s < NS; ++s)
                {
                    uint32_t const o = i0 + kg < iters ? sc_lane[s] + off : kOob;
                    uint32_t const sv = buffer_load_u16(sc_rsrc, o);
                    uint32_t const zv = ZERO ? (uint32_t) buffer_load_u16(zr_rsrc, o) : 0u;
                    dst[s][seg] = sv | (zv << 16);
                }
            }
        }
    };

    u32x4 const ones = {E::kOnes, E::kOnes, E::kOnes, E::kOnes};
    NibbleConsts const nib = fine_nibble_consts<DT>();
    f32x4 const zero4 = {0.f, 0.f, 0.f, 0.f};
    auto expand = [&](u32x4 const& wv, int j) -> u32x4
    {
        if constexpr (BITS == 4)
            return u32x4{expand_int4_fine_reg<DT>(wv[j], 0, nib), expand_int4_fine_reg<DT>(wv[j], 1, nib),
                expand_int4_fine_reg<DT>(wv[j], 2, nib), expand_int4_fine_reg<DT>(wv[j], 3, nib)};
        else
            return expand_int8<DT>(wv[2 * j], wv[2 * j + 1]);
    };

    f32x4 total[NS][RT]; // finished sums (group scales) / running P (per-channel)
    f32x4 S[RT];         // row sums of the group at hand / of all of K (per-channel)
#pragma unroll
    for (int s = 0; s < NS; ++s)
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
            total[s][rt] = zero4;
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
        S[rt] = zero4;

    int const a_lane_off = (c * 4 + (kg ^ frag_swizzle(c >> 2))) * 16 + wave * UNIT_BYTES;
    f32x4 P[NS][RT];
    // one unit of a tile row (two slabs of 32 rows of K): every activation fragment is read once and feeds all strips
    auto compute = [&](u32x4 const* stage, u32x4 const(&wv)[NS], int u, int unit)
    {
        char const* const base = reinterpret_cast<char const*>(stage) + a_lane_off;
#pragma unroll
        for (int jj = 0; jj < 2; ++jj)
        {
            int const j = unit * 2 + jj, seg = j / SEG_SLABS;
            bool const begin = j % SEG_SLABS == 0;
            u32x4 av[RT];
#pragma unroll
            for (int rt = 0; rt < RT; ++rt)
                av[rt] = *reinterpret_cast<u32x4 const*>(base + (jj * RT + rt) * 1024);
#pragma unroll
            for (int s = 0; s < NS; ++s)
            {
                u32x4 const b = expand(wv[s], j);
#pragma unroll
                for (int rt = 0; rt < RT; ++rt)
                {
                    if constexpr (PER_CHANNEL)
                        total[s][rt] = E::mma(av[rt], b, total[s][rt]);
                    else
                        P[s][rt] = E::mma(av[rt], b, begin ? zero4 : P[s][rt]);
                }
            }
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) // row sums, once per tile row
                S[rt] = E::mma(av[rt], ones, (begin && !PER_CHANNEL) ? zero4 : S[rt]);
            if constexpr (!PER_CHANNEL)
            {
                if (j % SEG_SLABS == SEG_SLABS - 1)
                {
#pragma unroll
                    for (int s = 0; s < NS; ++s)
                    {
                        // the lanes (u, c) hold this tile row's scale and zero for column c
                        uint32_t const got = (uint32_t) __shfl((int) sz[s][seg], u * 16 + c);
                        float const sc = E::from_bits((uint16_t) (got & 0xFFFFu));
                        float const cc = __builtin_fmaf(-OFF, sc, ZERO ? E::from_bits((uint16_t) (got >> 16)) : 0.f);
#pragma unroll
                        for (int rt = 0; rt < RT; ++rt)
#pragma unroll
                            for (int r = 0; r < 4; ++r)
                                total[s][rt][r]
                                    = __builtin_fmaf(sc, P[s][rt][r], __builtin_fmaf(cc, S[rt][r], total[s][rt][r]));
                    }
                }
            }
        }
    };

    // ---- main loop: four tile rows at a time (the scales of four come in one request); unit h sits in stage h % STAGES ----
    auto stage_of = [&](int h) -> u32x4*
    { return h % STAGES == 0 ? stage0 : (h % STAGES == 1 ? stage1 : (h % STAGES == 2 ? stage2 : stage3)); };
    fetch_sz(sz, 0);
#pragma unroll
    for (int h = 0; h < STAGES; ++h)
        dma_a(stage_of(h), h / UNITS, h % UNITS);
    fetch_w(w[0], 0);
    fetch_w(w[1], 1);
    for (int i0 = 0; i0 < iters; i0 += 4)
    {
#pragma unroll
        for (int u = 0; u < 4; ++u)
        {
            int const i = i0 + u;
            if (i >= iters)
                break;
#pragma unroll
            for (int s = 0; s < NS; ++s) // nothing of the next weights is computed (and waited for) before this point
                asm volatile("" : "+v"(w[u & 1][s]));
#pragma unroll
            for (int unit = 0; unit < UNITS; ++unit)
            {
                int const h = u * UNITS + unit, next = h + STAGES; // 4 * UNITS is a multiple of STAGES
                compute(stage_of(h), w[u & 1], u, unit);
                __builtin_amdgcn_sched_barrier(0);
                dma_a(stage_of(h), i0 + next / UNITS, next % UNITS);
                __builtin_amdgcn_sched_barrier(0);
            }
            fetch_w(w[u & 1], i + 2);
            if (u == 1)
                fetch_sz(sz_next, i0 + 4);
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int s = 0; s < NS; ++s)
#pragma unroll
            for (int seg = 0; seg < SEGS; ++seg)
                sz[s][seg] = sz_next[s][seg];
    }

    // ---- the wavefronts' sums, in a fixed order: w + (w + 4) for eight wavefronts, then 0 + 1 + 2 + 3 ----
    // (the stages are free once every wavefront has left the loop and its last, out-of-range requests have landed)
    auto red = [&](int part) -> f32x4* // NS * RT blocks of 64 lanes
    { return reinterpret_cast<f32x4*>(part & 2 ? stage1 : stage0) + (part & 1) * (NS * RT * 64); };
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if constexpr (PER_CHANNEL) // sum a * q = P - OFFSET * S; the column's scale follows below
    {
#pragma unroll
        for (int s = 0; s < NS; ++s)
#pragma unroll
            for (int rt = 0; rt < RT; ++rt)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    total[s][rt][r] = __builtin_fmaf(-OFF, S[rt][r], total[s][rt][r]);
    }
    static_assert(WAVES == 4 || WAVES == 8, "four partial sums per element meet in LDS");
    if constexpr (WAVES == 8)
    {
        if (wave >= 4)
        {
#pragma unroll
            for (int s = 0; s < NS; ++s)
#pragma unroll
                for (int rt = 0; rt < RT; ++rt)
                    red(wave - 4)[(s * RT + rt) * 64 + lane] = total[s][rt];
        }
        __syncthreads();
        if (wave < 4)
        {
#pragma unroll
            for (int s = 0; s < NS; ++s)
#pragma unroll
                for (int rt = 0; rt < RT; ++rt)
                    total[s][rt] += red(wave)[(s * RT + rt) * 64 + lane];
        }
    }
    if (wave < 4)
    {
#pragma unroll
        for (int s = 0; s < NS; ++s)
#pragma unroll
            for (int rt = 0; rt < RT; ++rt)
                red(wave)[(s * RT + rt) * 64 + lane] = total[s][rt];
    }
    __syncthreads();
    auto sum_of = [&](int slot, int l) -> f32x4
    {
        int const at = slot * 64 + l;
        return ((red(0)[at] + red(1)[at]) + red(2)[at]) + red(3)[at];
    };

    uint16_t* const out16 = static_cast<uint16_t*>(tail.out);
    for (int e = threadIdx.x; e < NS * RT * 64; e += WAVES * 64)
    {
        int const slot = e >> 6, l = e & 63, s = slot / RT, rt = slot % RT;
        int const strip = group * NS + s;
        if (strip >= strips)
            continue;
        f32x4 v = sum_of(slot, l);
        // not finite: a row with an infinite activation.  The 64 lanes hold one 16 x 16 tile as the matrix core writes it, so
        // this wavefront forms the tile's plain sums by itself.
        if (__builtin_expect(__any(!is_finite((v[0] + v[1]) + (v[2] + v[3]))), 0))
        {
            // (values the compiler cannot tell from others: their arithmetic moved in front of the main loop otherwise)
            int lane0 = l, strip0 = __builtin_amdgcn_readfirstlane(strip), row0 = __builtin_amdgcn_readfirstlane(m0 + rt * 16);
            asm volatile("" : "+v"(lane0), "+s"(strip0), "+s"(row0));
            uint32_t const w_at[1] = {((uint32_t) strip0 * (uint32_t) k_tiles * 64u + (uint32_t) lane0) * 16u};
            uint32_t const sc_at[1] = {(uint32_t) (strip0 * 16 + (lane0 & 15)) * 2u};
            f32x4 plain[1][1] = {{zero4}};
            plain_sums<DT, BITS, GROUP, ZERO, 1, 1>(
                plain, act_rsrc, w_rsrc, sc_rsrc, zr_rsrc, w_at, sc_at, lane0, row0, m, n, k, 0, kt_begin, kt_end, 1);
#pragma unroll
            for (int r = 0; r < 4; ++r)
                v[r] = is_finite(v[r]) ? v[r] : plain[0][0][r];
        }
        int const col = strip * 16 + (l & 15);
        if constexpr (PER_CHANNEL)
        {
            float const sc = E::load(scales, col);
            v[0] *= sc, v[1] *= sc, v[2] *= sc, v[3] *= sc;
        }
        float const bias = (tail.bias && !tail.partial) ? E::load(tail.bias, col) : 0.f;
#pragma unroll
        for (int r = 0; r < 4; ++r)
        {
            int const row = m0 + rt * 16 + (l >> 4) * 4 + r;
            if (row >= m)
                continue;
            size_t const at = (size_t) row * n + col;
            if (tail.partial)
            {
                tail.partial[(size_t) blockIdx.y * ((size_t) m * n) + at] = v[r];
                continue;
            }
            out16[at] = E::store(__builtin_fmaf(tail.alpha, v[r], bias));
        }
    }
}

template <int DT, int BITS, int GROUP, bool ZERO, int RT, int NS, int WAVES>
int launch_mid_variant(MatmulProblem const& p, MidPlan const& plan, hipStream_t stream)
{
    int const k_tiles = p.k / (BITS == 4 ? 128 : 64), strips = p.n / kTileN;
    int const groups = (strips + NS - 1) / NS, groups_per_xcd = (groups + 7) / 8;
    int const tiles_m = (p.m + RT * 16 - 1) / (RT * 16);
    int const splits = plan.splits;
    MidTail const tail{p.bias, p.out, splits > 1 ? static_cast<float*>(p.workspace) : nullptr, p.alpha, p.m,
        (k_tiles + splits - 1) / splits};
    note_launch("mid rt=%d ns=%d waves=%d splits=%d", RT, NS, WAVES, splits);
    hipLaunchKernelGGL((mid_kernel<DT, BITS, GROUP, ZERO, RT, NS, WAVES>),
        dim3((unsigned) (groups_per_xcd * 8 * tiles_m), (unsigned) splits), dim3(WAVES * 64), 0, stream, p.weight, p.act,
        p.scales, p.zeros, k_tiles, strips, groups_per_xcd, p.n, p.k, tiles_m, tail);
    if (splits > 1)
    {
        size_t const count = (size_t) p.m * p.n;
        hipLaunchKernelGGL((gemm_finish_partial<DT>), dim3((unsigned) ((count / 4 + 255) / 256)), dim3(256), 0, stream,
            p.out, tail.partial, p.bias, p.alpha, p.m, p.n, splits);
    }
    hipError_t err = hipGetLastError();
    if (err != hipSuccess)
        return fail(WOQ_ERR_RUNTIME, "mid kernel launch failed: %s", hipGetErrorString(err));
    return WOQ_OK;
}

template <int DT, int BITS, int GROUP, bool ZERO>
int launch_mid_shaped(MatmulProblem const& p, MidPlan const& plan, hipStream_t s)
{
#define WOQ_MID(RT_, NS_, WAVES_)                                                                                      \
    if (plan.rt == RT_ && plan.ns == NS_ && plan.waves == WAVES_)                                                      \
        return launch_mid_variant<DT, BITS, GROUP, ZERO, RT_, NS_, WAVES_>(p, plan, s);
#define WOQ_MID_RT(RT_)                                                                                                \
    WOQ_MID(RT_, 1, 8)                                                                                                 \
    WOQ_MID(RT_, 2, 8)                                                                                                 \
    if constexpr (GROUP == 0 || RT_ < (GROUP == 64 ? 3 : 4)) /* more sums than registers beyond (best_mid_plan) */    \
    {                                                                                                                  \
        WOQ_MID(RT_, 4, 4)                                                                                             \
        WOQ_MID(RT_, 4, 8)                                                                                             \
    }
    if constexpr (BITS == 4) // (int8: the other streaming kernels are as fast)
    {
        WOQ_MID_RT(1)
    }
    WOQ_MID_RT(2)
    WOQ_MID_RT(3)
    WOQ_MID_RT(4)
#undef WOQ_MID_RT
#undef WOQ_MID
    return fail(WOQ_ERR_UNSUPPORTED, "mid kernel shape rt=%d ns=%d waves=%d is not instantiated", plan.rt, plan.ns, plan.waves);
}

template <int DT, int BITS>
int launch_mid_typed(MatmulProblem const& p, MidPlan const& plan, void* stream)
{
    auto s = static_cast<hipStream_t>(stream);
    if (plan.splits > 1 && (!p.workspace || p.workspace_bytes < split_partial_bytes(p.m, p.n, plan.splits)))
        return fail(WOQ_ERR_WORKSPACE, "split-K needs %zu workspace bytes", split_partial_bytes(p.m, p.n, plan.splits));
    if (p.group_size == 0)
        return launch_mid_shaped<DT, BITS, 0, false>(p, plan, s);
    if constexpr (BITS == 4)
    {
        if (p.group_size == 64)
            return p.zeros ? launch_mid_shaped<DT, BITS, 64, true>(p, plan, s) : launch_mid_shaped<DT, BITS, 64, false>(p, plan, s);
        if (p.group_size == 128)
            return p.zeros ? launch_mid_shaped<DT, BITS, 128, true>(p, plan, s)
                           : launch_mid_shaped<DT, BITS, 128, false>(p, plan, s);
    }
    return fail(WOQ_ERR_UNSUPPORTED, "mid kernel: group_size %d", p.group_size);
}

} // namespace woq
