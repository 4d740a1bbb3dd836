// The prefill's GEMMs for a short run (crates/graph/src/prefill.rs:218-413), where prefill_gemm's
// 256 x 128 tiles leave most of the chip idle: a wave to a workgroup, each its own strips of W against
// its own tiles of X, both straight from memory into registers many k-blocks ahead of their
// products. The epilogues are prefill_gemm's, and each output is the same MFMA chain over its
// k-blocks in order, so that a run's rows come out the same bits whichever kernel takes them.
#include "prefill_kernels.hpp"

#include <math.h>

#include "dispatch.hpp"

namespace tgx {

namespace {

constexpr int STRIP = 16;                       // W rows a strip
constexpr int SPAN = 128, SPAN_STRIPS = 8;      // the columns a sum of squares spans, and their strips
constexpr int MAX_SPANS = 2048 / SPAN;          // a norm's row has hidden <= 2048 columns

// SPANS spans of row m of f32 [M_pad][K], from span j0, a lane to its 4 columns of each strip, and
// each span's sum of squares (add_squares' order), the same in the row's four lanes.
template <int SPANS>
struct SpanSquares {
    float4 v[SPANS][SPAN_STRIPS];
    __device__ __forceinline__ void load(const float* rows, int m, int K, int j0) {
        const float* at = rows + (size_t)m * K + j0 * SPAN + threadIdx.x % WAVE / 16 * 4;
#pragma unroll
        for (int j = 0; j < SPANS; ++j)
#pragma unroll
            for (int s = 0; s < SPAN_STRIPS; ++s) v[j][s] = *reinterpret_cast<const float4*>(at + j * SPAN + s * STRIP);
    }
    __device__ __forceinline__ float sum(int j) const {
        float c = 0.f;
#pragma unroll
        for (int s = 0; s < SPAN_STRIPS; ++s) c = add_squares(c, v[j][s].x, v[j][s].y, v[j][s].z, v[j][s].w);
        c += lane_xor16(c);
        return c + lane_xor32(c);
    }
};

// The q/k/v epilogue of one 16 x 16 tile: a lane's four rows of a strip are two RoPE pairs
// (qkv_row_of), of row m at `pos` of cache block `block` (`held`: a row of the run, inside the
// cache), whose RMSNorm scale is rs; cs and sn the pairs' rotations. Lanes l and l ^ 16 run it
// together.
template <int D>
__device__ __forceinline__ void store_qkv(const PrefillArgs& a, const GemmArgs& g, int strip, int m, bool held, uint32_t pos, uint32_t block,
                                          const f32x4& acc, float rs, float2 cs, float2 sn) {
    const int H = a.heads, KV = a.kv_heads, quad = threadIdx.x % WAVE / 16;
    const int head = strip / (D / 16);
    const int e = strip % (D / 16) * 8 + quad * 2;
    const int d0 = (quad & 1) ? e - 2 + D / 2 : e;  // after quad_halves' trade
    float lo[2], hi[2];                              // dimensions e + k and e + k + D / 2
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        lo[k] = acc[2 * k] * rs;
        hi[k] = acc[2 * k + 1] * rs;
        if (head < H + KV && a.rope) rotate_pair(lo[k], hi[k], k ? cs.y : cs.x, k ? sn.y : sn.x);
    }
    const float qs = head < H ? log2_scale(a.scale) : 1.f;  // q in the attention softmax's units
    const uint2 w4 = quad_halves(pack_bf16x2(lo[0] * qs, lo[1] * qs), pack_bf16x2(hi[0] * qs, hi[1] * qs));
    if (!held) return;
    if (head < H) {
        *reinterpret_cast<uint2*>(g.q + ((size_t)m * H + head) * D + d0) = w4;
        return;
    }
    if (block >= (uint32_t)a.nblocks) return;
    const int kv = head < H + KV ? head - H : head - H - KV;
    constexpr int TILE = kv_tile(D);
    uint16_t* tl = g.kv + ((size_t)block * KV + kv) * 2 * TILE;
    const int pp = (int)(pos % BLOCK_TOKENS);
    if (head < H + KV) {
        *reinterpret_cast<uint2*>(tl + key_index(pp, d0, D)) = w4;
    } else {
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            tl[TILE + value_index(pp, e + k)] = (uint16_t)bf16_bits(lo[k]);
            tl[TILE + value_index(pp, e + k + D / 2)] = (uint16_t)bf16_bits(hi[k]);
        }
    }
}

// ---------------------------------------------------------------------------------------------
// prefill_direct: a unit of SW strips of W (gate/up: a gate strip and its up strip) by TT tiles of 16
// rows of X to a wave, DEPTH k-blocks of both in flight (a divisor of every K / 32, K a multiple of
// 1024). What bounds a run this short is the chain of k-blocks an output is, and one CU's rate from L2
// (145 GB/s): the strips and tiles are spread over every CU, and each wave keeps 32 to 48 loads of 1 KiB
// in flight with no barrier and no other wave to wait for. A unit's tiles sit on one XCD (workgroup
// id % 8), so that its W comes from memory once. At 57 rows of the backbone, us a launch against
// prefill_gemm's 4 and 5 workgroups: down_proj 77.1 -> 5.7, q/k/v 27.4 -> 5.3. Twice the loads in flight
// (DEPTH 32, the operands in AGPRs) measured the same. o_proj stays with prefill_ring, whose workgroups
// hold whole spans: with gate/up taking its rows' sums of squares from the rows, o_proj 7.0 -> 4.3 but
// gate/up 7.9 -> 11.7.
// q/k/v also needs its rows' sums of squares over every column, which no one wave of down_proj had: waves
// beside the GEMM's take them from the rows (g.rows, SPANS = K / 128 spans), half a tile's spans to a
// wave, and pass them on through LDS (in the GEMM's own wave they cost 3 us a launch).
template <int EPI, int TT>
constexpr int direct_waves() {
    return EPI == EPI_QKV ? 1 + 2 * TT : 1;
}
template <int EPI, int WR, int SW, int TT, int DEPTH, int D, int SPANS>
__global__ void __launch_bounds__((direct_waves<EPI, TT>() * WAVE)) prefill_direct(PrefillArgs a, GemmArgs g, int groups) {
    constexpr bool SCALED = !residual_epilogue(EPI);
    __shared__ float span_sq[EPI == EPI_QKV ? SPANS * 16 * TT : 1];  // [SPANS][16 TT]
    const bool scaled = EPI == EPI_QKV ? (bool)g.rows : SCALED && g.row_sq;  // uniform
    static_assert(32 % DEPTH == 0, "the k-blocks come in whole depths");
    static_assert(EPI != EPI_SILU || SW == 2, "gate/up takes a gate strip and its up strip");
    const int lane = threadIdx.x % WAVE, quad = lane / 16, col = lane % 16;
    const int turn = blockIdx.x / 8;
    const int unit = turn / groups * 8 + blockIdx.x % 8, t0 = turn % groups * TT;
    if constexpr (EPI == EPI_QKV) {
        const int helper = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE) - 1;
        if (helper >= 0) {
            if (scaled) {
                const int t = helper % TT, j0 = helper / TT * (SPANS / 2);
#pragma unroll
                for (int j = j0; j < j0 + SPANS / 2; j += 4) {  // four spans' loads in flight
                    SpanSquares<4> sq;
                    sq.load(g.rows, (t0 + t) * 16 + col, g.K, j);
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const float v = sq.sum(i);
                        if (quad == 0) span_sq[(j + i) * 16 * TT + t * 16 + col] = v;
                    }
                }
            }
            __syncthreads();
            return;
        }
    }
    const int kblocks = g.K / 32;
    int strip[SW];
#pragma unroll
    for (int s = 0; s < SW; ++s) strip[s] = EPI == EPI_SILU ? (s ? unit + g.N / 32 : unit) : unit * SW + s;

    // What the epilogue reads of its rows goes first: gate/up's sums of squares, their residual, their
    // places.
    float4 parts[TT][SPANS ? SPANS / 4 : 1];
    uint32_t pos[TT], slot[TT];
    f32x4 acc[SW][TT];
#pragma unroll
    for (int t = 0; t < TT; ++t) {
        const int m = (t0 + t) * 16 + col;
        if (EPI == EPI_SILU && scaled) {
#pragma unroll
            for (int i = 0; i < SPANS / 4; ++i) parts[t][i] = *reinterpret_cast<const float4*>(g.row_sq + (size_t)m * SPANS + 4 * i);
        }
        if (EPI == EPI_QKV) {
            pos[t] = a.tok_pos[m];
            slot[t] = a.tok_slot[m];
        }
#pragma unroll
        for (int s = 0; s < SW; ++s) {
            acc[s][t] = f32x4{0.f, 0.f, 0.f, 0.f};
            if (residual_epilogue(EPI)) {  // rows past M read row M - 1, never stored
                const float4 r = *reinterpret_cast<const float4*>(g.residual + (size_t)min(m, a.M - 1) * g.N + strip[s] * STRIP + quad * 4);
                acc[s][t] = f32x4{r.x, r.y, r.z, r.w};
            }
        }
    }
    f32x4 residual[SW][TT];
    if (EPI == EPI_RESIDUAL) {  // added after the products
#pragma unroll
        for (int s = 0; s < SW; ++s)
#pragma unroll
            for (int t = 0; t < TT; ++t) {
                residual[s][t] = acc[s][t];
                acc[s][t] = f32x4{0.f, 0.f, 0.f, 0.f};
            }
    }
    float4 gain[SW];
    if (residual_epilogue(EPI)) {
#pragma unroll
        for (int s = 0; s < SW; ++s)
            gain[s] = *reinterpret_cast<const float4*>((g.next_gain ? g.next_gain : g.residual) + strip[s] * STRIP + quad * 4);
    }

    // The operands: a strip's (or tile's) k-blocks follow each other, at a uniform address plus the
    // lane's offset.
    const uint32_t wlane = (uint32_t)fragment_index<WR>(0, 0, kblocks, lane), xlane = (uint32_t)lane * 8;
    uint4 wf[DEPTH][SW], xf[DEPTH][TT];
    auto fetch = [&](int kb, int d) __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < SW; ++s)
            wf[d][s] = *reinterpret_cast<const uint4*>(g.w + ((size_t)strip[s] * kblocks * 512 + (size_t)kb * WR * 32) + wlane);
#pragma unroll
        for (int t = 0; t < TT; ++t)
            xf[d][t] = *reinterpret_cast<const uint4*>(g.x + ((size_t)(t0 + t) * kblocks + kb) * 512 + xlane);
    };
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
        fetch(d, d);
        __builtin_amdgcn_sched_barrier(0);  // k-block by k-block: the first product waits for the first loads only
    }
    auto products = [&](int d) __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < SW; ++s)
#pragma unroll
            for (int t = 0; t < TT; ++t) acc[s][t] = mfma16(wf[d][s], xf[d][t], acc[s][t]);
    };
    for (int kb = DEPTH; kb < kblocks; kb += DEPTH) {
#pragma unroll
        for (int d = 0; d < DEPTH; ++d) {
            products(d);
            fetch(kb + d, d);
            __builtin_amdgcn_sched_barrier(0);  // each refill stays where it is, DEPTH k-blocks ahead of its use
        }
    }
    // The q/k/v rows' cache blocks and RoPE values, behind the last loads: they land beside the last
    // products.
    uint32_t block[TT];
    float2 cs[SW][TT], sn[SW][TT];
    bool held[TT];
    if constexpr (EPI == EPI_QKV) {
#pragma unroll
        for (int t = 0; t < TT; ++t) {
            const int m = (t0 + t) * 16 + col;
            held[t] = m < a.M && pos[t] < (uint32_t)a.capacity && slot[t] < (uint32_t)a.nslots;
            const uint32_t p = held[t] ? pos[t] : 0, sl = held[t] ? slot[t] : 0;
            block[t] = a.table[(size_t)sl * a.max_blocks + p / BLOCK_TOKENS];
#pragma unroll
            for (int s = 0; s < SW; ++s) {
                const int e = strip[s] % (D / 16) * 8 + quad * 2;
                cs[s][t] = sn[s][t] = make_float2(0.f, 0.f);
                if (a.rope) {
                    cs[s][t] = *reinterpret_cast<const float2*>(a.cos + (size_t)p * (D / 2) + e);
                    sn[s][t] = *reinterpret_cast<const float2*>(a.sin + (size_t)p * (D / 2) + e);
                }
            }
        }
    }
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) products(d);
    if constexpr (EPI == EPI_QKV) __syncthreads();  // the sums of squares

    // The epilogue: tile (s, t) holds W rows 16 strip + 4 quad + i against X row 16 (t0 + t) + col.
    if constexpr (residual_epilogue(EPI)) {
#pragma unroll
        for (int s = 0; s < SW; ++s) {
            const int n = strip[s] * STRIP + quad * 4;
#pragma unroll
            for (int t = 0; t < TT; ++t) {
                const int m = (t0 + t) * 16 + col;
                float4 o = make_float4(acc[s][t][0], acc[s][t][1], acc[s][t][2], acc[s][t][3]);
                if (EPI == EPI_RESIDUAL) {
                    o.x = residual[s][t][0] + acc[s][t][0];
                    o.y = residual[s][t][1] + acc[s][t][1];
                    o.z = residual[s][t][2] + acc[s][t][2];
                    o.w = residual[s][t][3] + acc[s][t][3];
                }
                if (m < a.M) *reinterpret_cast<float4*>(g.out + (size_t)m * g.N + n) = o;
                if (g.next_gain && m < a.M)
                    *reinterpret_cast<uint2*>(g.out_n + act_index(m, n, g.N)) =
                        make_uint2(pack_bf16x2(o.x * gain[s].x, o.y * gain[s].y), pack_bf16x2(o.z * gain[s].z, o.w * gain[s].w));
            }
        }
    } else {
#pragma unroll
        for (int t = 0; t < TT; ++t) {
            const int m = (t0 + t) * 16 + col;
            float rs = 1.f;
            if (scaled) {
                float total = 0.f;
#pragma unroll
                for (int j = 0; j < SPANS; ++j) {
                    if constexpr (EPI == EPI_QKV) {
                        total += span_sq[(j * TT + t) * 16 + col];
                    } else {
                        const float4 p = parts[t][j / 4];
                        total += j % 4 == 0 ? p.x : j % 4 == 1 ? p.y : j % 4 == 2 ? p.z : p.w;
                    }
                }
                rs = rms_scale(total, g.K, a.eps);
            }
            if constexpr (EPI == EPI_SILU) {
                const SiluRow silu_row(rs);
                float v[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) v[i] = silu_row(acc[0][t][i], acc[SW - 1][t][i]);
                if (m < a.M)
                    *reinterpret_cast<uint2*>(g.mlp + act_index(m, strip[0] * STRIP + quad * 4, g.N / 2)) =
                        make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
            } else {
#pragma unroll
                for (int s = 0; s < SW; ++s)
                    store_qkv<D>(a, g, strip[s], m, held[t], pos[t], block[t], acc[s][t], rs, cs[s][t], sn[s][t]);
            }
        }
    }
}

// ---------------------------------------------------------------------------------------------
// prefill_ring: four waves to a workgroup, each its own SW strips of W against the same TT tiles of
// 16 rows of X. A stage is G k-blocks: each wave's G SW fragments of W straight into registers (no
// other wave reads them), and its share of the tiles' G TT fragments into a ring of R LDS slots by
// direct global-to-LDS loads. R stages are in flight, in stage order, so a wave's count of loads in
// flight says which have landed, and the barrier after its wait says the same of every wave's. A
// stage's tiles are read from LDS while the stage before is multiplied. K / 32 is a multiple of 32:
// whole turns of R stages, the last one with nothing left to fetch. A workgroup's 128 columns are one
// span of a sum of squares. What bounds it: a k-block takes a CU 290 cycles at two tiles (10 KiB of
// operands; 16 or 240 workgroups, R 4 or 8 alike) and 640 at eight (16 KiB), and past a workgroup a
// CU the operands come from L2 at 18.5 TB/s in all (whole launches, start and epilogue in them, average
// 9 to 12 by the counters, gate/up and down_proj at 300 and 1167 rows). us a launch at the backbone
// against prefill_gemm: 57 rows o_proj 25.1 -> 7.0, gate/up 18.9 -> 7.9; 960 rows q/k/v 27.9 -> 12.5,
// o_proj 27.9 -> 8.8, gate/up 20.4 -> 18.7, down_proj 77.1 -> 20.9; 2048 rows 28.3 -> 16.6, 29.4 -> 12.0,
// 33.7 -> 32.4, 78.2 -> 25.2; 8192 rows down_proj 96.1 -> 77.9.
constexpr int RING_WAVES = 4;

template <int SW, int TT, int G, int R>
struct RingTile {
    static constexpr int XL = G * TT / RING_WAVES;  // a wave's loads to LDS a stage
    static constexpr int LOADS = G * SW + XL;       // all its loads
    // The ring (the residual epilogue's rows take its place, HALF tiles at a time), then the rows'
    // scales.
    static constexpr int HALF = TT < 4 ? TT : TT % 4 ? 3 : 4;
    static constexpr int ROW_FLOATS = SPAN + 4;  // 16 rows' quads on different banks
    static constexpr size_t RING_BYTES = (size_t)R * G * TT * 1024, ROW_BYTES = (size_t)16 * HALF * ROW_FLOATS * 4;
    static constexpr size_t LDS = (RING_BYTES > ROW_BYTES ? RING_BYTES : ROW_BYTES) + 16 * TT * sizeof(float);
    static_assert(XL * RING_WAVES == G * TT, "the tiles' fragments split evenly over the waves");
    static_assert(32 % (G * R) == 0, "the k-blocks come in whole turns of the ring");
};

// The workgroup's tile (nb, mb): each XCD (workgroup id % 8) takes a contiguous eighth of the tiles,
// in groups of GROUP_M bands of rows by every block of W, so that an XCD's L2 holds what its
// workgroups share.
template <int GROUP_M>
__device__ __forceinline__ void ring_tile_of(int NB, int MB, int& nb, int& mb) {
    const int total = NB * MB, id = blockIdx.x;
    const int v = total % 8 == 0 ? (id % 8) * (total / 8) + id / 8 : id;
    const int group = v / (GROUP_M * NB), in = v % (GROUP_M * NB);
    const int rows = min(GROUP_M, MB - group * GROUP_M);  // the last group may be short
    mb = group * GROUP_M + in % rows;
    nb = in / rows;
}

template <int N>
__device__ __forceinline__ void wait_loads(int n) {  // at most n (known once unrolled) of the wave's loads in flight
    if constexpr (N == 0) {
        wait_vm_seen<0>();
    } else {
        if (n >= N)
            wait_vm_seen<N>();
        else
            wait_loads<N - 1>(n);
    }
}

// Three tiles come four k-blocks a stage (a wave's share of fewer is not whole), whose operands are more
// registers than two waves to a SIMD leave.
template <int EPI, int WR, int SW, int TT, int G, int R, int D>
__global__ void __launch_bounds__(RING_WAVES * WAVE) __attribute__((amdgpu_waves_per_eu(TT == 3 ? 1 : 2)))
prefill_ring(PrefillArgs a, GemmArgs g, int NB, int MB) {
    using T = RingTile<SW, TT, G, R>;
    constexpr bool SCALED = !residual_epilogue(EPI);
    constexpr int ROWS = 16 * TT, LOADS = T::LOADS;
    static_assert(EPI != EPI_SILU || SW == 2, "gate/up takes a gate strip and its up strip");
    static_assert(!residual_epilogue(EPI) || RING_WAVES * SW == SPAN_STRIPS, "a workgroup's columns are one span of a sum of squares");
    static_assert(ROWS <= RING_WAVES * WAVE, "a thread to a row");
    static_assert(EPI != EPI_QKV || TT % 3, "the rows' places are read within the padded rows");
    extern __shared__ uint4 xs[];  // [R][G][TT tiles][64 lanes]
    float* scales = reinterpret_cast<float*>(reinterpret_cast<char*>(xs) + T::LDS) - ROWS;  // [ROWS]
    int nb, mb;
    ring_tile_of<8>(NB, MB, nb, mb);
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE), lane = threadIdx.x % WAVE, quad = lane / 16, col = lane % 16;
    const int m0 = mb * ROWS, kblocks = g.K / 32;
    int strip[SW];
#pragma unroll
    for (int s = 0; s < SW; ++s) {
        const int unit = nb * RING_WAVES + w;
        strip[s] = EPI == EPI_SILU ? (s ? unit + g.N / 32 : unit) : unit * SW + s;
    }
    // The rows' sums of squares (a thread to a row) and places go first, the stages behind them.
    float4 parts[MAX_SPANS / 4];
    const bool scaled = SCALED && g.row_sq && threadIdx.x < ROWS;
    if (scaled) {
        const float* row = g.row_sq + (size_t)(TT % 3 ? m0 + threadIdx.x : min((uint32_t)m0 + threadIdx.x, (uint32_t)a.M_pad - 1u)) * (g.K / SPAN);
#pragma unroll
        for (int i = 0; i < MAX_SPANS / 4; ++i) parts[i] = *reinterpret_cast<const float4*>(row + 4 * min(i, g.K / SPAN / 4 - 1));
    }
    uint32_t pos[TT], slot[TT];
    if constexpr (EPI == EPI_QKV) {
#pragma unroll
        for (int t = 0; t < TT; ++t) {
            pos[t] = a.tok_pos[m0 + 16 * t + col];
            slot[t] = a.tok_slot[m0 + 16 * t + col];
        }
    }
    // The accumulators start at zero, or with EPI_RESIDUAL_IN at the residual rows (rows past M read
    // row M - 1, never stored).
    f32x4 acc[SW][TT];
    auto residual_of = [&](int s, int t) __attribute__((always_inline)) {
        const float4 r = *reinterpret_cast<const float4*>(g.residual + (size_t)min(m0 + 16 * t + col, a.M - 1) * g.N + strip[s] * STRIP + quad * 4);
        return f32x4{r.x, r.y, r.z, r.w};
    };
#pragma unroll
    for (int s = 0; s < SW; ++s)
#pragma unroll
        for (int t = 0; t < TT; ++t) acc[s][t] = EPI == EPI_RESIDUAL_IN ? residual_of(s, t) : f32x4{0.f, 0.f, 0.f, 0.f};
    __builtin_amdgcn_sched_barrier(0);

    const uint32_t wlane = (uint32_t)fragment_index<WR>(0, 0, kblocks, lane);
    uint4 wf[R][G][SW];
    // Stage st into slot r (st % R): fragment f of the stage's G TT is k-block f / TT of tile f % TT;
    // wave w loads fragments XL w .. XL w + XL - 1.
    auto fetch = [&](int st, int r) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < G; ++k)
#pragma unroll
            for (int s = 0; s < SW; ++s) {
                typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
                const uint16_t* p = g.w + ((size_t)strip[s] * kblocks * 512 + (size_t)(st * G + k) * WR * 32) + wlane;
                wf[r][k][s] = __builtin_bit_cast(uint4, *(const __attribute__((address_space(1))) u32x4*)p);
            }
#pragma unroll
        for (int j = 0; j < T::XL; ++j) {
            const int f = w * T::XL + j;
            // Three or six tiles may go past the padded rows: the last tile again, never stored.
            const int tile = TT % 3 ? m0 / 16 + f % TT : __builtin_amdgcn_readfirstlane(min(m0 / 16 + f % TT, a.M_pad / 16 - 1));
            load_to_lds(g.x + ((size_t)tile * kblocks + st * G + f / TT) * 512 + lane * 8, &xs[(r * G * TT + f) * 64]);
        }
    };
    // Each stage stays behind the stage before (the waits count loads in issue order).
#pragma unroll
    for (int r = 0; r < R; ++r) {
        fetch(r, r);
        __builtin_amdgcn_sched_barrier(0);
    }
    // Stage 0 landed, every wave's; the scales into LDS by a store the compiler cannot see (it would
    // wait for every load to LDS in flight before it).
    if (SCALED && threadIdx.x < ROWS) {
        float rs = 1.f;
        if (scaled) {
            float total = 0.f;
#pragma unroll
            for (int i = 0; i < MAX_SPANS / 4; ++i) {
                if (i >= g.K / SPAN / 4) break;
                total += parts[i].x;
                total += parts[i].y;
                total += parts[i].z;
                total += parts[i].w;
            }
            rs = rms_scale(total, g.K, a.eps);
        }
        asm volatile("ds_write_b32 %0, %1" ::"v"(lds_offset(&scales[threadIdx.x])), "v"(rs) : "memory");
    }
    wait_vm_seen<(R - 1) * LOADS>();
    stage_barrier();
    uint4 xf[2][G * TT];
    auto read = [&](int r, uint4 (&x)[G * TT]) __attribute__((always_inline)) {
#pragma unroll
        for (int f = 0; f < G * TT; ++f) x[f] = lds_read16(&xs[(r * G * TT + f) * 64 + lane]);
    };
    read(0, xf[0]);
    // A step: slot r's stage multiplied while the next stage's tiles are read; `after` loads may be in
    // flight past the next stage's (negative: there is no next stage).
    auto step = [&](int r, int after) __attribute__((always_inline)) {
        const int b = r % 2;
        lds_landed(xf[b]);
        if (after >= 0) {
            // The barrier also says every wave has its tiles of slot r, which the fetch after this
            // step refills.
            wait_loads<(R - 2) * LOADS>(after);
            stage_barrier();
            read((r + 1) % R, xf[1 - b]);
        }
#pragma unroll
        for (int k = 0; k < G; ++k)
#pragma unroll
            for (int s = 0; s < SW; ++s)
#pragma unroll
                for (int t = 0; t < TT; ++t) acc[s][t] = mfma16(wf[r][k][s], xf[b][k * TT + t], acc[s][t]);
    };
    static_assert(R % 2 == 0, "a turn starts on the first buffer of tiles");
    const int stages = kblocks / G;
    for (int st = R; st < stages; st += R) {
#pragma unroll
        for (int r = 0; r < R; ++r) {
            step(r, (R - 2) * LOADS);
            fetch(st + r, r);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
        step(r, (R - 2 - r) * LOADS);
        __builtin_amdgcn_sched_barrier(0);
    }

    // The epilogue: tile (s, t) holds W rows 16 strip + 4 quad + i against X row m0 + 16 t + col.
    if constexpr (residual_epilogue(EPI)) {
        f32x4 r[SW][TT];
        float4 gain[SW];
#pragma unroll
        for (int s = 0; s < SW; ++s) {
            gain[s] = *reinterpret_cast<const float4*>((g.next_gain ? g.next_gain : g.residual) + strip[s] * STRIP + quad * 4);
#pragma unroll
            for (int t = 0; t < TT; ++t) r[s][t] = EPI == EPI_RESIDUAL ? residual_of(s, t) : f32x4{0.f, 0.f, 0.f, 0.f};
        }
        // With next_gain the rows pass through LDS, in the ring's place (every wave done with it), HALF
        // tiles at a time: a thread to a row's quad adds its squares over the span's strips in order.
        float* row_values = reinterpret_cast<float*>(xs);  // [16 HALF][ROW_FLOATS]
        constexpr int HALF = T::HALF;
        static_assert(16 * HALF * 4 <= RING_WAVES * WAVE, "a thread to a row's quad");
#pragma unroll
        for (int h = 0; h < TT; h += HALF) {
            if (g.next_gain) __syncthreads();
#pragma unroll
            for (int t = h; t < h + HALF; ++t) {
                const int m = m0 + 16 * t + col;
                uint32_t normed[SW][2];
#pragma unroll
                for (int s = 0; s < SW; ++s) {
                    const int n = strip[s] * STRIP + quad * 4;
                    float4 o = make_float4(acc[s][t][0], acc[s][t][1], acc[s][t][2], acc[s][t][3]);
                    if (EPI == EPI_RESIDUAL) o = make_float4(r[s][t][0] + o.x, r[s][t][1] + o.y, r[s][t][2] + o.z, r[s][t][3] + o.w);
                    normed[s][0] = pack_bf16x2(o.x * gain[s].x, o.y * gain[s].y);
                    normed[s][1] = pack_bf16x2(o.z * gain[s].z, o.w * gain[s].w);
                    if (m < a.M) *reinterpret_cast<float4*>(g.out + (size_t)m * g.N + n) = o;
                    if (g.next_gain)
                        *reinterpret_cast<float4*>(row_values + (16 * (t - h) + col) * T::ROW_FLOATS + (w * SW + s) * STRIP + quad * 4) = o;
                }
                if (!g.next_gain) continue;  // uniform
                static_assert(SW == 2, "two strips trade halves");
                const uint4 both = pair_blocks(normed[0], normed[1]);
                if (m < a.M) *reinterpret_cast<uint4*>(g.out_n + act_index(m, strip[quad & 1] * STRIP + (quad & 2) * 4, g.N)) = both;
            }
            if (!g.next_gain) continue;
            __syncthreads();
            const int row = threadIdx.x / 4;
            if (row >= 16 * HALF) continue;
            float c = 0.f;
#pragma unroll
            for (int s = 0; s < SPAN_STRIPS; ++s) {
                const float4 o = *reinterpret_cast<const float4*>(row_values + row * T::ROW_FLOATS + s * STRIP + threadIdx.x % 4 * 4);
                c = add_squares(c, o.x, o.y, o.z, o.w);
            }
            c += dpp_move<0xB1>(c);  // quad_perm [1, 0, 3, 2]
            c += dpp_move<0x4E>(c);  // quad_perm [2, 3, 0, 1]
            const int m = m0 + 16 * h + row;
            if (threadIdx.x % 4 == 0 && m < a.M) g.out_sq[(size_t)m * (g.N / SPAN) + nb] = c;
        }
    } else {
#pragma unroll
        for (int t = 0; t < TT; ++t) {
            const int m = m0 + 16 * t + col;
            const float rs = scales[16 * t + col];
            if constexpr (EPI == EPI_SILU) {
                const SiluRow silu_row(rs);
                float v[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) v[i] = silu_row(acc[0][t][i], acc[SW - 1][t][i]);
                if (m < a.M)
                    *reinterpret_cast<uint2*>(g.mlp + act_index(m, strip[0] * STRIP + quad * 4, g.N / 2)) =
                        make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
            } else {
                const bool held = m < a.M && pos[t] < (uint32_t)a.capacity && slot[t] < (uint32_t)a.nslots;
                const uint32_t p = held ? pos[t] : 0;
                const uint32_t block = a.table[(size_t)(held ? slot[t] : 0) * a.max_blocks + p / BLOCK_TOKENS];
#pragma unroll
                for (int s = 0; s < SW; ++s) {
                    const int e = strip[s] % (D / 16) * 8 + quad * 2;
                    float2 cs = make_float2(0.f, 0.f), sn = cs;
                    if (a.rope) {
                        cs = *reinterpret_cast<const float2*>(a.cos + (size_t)p * (D / 2) + e);
                        sn = *reinterpret_cast<const float2*>(a.sin + (size_t)p * (D / 2) + e);
                    }
                    store_qkv<D>(a, g, strip[s], m, held, p, block, acc[s][t], rs, cs, sn);
                }
            }
        }
    }
}

template <int EPI, int WR, int SW, int TT, int DEPTH, int D, int SPANS>
void direct(const char* label, const PrefillArgs& a, const GemmArgs& g, hipStream_t stream, DispatchTimer* timer) {
    const int units = g.N / STRIP / SW, tiles = (a.M + 15) / 16, groups = (tiles + TT - 1) / TT;
    dispatch(label, prefill_direct<EPI, WR, SW, TT, DEPTH, D, SPANS>, dim3(units * groups), dim3(direct_waves<EPI, TT>() * WAVE), 0,
             stream, timer, a, g, groups);
}

template <int EPI, int WR, int TT, int G, int R, int D>
void ring(const char* label, const PrefillArgs& a, const GemmArgs& g, hipStream_t stream, DispatchTimer* timer) {
    constexpr int SW = 2;
    const int NB = g.N / STRIP / (RING_WAVES * SW), MB = (a.M + 16 * TT - 1) / (16 * TT);
    dispatch(label, prefill_ring<EPI, WR, SW, TT, G, R, D>, dim3(NB * MB), dim3(RING_WAVES * WAVE), RingTile<SW, TT, G, R>::LDS, stream, timer,
             a, g, NB, MB);
}

// The workgroups prefill_ring takes for M rows in tiles of 16 TT.
int ring_groups(int M, int N, int TT) { return N / SPAN * ((M + 16 * TT - 1) / (16 * TT)); }

// The tiles a workgroup, of the `n` counts in tts (fewest first), by which M rows take the fewest rounds of
// a workgroup to each of the 256 CUs; the fewest tiles among equals, the shortest chain a k-block. us by
// 1 / 2 / 3 / 4 / 6 / 8 tiles: down_proj at 500 rows 18.3 / 19.6 / 22.5 / 24.0 / 27.3 / 38.1, 960 rows 30.4 /
// 20.6 / 22.2 / 23.4 / 30.1 / 38.4, 1167 rows - / 28.9 / 22.5 / 23.8 / 29.9 / 38.7, 2000 rows - / 38.0 / 39.2 /
// 26.0 / 31.1 / 38.4, 2600 rows - / - / 41.6 / 37.8 / 32.9 / 39.8, 4000 rows - / - / 60.2 / 48.5 / 50.2 / 44.0, 5000
// rows - / - / 78.0 / 62.2 / 53.7 / 59.7; gate/up at 300 rows 14.7 by two, 12.8 by four, 11.4 by six, 12.3 by
// eight, 500 rows 18.9 / 14.0 / 15.6 / 12.5, 768 rows 23.8 / 20.2 / 17.4 / 18.0, 1167 rows 34.5 / 29.2 / 28.3 /
// 27.0.
int fewest_rounds(int M, int N, const int* tts, int n) {
    int best = tts[0], rounds = (ring_groups(M, N, best) + 255) / 256;
    for (int i = 1; i < n; ++i) {
        const int r = (ring_groups(M, N, tts[i]) + 255) / 256;
        if (r < rounds) {
            best = tts[i];
            rounds = r;
        }
    }
    return best;
}

// The ring while its operands, read again by each workgroup, cost less than prefill_gemm's 256 x 128 tiles
// leave idle (down_proj 77.9 against 96.1 us at 8192 rows, 158 against 139 at 16384; gate/up 32.3 against
// 31.9 at 1600, 36.1 against 34.5 at 2000). q/k/v, whose epilogue leaves no registers for more, takes two
// tiles or four with a k-block a stage (4096 rows 23.3 against 26.8 with two; 8192: 39.5, prefill_gemm
// 43.8; 16384: 74.5, 70).
template <int EPI, int WR, int D>
hipError_t ring_by_rows(const char* label, const PrefillArgs& a, int strip_rows, const GemmArgs& g, hipStream_t stream, DispatchTimer* timer) {
    if constexpr (EPI == EPI_QKV) {
        if (ring_groups(a.M, g.N, 2) <= 256)
            ring<EPI, WR, 2, 2, 4, D>(label, a, g, stream, timer);
        else if (ring_groups(a.M, g.N, 4) <= 1280)
            ring<EPI, WR, 4, 1, 8, D>(label, a, g, stream, timer);
        else
            return launch_prefill_gemm(a, EPI, strip_rows, g, stream, timer);
    } else {
        if (ring_groups(a.M, g.N, 8) > 768) return launch_prefill_gemm(a, EPI, strip_rows, g, stream, timer);
        constexpr int tts[] = {1, 2, 3, 4, 6, 8}, pairs[] = {2, 4, 6, 8};
        int tt = residual_epilogue(EPI) ? fewest_rounds(a.M, g.N, tts, 6) : fewest_rounds(a.M, g.N, pairs, 4);
        // Two full rounds of six tiles against eight's round and a half: o_proj 29.1 against 28.1 us at 6000
        // rows (5000 rows, the second round less full: 23.9 against 26.8).
        const int six = ring_groups(a.M, g.N, 6);
        if (residual_epilogue(EPI) && tt == 6 && six > 256 && six * 8 > (six + 255) / 256 * 256 * 7) tt = 8;
        if constexpr (residual_epilogue(EPI)) {
            if (tt == 1) ring<EPI, WR, 1, 4, 4, D>(label, a, g, stream, timer);
            if (tt == 3) ring<EPI, WR, 3, 4, 4, D>(label, a, g, stream, timer);
        }
        if (tt == 2) ring<EPI, WR, 2, 2, 4, D>(label, a, g, stream, timer);
        if (tt == 4) ring<EPI, WR, 4, 2, 4, D>(label, a, g, stream, timer);
        if (tt == 6) ring<EPI, WR, 6, 2, 4, D>(label, a, g, stream, timer);
        if (tt == 8) ring<EPI, WR, 8, 1, 4, D>(label, a, g, stream, timer);
    }
    return hipGetLastError();
}

template <int EPI, int WR, int D = HEAD_DIM>
hipError_t projection(const char* label, const PrefillArgs& a, int strip_rows, const GemmArgs& g, hipStream_t stream, DispatchTimer* timer) {
    if constexpr (EPI == EPI_QKV) {
        if (prefill_by_rows(a.M, a.hidden)) {
            if (g.K == 2048)
                direct<EPI, WR, 2, 1, 16, D, 16>(label, a, g, stream, timer);
            else
                direct<EPI, WR, 2, 1, 16, D, 8>(label, a, g, stream, timer);
            return hipGetLastError();
        }
    } else if constexpr (EPI == EPI_SILU) {
        // A pair of strips by a tile up to two tiles (4.7 us at 16 rows where the ring takes 7.9; 6.2 at
        // 32), the ring past that (at 57 rows 8.0, the pair by a tile 9.2).
        if (a.M <= 32) {
            if (g.K == 2048)
                direct<EPI, WR, 2, 1, 16, D, 16>(label, a, g, stream, timer);
            else
                direct<EPI, WR, 2, 1, 16, D, 8>(label, a, g, stream, timer);
            return hipGetLastError();
        }
    } else if constexpr (EPI == EPI_RESIDUAL) {
        if (prefill_by_rows(a.M, a.hidden)) {
            // A strip by a tile to a wave while those waves are at most three to a CU, two by two past
            // that (at 128 rows, 512 waves: 8.0 us against 10.7; at 256 rows: 13.6 against 10.4).
            if (g.N / STRIP * ((a.M + 15) / 16) <= 768)
                direct<EPI, WR, 1, 1, 16, D, 0>(label, a, g, stream, timer);
            else
                direct<EPI, WR, 2, 2, 8, D, 0>(label, a, g, stream, timer);
            return hipGetLastError();
        }
    }
    return ring_by_rows<EPI, WR, D>(label, a, strip_rows, g, stream, timer);
}

}  // namespace

hipError_t launch_prefill_projection(const PrefillArgs& a, int epi, int strip_rows, const GemmArgs& g, hipStream_t stream,
                                     DispatchTimer* timer) {
    if (g.K <= 0 || g.K % 1024 || g.N <= 0 || g.N % 256 || a.M_pad % 256 || a.M <= 0 || a.M > a.M_pad) return hipErrorInvalidValue;
    if (residual_epilogue(epi) ? strip_rows != 4 && strip_rows != 16 : strip_rows != QKV_ROWS || g.K > MAX_SPANS * SPAN)
        return hipErrorInvalidValue;
    switch (epi) {
        case EPI_QKV:
            if (a.head_dim == 128) return projection<EPI_QKV, QKV_ROWS, 128>("prefill_qkv", a, strip_rows, g, stream, timer);
            if (a.head_dim == 64) return projection<EPI_QKV, QKV_ROWS, 64>("prefill_qkv", a, strip_rows, g, stream, timer);
            return hipErrorInvalidValue;
        case EPI_SILU: return projection<EPI_SILU, QKV_ROWS>("prefill_gate_up", a, strip_rows, g, stream, timer);
        case EPI_RESIDUAL_IN:
            return strip_rows == 4 ? projection<EPI_RESIDUAL_IN, 4>("prefill_o", a, strip_rows, g, stream, timer)
                                   : projection<EPI_RESIDUAL_IN, 16>("prefill_o", a, strip_rows, g, stream, timer);
        case EPI_RESIDUAL:
            return strip_rows == 4 ? projection<EPI_RESIDUAL, 4>("prefill_down", a, strip_rows, g, stream, timer)
                                   : projection<EPI_RESIDUAL, 16>("prefill_down", a, strip_rows, g, stream, timer);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace tgx
