// Gate and up with SwiGLU at 1..32 token rows (the GLU forward of solution/mlp.py:69-71 where the
// call is bound by unpacking the weights once): h = fp16(silu(gate) up) with gate and up as the
// forward kernels form them, no split over work-groups.
//
// A work-group (8 waves) owns RT row tiles of 16 rows of both weights. Waves 0..3 take gate's tiles,
// waves 4..7 up's, so a wave holds one weight; the four waves of a weight take the contraction's
// 128-wide super-steps in turn and their fp32 tiles are summed through LDS in wave order. X of a
// super-step comes from L2 straight into registers, once per weight: no LDS, no barrier per step.
// With all eight waves along the contraction and both weights' tiles in each (the small-M kernel's
// layout) a wave held twice the tiles: at two token blocks no more than 6 fitted the registers, 48
// rows of each weight, which a 7B MLP has 395 of for 256 CUs; and its 28 super-steps left half the
// waves idle in the last of four rounds. Graph-replayed, gate+up, us: 7B at 3 / 16 / 32 rows 25.4 /
// 25.9 / 43.4 -> 22.6 / 26.2 / 33.9, 1.5B 10.0 / 11.2 / 13.9 -> 8.9 / 10.5 / 14.0 (4 rows the first),
// [13824, 5120] at 16 rows 31.2 -> 30.1, [4864, 896] 8.0 -> 5.8. Its launches' row tiles and the
// line to the MFMA tiles: glu_small_m in capi.hip. At 16 rows of 7B the unpacking (24
// instructions per 8 weights a lane, an instruction every 4 to 5 cycles a SIMD) takes about two
// thirds of the time, the loads alone the same.
//
// Per super-step a lane loads 16 packed bytes (32 weights of one block) of each of its RT rows and
// the matching 64 bytes of X of each 16-token block; MFMA t (v_mfma_f32_16x16x32_f16, A = weights,
// B = X^T) contracts lane group g's dword t, k = k0 + 32 g + 8 t + e. The packed bytes and statistics
// of the next super-step are in flight while one is computed; X has one set of registers, refilled
// during the last row tile.
#include <type_traits>

#include "gemm_common.h"

namespace dk {

constexpr int kSgThreads = 512;
constexpr int kSgStep = 128;   // contraction per super-step
constexpr int kSgWaves = 4;    // waves per weight
__host__ __device__ constexpr int skinny_glu_pad(int rt) { return 16 * rt + 1; }  // floats of a staged token row
__host__ __device__ constexpr size_t skinny_glu_smem_bytes(int mt, int rt) {
    return (size_t)2 * kSgWaves * 16 * mt * skinny_glu_pad(rt) * 4;
}

template <int MT, bool NESTED, int RT>
__global__ __launch_bounds__(kSgThreads) void nf4_skinny_glu_kernel(const FwdArgs a) {
    constexpr int ROWS = 16 * RT;                      // rows of each weight
    constexpr int PAD = skinny_glu_pad(RT);
    __shared__ float2_t lut2[512];  // byte-pair code books: gate's, up's
    __shared__ float c2[512];       // nested statistics: the code2 tables
    extern __shared__ __attribute__((aligned(16))) float red[];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int sel = wave >> 2, kw = wave & 3;  // this wave's weight, and its place in the contraction
    const int i = lane & 15, g = lane >> 4;
    const NF4Dev& W = a.g[sel].w;
    const int M = a.m, K = a.k, N = (int)W.n, ldx = (int)a.ldx;
    const int n0 = (int)blockIdx.x * ROWS;

    // this thread's entries of the tables of its weight's half (written to LDS once the first
    // super-step's loads are on their way too)
    const int ht = tid & 255;
    const float book_hi = W.code[ht >> 4], book_lo = W.code[ht & 15];
    const float c2v = NESTED ? W.code2[ht] : 0.0f;
    const float offset = NESTED ? *W.offset : 0.0f;
    const rsrc_t wrs = make_rsrc(W.packed, W.packed_bytes);
    const rsrc_t ars = make_rsrc(NESTED ? (const void*)W.absmax8 : (const void*)W.absmaxf, W.absmax_bytes);
    const rsrc_t a2rs = make_rsrc(W.absmax2, NESTED ? W.absmax2_bytes : 0u);
    const rsrc_t xrs = make_rsrc(a.x, a.x_bytes);
    const uint32_t bs_shift = W.bs_shift, bs2_shift = W.bs2_shift;

    // this lane's rows (A row i of tile r) and token rows (B column i of token block b)
    uint32_t wbase[RT];
    bool rok[RT];
#pragma unroll
    for (int r = 0; r < RT; ++r) {
        const int row = n0 + 16 * r + i;
        rok[r] = row < N;
        wbase[r] = (uint32_t)(rok[r] ? row : 0) * (uint32_t)K + 32u * (uint32_t)g;  // flat element index
    }
    uint32_t xbase[MT];  // byte offset of the token row (past m: bit 31, reads zeros)
#pragma unroll
    for (int b = 0; b < MT; ++b) xbase[b] = off_if(16 * b + i < M, (uint32_t)((16 * b + i) * ldx + 32 * g) * 2u);

    const int total = (K + kSgStep - 1) / kSgStep;
    float4_t acc[RT][MT];
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int b = 0; b < MT; ++b) acc[r][b] = float4_t{};

    struct Step {
        u32x4_t p[RT];
        float s[RT];
        uint32_t q8[RT];  // nested: absmax codes (the scale is completed after the wait)
    };
    u32x4_t x[MT][4];
    auto load = [&](int ss, Step& st) __attribute__((always_inline)) {
        const bool kok = ss < total && ss * kSgStep + 32 * g < K;  // k % 32 == 0: wholly in or out
#pragma unroll
        for (int r = 0; r < RT; ++r) {
            const uint32_t el = wbase[r] + (uint32_t)ss * kSgStep;
            st.p[r] = bload128(wrs, off_if(kok && rok[r], el >> 1));
            const uint32_t blk = el >> bs_shift;
            if constexpr (NESTED) {
                st.q8[r] = bload8(ars, off_if(kok && rok[r], blk));
                st.s[r] = bloadf(a2rs, off_if(kok && rok[r], (blk >> bs2_shift) * 4u));
            } else {
                st.s[r] = bloadf(ars, off_if(kok && rok[r], blk * 4u));
            }
        }
    };
    // piece t of X of a super-step (past the contraction: zeros)
    auto load_x = [&](int ss, int t) __attribute__((always_inline)) {
        const bool kok = ss < total && ss * kSgStep + 32 * g < K;
#pragma unroll
        for (int b = 0; b < MT; ++b)
            x[b][t] = bload128(xrs, kok ? xbase[b] + (uint32_t)(ss * kSgStep + 8 * t) * 2u : 0x80000000u);
    };

    Step sa, sb;
    load(kw, sa);
#pragma unroll
    for (int t = 0; t < 4; ++t) load_x(kw, t);
    lut2[tid] = float2_t{book_hi, book_lo};
    if (NESTED) c2[tid] = c2v;
    __syncthreads();

    // The main loop and the staging of its sums, once per weight: the code book's place in LDS is then
    // a constant (copies of the loop alone would merge their accumulators, through spills).
    auto run = [&](auto SEL) __attribute__((always_inline)) {
        // Row tile r, MFMA t is item 4 r + t, its code-book values read while the item before is
        // packed, one wait an item (as in the small-M kernel).
        auto compute = [&](Step& st, int next) __attribute__((always_inline)) {
#pragma unroll
            for (int r = 0; r < RT; ++r) {
                if constexpr (NESTED) st.s[r] = c2[256 * SEL.value + st.q8[r]] * st.s[r] + offset;  // two roundings (no contraction)
                if (!rok[r]) st.s[r] = 0.0f;
            }
            float v[2][8];
            auto look = [&](int item) __attribute__((always_inline)) {
                const uint32_t w = st.p[item / 4][item % 4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float2_t cv = *(const float2_t*)((const char*)lut2 + 2048 * SEL.value + byte_x8(w, e));
                    v[item % 2][2 * e] = cv.x;
                    v[item % 2][2 * e + 1] = cv.y;
                }
            };
            look(0);
#pragma unroll
            for (int item = 0; item < 4 * RT; ++item) {
                const int r = item / 4, t = item % 4;
                if (item + 1 < 4 * RT) look(item + 1);
                __builtin_amdgcn_sched_barrier(0);
                if (item + 1 < 4 * RT) wait_lgkmcnt<4>();
                else wait_lgkmcnt<0>();
                __builtin_amdgcn_sched_barrier(0);
                const half8_t av = __builtin_bit_cast(half8_t, pack_half8(v[item % 2], st.s[r]));
#pragma unroll
                for (int b = 0; b < MT; ++b) {
                    const u32x4_t xv = x[b][t];
                    acc[r][b] = mfma16x16x32(av, __builtin_bit_cast(half8_t, xv), acc[r][b]);
                }
                if (r == RT - 1) {
                    __builtin_amdgcn_sched_barrier(0);
                    load_x(next, t);
                }
            }
        };
        int ss = kw;
        while (ss < total) {
            load(ss + kSgWaves, sb);
            __builtin_amdgcn_sched_barrier(0);
            compute(sa, ss + kSgWaves);
            __builtin_amdgcn_sched_barrier(0);
            if (ss + kSgWaves >= total) break;
            load(ss + 2 * kSgWaves, sa);
            __builtin_amdgcn_sched_barrier(0);
            compute(sb, ss + 2 * kSgWaves);
            __builtin_amdgcn_sched_barrier(0);
            ss += 2 * kSgWaves;
        }

        // lane holds D[4 g + q][i] of tile r, token block b: weight row n0 + 16 r + 4 g + q, token
        // 16 b + i. Staged as red[wave][token][row]; each thread then sums the four waves of gate and
        // of up for its outputs.
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
            for (int b = 0; b < MT; ++b)
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    red[(wave * 16 * MT + 16 * b + i) * PAD + 16 * r + 4 * g + q] = acc[r][b][q];
    };
    if (sel == 0) run(std::integral_constant<int, 0>{});
    else run(std::integral_constant<int, 1>{});
    __syncthreads();
    for (int o = tid; o < 16 * MT * ROWS; o += kSgThreads) {
        const int m = o / ROWS, row = o - m * ROWS;  // consecutive threads: consecutive rows
        const int n = n0 + row;
        if (m >= M || n >= N) continue;
        float v[2];
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            v[s] = 0.0f;
#pragma unroll
            for (int w = 0; w < kSgWaves; ++w) v[s] += red[((kSgWaves * s + w) * 16 * MT + m) * PAD + row];
            if (a.g[s].bias != nullptr) v[s] += (float)a.g[s].bias[n];
        }
        // gate and up rounded to fp16 (their outputs), then the SwiGLU kernel's arithmetic
        const uint32_t g2 = pack_half2(v[0], 0.0f), u2 = pack_half2(v[1], 0.0f);
        if (a.g[0].y != nullptr) *(uint16_t*)(a.g[0].y + (int64_t)m * a.g[0].ldy + n) = (uint16_t)g2;
        if (a.g[1].y != nullptr) *(uint16_t*)(a.g[1].y + (int64_t)m * a.g[1].ldy + n) = (uint16_t)u2;
        *(uint16_t*)(a.h + (int64_t)m * a.ldh + n) = (uint16_t)swiglu_fwd2(g2, u2);
    }
}

template <int MT, int RT>
static hipError_t launch_skinny_glu_t(const FwdArgs& a, int grid, hipStream_t s) {
    const size_t lds = skinny_glu_smem_bytes(MT, RT);
    const void* fn = a.nested ? (const void*)nf4_skinny_glu_kernel<MT, true, RT> : (const void*)nf4_skinny_glu_kernel<MT, false, RT>;
    const hipError_t e = allow_dynamic_lds(fn, lds);
    if (e != hipSuccess) return e;
    if (a.nested) hipLaunchKernelGGL((nf4_skinny_glu_kernel<MT, true, RT>), dim3(grid), dim3(kSgThreads), lds, s, a);
    else hipLaunchKernelGGL((nf4_skinny_glu_kernel<MT, false, RT>), dim3(grid), dim3(kSgThreads), lds, s, a);
    return hipGetLastError();
}

template <int RT>
static hipError_t launch_skinny_glu_rt(const FwdArgs& a, int grid, hipStream_t s) {
    if (a.m <= 16) return launch_skinny_glu_t<1, RT>(a, grid, s);
    return launch_skinny_glu_t<2, RT>(a, grid, s);
}

// grid work-groups of 16 * row_tiles rows of both weights
hipError_t launch_skinny_glu(const FwdArgs& a, int row_tiles, int grid, hipStream_t s) {
    if (a.m < 1 || a.m > kSkinnyMaxM || !a.glu || a.ngroups != 2 || a.g[0].w.n != a.g[1].w.n || a.h == nullptr ||
        a.splits != 1 || a.g[0].lora_u != nullptr || a.g[1].lora_u != nullptr)
        return hipErrorInvalidValue;
    switch (row_tiles) {
        case 1: return launch_skinny_glu_rt<1>(a, grid, s);
        case 2: return launch_skinny_glu_rt<2>(a, grid, s);
        case 3: return launch_skinny_glu_rt<3>(a, grid, s);
        case 4: return launch_skinny_glu_rt<4>(a, grid, s);
        case 5: return launch_skinny_glu_rt<5>(a, grid, s);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace dk
