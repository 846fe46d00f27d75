// Linears on unquantized weights: bf16 on v_mfma_f32_16x16x32_bf16 (a weight-streaming kernel for up to 64 rows, a
// 128 x 128 tile kernel above that; kern_gemm_mfma.hip has the 256-row tiles for prompts), and a true f32 form for
// models that run in 32 bits.  All of them share the epilogues of LinearEpilogue.
// The matrix instruction takes the weight tile as its first operand, so lane l of an accumulator tile holds row
// l % 16 of the output and its columns 4 (l / 16) .. + 3.
#include <algorithm>
#include <type_traits>

#include "device_utils.hpp"
#include "kernels.hpp"
#include "linear_epilogue.hpp"

namespace fa {
namespace k {
using namespace fa::dev;

int g_linear_form = 0;        // tuning: 2 keeps the large-tile kernel out, 3 norms in front of the linears; grouped rows: 4 streamed
                              // weights, 5 128 x 128 tiles, 6 large tiles whatever the rows

namespace {

// ------------------------------------------------------------------ up to 64 rows
// A block owns NTW column tiles.  Its eight wavefronts take every eighth pair of k tiles, two pairs at a time under way: the weight
// tiles in registers, the activation rows' 128 bytes of a pair in LDS, eight neighbouring lanes to a row.  The
// sums meet in LDS in a fixed order.  row_of(i): the activation row behind row i of the block's rows (i < m; others repeat the last
// one and are never stored) and the output row.
// What bounds it is the weights' way from memory, as long as the rows do not stand in it: the matrix instruction wants a lane to
// hold 16 bytes of its own row, and loaded that way into registers four neighbouring lanes touch four cache lines, which the
// address unit serves one per cycle (64 cycles an instruction instead of 16).  In microseconds, loaded so and staged, with 4, 16
// and 32 rows: 2048 -> 2048 4.6, 6.0, 8.0 and 4.1, 4.7, 5.7; 2048 -> 6176 6.7, 9.3, 9.5 and 6.1, 6.6, 8.1; 8192 -> 2048 10.0,
// 15.1, 21.1 and 9.1, 11.5, 15.3; 4096 -> 32000 47, 45, 50 and 42, 42, 47 (6.3 TB/s).  33 to 64 rows, whole prompts of 33, 48 and
// 64 rows through four layers of width 2048 373, 397, 421 and 335, 343, 353, of 4096 574, 620, 670 and 504, 524, 548.  What the
// epilogue reads from memory is requested ahead of the weights (0.7 us of the residual form at 4.5).
// Loads of rows are buffer loads: behind a global load into LDS, which the compiler takes for one that LDS answers, it waits for
// everything instead of counting.  (Worth up to 2 %, and that with 33 to 48 rows of width 4096: while one wavefront waited for both
// pairs, the block's other seven had theirs under way.)  A pair's rows are requested ahead of its weights, so that they are read back
// while those travel.
constexpr int kRowWaves = 8, kRowPairs = 2;          // wavefronts of a block; pairs of k tiles under way in each
constexpr uint32_t row_stage_bytes(int mt) { return mt * 2048; }     // rows of one pair
constexpr uint32_t row_lds_bytes(int mt, int ntw) {
    const uint32_t stage = kRowWaves * kRowPairs * row_stage_bytes(mt), sums = kRowWaves * mt * ntw * 1024;
    return stage > sums ? stage : sums;
}
typedef __attribute__((address_space(1))) const void *gptr;
typedef __attribute__((address_space(3))) void *lptr;

// No load moves across this one (in the program; it is no instruction).
__device__ __forceinline__ void loads_stay() { asm volatile("" ::: "memory"); }
// This wavefront's loads but the N youngest have landed, those into LDS too.  N counts what was issued since: loads_stay keeps it there.
template <int N>
__device__ __forceinline__ void loads_wait() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
// The operand fragments of MT row tiles of a staged pair: k tile h of row tile i at at[h] + BASE + 2048 i.  Assembly, because the
// compiler would wait for every load into LDS that is under way ahead of any read.
template <int BASE>
__device__ __forceinline__ void stage_read(v4i (&a)[1][2], const uint32_t (&at)[2]) {
    asm volatile("ds_read_b128 %0, %2 offset:%4\n\tds_read_b128 %1, %3 offset:%4\n\ts_waitcnt lgkmcnt(0)"
                 : "=&v"(a[0][0]), "=&v"(a[0][1])
                 : "v"(at[0]), "v"(at[1]), "n"(BASE)
                 : "memory");
}
template <int BASE>
__device__ __forceinline__ void stage_read(v4i (&a)[2][2], const uint32_t (&at)[2]) {
    asm volatile("ds_read_b128 %0, %4 offset:%6\n\tds_read_b128 %1, %5 offset:%6\n\t"
                 "ds_read_b128 %2, %4 offset:%7\n\tds_read_b128 %3, %5 offset:%7\n\ts_waitcnt lgkmcnt(0)"
                 : "=&v"(a[0][0]), "=&v"(a[0][1]), "=&v"(a[1][0]), "=&v"(a[1][1])
                 : "v"(at[0]), "v"(at[1]), "n"(BASE), "n"(BASE + 2048)
                 : "memory");
}
template <int BASE>
__device__ __forceinline__ void stage_read(v4i (&a)[4][2], const uint32_t (&at)[2]) {
    asm volatile("ds_read_b128 %0, %8 offset:%10\n\tds_read_b128 %1, %9 offset:%10\n\t"
                 "ds_read_b128 %2, %8 offset:%11\n\tds_read_b128 %3, %9 offset:%11\n\t"
                 "ds_read_b128 %4, %8 offset:%12\n\tds_read_b128 %5, %9 offset:%12\n\t"
                 "ds_read_b128 %6, %8 offset:%13\n\tds_read_b128 %7, %9 offset:%13\n\ts_waitcnt lgkmcnt(0)"
                 : "=&v"(a[0][0]), "=&v"(a[0][1]), "=&v"(a[1][0]), "=&v"(a[1][1]), "=&v"(a[2][0]), "=&v"(a[2][1]), "=&v"(a[3][0]), "=&v"(a[3][1])
                 : "v"(at[0]), "v"(at[1]), "n"(BASE), "n"(BASE + 2048), "n"(BASE + 4096), "n"(BASE + 6144)
                 : "memory");
}

// Up to four rows that are still ahead of their norm: the block norms them itself, two wavefronts to a row, while its first weights
// travel, and keeps them in LDS (pitch below), so that the norm needs no launch in front of this one.  V: four values per thread
// and step of 512 columns.  4 rows, the norm's launch and this one against this one alone: 2048 -> 6176 9.4,
// 8.1 us; 2048 -> 1360 7.2, 5.8; 2048 -> 16384 16.0, 14.5; 4096 -> 12352 22.6, 21.2.
constexpr uint32_t kNormRows = 4;
__host__ __device__ constexpr uint32_t normed_pitch(uint32_t k_pad) { return k_pad * 2 + 32; }     // rows in different banks
template <int V>
struct RowsAhead {
    v4f x[V], w[V];
};
template <int V>
__device__ __forceinline__ void norm_rows_load(const NormAhead &nm, uint32_t m, RowsAhead<V> &ra) {
    const uint32_t row = __builtin_amdgcn_readfirstlane(threadIdx.x / 128);
    if (row >= m) return;
    const float *x = nm.x + (uint64_t)row * nm.hidden;
#pragma unroll
    for (int i = 0; i < V; ++i) {
        const uint32_t c = (threadIdx.x % 128) * 4 + i * 512, from = c < nm.hidden ? c : nm.hidden - 4;
        ra.x[i] = *(const v4f *)(x + from);
        ra.w[i] = *(const v4f *)(nm.w + from);
    }
}
// The rows' sums meet in `meet` [2 x 8]; two barriers, the normed rows are not yet published.
template <int V>
__device__ __forceinline__ void norm_rows_store(const NormAhead &nm, uint32_t m, uint32_t k_pad, RowsAhead<V> &ra, float *meet, uint8_t *rows) {
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), row = wave / 2;
    float sum = 0.0f, sq = 0.0f, mean = 0.0f;
    if (row < m && !nm.rms) {
#pragma unroll
        for (int i = 0; i < V; ++i)
            if ((threadIdx.x % 128) * 4 + i * 512 < nm.hidden) sum += (ra.x[i][0] + ra.x[i][1]) + (ra.x[i][2] + ra.x[i][3]);
        sum = wave_sum_dpp(sum);
    }
    if (threadIdx.x % 64 == 0) meet[wave] = sum;
    __syncthreads();
    if (row < m) {
        mean = nm.rms ? 0.0f : (meet[row * 2] + meet[row * 2 + 1]) / (float)nm.hidden;
#pragma unroll
        for (int i = 0; i < V; ++i) {
            if ((threadIdx.x % 128) * 4 + i * 512 >= nm.hidden) continue;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                ra.x[i][e] -= mean;
                sq = fmaf(ra.x[i][e], ra.x[i][e], sq);
            }
        }
        sq = wave_sum_dpp(sq);
    }
    if (threadIdx.x % 64 == 0) meet[8 + wave] = sq;
    __syncthreads();
    if (row >= m) return;
    const float rstd = 1.0f / sqrtf((meet[8 + row * 2] + meet[8 + row * 2 + 1]) / (float)nm.hidden + nm.eps);
#pragma unroll
    for (int i = 0; i < V; ++i) {
        const uint32_t c = (threadIdx.x % 128) * 4 + i * 512;
        if (c >= k_pad) continue;
        const v4f y = c < nm.hidden ? ra.x[i] * rstd * ra.w[i] : v4f{0.f, 0.f, 0.f, 0.f};
        *(v2u *)(rows + row * normed_pitch(k_pad) + c * 2) = v2u{f32x2_to_bf16x2(y[0], y[1]), f32x2_to_bf16x2(y[2], y[3])};
    }
}

// NORM: 0 rows of `a`, otherwise V of the rows that `nm` names
template <int MT, int NTW, int MODE, int NORM, typename RowOf>
__device__ __forceinline__ void linear_rows(const uint16_t *__restrict__ a, uint64_t lda, const uint8_t *__restrict__ w_batch, uint32_t m,
                                            uint32_t n, uint32_t n_tiles, uint32_t k_tiles, uint32_t batch, const LinearEpilogue &ep, const NormAhead &nm,
                                            uint8_t *lds, RowOf row_of) {
    static_assert(NORM == 0 || MT == 1, "rows that the block norms are few");
    static_assert(!is_glu(MODE) || NTW % 2 == 0, "gate and up are neighbouring tiles");
    constexpr int NT = MT * NTW, STEP = is_glu(MODE) ? 2 : 1, SINCE = 2 * (NORM ? 0 : MT) + 4 * NTW;      // issued since a slot's rows
    static_assert(NT <= kRowWaves * STEP, "a wavefront finishes one tile, or one gate and its up");
    const int lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    const uint32_t nt0 = blockIdx.x * NTW, pairs = k_tiles / 2;
    const uint32_t cnt = pairs > (uint32_t)wave ? (pairs - wave + kRowWaves - 1) / kRowWaves : 0;
    // load x of a row tile: rows 8 x .. + 7, lane l brings piece (l % 8) ^ (l / 8) of row l / 8, so that the 16 lanes an LDS
    // read serves together (eight rows of two neighbouring k groups) find theirs in different banks
    [[maybe_unused]] uint32_t a_at[MT][2];
    [[maybe_unused]] const __amdgpu_buffer_rsrc_t a_all = __builtin_amdgcn_make_buffer_rsrc((void *)a, 0, -1, 0x00020000);
    [[maybe_unused]] RowsAhead<NORM ? NORM : 1> ra;
    if constexpr (NORM != 0) norm_rows_load(nm, m, ra);
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int x = 0; x < (NORM ? 0 : 2); ++x) {
            const uint32_t r = i * 16 + x * 8 + lane / 8;
            a_at[i][x] = row_of(r < m ? r : m - 1).x * (uint32_t)lda * 2 + ((lane % 8) ^ (lane / 8)) * 16;
        }
    gptr w_all = (gptr)w_batch;
    asm volatile("" : "+s"(w_all));                  // (of a pointer that nothing else names, loads could pass loads_stay)
    const uint8_t *w_src[NTW];
#pragma unroll
    for (int j = 0; j < NTW; ++j) w_src[j] = (const uint8_t *)w_all + (uint64_t)(nt0 + j < n_tiles ? nt0 + j : n_tiles - 1) * k_tiles * 1024 + lane * 16;
    uint8_t *stage = lds + wave * (kRowPairs * row_stage_bytes(MT));
    const uint32_t r16 = lane % 16, at0 = (uint32_t)(uintptr_t)(lptr)stage + (r16 / 8) * 1024 + (r16 % 8) * 128;
    const uint32_t at[2] = {at0 + (((uint32_t)lane / 16) ^ (r16 % 8)) * 16, at0 + ((4 + (uint32_t)lane / 16) ^ (r16 % 8)) * 16};
    // normed rows: k group lane / 16 of row lane % 16; rows at or past m read row 0 and are never stored
    uint8_t *normed = lds + kRowWaves * NT * 1024;
    [[maybe_unused]] const uint8_t *own_row = normed + (r16 < m ? r16 : 0) * normed_pitch(k_tiles * 32) + lane / 16 * 16;
    // the tile this wavefront finishes
    const uint32_t t = wave * STEP, row = t / NTW * 16 + r16, tile = nt0 + t % NTW;
    const bool own = t < (uint32_t)NT && row < m && tile < n_tiles;
    const uint32_t out_row = own ? row_of(row).y : 0, col = (is_glu(MODE) ? tile / 2 : tile) * 16 + 4 * (lane / 16);
    const EpilogueAhead ahead = own ? epilogue_ahead<MODE>(ep, out_row, col, n, batch) : EpilogueAhead{};
    __builtin_amdgcn_sched_barrier(0);

    v4f acc[MT][NTW];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NTW; ++j) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};
    v4i bv[kRowPairs][2][NTW];
    auto load = [&](int s, uint32_t it) {            // past the end: the wavefront's last pair again, so that the number under way is the same
        const uint32_t p = cnt ? wave + (it < cnt ? it : cnt - 1) * kRowWaves : 0;
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int x = 0; x < (NORM ? 0 : 2); ++x)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(a_all, (lptr)(stage + s * row_stage_bytes(MT) + i * 2048 + x * 1024), 16, a_at[i][x], p * 128, 0, 0);
        loads_stay();
#pragma unroll
        for (int j = 0; j < NTW; ++j)
#pragma unroll
            for (int h = 0; h < 2; ++h) bv[s][h][j] = stream_load<true>((const v4i *)(w_src[j] + (uint64_t)p * 2048 + h * 1024));
        loads_stay();
    };
    auto mul = [&](auto sc, uint32_t it) {
        constexpr int s = decltype(sc)::value;
        v4i av[MT][2];
        if constexpr (NORM != 0) {
#pragma unroll
            for (int h = 0; h < 2; ++h) av[0][h] = *(const v4i *)(own_row + (wave + it * kRowWaves) * 128 + h * 64);
        } else {
            stage_read<s * (int)row_stage_bytes(MT)>(av, at);
        }
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int j = 0; j < NTW; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, bv[s][h][j]), __builtin_bit_cast(v8bf, av[i][h]),
                                                                        acc[i][j], 0, 0, 0);
    };
    static_assert(kRowPairs == 2, "two slots are written out below");
    // (ahead of a norm also in wavefronts without a pair, who load the first one, and nobody reads it: behind a branch nothing could
    // count these loads, and the norm would wait for them instead of for its rows)
    if (NORM != 0 || cnt != 0) {
        load(0, 0);
        load(1, 1);
    }
    if constexpr (NORM != 0) {
        __builtin_amdgcn_sched_barrier(0);
        norm_rows_store(nm, m, k_tiles * 32, ra, (float *)(normed + kNormRows * normed_pitch(k_tiles * 32)), normed);
        __syncthreads();
    }
    if (cnt != 0) {
        uint32_t it = 0;
        for (; it + 2 < cnt; it += 2) {
            // the reads of a slot are complete (stage_read waits) before it is loaded again
            loads_wait<SINCE>();
            mul(std::integral_constant<int, 0>{}, it);
            __builtin_amdgcn_sched_barrier(0);
            load(0, it + 2);
            __builtin_amdgcn_sched_barrier(0);
            loads_wait<SINCE>();
            mul(std::integral_constant<int, 1>{}, it + 1);
            __builtin_amdgcn_sched_barrier(0);
            load(1, it + 3);
            __builtin_amdgcn_sched_barrier(0);
        }
        loads_wait<SINCE>();
        mul(std::integral_constant<int, 0>{}, it);
        loads_wait<0>();
        if (it + 1 < cnt) mul(std::integral_constant<int, 1>{}, it + 1);
    }
    loads_wait<0>();                                 // (no load into LDS is under way any more)
    v4f(*red)[NT][64] = (v4f(*)[NT][64])lds;
    if constexpr (NORM == 0) __syncthreads();        // nobody reads staged rows any more
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NTW; ++j) red[wave][i * NTW + j][lane] = acc[i][j];
    __syncthreads();
    if (!own) return;
    auto total = [&](int u) {
        v4f r = red[0][u][lane];
#pragma unroll
        for (int q = 1; q < kRowWaves; ++q) r += red[q][u][lane];
        return r;
    };
    const v4f x = total(t);
    epilogue_store4<MODE, true>(ep, out_row, col, n, batch, x, STEP == 2 ? total(t + 1) : x, ahead);
}

template <int MT, int NTW, int MODE>
__global__ void __launch_bounds__(kRowWaves * 64)
    linear_rows_kernel(const uint16_t *__restrict__ a, uint64_t lda, uint64_t a_batch, const uint8_t *__restrict__ w, uint32_t m,
                       uint32_t n, uint32_t n_tiles, uint32_t k_tiles, LinearEpilogue ep) {
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const uint32_t batch = blockIdx.y;
    linear_rows<MT, NTW, MODE, 0>(a + batch * a_batch, lda, w + (uint64_t)batch * n_tiles * k_tiles * 1024, m, n, n_tiles, k_tiles, batch, ep,
                                  NormAhead{}, lds, [](uint32_t r) { return make_uint2(r, r); });
}

template <int V, int NTW, int MODE>
__global__ void __launch_bounds__(kRowWaves * 64)
    linear_normed_rows_kernel(NormAhead nm, const uint8_t *__restrict__ w, uint32_t m, uint32_t n, uint32_t n_tiles, uint32_t k_tiles, LinearEpilogue ep) {
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    linear_rows<1, NTW, MODE, V>(nullptr, 0, w, m, n, n_tiles, k_tiles, 0, ep, nm, lds, [](uint32_t r) { return make_uint2(r, r); });
}

// The rows of a group, up to 16 MT at a time (its weights then come from the caches again); groups without rows cost a
// launch slot only.
template <int MT, int NTW, int MODE>
__global__ void __launch_bounds__(kRowWaves * 64)
    linear_rows_grouped_kernel(const uint16_t *__restrict__ a, uint64_t lda, const uint8_t *__restrict__ w, uint32_t n, uint32_t n_tiles,
                               uint32_t k_tiles, RowGroups rg, LinearEpilogue ep) {
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const uint32_t group = blockIdx.y;
    uint32_t m = rg.count[group];
    m = m < rg.pitch ? m : rg.pitch;
    const uint8_t *wg = w + (uint64_t)group * n_tiles * k_tiles * 1024;
    for (uint32_t r0 = 0; r0 < m; r0 += 16 * MT) {
        const uint32_t left = m - r0;
        const uint32_t *list = rg.list + (uint64_t)group * rg.pitch + r0;
        auto row_of = [&](uint32_t r) {
            const uint32_t e = list[r];
            return make_uint2(e / rg.a_div, e);
        };
        if (r0) __syncthreads();
        if (MT == 1 || left <= 16) linear_rows<1, NTW, MODE, 0>(a, lda, wg, left < 16 ? left : 16, n, n_tiles, k_tiles, 0, ep, NormAhead{}, lds, row_of);
        else if (MT == 2 || left <= 32) linear_rows<(MT < 2 ? MT : 2), NTW, MODE, 0>(a, lda, wg, left < 32 ? left : 32, n, n_tiles, k_tiles, 0, ep, NormAhead{}, lds, row_of);
        else linear_rows<MT, NTW, MODE, 0>(a, lda, wg, left < 16 * MT ? left : 16 * MT, n, n_tiles, k_tiles, 0, ep, NormAhead{}, lds, row_of);
    }
}

// ------------------------------------------------------------------ 128 x 128 tiles
// Four wavefronts in 2 x 2, 64 x 64 each; a stage is two k tiles (64 values), double-buffered through registers.  LDS
// holds operand tiles in the instruction's lane order; the activation rows of k-group g are rotated by 4 g (+ 2 for the
// second k tile) so that the eight lanes that fetch one row's 128 bytes store to different banks.
template <int MODE, bool GROUPED = false>
__global__ void __launch_bounds__(256)
    linear_tile_kernel(const uint16_t *__restrict__ a, uint64_t lda, uint64_t a_batch, const uint8_t *__restrict__ w, uint32_t m,
                       uint32_t n, uint32_t n_tiles, uint32_t k_tiles, LinearEpilogue ep, RowGroups rg) {
    __shared__ __attribute__((aligned(16))) uint8_t lds_a[2][2][8 * 1024], lds_b[2][2][8 * 1024];   // [buffer][k tile]
    const int tid = threadIdx.x, lane = tid % 64, wave = tid / 64, wm = wave / 2, wn = wave % 2;
    uint32_t m0 = blockIdx.y * 128, nt0 = blockIdx.x * 8, batch = blockIdx.z;
    const uint32_t *list = nullptr;
    if constexpr (GROUPED) {
        uint32_t tile, column;
        if (!group_tile(rg, blockIdx.x, 128, (n_tiles + 7) / 8, &batch, &tile, &column)) return;
        m0 = tile * 128;
        nt0 = column * 8;
        m = rg.count[batch];
        list = rg.list + (uint64_t)batch * rg.pitch;
    }
    const uint8_t *ab = (const uint8_t *)(GROUPED ? a : a + batch * a_batch);
    const uint8_t *wb = w + (uint64_t)batch * n_tiles * k_tiles * 1024;
    uint32_t a_row[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t row = m0 + threadIdx.x / 8 + 32 * i;
        a_row[i] = row < m ? row : m - 1;
        if constexpr (GROUPED) a_row[i] = list[a_row[i]] / rg.a_div;
    }
    v4u as[4], bs[4];
    const int piece = tid % 8, kt2 = piece / 4, kg = piece % 4;
    auto fetch = [&](uint32_t kt) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            as[i] = *(const v4u *)(ab + (uint64_t)a_row[i] * lda * 2 + (uint64_t)kt * 64 + piece * 16);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int c = tid + 256 * i;                 // 16-byte chunk of the stage: column tile c / 128, then k tile, then lane
            uint32_t nt = nt0 + c / 128;
            nt = nt < n_tiles ? nt : n_tiles - 1;
            bs[i] = *(const v4u *)(wb + ((uint64_t)nt * k_tiles + kt) * 1024 + (c % 128) * 16);
        }
    };
    auto put = [&](int buf) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int r = tid / 8 + 32 * i;
            *(v4u *)&lds_a[buf][kt2][(r / 16) * 1024 + (kg * 16 + ((r + 4 * kg + 2 * kt2) & 15)) * 16] = as[i];
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int c = tid + 256 * i;
            *(v4u *)&lds_b[buf][(c % 128) / 64][(c / 128) * 1024 + (c % 64) * 16] = bs[i];
        }
    };
    v4f acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};
    fetch(0);
    put(0);
    __syncthreads();
    for (uint32_t kt = 0; kt < k_tiles; kt += 2) {
        const int buf = (kt / 2) & 1;
        const bool more = kt + 2 < k_tiles;
        if (more) fetch(kt + 2);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            v8bf av[4], bv[4];
            const int g = lane / 16, pos = (g * 16 + ((lane % 16 + 4 * g + 2 * h) & 15)) * 16;
#pragma unroll
            for (int i = 0; i < 4; ++i) av[i] = *(const v8bf *)&lds_a[buf][h][(wm * 4 + i) * 1024 + pos];
#pragma unroll
            for (int j = 0; j < 4; ++j) bv[j] = *(const v8bf *)&lds_b[buf][h][(wn * 4 + j) * 1024 + lane * 16];
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bv[j], av[i], acc[i][j], 0, 0, 0);
        }
        if (more) put(buf ^ 1);
        __syncthreads();
    }
    constexpr int STEP = is_glu(MODE) ? 2 : 1;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        uint32_t row = m0 + (wm * 4 + i) * 16 + lane % 16;
        if (row >= m) continue;
        if constexpr (GROUPED) row = list[row];
#pragma unroll
        for (int j = 0; j < 4; j += STEP) {
            const uint32_t nt = nt0 + wn * 4 + j;
            if (nt >= n_tiles) continue;
            const uint32_t tile = is_glu(MODE) ? nt / 2 : nt;
            epilogue_store4<MODE>(ep, row, tile * 16 + 4 * (lane / 16), n, GROUPED ? 0 : batch, acc[i][j], acc[i][j + STEP - 1]);
        }
    }
}

// ------------------------------------------------------------------ f32
// 64 x 64 outputs per block, 16 k per slab; thread (ty, tx) owns rows 4 ty .. + 3 of columns tx, tx + 16, tx + 32, tx + 48,
// so a gate column and its up column (the neighbouring tile of 16) sit in one thread.
template <int MODE, bool GROUPED = false>
__global__ void __launch_bounds__(256)
    linear_f32_kernel(const float *__restrict__ a, uint64_t lda, uint64_t a_batch, const float *__restrict__ w, uint32_t m, uint32_t n,
                      uint32_t n_tiles, uint32_t k_pad, LinearEpilogue ep, RowGroups rg) {
    __shared__ float as[16][68], bs[16][68];
    const int tid = threadIdx.x, tx = tid % 16, ty = tid / 16;
    const uint32_t m0 = blockIdx.y * 64, n0 = blockIdx.x * 64, batch = blockIdx.z, n_rows = n_tiles * 16;
    const float *ab = GROUPED ? a : a + batch * a_batch, *wb = w + (uint64_t)batch * n_rows * k_pad;
    const uint32_t *list = nullptr;
    if constexpr (GROUPED) {
        m = rg.count[batch];
        list = rg.list + (uint64_t)batch * rg.pitch;
        if (m0 >= m) return;
    }
    const int r = tid / 4, c = (tid % 4) * 4;
    uint32_t ar = m0 + r < m ? m0 + r : m - 1;
    const uint32_t br = n0 + r < n_rows ? n0 + r : n_rows - 1;
    if constexpr (GROUPED) ar = list[ar] / rg.a_div;
    float acc[4][4] = {};
    for (uint32_t k0 = 0; k0 < k_pad; k0 += 16) {
        float va[4], vb[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            va[e] = ab[(uint64_t)ar * lda + k0 + c + e];
            vb[e] = wb[(uint64_t)br * k_pad + k0 + c + e];
        }
        __syncthreads();
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            as[c + e][r] = va[e];
            bs[c + e][r] = vb[e];
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < 16; ++q)
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] = __builtin_fmaf(as[q][ty * 4 + i], bs[q][tx + 16 * j], acc[i][j]);
    }
    constexpr int STEP = is_glu(MODE) ? 2 : 1;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        uint32_t row = m0 + ty * 4 + i;
        if (row >= m) continue;
        if constexpr (GROUPED) row = list[row];
#pragma unroll
        for (int j = 0; j < 4; j += STEP) {
            const uint32_t nt = n0 / 16 + j;
            if (nt >= n_tiles) continue;
            const uint32_t col = (is_glu(MODE) ? nt / 2 : nt) * 16 + tx;
            if (col < n) epilogue_store1<MODE>(ep, row, col, GROUPED ? 0 : batch, acc[i][j], acc[i][j + STEP - 1]);
        }
    }
}

template <typename SRC, typename DST>
__global__ void __launch_bounds__(256)
    pack_linear_kernel(const SRC *__restrict__ src, uint64_t row_stride, uint64_t col_stride, uint32_t rows, uint32_t cols,
                       DST *__restrict__ dst, uint32_t k_tiles, uint32_t n0, uint32_t group, uint32_t pitch, uint32_t k0) {
    const uint64_t total = (uint64_t)rows * cols;
    for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (uint64_t)gridDim.x * 256) {
        const uint32_t r = (uint32_t)(i / cols), c = (uint32_t)(i % cols);
        const uint32_t nr = n0 + (r / group) * pitch + r % group;
        const SRC v = src[r * row_stride + c * col_stride];
        const uint32_t kc = k0 + c;
        if constexpr (sizeof(DST) == 4) {
            float f;
            if constexpr (sizeof(SRC) == 4) f = v;
            else f = bf16_to_f32(v);
            dst[(uint64_t)nr * k_tiles * 32 + kc] = f;
        } else {
            uint16_t h;
            if constexpr (sizeof(SRC) == 4) h = f32_to_bf16(v);
            else h = v;
            dst[((uint64_t)(nr / 16) * k_tiles + kc / 32) * 512 + (((kc % 32) / 8) * 16 + nr % 16) * 8 + kc % 8] = h;
        }
    }
}

// LDS beyond 64 KiB has to be asked for once
template <typename K>
void allow_lds(K kernel, uint32_t bytes) {
    if (bytes > 65536) (void)hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
}
// The rows are addressed by 32-bit byte offsets
bool rows_reach(uint64_t rows, uint64_t lda) { return rows * lda * 2 <= 1ull << 32; }
template <int MT, int NTW, int MODE>
void launch_rows(const uint16_t *a, uint64_t lda, uint64_t a_batch, uint64_t m, const LinearWeight &w, const LinearEpilogue &ep, hipStream_t s) {
    constexpr uint32_t lds = row_lds_bytes(MT, NTW);
    static const bool allowed = (allow_lds(&linear_rows_kernel<MT, NTW, MODE>, lds), true);
    (void)allowed;
    linear_rows_kernel<MT, NTW, MODE><<<dim3((w.n_tiles + NTW - 1) / NTW, w.batches), kRowWaves * 64, lds, s>>>(
        a, lda, a_batch, (const uint8_t *)w.w, (uint32_t)m, w.n, w.n_tiles, w.k_tiles, ep);
}
template <int MT, int NTW, int MODE>
void launch_rows_grouped(const uint16_t *a, uint64_t lda, const LinearWeight &w, const RowGroups &rg, const LinearEpilogue &ep, hipStream_t s) {
    constexpr uint32_t lds = row_lds_bytes(MT, NTW);
    static const bool allowed = (allow_lds(&linear_rows_grouped_kernel<MT, NTW, MODE>, lds), true);
    (void)allowed;
    linear_rows_grouped_kernel<MT, NTW, MODE><<<dim3((w.n_tiles + NTW - 1) / NTW, rg.groups), kRowWaves * 64, lds, s>>>(
        a, lda, (const uint8_t *)w.w, w.n, w.n_tiles, w.k_tiles, rg, ep);
}

// Two tiles per block as soon as one tile each does not fit the device at once, so that the rows cross the L2 half as
// often (4096 -> 6144 with 4, 16, 32 rows 11.0, 12.6, 16.4 and 10.0, 11.0, 13.1 us; 2048 -> 4096, which fits, 4.7, 5.1, 6.2 and
// 5.5, 6.1, 7.5).  Four: behind two in nearly every shape (4096 -> 28672 with 32 rows 45.1 and 45.9).  Up to
// four rows are hardly in the way, and four rounds of single tiles end more evenly (4096 -> 28672 38.9 and 36.4).
bool two_tiles(bool glu, const LinearWeight &w, uint64_t m, int num_cus) {
    const uint64_t tiles = (uint64_t)w.n_tiles * w.batches, cus = (uint64_t)num_cus;
    return glu || (tiles > cus && (m > 4 || tiles < 4 * cus));
}

template <int V, int NTW, int MODE>
void launch_normed_rows(const NormAhead &nm, uint64_t m, const LinearWeight &w, const LinearEpilogue &ep, hipStream_t s) {
    const uint32_t lds = kRowWaves * NTW * 1024 + kNormRows * normed_pitch(w.k_tiles * 32) + 64;
    linear_normed_rows_kernel<V, NTW, MODE><<<(w.n_tiles + NTW - 1) / NTW, kRowWaves * 64, lds, s>>>(nm, (const uint8_t *)w.w, (uint32_t)m, w.n, w.n_tiles,
                                                                                              w.k_tiles, ep);
}
template <int MODE>
void launch_normed(const NormAhead &nm, uint64_t m, const LinearWeight &w, const LinearEpilogue &ep, int num_cus, hipStream_t s) {
    const bool two = two_tiles(is_glu(MODE), w, m, num_cus), wide = w.k_tiles * 32 > 2048;
    if constexpr (!is_glu(MODE))
        if (!two) return wide ? launch_normed_rows<8, 1, MODE>(nm, m, w, ep, s) : launch_normed_rows<4, 1, MODE>(nm, m, w, ep, s);
    wide ? launch_normed_rows<8, 2, MODE>(nm, m, w, ep, s) : launch_normed_rows<4, 2, MODE>(nm, m, w, ep, s);
}

template <int MODE>
void launch_bf16(const uint16_t *a, uint64_t lda, uint64_t a_batch, uint64_t m, const LinearWeight &w, const LinearEpilogue &ep,
                 int num_cus, hipStream_t s, const SplitKArea *sk) {
    const uint8_t *wt = (const uint8_t *)w.w;
    if (m <= 64 && rows_reach(m, lda)) {
        const bool two = two_tiles(is_glu(MODE), w, m, num_cus);
        if (m <= 16) {
            if constexpr (!is_glu(MODE))
                if (!two) return launch_rows<1, 1, MODE>(a, lda, a_batch, m, w, ep, s);
            return launch_rows<1, 2, MODE>(a, lda, a_batch, m, w, ep, s);
        }
        if (m <= 32) {
            if constexpr (!is_glu(MODE))
                if (!two) return launch_rows<2, 1, MODE>(a, lda, a_batch, m, w, ep, s);
            return launch_rows<2, 2, MODE>(a, lda, a_batch, m, w, ep, s);
        }
        if constexpr (!is_glu(MODE))
            if (!two) return launch_rows<4, 1, MODE>(a, lda, a_batch, m, w, ep, s);
        return launch_rows<4, 2, MODE>(a, lda, a_batch, m, w, ep, s);
    }
    if (MODE != LinearEpilogue::kHeadGate && g_linear_form != 2 && gemm_bf16_big_applies(lda, m, w)) return gemm_bf16_big(a, m, w, ep, num_cus, s, sk);
    const dim3 grid((w.n_tiles + 7) / 8, (unsigned)((m + 127) / 128), w.batches);
    linear_tile_kernel<MODE><<<grid, 256, 0, s>>>(a, lda, a_batch, wt, (uint32_t)m, w.n, w.n_tiles, w.k_tiles, ep, RowGroups{});
}

// Grouped rows: by the rows a group gets on average.  Few: weights streamed past them; a hundred and more: large tiles
// (16 experts of width 4096 and size 5376, 4 a token, passes of three layers, ms for 32 / 64 / 256 / 512 / 1024 rows: streamed 1.05 /
// 1.28 / 2.54 / 4.07 / 7.32, 128 x 128 tiles 1.13 / 1.20 / 1.54 / 1.92 / 2.87, large tiles 1.18 / 1.28 / 1.68 / 1.81 / 2.39).
template <int MODE>
void launch_grouped_bf16(const uint16_t *a, uint64_t lda, const LinearWeight &w, const RowGroups &rg, const LinearEpilogue &ep, int num_cus, hipStream_t s) {
    const uint8_t *wt = (const uint8_t *)w.w;
    constexpr bool GLU = is_glu(MODE);
    const uint64_t mean = (rg.likely ? rg.likely : rg.entries) / rg.groups;
    const int form = g_linear_form;
    if ((form == 4 || (form != 5 && form != 6 && mean <= 10)) && rows_reach((rg.entries + rg.a_div - 1) / rg.a_div, lda)) {
        const bool two = GLU || (uint64_t)w.n_tiles * std::min(rg.groups, rg.entries) >= 2 * (uint64_t)num_cus;
        const int mt = rg.most <= 16 ? 1 : mean <= 8 ? 2 : 4;
        if constexpr (!GLU)
            if (!two) {
                if (mt == 1) launch_rows_grouped<1, 1, MODE>(a, lda, w, rg, ep, s);
                else if (mt == 2) launch_rows_grouped<2, 1, MODE>(a, lda, w, rg, ep, s);
                else launch_rows_grouped<4, 1, MODE>(a, lda, w, rg, ep, s);
                return;
            }
        if (mt == 1) launch_rows_grouped<1, 2, MODE>(a, lda, w, rg, ep, s);
        else if (mt == 2) launch_rows_grouped<2, 2, MODE>(a, lda, w, rg, ep, s);
        else launch_rows_grouped<4, 2, MODE>(a, lda, w, rg, ep, s);
        return;
    }
    if (form == 6 || (form != 5 && mean >= 112 && lda == (uint64_t)w.k_tiles * 32 && w.n_tiles >= 14)) return gemm_bf16_big_grouped(a, w, rg, ep, num_cus, s);
    const uint32_t tiles = rg.entries / 128 + std::min(rg.groups, rg.entries);
    linear_tile_kernel<MODE, true><<<tiles * ((w.n_tiles + 7) / 8), 256, 0, s>>>(a, lda, 0, wt, 0, w.n, w.n_tiles, w.k_tiles, ep, rg);
}

template <int MODE>
void launch_grouped_f32(const float *a, uint64_t lda, const LinearWeight &w, const RowGroups &rg, const LinearEpilogue &ep, hipStream_t s) {
    const dim3 grid((w.n_tiles + 3) / 4, (unsigned)((rg.most + 63) / 64), rg.groups);
    linear_f32_kernel<MODE, true><<<grid, 256, 0, s>>>(a, lda, 0, (const float *)w.w, 0, w.n, w.n_tiles, w.k_tiles * 32, ep, rg);
}

template <int MODE>
void launch_f32(const float *a, uint64_t lda, uint64_t a_batch, uint64_t m, const LinearWeight &w, const LinearEpilogue &ep, hipStream_t s) {
    const dim3 grid((w.n_tiles + 3) / 4, (unsigned)((m + 63) / 64), w.batches);
    linear_f32_kernel<MODE><<<grid, 256, 0, s>>>(a, lda, a_batch, (const float *)w.w, (uint32_t)m, w.n, w.n_tiles, w.k_tiles * 32, ep, RowGroups{});
}

}  // namespace

void linear_bf16(const uint16_t *a, uint64_t lda, uint64_t a_batch, uint64_t m, const LinearWeight &w, const LinearEpilogue &ep,
                 int num_cus, hipStream_t s, const SplitKArea *sk) {
    if (m == 0) return;
    switch (ep.mode) {
        case LinearEpilogue::kResidual: return launch_bf16<LinearEpilogue::kResidual>(a, lda, a_batch, m, w, ep, num_cus, s, sk);
        case LinearEpilogue::kGlu: return launch_bf16<LinearEpilogue::kGlu>(a, lda, a_batch, m, w, ep, num_cus, s, sk);
        case LinearEpilogue::kSiluGlu: return launch_bf16<LinearEpilogue::kSiluGlu>(a, lda, a_batch, m, w, ep, num_cus, s, sk);
        case LinearEpilogue::kSoftcap: return launch_bf16<LinearEpilogue::kSoftcap>(a, lda, a_batch, m, w, ep, num_cus, s, sk);
        case LinearEpilogue::kHeadGate: return launch_bf16<LinearEpilogue::kHeadGate>(a, lda, a_batch, m, w, ep, num_cus, s, sk);
        case LinearEpilogue::kXielu: return launch_bf16<LinearEpilogue::kXielu>(a, lda, a_batch, m, w, ep, num_cus, s, sk);
        default: return launch_bf16<LinearEpilogue::kStore>(a, lda, a_batch, m, w, ep, num_cus, s, sk);
    }
}

// Up to what the LDS and a thread's registers hold of the rows, and while the blocks that norm the same rows again cost less than
// the launch (4 rows, us, with the launch and without: 896 blocks at k of 4096 42.9 and 42.2, 2000 at 2048 25.4 and 24.7, 2000 at 4096
// 44.6 and 46.3).
bool linear_norms_rows(uint64_t m, uint64_t hidden, const LinearWeight &w, int mode, int num_cus) {
    const uint64_t k_pad = (uint64_t)w.k_tiles * 32, ntw = two_tiles(is_glu(mode), w, m, num_cus) ? 2 : 1, blocks = (w.n_tiles + ntw - 1) / ntw;
    return linear_norms_mode(mode) && m <= kNormRows && hidden % 4 == 0 && hidden <= k_pad && k_pad <= 4096 && blocks * k_pad <= 5 << 20 && w.batches == 1 && g_linear_form != 3;
}

void linear_normed_bf16(const NormAhead &nm, uint64_t m, const LinearWeight &w, const LinearEpilogue &ep, int num_cus, hipStream_t s) {
    if (m == 0) return;
    switch (ep.mode) {
        case LinearEpilogue::kGlu: return launch_normed<LinearEpilogue::kGlu>(nm, m, w, ep, num_cus, s);
        case LinearEpilogue::kSiluGlu: return launch_normed<LinearEpilogue::kSiluGlu>(nm, m, w, ep, num_cus, s);
        case LinearEpilogue::kSoftcap: return launch_normed<LinearEpilogue::kSoftcap>(nm, m, w, ep, num_cus, s);
        case LinearEpilogue::kXielu: return launch_normed<LinearEpilogue::kXielu>(nm, m, w, ep, num_cus, s);
        case LinearEpilogue::kStore: return launch_normed<LinearEpilogue::kStore>(nm, m, w, ep, num_cus, s);
        default: static_assert(!linear_norms_mode(LinearEpilogue::kResidual) && !linear_norms_mode(LinearEpilogue::kHeadGate) &&
                               !linear_norms_mode(LinearEpilogue::kSquaredRelu), "the modes above are those of the predicate");
    }
}

void linear_f32(const float *a, uint64_t lda, uint64_t a_batch, uint64_t m, const LinearWeight &w, const LinearEpilogue &ep, hipStream_t s) {
    if (m == 0) return;
    switch (ep.mode) {
        case LinearEpilogue::kResidual: return launch_f32<LinearEpilogue::kResidual>(a, lda, a_batch, m, w, ep, s);
        case LinearEpilogue::kGlu: return launch_f32<LinearEpilogue::kGlu>(a, lda, a_batch, m, w, ep, s);
        case LinearEpilogue::kSiluGlu: return launch_f32<LinearEpilogue::kSiluGlu>(a, lda, a_batch, m, w, ep, s);
        case LinearEpilogue::kSoftcap: return launch_f32<LinearEpilogue::kSoftcap>(a, lda, a_batch, m, w, ep, s);
        case LinearEpilogue::kHeadGate: return launch_f32<LinearEpilogue::kHeadGate>(a, lda, a_batch, m, w, ep, s);
        case LinearEpilogue::kXielu: return launch_f32<LinearEpilogue::kXielu>(a, lda, a_batch, m, w, ep, s);
        default: return launch_f32<LinearEpilogue::kStore>(a, lda, a_batch, m, w, ep, s);
    }
}

void linear_grouped_bf16(const uint16_t *a, uint64_t lda, const LinearWeight &w, const RowGroups &rg, const LinearEpilogue &ep, int num_cus,
                         hipStream_t s) {
    if (rg.entries == 0 || rg.groups == 0) return;
    if (ep.mode == LinearEpilogue::kSquaredRelu) launch_grouped_bf16<LinearEpilogue::kSquaredRelu>(a, lda, w, rg, ep, num_cus, s);
    else if (ep.mode == LinearEpilogue::kSiluGlu) launch_grouped_bf16<LinearEpilogue::kSiluGlu>(a, lda, w, rg, ep, num_cus, s);
    else launch_grouped_bf16<LinearEpilogue::kStore>(a, lda, w, rg, ep, num_cus, s);
}

void linear_grouped_f32(const float *a, uint64_t lda, const LinearWeight &w, const RowGroups &rg, const LinearEpilogue &ep, hipStream_t s) {
    if (rg.entries == 0 || rg.groups == 0) return;
    if (ep.mode == LinearEpilogue::kSquaredRelu) launch_grouped_f32<LinearEpilogue::kSquaredRelu>(a, lda, w, rg, ep, s);
    else if (ep.mode == LinearEpilogue::kSiluGlu) launch_grouped_f32<LinearEpilogue::kSiluGlu>(a, lda, w, rg, ep, s);
    else launch_grouped_f32<LinearEpilogue::kStore>(a, lda, w, rg, ep, s);
}

void pack_linear(const void *src, int src_f32, uint64_t row_stride, uint64_t col_stride, uint32_t rows, uint32_t cols, void *dst,
                 int dst_f32, uint32_t k_tiles, uint32_t n0, uint32_t group, uint32_t pitch, hipStream_t s, uint32_t k0) {
    const uint64_t total = (uint64_t)rows * cols;
    if (total == 0) return;
    const unsigned grid = (unsigned)std::min<uint64_t>((total + 255) / 256, 8192);
    if (src_f32 && dst_f32)
        pack_linear_kernel<float, float><<<grid, 256, 0, s>>>((const float *)src, row_stride, col_stride, rows, cols, (float *)dst, k_tiles, n0, group, pitch, k0);
    else if (src_f32)
        pack_linear_kernel<float, uint16_t><<<grid, 256, 0, s>>>((const float *)src, row_stride, col_stride, rows, cols, (uint16_t *)dst, k_tiles, n0, group, pitch, k0);
    else if (dst_f32)
        pack_linear_kernel<uint16_t, float><<<grid, 256, 0, s>>>((const uint16_t *)src, row_stride, col_stride, rows, cols, (float *)dst, k_tiles, n0, group, pitch, k0);
    else
        pack_linear_kernel<uint16_t, uint16_t><<<grid, 256, 0, s>>>((const uint16_t *)src, row_stride, col_stride, rows, cols, (uint16_t *)dst, k_tiles, n0, group, pitch, k0);
}

}  // namespace k
}  // namespace fa
