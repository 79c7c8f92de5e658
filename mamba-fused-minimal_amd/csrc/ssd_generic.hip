// SSD chunk-state contraction (optionally with the recurrence) for whatever the bf16 kernels do not take: fp32 and fp16
// inputs, any headdim, dstate, chunk size and alignment, with the accuracy of fp32 products and sums.
//
// The fp32 matrix instructions (256 flop per clock and compute unit) are a sixteenth of bf16's, so an operand enters as the
// sum of bf16 values: the product x * w and an fp32 B as three (all 24 bits), an f16 B as two, a bf16 B as itself, and
// v_mfma_f32_16x16x32_bf16 multiplies all pairs of parts but those below 2^-24 of the largest: 6, 5 or 3 instructions of 16 clocks
// where the fp32 ones take 256.  Each adds 32 products at a time, so the sums round less often: error against 64 bits 0.58 -
// 0.75e-7 where the fp32 instructions left 0.66 - 1.3e-7 (fp32, fp16 and odd sizes, fast and slow decays).  Where a sum is not finite
// (an infinite input, or one too large for its parts, kLift) the fp32 instructions do the wave's tokens again.
//
// What bounds it: the vector instructions, most of them the splitting of operands.  Of a SIMD's 37.8 K clocks at 2 x 2048 x 24 heads,
// fp32, they issue for 21.8 K, the matrix unit is busy for 9.2 K and the waves' waits overlap with little of either; fp16, 2 x 3001 x 24:
// 30.4 K and 11.5 K of 51.8 K (hardware counters).  For small calls it is a wave's start and the adding up at the end: 2 x 1900 x 15 x 48 x
// 96 in chunks of 64 has 1.8 waves a SIMD, vector instructions for 8.4 K and matrix instructions for 1.5 K of 23.4 K clocks.
// Chunk states, fp32 matrix instructions / this: fp16, 2 x 3001 tokens x 24 heads x 64 x 128 31.5 / 24.3 us, 8 x 3001 x 48 188 / 120;
// fp32, 2 x 2048 x 24 20.4 / 18.6; 1024 x 8 x 64 x 64 8.6 / 6.3.  A lane loads A consecutive headdim elements of eight tokens' x
// rows and S consecutive dstate elements of their B rows, and its eight tokens of one row or column *are* the operand layout: lane i
// of a 16-lane group stands for rows A i .. A i + A-1 and columns S i .. S i + S-1 of the tile, the four lane groups for eight
// consecutive tokens each, and matrix instruction (r, s) multiplies the r-th elements of the x vectors with the s-th of the B
// vectors.  No LDS on the way in, no barrier in the loop, whole rows per load; the accumulators of one lane are S consecutive
// columns, so rows leave as vectors as well.
//
// Tiles and chunks too small to repay the splitting (PARTS, generic_way in ssd_cost.h) and the walk over a sequence's chunks
// (FUSED: one chunk, or a 16-bit out without room for chunk states) keep the fp32 matrix instructions, the walk because with the
// parts beside the running state a 64 x 64 tile leaves one wave a SIMD: fp32 instructions / parts (fp16, 8 x 3000 x 48 x 64 x 128
// 234 / 242 us, 8 x 102 x 76 x 128 x 128 47 / 64, 8 x 2000 x 60 x 40 x 40 in chunks of 100 114 / 134).
//
// One workgroup owns a (16 A) x (16 S) tile of one (batch, head) and chunk; its SPLIT = 4 waves take a quarter of the
// chunk's tokens each and add up through LDS, after which wave v holds accumulator q = v of every instruction.  In
// fused mode it walks the chunks with the state in registers.  Short chunks leave a quarter too little to do between
// a wave's start and the adding up: there a wave owns a tile by itself (SPLIT = 1).  Rows and columns past the edge of an
// odd headdim or dstate are not loaded: the last lanes' vectors move up to end at the edge and repeat rows that their
// neighbours also compute.  Both store them, the same bits: a sum's order does not depend on the wave or lane that forms it.  (Not
// where only one of the two has done its tokens again in fp32: either sum is then stored, both with the accuracy stated above.)
//
// Reference semantics: kernels/ssd_chunk_state.py:97-173, kernels/ssd_state_passing.py:27-84.
#include "ssd_cost.h"
#include "ssd_tile.h"

#include <algorithm>

namespace ssd {
namespace generic {

using tile::f32x4;
using tile::static_for;

// K consecutive elements as they lie in memory, in whole registers: they stay packed until they are used, a group of
// loads later (as an array of 16-bit elements the compiler takes them apart, and so waits for them, at the load).
template <int K, typename T>
struct Row {
    static constexpr int kWords = (K * (int)sizeof(T) + 3) / 4;
    uint32_t w[kWords];
};

template <int K, typename T>
__device__ __forceinline__ Row<K, T> load_row(const T *q)
{
    Row<K, T> r;
    // element-aligned: the device takes unaligned vector loads
    if constexpr (K * sizeof(T) % 4 == 0) {
        __builtin_memcpy(r.w, q, K * sizeof(T));
    } else {
        if constexpr (K > 1) __builtin_memcpy(r.w, q, 4);
        uint16_t last;
        __builtin_memcpy(&last, q + K - 1, 2);
        r.w[r.kWords - 1] = last;
    }
    return r;
}
template <int J, typename T, int K>
__device__ __forceinline__ float element(const Row<K, T> &r)
{
    if constexpr (sizeof(T) == 4) return __builtin_bit_cast(float, r.w[J]);
    else if constexpr (std::is_same<T, _Float16>::value) return (float)__builtin_bit_cast(_Float16, (uint16_t)(r.w[J / 2] >> (J % 2 * 16)));
    else return __builtin_bit_cast(float, J % 2 ? r.w[J / 2] & 0xffff0000u : r.w[J / 2] << 16);
}

template <int K>
__device__ __forceinline__ void load_state(float (&v)[K], const void *base, int64_t off, int dt)
{
    if (dt == DT_F32) {
        __builtin_memcpy(v, (const float *)base + off, sizeof(v));
    } else {
#pragma unroll
        for (int j = 0; j < K; ++j) v[j] = load_as_f32(base, off + j, dt);
    }
}
template <int K>
__device__ __forceinline__ void store_state(void *base, int64_t off, int dt, const float (&v)[K])
{
    if (dt == DT_F32) {
        __builtin_memcpy((float *)base + off, v, sizeof(v));
    } else {
        uint16_t h[K];
#pragma unroll
        for (int j = 0; j < K; ++j) h[j] = dt == DT_BF16 ? f32_to_bf16_bits(v[j]) : __builtin_bit_cast(uint16_t, (_Float16)v[j]);
        __builtin_memcpy((uint16_t *)base + off, h, sizeof(h));
    }
}

constexpr int kWaves = 4;
constexpr int kWindow = 64;      // walk: tokens whose weights a wave computes at once, one per lane
// walk: matrix steps of four tokens whose rows are loaded together, a group ahead of their use: a group's matrix instructions
// (32 clocks each) have to last for a load's way from memory
constexpr int group_of(int tiles) { return tiles >= 12 ? 4 : 2; }
constexpr int kStep = 32;        // tokens of a bf16 matrix instruction

// Eight fp32 values as the sum of PARTS bf16 ones each (three hold all 24 bits of a value, two the 11 bits of an f16), every
// part the rest rounded to nearest.
using tile::bf16x8;
template <int PARTS>
__device__ __forceinline__ void split(const float (&v)[8], bf16x8 (&parts)[PARTS])
{
    float rest[8];
#pragma unroll
    for (int t = 0; t < 8; ++t) rest[t] = v[t];
#pragma unroll
    for (int q = 0; q < PARTS; ++q) {
        tile::u32x4 packed;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            uint32_t two = tile::pack_bf16(rest[2 * t], rest[2 * t + 1]);
            asm volatile("" : "+v"(two));      // keeps the compiler from converting a second time
            packed[t] = two;
            if (q + 1 < PARTS) {
                rest[2 * t] -= __builtin_bit_cast(float, two << 16);
                rest[2 * t + 1] -= __builtin_bit_cast(float, two & 0xffff0000u);
            }
        }
        parts[q] = __builtin_bit_cast(bf16x8, packed);
    }
}
// parts of an element of B: a bf16 is one, an f16 two, an fp32 three
template <typename T> constexpr int kBParts = sizeof(T) == 4 ? 3 : std::is_same<T, _Float16>::value ? 2 : 1;
// Three parts hold 24 bits only down to 2^-109, below that the last one is subnormal: x * w and an fp32 B are split 2^24 times as
// large, which reaches down to the smallest normal fp32 value, and the sums are scaled back.
constexpr float kLift = 0x1p24f;
template <typename T> constexpr float kBLift = kBParts<T> == 3 ? kLift : 1.f;

template <int A, int S, typename T, int SPLIT, bool FUSED, bool PARTS>
__global__ void __launch_bounds__(64 * kWaves, 2) generic_kernel(const Params p, int first_group)
{
    // partial tiles: accumulator q of the wave that owns it, from each of the three others
    constexpr int SV = S == 3 ? 4 : S;
    constexpr int kGroup = group_of(A * S);
    constexpr int kParts = SPLIT == 1 ? 1 : kWaves;
    __shared__ __align__(16) float part[kParts][kWaves - 1][SPLIT == 1 ? 1 : A][SPLIT == 1 ? 1 : 64][SV];
    static_assert(SPLIT == kWaves || (SPLIT == 1 && !FUSED), "all waves of a workgroup on one tile, or one each");
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int sub = lane >> 4, col = lane & 15;      // token of a step, vector of a row

    // Consecutive workgroups land on consecutive XCDs: give each XCD a contiguous run of tiles, so that the tiles that
    // share x (the column tiles of a head) and B (the heads of a group) share an L2.
    const int per_xcd = gridDim.x >> 3;
    int item = first_group + (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
    if (SPLIT == 1) item = item * kWaves + wv;
    if (item >= p.n_items) return;
    const int n_pt = (p.headdim + 16 * A - 1) / (16 * A), n_nt = (p.dstate + 16 * S - 1) / (16 * S);
    const int nt = item % n_nt; item /= n_nt;
    const int pt = item % n_pt; item /= n_pt;
    const int h = item % p.nheads; item /= p.nheads;
    int b, c_begin, c_end;
    if (FUSED) { b = item; c_begin = 0; c_end = p.C; }
    else { b = item / p.C; c_begin = item - b * p.C; c_end = c_begin + 1; }

    const int L = p.seqlen, Q = p.Q;
    const int g = h / (p.nheads / p.ngroups);
    const float *dtb = p.dt + b * p.sdt_b + h * p.sdt_h;
    const float *dab = p.dacs + b * p.sda_b + h * p.sda_h;
    const int32_t *sqb = p.seq ? p.seq + b * p.ssq_b : nullptr;
    // A <= headdim and S <= dstate (launcher): every vector lies inside its row
    const T *xl = (const T *)p.x + b * p.sx_b + h * p.sx_h + min(pt * 16 * A + col * A, p.headdim - A);
    const T *Bl = (const T *)p.B + b * p.sB_b + g * p.sB_g + min(nt * 16 * S + col * S, p.dstate - S);

    // what this lane holds of the finished tile: rows row(q) .. row(q) + A-1 of its accumulators q, columns
    // ncol .. ncol + S-1
    auto row_first = [&](int q) { return pt * 16 * A + (sub * 4 + q) * A; };
    const int ncol_first = nt * 16 * S + col * S, ncol = min(ncol_first, p.dstate - S);
    const int row = min(row_first(wv), p.headdim - A);
    const bool mine = row_first(wv) < p.headdim && ncol_first < p.dstate;

    float st[A][S];
    if constexpr (FUSED) {
#pragma unroll
        for (int r = 0; r < A; ++r) {
#pragma unroll
            for (int s = 0; s < S; ++s) st[r][s] = 0.f;
            if (mine) {
                if (p.init) load_state<S>(st[r], p.init, b * p.sin_b + h * p.sin_h + (int64_t)(row + r) * p.sin_p + ncol, p.dt_init);
                store_state<S>(p.out, b * p.so_b + h * p.so_h + (int64_t)(row + r) * p.so_p + ncol, p.dt_out, st[r]);
            }
        }
    }
    int32_t prev_id = 0;

    for (int c = c_begin; c < c_end; ++c) {
        const int t0 = c * Q, qlen = min(Q, L - t0);
        const int quarter = (qlen + 4 * SPLIT - 1) / (4 * SPLIT) * 4;
        const int k_begin = SPLIT == 1 ? 0 : wv * quarter, k_end = min(qlen, k_begin + quarter);
        const float last = dab[c * p.sda_c + (int64_t)(Q - 1) * p.sda_k];
        const int32_t id_last = sqb ? sqb[(int64_t)(t0 + qlen - 1) * p.ssq_l] : 0;
        const T *xc = xl + (int64_t)t0 * p.sx_l, *Bc = Bl + (int64_t)t0 * p.sB_l;

        f32x4 acc[A][S];
#pragma unroll
        for (int r = 0; r < A; ++r)
#pragma unroll
            for (int s = 0; s < S; ++s) acc[r][s] = f32x4{0.f, 0.f, 0.f, 0.f};

        if constexpr (!PARTS) {
        // fp32 matrix instructions, steps of four tokens, one per lane group
        for (int w0 = k_begin; w0 < k_end; w0 += kWindow) {
            const int steps = (min(kWindow, k_end - w0) + 3) >> 2;
            const T *xw = xc + (int64_t)(w0 + sub) * p.sx_l, *Bw = Bc + (int64_t)(w0 + sub) * p.sB_l;

            Row<A, T> xr[2][kGroup];
            Row<S, T> br[2][kGroup];
            auto load = [&](int grp, int buf) {
#pragma unroll
                for (int i = 0; i < kGroup; ++i) {
                    const int step = grp * kGroup + i;
                    const bool in = w0 + step * 4 + sub < k_end;      // elsewhere: the chunk's first token, not used
                    xr[buf][i] = load_row<A>(in ? xw + (int64_t)(step * 4) * p.sx_l : xc);
                    br[buf][i] = load_row<S>(in ? Bw + (int64_t)(step * 4) * p.sB_l : Bc);
                }
            };
            // the first rows and the weights' inputs travel together: without the fence the compiler puts the weights'
            // loads, and the wait for them, in front
            load(0, 0);
            asm volatile("" ::: "memory");
            const int kl = min(w0 + lane, k_end - 1);      // lanes past the end repeat the last token; nobody asks them
            const float da_k = dab[c * p.sda_c + (int64_t)kl * p.sda_k], dt_k = dtb[c * p.sdt_c + (int64_t)kl * p.sdt_k];
            const int32_t id_k = sqb ? sqb[(int64_t)(t0 + kl) * p.ssq_l] : 0;
            float ex = last - da_k;
            if (p.clamp) ex = fminf(ex, 0.f);
            float w = __expf(ex) * dt_k;
            if (id_k != id_last) w = 0.f;
#pragma unroll
            for (int grp = 0; grp < kWindow / 4 / kGroup; ++grp) {
                if (grp * kGroup >= steps) break;
                // always, past the last step too (the chunk's first token then): a branch around it drains the queue
                if (grp + 1 < kWindow / 4 / kGroup) load(grp + 1, (grp + 1) & 1);
#pragma unroll
                for (int i = 0; i < kGroup; ++i) {
                    const int k = (grp * kGroup + i) * 4 + sub;
                    const bool in = w0 + k < k_end;
                    const float wk = __shfl(w, k);
                    Row<A, T> xv = xr[grp & 1][i];
                    Row<S, T> bv = br[grp & 1][i];
                    // not before here: a conversion moved up to the load would wait for it
#pragma unroll
                    for (int j = 0; j < xv.kWords; ++j) asm volatile("" : "+v"(xv.w[j]));
#pragma unroll
                    for (int j = 0; j < bv.kWords; ++j) asm volatile("" : "+v"(bv.w[j]));
                    float xs[A], bs[S];
                    static_for<A>([&](auto r) { xs[r.value] = in ? element<r.value>(xv) * wk : 0.f; });
                    static_for<S>([&](auto s) { bs[s.value] = in ? element<s.value>(bv) : 0.f; });
#pragma unroll
                    for (int r = 0; r < A; ++r)
#pragma unroll
                        for (int s = 0; s < S; ++s) acc[r][s] = __builtin_amdgcn_mfma_f32_16x16x4f32(xs[r], bs[s], acc[r][s], 0, 0, 0);
                }
            }
        }
        } else {
        // Steps of 32 tokens: lane group `sub` holds the tokens 8 sub + t, t = 0 .. 7, of its rows and columns.  The rows of the
        // next step are on their way while a step is multiplied, the inputs of the weights (one token per lane) a window of
        // two steps ahead.
        const int steps = k_begin < k_end ? (k_end - k_begin + kStep - 1) / kStep : 0;
        Row<A, T> xr[8];
        Row<S, T> br[8];
        auto place = [&](int st, int t) {
            const int k = k_begin + st * kStep + 8 * sub + t;
            return (int64_t)(k < k_end ? k : 0);      // elsewhere: the chunk's first token, not used
        };
        auto load_x = [&](int st) {
#pragma unroll
            for (int t = 0; t < 8; ++t) xr[t] = load_row<A>(xc + place(st, t) * p.sx_l);
        };
        auto load_B = [&](int st) {
#pragma unroll
            for (int t = 0; t < 8; ++t) br[t] = load_row<S>(Bc + place(st, t) * p.sB_l);
        };
        float da_k = 0.f, dt_k = 0.f;
        int32_t id_k = 0;
        auto load_weights = [&](int window) {
            const int kl = min(k_begin + window * 2 * kStep + lane, k_end - 1);      // lanes past the end repeat the last token; nobody asks them
            da_k = dab[c * p.sda_c + (int64_t)kl * p.sda_k];
            dt_k = dtb[c * p.sdt_c + (int64_t)kl * p.sdt_k];
            id_k = sqb ? sqb[(int64_t)(t0 + kl) * p.ssq_l] : 0;
        };
        auto weight = [&](int window) {      // zero for tokens past the end
            float ex = last - da_k;
            if (p.clamp) ex = fminf(ex, 0.f);
            const float w = __expf(ex) * dt_k;
            return id_k != id_last || k_begin + window * 2 * kStep + lane >= k_end ? 0.f : w;
        };
        // row r of the step's x rows times the weights, column s of its B rows, as fp32 values (tokens past the end: zero times
        // whatever the first token holds)
        auto products = [&](int st, float w, auto r, float (&v)[8]) {
#pragma unroll
            for (int t = 0; t < 8; ++t) v[t] = element<decltype(r)::value>(xr[t]) * __shfl(w, (st * kStep + 8 * sub + t) & 63);
        };
        auto columns = [&](auto s, float (&v)[8]) {
#pragma unroll
            for (int t = 0; t < 8; ++t) v[t] = element<decltype(s)::value>(br[t]);
        };
        if (steps > 0) {
            load_x(0);
            load_B(0);
            load_weights(0);
        }
        float w = 0.f;
        for (int st = 0; st < steps; ++st) {
            if ((st & 1) == 0) {
                w = kLift * weight(st >> 1);
                load_weights((st >> 1) + 1);
            }
            const int next = min(st + 1, steps - 1);      // behind the last step: that one again, not used
            bf16x8 xp[A][3];
            static_for<A>([&](auto r) {
                float v[8];
                products(st, w, r, v);
                split<3>(v, xp[r.value]);
            });
            load_x(next);
            static_for<S>([&](auto s) {
                float v[8];
                columns(s, v);
                if constexpr (kBLift<T> != 1.f)
#pragma unroll
                    for (int t = 0; t < 8; ++t) v[t] *= kBLift<T>;
                bf16x8 bp[kBParts<T>];
                split<kBParts<T>>(v, bp);
                if constexpr (s.value == S - 1) load_B(next);
#pragma unroll
                for (int q = kBParts<T> - 1; q >= 0; --q)       // the smallest products first; those below 2^-24 of the largest not at all
#pragma unroll
                    for (int u = 2 - q; u >= 0; --u)
#pragma unroll
                        for (int r = 0; r < A; ++r) acc[r][s.value] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xp[r][u], bp[q], acc[r][s.value], 0, 0, 0);
            });
        }
        // An infinite value, or one that is infinite 2^24 times as large or as a bf16, leaves NaN in its rest, and so does one in the place
        // of a token past the end: where a sum is not finite this wave's tokens are added up once more by the fp32 instructions.
        float odd[4] = {0.f, 0.f, 0.f, 0.f};      // zero times every sum: NaN where one is not finite
#pragma unroll
        for (int r = 0; r < A; ++r)
#pragma unroll
            for (int s = 0; s < S; ++s)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    odd[q] = __builtin_fmaf(acc[r][s][q], 0.f, odd[q]);
                    acc[r][s][q] *= 1.f / (kLift * kBLift<T>);
                }
        if (!__all(odd[0] + odd[1] + odd[2] + odd[3] == 0.f)) {
#pragma unroll
            for (int r = 0; r < A; ++r)
#pragma unroll
                for (int s = 0; s < S; ++s) acc[r][s] = f32x4{0.f, 0.f, 0.f, 0.f};
            for (int st = 0; st < steps; ++st) {
                load_x(st);
                load_B(st);
                load_weights(st >> 1);
                w = weight(st >> 1);
                static_for<A>([&](auto r) {
                    float xs[8];
                    products(st, w, r, xs);
                    static_for<S>([&](auto s) {
                        float bs[8];
                        columns(s, bs);
#pragma unroll
                        for (int t = 0; t < 8; ++t)
                            if (k_begin + st * kStep + 8 * sub + t >= k_end) xs[t] = bs[t] = 0.f;
#pragma unroll
                        for (int t = 0; t < 8; ++t)
                            acc[r.value][s.value] = __builtin_amdgcn_mfma_f32_16x16x4f32(xs[t], bs[t], acc[r.value][s.value], 0, 0, 0);
                    });
                });
            }
        }
        }

        if constexpr (SPLIT == 1) {
            if (ncol_first >= p.dstate) return;
            static_for<kWaves>([&](auto qc) {
                constexpr int q = qc.value;
                if (row_first(q) >= p.headdim) return;
                const int row_q = min(row_first(q), p.headdim - A);
#pragma unroll
                for (int r = 0; r < A; ++r) {
                    float v[S];
#pragma unroll
                    for (int s = 0; s < S; ++s) v[s] = acc[r][s][q];
                    store_state<S>(p.states, b * p.sst_b + c * p.sst_c + h * p.sst_h + (int64_t)(row_q + r) * p.sst_p + ncol, p.dt_states, v);
                }
            });
            return;
        } else {
        // accumulator q of every wave goes to wave q
        static_for<kWaves>([&](auto qc) {
            constexpr int q = qc.value;
            if (q == wv) return;
            const int slot = wv < q ? wv : wv - 1;
#pragma unroll
            for (int r = 0; r < A; ++r)
#pragma unroll
                for (int s = 0; s < S; ++s) part[q][slot][r][lane][s] = acc[r][s][q];
        });
        __syncthreads();
        // every wave adds the four parts up in the order of the tokens, so that a row does not depend on the wave that
        // finishes it: rows that a moved-up vector repeats are stored by two waves (or workgroups), with the same bits
        float own[A][S];
        static_for<kWaves>([&](auto qc) {
            constexpr int q = qc.value;
            if (q != wv) return;
#pragma unroll
            for (int r = 0; r < A; ++r)
#pragma unroll
                for (int s = 0; s < S; ++s) {
                    auto of_wave = [&](int o) { return o == q ? acc[r][s][q] : part[q][o < q ? o : o - 1][r][lane][s]; };
                    own[r][s] = of_wave(0);
#pragma unroll
                    for (int o = 1; o < kWaves; ++o) own[r][s] += of_wave(o);
                }
        });
        if (FUSED) __syncthreads();      // the next chunk's partial tiles go to the same place

        if (p.states && mine)
#pragma unroll
            for (int r = 0; r < A; ++r)
                store_state<S>(p.states, b * p.sst_b + c * p.sst_c + h * p.sst_h + (int64_t)(row + r) * p.sst_p + ncol, p.dt_states, own[r]);
        if (FUSED) {
            float sc = __expf(last);
            if (sqb) {
                if (id_last != prev_id) sc = 0.f;
                prev_id = id_last;
            }
#pragma unroll
            for (int r = 0; r < A; ++r) {
#pragma unroll
                for (int s = 0; s < S; ++s) st[r][s] = sc * st[r][s] + own[r][s];
                if (!mine) continue;
                if (c < p.C - 1)
                    store_state<S>(p.out, b * p.so_b + (c + 1) * p.so_c + h * p.so_h + (int64_t)(row + r) * p.so_p + ncol, p.dt_out, st[r]);
                else store_state<S>(p.fin, b * p.sf_b + h * p.sf_h + (int64_t)(row + r) * p.sf_p + ncol, DT_F32, st[r]);
            }
        }
        }
    }
}

struct Shape { int a, sv, split; bool parts; int64_t grid; };

// A launch holds fewer than 2^32 threads: short chunks of many heads (chunk 1, 2^20 tokens x 64 heads) are more workgroups than that.
constexpr int64_t kMostGroups = 1 << 23;

template <int A, int S, typename T, int SPLIT, bool FUSED, bool PARTS>
hipError_t launch_k(const Params &p, const Shape &k, hipStream_t s)
{
    for (int64_t first = 0; first < k.grid; first += kMostGroups) {
        const dim3 grid((unsigned)std::min(k.grid - first, kMostGroups));
        hipLaunchKernelGGL((generic_kernel<A, S, T, SPLIT, FUSED, PARTS>), grid, dim3(64 * kWaves), 0, s, p, (int)first);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

template <int A, int S, typename T>
hipError_t launch(const Params &p, bool fused, const Shape &k, hipStream_t s)
{
    if (fused) return launch_k<A, S, T, kWaves, true, false>(p, k, s);
    if constexpr (A > 1 && S > 1)
        if (k.parts) return k.split == 1 ? launch_k<A, S, T, 1, false, true>(p, k, s) : launch_k<A, S, T, kWaves, false, true>(p, k, s);
    return k.split == 1 ? launch_k<A, S, T, 1, false, false>(p, k, s) : launch_k<A, S, T, kWaves, false, false>(p, k, s);
}

template <int A, int S>
hipError_t launch_t(const Params &p, bool fused, const Shape &k, hipStream_t s)
{
    if (p.dt_in == DT_F32) return launch<A, S, float>(p, fused, k, s);
    if (p.dt_in == DT_F16) return launch<A, S, _Float16>(p, fused, k, s);
    return launch<A, S, uint16_t>(p, fused, k, s);
}

template <int A>
hipError_t launch_s(const Params &p, bool fused, const Shape &k, hipStream_t s)
{
    switch (k.sv) {
        case 1: return launch_t<A, 1>(p, fused, k, s);
        case 2: return launch_t<A, 2>(p, fused, k, s);
        case 3: return launch_t<A, 3>(p, fused, k, s);
        default: return launch_t<A, 4>(p, fused, k, s);
    }
}

// elements per lane for `size` rows or columns in tiles of at most 16 x cap: as few tiles as possible, evenly filled
int per_lane(int size, int cap)
{
    const int tiles = (size + 16 * cap - 1) / (16 * cap);
    return (size + 16 * tiles - 1) / (16 * tiles);
}

}  // namespace generic

hipError_t launch_generic(const Params &p_in, bool fused, hipStream_t s)
{
    Params p = p_in;
    generic::Shape k{1, 1, generic::kWaves, false, 0};
    int64_t items = 0;
    const int64_t n_cu = p.n_cu > 0 ? p.n_cu : 256;
    if (!fused) {
        const int64_t tiles = (int64_t)p.batch * p.nheads * p.C * ((p.headdim + 63) / 64) * ((p.dstate + 63) / 64);
        const int b_parts = p.dt_in == DT_F32 ? 3 : p.dt_in == DT_F16 ? 2 : 1;
        const cost::GenericWay w = cost::generic_way(p.Q, generic::per_lane(p.headdim, 4), generic::per_lane(p.dstate, 4), b_parts,
                                                     p.dstate, (double)tiles / n_cu);
        k.split = w.quarters ? generic::kWaves : 1;
        k.parts = w.parts;
    }
    // the largest tile (operands loaded once per 16 A x 16 S) that still gives every compute unit four waves; with parts, one wave a
    // tile, the largest there is beyond chunks of 64 (5357 x 8 x 64 x 128, chunk 128, as 64 x 32: 15.0 us, 13.9)
    static const int caps[][2] = {{4, 4}, {4, 2}, {2, 2}};
    for (const auto &cap : caps) {
        k.a = generic::per_lane(p.headdim, cap[0]);
        k.sv = generic::per_lane(p.dstate, cap[1]);
        const int64_t n_pt = (p.headdim + 16 * k.a - 1) / (16 * k.a), n_nt = (p.dstate + 16 * k.sv - 1) / (16 * k.sv);
        items = (int64_t)p.batch * p.nheads * n_pt * n_nt * (fused ? 1 : p.C);
        if (items * k.split >= n_cu * generic::kWaves || (k.parts && k.split == 1 && p.Q > 64)) break;
    }
    if (items <= 0) return hipSuccess;
    if (items > 0x7fffffffLL - 64) return hipErrorInvalidValue;
    p.n_items = (int)items;
    const int64_t groups = k.split == 1 ? (items + generic::kWaves - 1) / generic::kWaves : items;
    k.grid = (groups + 7) / 8 * 8;
    switch (k.a) {
        case 1: return generic::launch_s<1>(p, fused, k, s);
        case 2: return generic::launch_s<2>(p, fused, k, s);
        case 3: return generic::launch_s<3>(p, fused, k, s);
        default: return generic::launch_s<4>(p, fused, k, s);
    }
}

}  // namespace ssd
