// SSD chunk-state contraction (optionally with the recurrence) on the fp32 matrix instructions, for whatever the bf16
// kernels do not take: fp32 and fp16 inputs, any headdim, dstate, chunk size and alignment.  The weighted x and B enter
// v_mfma_f32_16x16x4_f32 as fp32 values and every sum is fp32, so fp32 inputs keep fp32 accuracy.
//
// Where its time goes: the fp32 matrix instructions (256 flop per clock and compute unit, a sixteenth of bf16's) are the
// largest part -- fp32, batch 2 x 2048 tokens x 24 heads x 64 x 128: 1.6 GFLOP, 10 us, and 41 MB, 8 us; 21 us measured (an
// FMA kernel that staged both operands through LDS: 92 us); fp16, batch 8 x 3001 x 48 heads: 18.9 GFLOP in 187 us.  The
// matrix units are busy 56 % of that fp32 launch; a wave waits 64 % of its clocks to issue, with three of them on a SIMD, and
// 19 % in s_waitcnt, and the rest of the launch is where the waves of a SIMD start, or add up and store, together.  So the
// operands must cost next to no issue slots: a lane loads A consecutive headdim elements of one token's x row and S
// consecutive dstate elements of its B row with one load each, and that *is* the operand layout -- lane i of a 16-lane group
// stands for rows A i .. A i + A-1 and columns S i .. S i + S-1 of the tile, the four lane groups for four consecutive tokens,
// and matrix instruction (r, s) multiplies the r-th element of every x vector with the s-th of every B vector.  No LDS on the
// way in, no barrier in the loop, whole rows per load; the accumulators of one lane are S consecutive columns, so rows leave
// as vectors as well.
//
// One workgroup owns a (16 A) x (16 S) tile of one (batch, head) and chunk; its SPLIT = 4 waves take a quarter of the
// chunk's tokens each and add up through LDS, after which wave v holds accumulator q = v of every instruction.  In
// fused mode it walks the chunks with the state in registers.  Short chunks leave a quarter too little to do between
// a wave's start and the adding up: there a wave owns a tile by itself (SPLIT = 1).  Rows and columns past the edge of an
// odd headdim or dstate are not loaded: the last lanes' vectors move up to end at the edge and repeat rows that their
// neighbours also compute.  Both store them, the same bits: a sum's order does not depend on the wave or lane that forms it.
//
// Reference semantics: kernels/ssd_chunk_state.py:97-173, kernels/ssd_state_passing.py:27-84.
#include "ssd_tile.h"

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
constexpr int kWindow = 64;      // tokens whose weights a wave computes at once, one per lane
// matrix steps of four tokens whose rows are loaded together, a group ahead of their use: a group's matrix instructions
// (32 clocks each) have to last for a load's way from memory
constexpr int group_of(int tiles) { return tiles >= 12 ? 4 : 2; }

template <int A, int S, typename T, int SPLIT, bool FUSED>
__global__ void __launch_bounds__(64 * kWaves, FUSED ? 2 : 3) generic_kernel(const Params p)
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
    int item = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
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

struct Shape { int a, sv, split; int64_t grid; };

template <int A, int S, typename T>
hipError_t launch(const Params &p, bool fused, const Shape &k, hipStream_t s)
{
    const dim3 grid((unsigned)k.grid), block(64 * kWaves);
    if (fused) hipLaunchKernelGGL((generic_kernel<A, S, T, kWaves, true>), grid, block, 0, s, p);
    else if (k.split == 1) hipLaunchKernelGGL((generic_kernel<A, S, T, 1, false>), grid, block, 0, s, p);
    else hipLaunchKernelGGL((generic_kernel<A, S, T, kWaves, false>), grid, block, 0, s, p);
    return hipGetLastError();
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
    generic::Shape k{1, 1, generic::kWaves, 0};
    int64_t items = 0;
    const int64_t n_cu = p.n_cu > 0 ? p.n_cu : 256;
    // One wave per tile where a quarter of a chunk is too little (chunk 64, batch 2 x 1900 tokens x 15 heads x 48 x 96:
    // 13.5 against 16.6 us; chunk 100: 16.9 against 14.1) and where 64 x 64 tiles alone give every SIMD six waves (fp16,
    // batch 8 x 3001 x 48 heads x 64 x 128: chunk 256 187 against 198 us, chunk 128 203 against 247; half of it, four and a
    // half waves: 105 against 101).
    const int64_t big_tiles = (int64_t)p.batch * p.nheads * p.C * ((p.headdim + 63) / 64) * ((p.dstate + 63) / 64);
    if (!fused && (p.Q <= 64 || big_tiles >= 24 * n_cu)) k.split = 1;
    // the largest tile (operands loaded once per 16 A x 16 S) that still gives every compute unit four waves
    static const int caps[][2] = {{4, 4}, {4, 2}, {2, 2}};
    for (const auto &cap : caps) {
        k.a = generic::per_lane(p.headdim, cap[0]);
        k.sv = generic::per_lane(p.dstate, cap[1]);
        const int64_t n_pt = (p.headdim + 16 * k.a - 1) / (16 * k.a), n_nt = (p.dstate + 16 * k.sv - 1) / (16 * k.sv);
        items = (int64_t)p.batch * p.nheads * n_pt * n_nt * (fused ? 1 : p.C);
        if (items * k.split >= n_cu * generic::kWaves) break;
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
