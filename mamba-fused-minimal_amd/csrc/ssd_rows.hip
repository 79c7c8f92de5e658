// Row kernel: a workgroup owns KR slices of 16 state rows (headdim rows of one or several heads that share a (batch,
// group) and therefore B) times all dstate columns, and walks the sequence with the running state in its accumulators
// (gfx950).
//
// Loading waves and multiplying waves.  Some waves fetch and prepare, four waves multiply and store; they meet once per
// round of four 32-token steps, in a double buffer of LDS.
//   * One wave turns dt and dA_cumsum into the weights of a round, a round ahead of their use.
//   * A wave that loads x takes one or two slices of every round: it requests their rows into registers several rounds ahead,
//     forms x * w in fp32 and its split into bf16 hi + bf16 lo (two products keep about 16 mantissa bits of x * w).  A lane
//     holds eight tokens of eight (or four) rows, so that packing two tokens of a row into one register is also the
//     transposition the matrix instructions want.
//   * A wave that loads B takes one step (dstate 64: two) of every round and turns 8 x 8 elements per lane.
//   * A multiplying wave owns a quarter of the dstate columns of every slice; both operands lie in LDS as it needs them, 16
//     bytes a lane.  D[p][n] accumulates in registers.  At a chunk boundary it stores the accumulators as the state entering
//     the chunk and multiplies them by exp(dA_chunk).
// Every x element is scaled and split once per workgroup and every B element is read once from LDS, whatever the number
// of slices, so the rows per workgroup can follow the number of compute units: the launcher takes the KR that leaves the
// compute units evenly loaded.  No workgroup waits for another one and no state is read back.
//
// Measured (inputs from memory, before / with this kernel): 8 x 2048 x 24 heads 48.4 / 35.3 us, 2048 x 80 heads 29.0 / 26.2,
// 8 x 2048 x 24 in chunks of 128 64.9 / 42.7.  What bounds it: the rows of x that a workgroup reads are narrow (160 bytes of a
// 10 KB token row with five slices), and it reads the same columns to the end: 4.0 - 4.6 TB/s of the 5.5 that wider, moving
// requests reach (the loads alone 84 us of 177 at 4 x 8192 x 80), and a workgroup on a busy memory channel finishes last.  No unit of a
// compute unit is full: at 8 x 2048 x 24 (three slices) the matrix unit is busy a fifth of the launch, vector instructions issue for a
// third, LDS instructions for a sixth, and the waves spend 43 % of their time in waits (hardware counters).  With two slices a
// workgroup loads 64 KB of B for 16 KB of x: at 2048 x 80, on the 160 compute units that have one, the same shares are a fifth, a third, a sixth and 45 %.
//
// Reference semantics: kernels/ssd_chunk_state.py:97-173, kernels/ssd_state_passing.py:27-84,
// kernels/fused_globalbar.py:16-198 (same math, one launch).
#include "ssd_tile.h"

#include <algorithm>

namespace ssd {
namespace rows {

using namespace tile;

constexpr int kRound = 4;           // steps per round
constexpr int kStepTokens = 32, kRoundTokens = kRound * kStepTokens;

// LDS: two buffers of kRound slots.  A slot holds the operands of a step as blocks of 1 KB -- 16 rows or columns times 32
// tokens, the eight tokens of lane group kg at place i at 256 kg + 16 i --: hi of every slice, lo of every slice, B.  Inside a
// quarter of a block the places are XORed (x_swizzle, b_swizzle), which keeps the 16 lanes that write together on different
// banks.
// Which tokens of a round meet in a step is free, as long as x and B agree: group kg of step j takes the tokens
// 16 t + 4 j + kg, t = 0 .. 7, so that load t of a wave covers consecutive token rows.
template <int KR, int NT> constexpr int slot_bytes() { return (2 * KR + NT) * 1024; }
// Rows a lane of an x wave holds, the lanes that hold a token's rows, and the waves that take the 16 token groups.  The rows
// of a token lie side by side in the lanes of one wave: where the slices' heads do in memory, a load touches each line once.
template <int KR> constexpr int rows_per_lane() { return KR <= 3 ? 4 : 8; }
template <int KR> constexpr int token_lanes() { return 16 * KR / rows_per_lane<KR>(); }
template <int KR> constexpr int x_waves() { return (16 + 64 / token_lanes<KR>() - 1) / (64 / token_lanes<KR>()); }
template <int NT> constexpr int b_waves() { return NT == 8 ? 4 : 2; }
template <int KR, int NT> constexpr int n_threads() { return 64 * (4 + x_waves<KR>() + b_waves<NT>() + 1); }
// behind the slots: the weights of two rounds, one row of kRoundTokens per slice in the order of the groups; the slices' chunk decays of four rounds
template <int KR, int NT> constexpr int weights_at() { return 2 * kRound * slot_bytes<KR, NT>(); }
template <int KR, int NT> constexpr int decays_at() { return weights_at<KR, NT>() + 2 * KR * kRoundTokens * 4; }
template <int KR, int NT> constexpr int lds_bytes() { return decays_at<KR, NT>() + 4 * 8 * 4; }
template <int KR> __device__ __forceinline__ int x_swizzle(int slice, int kg) { return (slice + KR * kg) & (rows_per_lane<KR>() - 1); }
template <int NT> __device__ __forceinline__ int b_swizzle(int quarter, int kg)
{
    return NT == 8 ? (quarter & 1) | ((quarter >> 1) << 3) : (quarter << 2) | (kg & 1);
}

template <int CTRL, int BANKS>
__device__ __forceinline__ float dpp_from(float old, float src)
{
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, old), __builtin_bit_cast(int, src),
                                                                 CTRL, 0xf, BANKS, false));
#else
    return old + src;
#endif
}

// Meeting point of the eight waves: this wave's LDS operations are done (vector-memory operations stay in flight).
__device__ __forceinline__ void meet() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

struct RowParams {
    Params p;
    int slices;           // 16-row slices of a (batch, group)
    int wg_per_group;     // workgroups of a (batch, group)
    int n_wg;             // batch * groups * wg_per_group
};

// F32: the passed states are stored in fp32, else in the 16-bit type that the parameters say
template <int KR, int NT, bool F32>
__global__ void __launch_bounds__((n_threads<KR, NT>()), ((n_threads<KR, NT>() + 255) / 256)) rows_kernel(const RowParams rp)
{
    constexpr int NB = NT / 4;                 // column blocks of a multiplying wave
    constexpr int kSlot = slot_bytes<KR, NT>();
    extern __shared__ __attribute__((aligned(16))) char lds[];
    const Params &p = rp.p;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);

    // consecutive workgroups of a (batch, group) sit on one XCD: they read the same B rows and neighbouring x rows
    const int per_xcd = (rp.n_wg + p.n_xcd - 1) / p.n_xcd;
    const int vwg = (int)(blockIdx.x % p.n_xcd) * per_xcd + (int)(blockIdx.x / p.n_xcd);
    if ((int)(blockIdx.x / p.n_xcd) >= per_xcd || vwg >= rp.n_wg) return;
    const int bg = vwg / rp.wg_per_group;
    const int slice0 = (vwg % rp.wg_per_group) * KR;
    const int b = bg / p.ngroups, g = bg % p.ngroups;
    const int heads = p.nheads / p.ngroups;
    const int n_sl = min(KR, rp.slices - slice0);                  // slices that exist
    const int rpc = p.Q / kRoundTokens;                  // rounds per chunk
    const int n_rounds = p.C * rpc;

    constexpr int kNowhere = (int)0x80000000u;                     // beyond every descriptor: the load returns zeros

    // A loading wave: rounds 0 .. n_rounds - 1 in order, the requests of kDepth rounds in flight.  (One way into the loop and
    // one out of it: a second one, as the compiler lays it out, would make the waits for the loads of a round count those of
    // the rounds behind it too.)
    auto pipeline = [&](auto depth, auto &loads, auto &&request, auto &&prepare) {
        constexpr int D = decltype(depth)::value;
        static_for<D>([&](auto kc) {
            request(loads[decltype(kc)::value]);
            __builtin_amdgcn_sched_barrier(0);
        });
        int r = 0;
        for (; r + D <= n_rounds; r += D)
            static_for<D>([&](auto kc) {
                constexpr int k = decltype(kc)::value;
                prepare(r + k, loads[k]);
                __builtin_amdgcn_sched_barrier(0);
                request(loads[k]);
                __builtin_amdgcn_sched_barrier(0);
                meet();
                __builtin_amdgcn_sched_barrier(0);      // (nothing of the next round, whose loads may be on their way, in front)
            });
        static_for<D - 1>([&](auto kc) {
            constexpr int k = decltype(kc)::value;
            if (r + k < n_rounds) {
                prepare(r + k, loads[k]);
                meet();
            }
        });
    };

    if (wave == 4 + x_waves<KR>() + b_waves<NT>()) {
        // ---- weights: lane = tokens lane and lane + 64 (= 16 t + group) of a round, for every slice ---------------------------------------
        int dtoff[KR], csoff[KR], lastoff[KR];
#pragma unroll
        for (int k = 0; k < KR; ++k) {
            const int hd = (slice0 + min(k, n_sl - 1)) * 16 / p.headdim;
            dtoff[k] = 4 * (hd * (int)p.sdt_h + lane * (int)p.sdt_k);
            csoff[k] = 4 * (hd * (int)p.sda_h + lane * (int)p.sda_k);
            lastoff[k] = 4 * (hd * (int)p.sda_h + (p.Q - 1) * (int)p.sda_k);
        }
        struct Loads {
            uint32_t dt[KR][2], cs[KR][2], last[KR];
            int id[2], id_last, id_prev;
        };
        const __amdgpu_buffer_rsrc_t rs_seq = make_rsrc(p.seq ? p.seq + b * p.ssq_b : nullptr, p.seq ? 0x7fffffffLL : 0);
        const int sq = 4 * (int)p.ssq_l;
        int t0 = 0, in_chunk = 0, first = 0;          // the next request's first token; the same in its chunk; of its chunk
        const char *dtb = (const char *)(p.dt + b * p.sdt_b + (int64_t)g * heads * p.sdt_h);
        const char *dab = (const char *)(p.dacs + b * p.sda_b + (int64_t)g * heads * p.sda_h);
        auto request = [&](Loads &d) {
            const bool any = first < p.seqlen;                   // past the last chunk: nothing (empty descriptors)
            const __amdgpu_buffer_rsrc_t rd = make_rsrc(dtb, any ? 0x7fffffffLL : 0), ra = make_rsrc(dab, any ? 0x7fffffffLL : 0);
#pragma unroll
            for (int k = 0; k < KR; ++k) {
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    d.dt[k][u] = __builtin_amdgcn_raw_buffer_load_b32(rd, dtoff[k], 4 * (in_chunk + 64 * u) * (int)p.sdt_k, 0);
                    d.cs[k][u] = __builtin_amdgcn_raw_buffer_load_b32(ra, csoff[k], 4 * (in_chunk + 64 * u) * (int)p.sda_k, 0);
                }
                d.last[k] = __builtin_amdgcn_raw_buffer_load_b32(ra, lastoff[k], 0, 0);
            }
#pragma unroll
            for (int u = 0; u < 2; ++u)
                d.id[u] = __builtin_amdgcn_raw_buffer_load_b32(rs_seq, min(t0 + lane + 64 * u, p.seqlen - 1) * sq, 0, 0);
            d.id_last = __builtin_amdgcn_raw_buffer_load_b32(rs_seq, 0, (min(first + p.Q, p.seqlen) - 1) * sq, 0);
            d.id_prev = __builtin_amdgcn_raw_buffer_load_b32(rs_seq, first > 0 ? 0 : kNowhere, first > 0 ? (min(first, p.seqlen) - 1) * sq : 0, 0);
            t0 += kRoundTokens;
            in_chunk += kRoundTokens;
            const bool next = in_chunk >= p.Q;
            in_chunk -= next ? p.Q : 0;
            first += next ? p.Q : 0;
            dtb += next ? 4 * p.sdt_c : 0;
            dab += next ? 4 * p.sda_c : 0;
        };
        const bool clamp = p.clamp;
        int left_use = p.seqlen;
        auto prepare = [&](int r, const Loads &d) {
            float *wtab = (float *)(lds + weights_at<KR, NT>()) + (r & 1) * KR * kRoundTokens + 8 * (lane & 15) + (lane >> 4);
            float *dtab = (float *)(lds + decays_at<KR, NT>()) + (r & 3) * 8;
#pragma unroll
            for (int k = 0; k < KR; ++k) {
                const float last = __builtin_bit_cast(float, d.last[k]);
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    const float e = last - __builtin_bit_cast(float, d.cs[k][u]);
                    const float wk = __expf(clamp ? fminf(e, 0.f) : e) * __builtin_bit_cast(float, d.dt[k][u]);
                    wtab[k * kRoundTokens + 4 * u] = ((lane + 64 * u < left_use) & (d.id[u] == d.id_last)) ? wk : 0.f;
                }
                const float dec = __expf(last);
                dtab[k] = d.id_last == d.id_prev ? dec : 0.f;      // (all lanes, the same value)
            }
            left_use -= kRoundTokens;
        };
        constexpr int D = KR >= 4 ? 3 : 4;
        Loads loads[D];
        pipeline(std::integral_constant<int, D>{}, loads, request, prepare);
        meet();
        return;
    }
    meet();               // the weights of round 0
    if (wave >= 4 + x_waves<KR>()) {
        // ---- B: a lane takes 8 tokens x 8 columns (16 bytes a load) ------------------------------------------------------
        constexpr int kCg = 2 * NT, kSteps = kRound / b_waves<NT>();       // column groups of eight; steps of a wave
        const int j = (wave - 4 - x_waves<KR>()) * kSteps + lane / (4 * kCg);      // step
        const int cg = lane % kCg, kg = (lane / kCg) & 3;
        const int Brb = (int)(2 * p.sB_l);
        const int boff = (4 * j + kg) * Brb + 16 * cg;
        // Columns of a multiplying wave's quarter in the places of its blocks: neighbouring columns in neighbouring registers
        // or lanes eight apart, see store_states.  Two blocks: place i < 8 of block t is column 4 i + t, i >= 8 column
        // 4 (i - 8) + 2 + t; one block: place 4 q + e is column 4 e + q.
        int at[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int quarter = NB == 2 ? cg >> 2 : cg >> 1;
            const int place = NB == 2 ? 8 * ((e >> 1) & 1) + 2 * (cg & 3) + (e >> 2) : 4 * (e & 3) + 2 * (cg & 1) + (e >> 2);
            const int block = NB == 2 ? 2 * quarter + (e & 1) : quarter;
            at[e] = j * kSlot + (2 * KR + block) * 1024 + 256 * kg + 16 * (place ^ b_swizzle<NT>(quarter, kg));
        }
        struct Loads { u32x4 v[8]; };
        int t0 = 0;                                    // the next request's first token
        const char *base = (const char *)p.B + 2 * ((int64_t)b * p.sB_b + (int64_t)g * p.sB_g);
        auto request = [&](Loads &d) {
            const int left = min(p.seqlen - t0, kRoundTokens);
            const __amdgpu_buffer_rsrc_t rs = make_rsrc(left > 0 ? base : (const char *)p.B, left > 0 ? left * Brb : 0);
#pragma unroll
            for (int t = 0; t < 8; ++t) d.v[t] = __builtin_amdgcn_raw_buffer_load_b128(rs, boff, 16 * t * Brb, 0);
            t0 += kRoundTokens;
            base += (int64_t)kRoundTokens * Brb;
        };
        auto prepare = [&](int r, const Loads &d) {
            char *slots = lds + (r & 1) * kRound * kSlot;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                u32x4 v;
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    v[q] = __builtin_amdgcn_perm(d.v[2 * q + 1][e >> 1], d.v[2 * q][e >> 1], (e & 1) ? 0x07060302 : 0x05040100);
                *(u32x4 *)(slots + at[e]) = v;
            }
        };
        constexpr int D = 3;
        Loads loads[D];
        pipeline(std::integral_constant<int, D>{}, loads, request, prepare);
        return;
    }
    if (wave >= 4) {
        // ---- x, weights: a lane takes 8 tokens x RPL rows of a slice ------------------------------------------------------
        constexpr int RPL = rows_per_lane<KR>(), kLanes = token_lanes<KR>(), kGroups = (16 + x_waves<KR>() - 1) / x_waves<KR>();
        typedef __attribute__((ext_vector_type(RPL / 2))) uint32_t Piece;
        const int group = (wave - 4) * kGroups + lane / kLanes;       // the lane's tokens of a round: 16 t + group
        const bool exists = lane < kGroups * kLanes && group < 16;
        const int slice = lane % kLanes / (16 / RPL), piece = lane % (16 / RPL), j = (group & 15) >> 2, kg = group & 3;
        const int xrb = (int)(2 * p.sx_l);
        const int row = (slice0 + min(slice, n_sl - 1)) * 16;
        const int xoff = exists && slice < n_sl ? group * xrb + 2 * ((row / p.headdim) * (int)p.sx_h + row % p.headdim) + 2 * RPL * piece : kNowhere;
        const int wrow = slice * kRoundTokens + 8 * (group & 15);
        int at[RPL];
#pragma unroll
        for (int e = 0; e < RPL; ++e)
            at[e] = j * kSlot + slice * 1024 + 256 * kg + 16 * ((RPL * piece + e) ^ x_swizzle<KR>(slice, kg));
        struct Loads { Piece x[8]; };
        int t0 = 0;                                    // the next request's first token
        const char *base = (const char *)p.x + 2 * ((int64_t)b * p.sx_b + (int64_t)g * heads * p.sx_h);
        auto request = [&](Loads &d) {
            const int left = min(p.seqlen - t0, kRoundTokens);
            const __amdgpu_buffer_rsrc_t rx = make_rsrc(left > 0 ? base : (const char *)p.x, left > 0 ? left * xrb : 0);
#pragma unroll
            for (int t = 0; t < 8; ++t) {
                if constexpr (RPL == 8) d.x[t] = __builtin_amdgcn_raw_buffer_load_b128(rx, xoff, 16 * t * xrb, 0);
                else d.x[t] = __builtin_amdgcn_raw_buffer_load_b64(rx, xoff, 16 * t * xrb, 0);
            }
            t0 += kRoundTokens;
            base += (int64_t)kRoundTokens * xrb;
        };
        auto prepare = [&](int r, const Loads &d) {
            char *slots = lds + (r & 1) * kRound * kSlot;
            const float *wtab = (const float *)(lds + weights_at<KR, NT>()) + (r & 1) * KR * kRoundTokens + wrow;
            const f32x4 wlo = *(const f32x4 *)wtab, whi = *(const f32x4 *)(wtab + 4);
            const float w[8] = {wlo.x, wlo.y, wlo.z, wlo.w, whi.x, whi.y, whi.z, whi.w};
#pragma unroll
            for (int e = 0; e < RPL; ++e) {
                u32x4 hi, lo;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const uint32_t a = d.x[2 * q][e >> 1], c = d.x[2 * q + 1][e >> 1];
                    const float x0 = __builtin_bit_cast(float, (e & 1) ? a & 0xffff0000u : a << 16);
                    const float x1 = __builtin_bit_cast(float, (e & 1) ? c & 0xffff0000u : c << 16);
                    uint32_t hp = pack_bf16(x0 * w[2 * q], x1 * w[2 * q + 1]);
                    asm volatile("" : "+v"(hp));      // keeps the compiler from converting the products a second time
                    hi[q] = hp;
                    lo[q] = pack_bf16(__builtin_fmaf(x0, w[2 * q], -__builtin_bit_cast(float, hp << 16)),
                                      __builtin_fmaf(x1, w[2 * q + 1], -__builtin_bit_cast(float, hp & 0xffff0000u)));
                }
                if (exists) {
                    *(u32x4 *)(slots + at[e]) = hi;
                    *(u32x4 *)(slots + KR * 1024 + at[e]) = lo;
                }
            }
        };
        constexpr int D = RPL == 8 ? 3 : 4;
        Loads loads[D];
        pipeline(std::integral_constant<int, D>{}, loads, request, prepare);
        return;
    }

    // ---- multiplying wave ------------------------------------------------------------------------------------
    const int i16 = lane & 15, kg = lane >> 4;
    f32x4 acc[KR][NB];
    int s_head[KR], s_p0[KR];
#pragma unroll
    for (int s = 0; s < KR; ++s) {
        const int row = (slice0 + min(s, n_sl - 1)) * 16;
        s_head[s] = row / p.headdim;
        s_p0[s] = row % p.headdim;
    }
    // acc[s][t][r]: row 4 kg + r of slice s; column of block t at lane i16 as the loading waves deal them.  Without initial
    // states the descriptor is empty and the loads return zeros.
    {
        const int es = p.dt_init == DT_F32 ? 4 : 2;
        const int64_t first = (int64_t)b * p.sin_b + (int64_t)g * heads * p.sin_h;
        const __amdgpu_buffer_rsrc_t ri = make_rsrc((const char *)p.init + first * es, p.init ? 0x7fffffffLL : 0);
        const int voff = 4 * kg * (int)p.sin_p + (NB == 2 ? 32 * wave + 4 * (i16 & 7) + 2 * (i16 >> 3) : 16 * wave + 4 * (i16 & 3) + (i16 >> 2));
        auto fill = [&](auto load) {
#pragma unroll
            for (int s = 0; s < KR; ++s) {
                const int soff = s_head[s] * (int)p.sin_h + s_p0[s] * (int)p.sin_p;
#pragma unroll
                for (int t = 0; t < NB; ++t)
#pragma unroll
                    for (int r = 0; r < 4; ++r) acc[s][t][r] = load(voff, soff + r * (int)p.sin_p + t);
            }
        };
        if (p.dt_init == DT_F32)
            fill([&](int v, int so) { return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(ri, 4 * v, 4 * so, 0)); });
        else if (p.dt_init == DT_BF16)
            fill([&](int v, int so) { return bf16_bits_to_f32(__builtin_amdgcn_raw_buffer_load_b16(ri, 2 * v, 2 * so, 0)); });
        else
            fill([&](int v, int so) { return (float)__builtin_bit_cast(_Float16, (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(ri, 2 * v, 2 * so, 0)); });
    }
    // After the exchange among the 16 lanes of a row group a lane holds four neighbouring columns of one row: with two
    // blocks the lanes < 8 take row 4 kg + 2 u and the others row 4 kg + 2 u + 1 (u = 0, 1), eight lanes writing 128
    // consecutive bytes; with one block lane 4 q + e takes row 4 kg + q, four lanes writing 64.
    const int st_row = NB == 2 ? 4 * kg + (i16 >> 3) : 4 * kg + (i16 >> 2);
    const int st_col = NB == 2 ? 32 * wave + 4 * (i16 & 7) : 16 * wave + 4 * (i16 & 3);
    constexpr int kPieces = KR * NB;
    auto piece = [&](auto pc) {
        constexpr int s = decltype(pc)::value / NB, u = decltype(pc)::value % NB;
        f32x4 v;
        if constexpr (NB == 2) {
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const float a = acc[s][t][2 * u], c = acc[s][t][2 * u + 1];
                v[t] = dpp_from<0x128, 0xc>(a, c);            // row_ror:8 into lanes 8..15
                v[2 + t] = dpp_from<0x128, 0x3>(c, a);        // ... into lanes 0..7
            }
        } else {
            float lo[2], hi[2];
#pragma unroll
            for (int r = 0; r < 2; ++r) {
                lo[r] = dpp_from<0x128, 0xc>(acc[s][0][r], acc[s][0][r + 2]);
                hi[r] = dpp_from<0x128, 0x3>(acc[s][0][r + 2], acc[s][0][r]);
            }
            v[0] = dpp_from<0x124, 0xa>(lo[0], lo[1]);            // row_ror:4: from lane - 4
            v[1] = dpp_from<0x12c, 0x5>(lo[1], lo[0]);            // row_ror:12: from lane + 4
            v[2] = dpp_from<0x124, 0xa>(hi[0], hi[1]);
            v[3] = dpp_from<0x12c, 0x5>(hi[1], hi[0]);
        }
        return v;
    };
    // piece pc of a (batch, group, chunk)'s states behind rs; slices that do not exist go nowhere
    auto put = [&](auto pc, auto f32, __amdgpu_buffer_rsrc_t rs, f32x4 v, int s_h, int s_p, bool bf16) {
        constexpr int s = decltype(pc)::value / NB, u = decltype(pc)::value % NB, es = decltype(f32)::value ? 4 : 2;
        const int soff = es * (s_head[s] * s_h + s_p0[s] * s_p);
        const int voff = s < n_sl ? es * ((st_row + 2 * u) * s_p + st_col) : kNowhere;
        if constexpr (decltype(f32)::value) {
            const u32x4 q = __builtin_bit_cast(u32x4, v);
            __builtin_amdgcn_raw_buffer_store_b128(q, rs, voff, soff, 0);
            asm volatile("s_nop 3" ::"v"(q) : "memory");
        } else {
            typedef __attribute__((ext_vector_type(2))) _Float16 h2;
            const h2 a = {(_Float16)v.x, (_Float16)v.y}, c = {(_Float16)v.z, (_Float16)v.w};
            const u32x2 q = {bf16 ? pack_bf16(v.x, v.y) : __builtin_bit_cast(uint32_t, a),
                             bf16 ? pack_bf16(v.z, v.w) : __builtin_bit_cast(uint32_t, c)};
            __builtin_amdgcn_raw_buffer_store_b64(q, rs, voff, soff, 0);
            asm volatile("s_nop 3" ::"v"(q) : "memory");
        }
    };
    char *const out_base = (char *)p.out + ((int64_t)b * p.so_b + (int64_t)g * heads * p.so_h) * (F32 ? 4 : 2);
    typedef std::integral_constant<bool, F32> OutF32;
    // operand blocks: 16 bytes a lane; the swizzle depends on the slice or on the wave's quarter
    int aoff[KR];
#pragma unroll
    for (int s = 0; s < KR; ++s) aoff[s] = s * 1024 + 256 * kg + 16 * (i16 ^ x_swizzle<KR>(s, kg));
    const int boff = (2 * KR + NB * wave) * 1024 + 256 * kg + 16 * (i16 ^ b_swizzle<NT>(wave, kg));
    // One round.  FIRST: of a chunk; the states entering it leave in the shadow of the matrix instructions, a piece every few
    // units (stored in one go they keep a wave from multiplying for 2300 of the 8800 clocks of a chunk of five slices: a
    // compute unit's stores take about 50 clocks per KB).
    auto round_of = [&](auto firstc, int r, int c) {
        constexpr bool FIRST = decltype(firstc)::value;
        const char *round = lds + (r & 1) * kRound * kSlot;
        // Operands travel kAhead units (a slice of a step: two reads, 2 NB matrix instructions) ahead of their use.
        constexpr int kUnits = kRound * KR, kAhead = 2;
        bf16x8 hi[kAhead + 1], lo[kAhead + 1], Bop[kAhead + 1][NB];      // (one slice: a unit is a step)
        auto fetch = [&](auto uc) {
            constexpr int u = decltype(uc)::value, st = u / KR, s = u % KR;
            const char *slot = round + st * kSlot;
            if constexpr (s == 0)
#pragma unroll
                for (int t = 0; t < NB; ++t) Bop[st % (kAhead + 1)][t] = *(const bf16x8 *)(slot + boff + 1024 * t);
            hi[u % (kAhead + 1)] = *(const bf16x8 *)(slot + aoff[s]);
            lo[u % (kAhead + 1)] = *(const bf16x8 *)(slot + KR * 1024 + aoff[s]);
        };
        f32x4 out[FIRST ? kPieces : 1];
        const __amdgpu_buffer_rsrc_t rs = make_rsrc(out_base + c * p.so_c * (F32 ? 4 : 2), 0x7fffffffLL);
        if constexpr (FIRST) {
            float dec[KR];
#pragma unroll
            for (int s = 0; s < KR; ++s) dec[s] = ((const float *)(lds + decays_at<KR, NT>()))[(r & 3) * 8 + s];
            static_for<kAhead>([&](auto uc) { fetch(uc); });
            static_for<kPieces>([&](auto pc) { out[decltype(pc)::value] = piece(pc); });
#pragma unroll
            for (int s = 0; s < KR; ++s)
#pragma unroll
                for (int t = 0; t < NB; ++t) acc[s][t] *= dec[s];
        } else {
            static_for<kAhead>([&](auto uc) { fetch(uc); });
        }
        static_for<kUnits>([&](auto uc) {
            constexpr int u = decltype(uc)::value, st = u / KR, s = u % KR;
            if constexpr (u + kAhead < kUnits) fetch(std::integral_constant<int, u + kAhead>{});
#pragma unroll
            for (int t = 0; t < NB; ++t)
                acc[s][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(hi[u % (kAhead + 1)], Bop[st % (kAhead + 1)][t], acc[s][t], 0, 0, 0);
#pragma unroll
            for (int t = 0; t < NB; ++t)
                acc[s][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(lo[u % (kAhead + 1)], Bop[st % (kAhead + 1)][t], acc[s][t], 0, 0, 0);
            if constexpr (FIRST && u % (4 / NB) == 0)            // kUnits / kPieces = 4 / NB
                put(std::integral_constant<int, u / (4 / NB)>{}, OutF32{}, rs, out[u / (4 / NB)], (int)p.so_h, (int)p.so_p, p.dt_out == DT_BF16);
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    int r = 0;
    for (int c = 0; c < p.C; ++c) {
        meet();
        round_of(std::true_type{}, r, c);
        ++r;
        for (int k = 1; k < rpc; ++k, ++r) {
            meet();
            round_of(std::false_type{}, r, c);
        }
    }
    const __amdgpu_buffer_rsrc_t rs = make_rsrc(p.fin + (int64_t)b * p.sf_b + (int64_t)g * heads * p.sf_h, 0x7fffffffLL);
    static_for<kPieces>([&](auto pc) { put(pc, std::true_type{}, rs, piece(pc), (int)p.sf_h, (int)p.sf_p, false); });
}

static bool aligned(const void *ptr, size_t a) { return ((uintptr_t)ptr % a) == 0; }

// a state tensor whose 16-byte (fp32) or 8-byte (16-bit) pieces are aligned and whose (batch, group, chunk) part is below 2 GiB
static bool states_ok(const void *ptr, int dt, int64_t strides_or, int64_t s_h, int64_t s_p, const Params &p)
{
    return aligned(ptr, dt == DT_F32 ? 16 : 8) && strides_or % 4 == 0 && s_h >= 0 && s_p >= 0 &&
           4 * ((p.nheads / p.ngroups) * s_h + p.headdim * s_p) < (1LL << 31);
}

static bool inputs_ok(const Params &p)
{
    if (p.dt_in != DT_BF16 || p.headdim % 16 || (p.dstate != 64 && p.dstate != 128) || p.Q % kRoundTokens) return false;
    if (!aligned(p.x, 16) || (p.sx_b | p.sx_l | p.sx_h) % 8 || !aligned(p.B, 16) || (p.sB_b | p.sB_l | p.sB_g) % 8) return false;
    // byte offsets within a step, chunk or row of sequence ids are 32 bits
    const int64_t heads = p.nheads / p.ngroups, lim = 1LL << 31;
    // (a token's heads lie within its pitch: what is past the last token is past the descriptor)
    if (p.sx_h < 0 || (heads - 1) * p.sx_h + p.headdim > p.sx_l || 2 * kRoundTokens * p.sx_l >= lim) return false;
    if (p.sB_l < p.dstate || 2 * kRoundTokens * p.sB_l >= lim) return false;
    if (p.sdt_h < 0 || p.sdt_k < 0 || 4 * (heads * p.sdt_h + p.Q * p.sdt_k) >= lim) return false;
    if (p.sda_h < 0 || p.sda_k < 0 || 4 * (heads * p.sda_h + p.Q * p.sda_k) >= lim) return false;
    if (p.seq && (p.ssq_l < 0 || 4 * p.seqlen * p.ssq_l >= lim)) return false;
    return true;
}

}  // namespace rows

bool rows_supported(const Params &p)
{
    using namespace rows;
    if (p.states || !p.out || !p.fin || !inputs_ok(p)) return false;
    if (!states_ok(p.out, p.dt_out, p.so_b | p.so_c | p.so_h | p.so_p, p.so_h, p.so_p, p)) return false;
    if (!states_ok(p.fin, DT_F32, p.sf_b | p.sf_h | p.sf_p, p.sf_h, p.sf_p, p)) return false;
    if (p.init && (p.sin_h < 0 || p.sin_p < 0 || 4 * ((p.nheads / p.ngroups) * p.sin_h + p.headdim * p.sin_p + p.dstate) >= (1LL << 31))) return false;
    return true;
}

template <int KR, int NT, bool F32>
static hipError_t launch_rows_k(const rows::RowParams &rp, dim3 grid, hipStream_t s)
{
    constexpr int lds = rows::lds_bytes<KR, NT>();
    static_assert(lds <= 160 * 1024, "LDS of a compute unit");
    static std::atomic<uint64_t> configured{0};
    const hipError_t e = ensure_dynamic_lds((const void *)rows::rows_kernel<KR, NT, F32>, lds, configured);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((rows::rows_kernel<KR, NT, F32>), grid, dim3(rows::n_threads<KR, NT>()), lds, s, rp);
    return hipGetLastError();
}

template <int KR>
static hipError_t launch_rows_r(const rows::RowParams &rp, dim3 grid, bool f32, hipStream_t s)
{
    if (rp.p.dstate == 128) return f32 ? launch_rows_k<KR, 8, true>(rp, grid, s) : launch_rows_k<KR, 8, false>(rp, grid, s);
    return f32 ? launch_rows_k<KR, 4, true>(rp, grid, s) : launch_rows_k<KR, 4, false>(rp, grid, s);
}

// kr: slices of 16 rows per workgroup, 1 .. kMaxRowSlices
hipError_t launch_rows(const Params &p_in, int kr, hipStream_t s)
{
    rows::RowParams rp;
    rp.p = p_in;
    Params &p = rp.p;
    rp.slices = (p.nheads / p.ngroups) * (p.headdim / 16);
    rp.wg_per_group = (rp.slices + kr - 1) / kr;
    rp.n_wg = p.batch * p.ngroups * rp.wg_per_group;
    if (rp.n_wg <= 0 || p.C <= 0) return hipSuccess;
    if (p.n_cu <= 0) p.n_cu = 256;
    p.n_xcd = p.n_cu >= 32 ? p.n_cu / 32 : 1;       // an XCD is 32 compute units on this part
    const dim3 grid((rp.n_wg + p.n_xcd - 1) / p.n_xcd * p.n_xcd);
    const bool f32 = p.dt_out == DT_F32;
    switch (kr) {
        case 1: return launch_rows_r<1>(rp, grid, f32, s);
        case 2: return launch_rows_r<2>(rp, grid, f32, s);
        case 3: return launch_rows_r<3>(rp, grid, f32, s);
        case 4: return launch_rows_r<4>(rp, grid, f32, s);
        case 5: return launch_rows_r<5>(rp, grid, f32, s);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace ssd
