// Stand-alone inter-chunk recurrence  s = exp(dA_c) * s + states_c  (exclusive scan written to `out`,
// inclusive last value to `final`).  Pure streaming: each lane owns VEC consecutive state elements of one
// (batch, head) and walks the chunks serially; the loads of states_c do not depend on the running state,
// so several chunks are kept in flight per lane to cover HBM latency.  Batch 4 x 80 heads x 32 chunks: 126 us for 703 MB.
//
// Reference semantics: kernels/ssd_state_passing.py:27-84.
#include "ssd_params.h"

namespace ssd {

typedef __attribute__((ext_vector_type(4))) float f32x4;

template <int VEC> struct Vals { float v[VEC]; };

template <int VEC>
__device__ __forceinline__ Vals<VEC> load_vals(const void *base, int64_t off, int dt)
{
    Vals<VEC> r;
    if (VEC == 4 && dt == DT_F32) {
        f32x4 q = *(const f32x4 *)((const float *)base + off);
        r.v[0] = q.x; r.v[1] = q.y; r.v[2] = q.z; r.v[3] = q.w;
    } else {
#pragma unroll
        for (int j = 0; j < VEC; ++j) r.v[j] = load_as_f32(base, off + j, dt);
    }
    return r;
}

template <int VEC>
__device__ __forceinline__ void store_vals(void *base, int64_t off, int dt, const Vals<VEC> &r)
{
    if (VEC == 4 && dt == DT_F32) {
        f32x4 q = {r.v[0], r.v[1], r.v[2], r.v[3]};
        *(f32x4 *)((float *)base + off) = q;
    } else {
#pragma unroll
        for (int j = 0; j < VEC; ++j) store_from_f32(base, off + j, dt, r.v[j]);
    }
}

// D = chunks in flight per lane.  The decays (and the sequence comparison) of 64 chunks are computed at once, one chunk
// per lane, and read back lane by lane: as scalar loads of their own they would have to be waited for one chunk after
// the other (scalar loads return out of order, so every wait for one drains those ahead of it).
template <int VEC, int D>
__global__ void __launch_bounds__(256) state_passing_kernel(const PassParams p)
{
    const int d0 = (blockIdx.x * blockDim.x + threadIdx.x) * VEC;
    const int h = blockIdx.y, b = blockIdx.z;
    const int lane = threadIdx.x & 63;
    const bool in = d0 < p.dim;
    // lanes past the end stay (the others read their decays): they repeat the last elements and store nothing
    const int e0 = in ? d0 : p.dim - VEC;
    const int64_t st_base = b * p.sst_b + h * p.sst_h + e0;
    const int64_t out_base = b * p.so_b + h * p.so_h + e0;
    const float *da = p.da + b * p.sda_b + h * p.sda_h;
    const int32_t *sq = p.seq ? p.seq + b * p.ssq_b : nullptr;

    Vals<VEC> s;
    if (p.init) s = load_vals<VEC>(p.init, b * p.sin_b + h * p.sin_h + e0, p.dt_init);
    else {
#pragma unroll
        for (int j = 0; j < VEC; ++j) s.v[j] = 0.f;
    }
    // `out` may be the buffer `states` lives in (slot c holds the chunk state of chunk c and receives the state that
    // enters chunk c): a lane only ever touches its own elements, reads slot c before it writes it, and memory
    // operations of one lane on one address keep their program order -- hence the first loads before the first store.
    // (Loads past the last chunk repeat it and are not used; lanes past the end read what others write and drop it.)
    auto last_id = [&](int c) { return sq[(int64_t)(min((c + 1) * p.Q, p.seqlen) - 1) * p.ssq_l]; };
    struct Decay { float da; int32_t id, before; };
    auto load_decay = [&](int c0) {
        const int c = min(c0 + lane, p.C - 1);
        Decay d{da[c * p.sda_c], 0, 0};
        if (sq) {
            d.id = last_id(c);
            d.before = c > 0 ? last_id(c - 1) : 0;
        }
        return d;
    };
    Decay ahead = load_decay(0);
    Vals<VEC> nxt[D];
    auto request = [&](int i, int c) { nxt[i] = load_vals<VEC>(p.states, st_base + (int64_t)min(c, p.C - 1) * p.sst_c, p.dt_states); };
#pragma unroll
    for (int i = 0; i < D; ++i) request(i, i);
    if (in) store_vals<VEC>(p.out, out_base, p.dt_out, s);
    static_assert(64 % D == 0, "a group of chunks has its decays in one window");
    for (int w0 = 0; w0 < p.C; w0 += 64) {
        const float scale = ahead.id == ahead.before ? __expf(ahead.da) : 0.f;
        ahead = load_decay(w0 + 64);
        auto step = [&](int i, int c) {
            const Vals<VEC> cur = nxt[i];
            const float sc = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, scale), c - w0));
            request(i, c + D);
#pragma unroll
            for (int j = 0; j < VEC; ++j) s.v[j] = sc * s.v[j] + cur.v[j];
        };
        const int c1 = min(w0 + 64, p.C - 1);      // chunks of this window that have one behind them
        int c0 = w0;
        for (; c0 + D <= c1; c0 += D) {
#pragma unroll
            for (int i = 0; i < D; ++i) {
                step(i, c0 + i);
                if (in) store_vals<VEC>(p.out, out_base + (int64_t)(c0 + i + 1) * p.so_c, p.dt_out, s);
            }
        }
        if (c1 == w0 + 64) continue;
        // the last chunks, up to D of them
#pragma unroll
        for (int i = 0; i < D; ++i) {
            const int c = c0 + i;
            if (c > c1) break;
            step(i, c);
            if (!in) continue;
            if (c < p.C - 1) store_vals<VEC>(p.out, out_base + (int64_t)(c + 1) * p.so_c, p.dt_out, s);
            else store_vals<VEC>(p.fin, b * p.sf_b + h * p.sf_h + e0, DT_F32, s);
        }
        break;
    }
}

hipError_t launch_state_passing(const PassParams &p, hipStream_t s)
{
    if (p.batch <= 0 || p.nheads <= 0 || p.dim <= 0 || p.C <= 0) return hipSuccess;
    auto al = [](const void *q, size_t a) { return q == nullptr || ((uintptr_t)q % a) == 0; };
    const bool vec = p.dim % 4 == 0 && al(p.states, 16) && al(p.out, 16) && al(p.fin, 16) && al(p.init, 16) &&
                     (p.sst_b | p.sst_c | p.sst_h | p.so_b | p.so_c | p.so_h | p.sf_b | p.sf_h | p.sin_b | p.sin_h) % 4 == 0;
    // One wave per workgroup, so that small launches spread over all compute units (256 lanes each: b=1 x 32768 tokens x 80
    // heads 131 against 121 us).
    auto launch = [&](auto kernel, int v, int lanes) {
        dim3 grid((p.dim + v * lanes - 1) / (v * lanes), p.nheads, p.batch), block(lanes);
        hipLaunchKernelGGL(kernel, grid, block, 0, s, p);
    };
    if (vec) {
        // Four chunks in flight per lane cover the latency of memory from a thousand waves on (4 / 8 / 16 in flight: 80
        // heads x 128 chunks, 2560 waves: 121 / 125 / 132 us).  With fewer waves and a long chain more of them do (16 heads x
        // 512 chunks, 512 waves: 156 / 128 / 108); with few chunks the requests past the last one only cost time (2 x 24
        // heads x 8 chunks: 5.9 / 6.3 / 9.8).
        const int64_t waves = ((int64_t)p.dim / 4 + 63) / 64 * p.nheads * p.batch;
        const int deep = waves >= 1024 ? 4 : p.C >= 64 ? 16 : p.C >= 16 ? 8 : 4;
        if (deep == 16) launch(state_passing_kernel<4, 16>, 4, 64);
        else if (deep == 8) launch(state_passing_kernel<4, 8>, 4, 64);
        else launch(state_passing_kernel<4, 4>, 4, 64);
    } else {
        launch(state_passing_kernel<1, 4>, 1, 256);
    }
    return hipGetLastError();
}

}  // namespace ssd
