// Which fused kernel for which problem: estimated durations of the kernel families, in microseconds.
//
// The families differ in how they spread the work, not in what they compute, so the choice is a matter of time only:
//   four-tile     one workgroup per unit (four state tiles sharing B) walks the whole sequence with the state in its
//                 accumulators: nothing is read back and nothing waits, but a unit is one compute unit's work;
//   token-split   one workgroup per tile, four waves splitting every chunk's tokens: the shortest chunk when tiles
//                 are scarce, four times the B traffic;
//   pair          a chunk-state launch over (unit, run of chunks) that fills every compute unit, then the streaming
//                 recurrence over what it wrote: three more passes over the states;
//   chain         work items of R chunks of a unit drawn from a ticket counter, linked by flags: fills every compute
//                 unit whatever the number of units, pays a start, a read-back per item and a link per item.
// The formulas are fits to one sweep of 36 shapes around the benchmark configurations (batch 1 - 32, 512 - 65 536
// tokens, 24 - 128 heads, dstate 64 / 128, chunk 128 / 256, 1 / 8 groups, with and without packed sequences) on an
// MI355X at steady clocks; every quantity is per compute unit, so another compute-unit count rescales them.  They
// are good to about 10 %, which is enough to rank the families; tests/test_cost_model_cpu.py holds the sweep and a
// second one of 18 other shapes that the fit has not seen, and checks that the family picked is never more than a few
// per cent slower than the best one the dispatcher could have picked.
// The constants (microseconds per unit-chunk, per link, the 5 TB/s of the streaming pair) are this one device's: an
// MI355X with 256 compute units in 8 XCDs of 32 at its steady clocks.  Another compute-unit count rescales them
// linearly and nothing has been measured at any other value; another part needs its own sweep.
#pragma once

#include <stdint.h>

namespace ssd {
namespace cost {

struct Problem {
    int64_t units;      // groups of four state tiles (32 headdim rows x dstate) that share (batch, group)
    int chunks;         // chunks per sequence
    int chunk_size, dstate;
    int n_cu;           // compute units of the device
};

// Time of one unit-chunk relative to dstate 128, chunk 256: the part that shrinks with the tile (arithmetic, x and B
// traffic) and the part that does not (per-chunk bookkeeping, the state's way out).  dstate 64: 0.71 measured, chunk
// 128: 0.75.
inline double work(const Problem &q) { return 0.45 + 0.55 * (q.dstate / 128.0) * (q.chunk_size / 256.0); }

inline int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

// Chain kernel with R chunks per item.  Throughput: a compute unit takes an item after the other, 8 us per unit-chunk
// at R = 4 (more links and read-backs per chunk below that), and the launch ends with its fullest compute unit, whose
// last item nothing overlaps; 15 us of start and drain.  Latency: the items of a unit form a chain whose links
// (flag, read-back, recurrence, store, acknowledge: 3 us) follow one another however many compute units there are.
inline double chain_us(const Problem &q, int R)
{
    const int64_t items_per_unit = ceil_div(q.chunks, R);
    const double per_item = (double)q.chunks / (double)items_per_unit;       // chunks of an average item
    const double items_per_cu = (double)(q.units * items_per_unit) / q.n_cu;
    const double rounds = (double)ceil_div(q.units * items_per_unit, q.n_cu);
    const double t_chunk = (R >= 4 ? 8.0 : R == 2 ? 8.4 : 10.0) * work(q);
    const double throughput = 15.0 + t_chunk * per_item * (items_per_cu > 0.95 * rounds ? items_per_cu : 0.95 * rounds);
    const double latency = 3.0 * (double)items_per_unit + t_chunk * per_item;
    return throughput > latency ? throughput : latency;
}

// The best R of {4, 2, 1} for the chain kernel, and its estimate.
inline int chain_chunks_per_item(const Problem &q, double *us)
{
    int best = 4;
    double t = chain_us(q, 4);
    for (int R = 2; R >= 1; --R) {
        const double c = chain_us(q, R);
        if (c < 0.97 * t) { t = c; best = R; }      // fewer links unless the gain is clear
    }
    if (us) *us = t;
    return best;
}

// Four-tile kernel: a wave walks its tile's chunks one after the other, 4.7 us each on an otherwise idle device and
// 7.1 us when every compute unit has a workgroup; beyond that workgroups share compute units and take turns at
// their instruction issue, and the launch lasts as long as the compute unit with the most of them.
inline double four_tile_us(const Problem &q)
{
    const double k = (double)q.units / q.n_cu;
    const double most = (double)ceil_div(q.units, q.n_cu);
    const double t_chunk = k <= 1.0 ? 4.7 + 2.4 * k : 7.1 * (1.0 + 0.95 * (most - 1.0) + 0.3 * (k - 1.0));
    return 4.0 + q.chunks * t_chunk * work(q);
}

// Token-split kernel: 2.35 us per chunk while every workgroup (one per tile) has a compute unit of its own; with w
// workgroups per compute unit 1.6 times that up to w = 1.5 and a further 1.1 times per workgroup beyond.  (Measured up
// to 32 chunks; longer sequences run about a third slower per chunk, but there this family is not a candidate.)
inline double token_split_us(const Problem &q)
{
    const double w = 4.0 * (double)q.units / q.n_cu;
    const double share = w <= 1.0 ? 1.0 : 1.6 + (w > 1.5 ? 1.1 * (w - 1.5) : 0.0);
    return 3.5 + q.chunks * 2.35 * share * work(q);
}

// Chunk-state launch + recurrence: x read and the chunk states written, then read, and the passed states written
// (read and write share the bandwidth: about 5 TB/s over the lot).
inline double pair_us(const Problem &q)
{
    const double x_bytes = (double)q.units * q.chunks * 256.0 * q.chunk_size;       // 4 tiles x 32 rows x Q x bf16
    const double s_bytes = (double)q.units * q.chunks * 512.0 * q.dstate;           // 4 tiles x 32 rows x N x fp32
    return 6.0 + (x_bytes + 3.0 * s_bytes) / 5.0e6 * (256.0 / q.n_cu);
}

// Few units: the pair, whatever the estimates say (they are fits to 24 and more heads and know the recurrence as a pure
// bandwidth).  The other families then leave most of the chip idle -- a unit's chunks are one serial chain in each of
// them -- where the chunk-state launch spreads over (tile, chunk) and the recurrence costs about 0.2 us a chunk.  dstate
// 128, chunk 256, headdim 64, batch 1, the faster of the others against the pair, us:
//     heads      4 chunks      8             16            32            64            128
//     4          11.3 /  7.8   19.3 /  9.0   43.0 / 11.0   63.9 / 15.1   91.5 / 25.1   142.1 /  39.6
//     16         11.6 /  8.9   19.8 / 11.0   45.2 / 17.0   66.4 / 26.7   90.7 / 34.9   142.1 /  59.9
//     32         12.0 / 10.6   21.5 / 15.8   46.6 / 24.9   65.2 / 31.7   92.1 / 57.2   100.5 / 114.2
//     48         13.0 / 13.1   22.3 / 20.6   46.3 / 28.6   65.2 / 42.7   95.7 / 86.5   154.8 / 174.6
//     80                       24.1 / 24.8   41.3 / 38.4
// (fewer than four chunks: 24 heads x 2, 7.6 / 8.3; no seq_idx).  The lines are drawn inside what was measured: up to a
// tenth as many units as compute units while there are fewer than three unit-chunks per compute unit, and any length below a
// twenty-fourth.  With dstate 64, chunk 128 or batches the pair is ahead inside them too (48 heads x 8 chunks of 128: as
// fast).  They are not where the pair stops paying: beyond them it is no candidate until there are 32 state-tile chunks per
// compute unit (choose in ssd_capi.hip), so that 32 heads x 64 chunks, 48 x 32, 48 x 64 and 24 x 64 (92.7 / 44.7) stay on the
// chain kernel although the table or the estimates have the pair ahead.
inline bool few_units(const Problem &q)
{
    if (q.chunks < 4) return false;
    return q.units * 24 <= q.n_cu || (q.units * 10 <= q.n_cu && q.units * q.chunks < 3 * (int64_t)q.n_cu);
}

// The same against the chain kernel for packed sequences (seq_idx): its chains are then as long as a sequence, and how
// long those are only the device knows, so the pair goes in front only where it does not lose (3 % at most) with four starts in
// every chunk.  The chain kernel's time is then about 35 us for a unit-chunk of work 1 while it runs items of four chunks
// (22 - 24 with shorter items, below 17 chunks of work 1), the pair's grows by 0.14 us a chunk and 0.022 a unit-chunk.  At
// the line, heads x chunks, five sequences / one start a chunk / four, chain kernel against pair, us:
//     dstate, chunk                fp32 out                                   bf16 out
//     128, 256      8 x 48         49.4 / 27.2   36.1 / 27.0   34.2 / 27.0    52.9 / 30.8   37.0 / 30.7   34.7 / 30.8
//                  12 x 48         54.4 / 31.1   36.2 / 30.9   34.6 / 30.8    59.3 / 34.4   36.9 / 34.3   34.7 / 34.3
//                  24 x 32         45.3 / 30.5   37.5 / 30.5   36.0 / 30.5    47.2 / 32.6   38.2 / 32.8   36.4 / 32.8
//                  48 x 17         39.1 / 30.5   37.4 / 30.3   35.3 / 30.0    40.0 / 30.2   37.9 / 30.0   35.9 / 30.1
//                  24 x 16         33.9 / 22.6   25.0 / 22.4   22.4 / 22.5    37.1 / 23.5   25.7 / 23.4   22.7 / 23.3
//     128, 128     24 x 23         35.7 / 24.1   27.6 / 24.5   25.6 / 24.3    38.0 / 27.0   28.3 / 26.8   26.4 / 26.9
//     64, 128      24 x 18         23.3 / 15.5   21.1 / 15.4   20.1 / 15.5    24.2 / 16.6   21.4 / 16.4   20.2 / 16.5
// and beyond it: 8 x 64 64.4 / 32.1, 36.1 / 32.0, 34.1 / 31.9, bf16 72.0 / 37.0, 36.7 / 36.9, 34.4 / 37.0; 12 x 64 bf16 35.4 /
// 40.1 with four starts; 48 x 16 32.5 / 28.9, 26.1 / 29.2, 23.6 / 29.1; 128, 128: 12 x 46 46.4 / 27.8, 27.6 / 27.8, 26.0 / 27.9;
// 16 x 128 98.1 / 63.2, 41.9 / 62.1, 40.6 / 61.8; 4 x 512 in 4, 16 and 64 sequences 260 / 127, 121 / 127 and 69 / 126.
//
// scan: the call with the scan's state half, whose consumer is a launch of its own behind the pair and costs it 0.1 us a
// unit-chunk, against the chain kernel's variant that computes that half (44 us with four starts a chunk).  At its line:
// 24 x 20 55.6 / 35.5, 46.0 / 35.2, 44.0 / 35.1; 20 x 27 59.1 / 43.7, 45.6 / 43.6, 44.1 / 43.4; 12 x 40 74.0 / 38.6, 49.4 / 38.5, 43.9 /
// 38.4; 8 x 57 86.9 / 41.8, 49.5 / 41.9, 43.7 / 41.3; 128, 128: 8 x 41 59.8 / 29.7, 34.1 / 29.7, 30.3 / 29.7; 64, 128: 16 x 19 30.9 /
// 22.0, 25.4 / 22.0, 24.3 / 21.9; beyond it: 24 x 32 59.7 / 49.8, 49.1 / 49.7, 45.0 / 49.5.
inline bool few_units_packed(const Problem &q, bool scan)
{
    if (!few_units(q)) return false;
    const double unit_chunks = (double)(q.units * q.chunks);
    if (scan && q.chunks / 200.0 + unit_chunks / (1.25 * q.n_cu) > work(q)) return false;
    if (chain_chunks_per_item(q, nullptr) < 4) return unit_chunks <= 0.75 * q.n_cu;
    return q.chunks / 95.0 + unit_chunks / (2.3 * q.n_cu) <= work(q);
}

}  // namespace cost
}  // namespace ssd
