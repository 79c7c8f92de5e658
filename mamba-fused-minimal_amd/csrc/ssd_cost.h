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
// long those are only the device knows, so the pair goes in front only where it does not lose with a sequence start in
// every chunk.  The chain kernel's time is then that of its busiest compute unit's items, the pair's grows with the
// chunks of a row and with all unit-chunks, so the two lines scale with the work of a unit-chunk.  At the lines, one start
// / four starts a chunk, chain kernel against pair, us:
//     dstate, chunk   heads x chunks   fp32 out                     bf16 out                     call with the scan's state half
//     128, 256         4 x 64          35.2 / 25.4   33.7 / 25.6    36.3 / 30.7   34.5 / 30.8    46.9 / 33.8   42.4 / 33.9
//                      8 x 57          37.7 / 30.9   34.0 / 30.8    38.7 / 34.1   34.3 / 34.0    49.4 / 42.5   43.6 / 41.9
//                     20 x 23          36.3 / 25.4   34.3 / 25.4    36.9 / 26.0   34.7 / 26.0    46.4 / 36.2   44.0 / 35.8
//     128, 128         8 x 41          26.4 / 22.5   24.6 / 22.5    27.2 / 25.4   25.5 / 25.4    34.0 / 32.4   30.4 / 32.5
//     64, 128          8 x 33          21.0 / 15.1   19.6 / 15.1    21.6 / 17.8   19.8 / 17.8    26.4 / 23.5   24.1 / 23.6
// and beyond them: 8 x 64 34.1 / 32.7 (four starts), bf16 34.4 / 37.3; 16 x 128 in 64 sequences 46.0 / 64.2; 4 x 512 in 4, 16
// and 64 sequences 260 / 127, 121 / 127 and 69 / 126.
inline bool few_units_packed(const Problem &q)
{
    return few_units(q) && q.units * 24 <= q.n_cu && q.chunks <= 64 * work(q) && (double)(q.units * q.chunks) <= 0.9 * work(q) * q.n_cu;
}

}  // namespace cost
}  // namespace ssd
