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
    int64_t units;      // groups of four state tiles (32 headdim rows x dstate) that share (batch, group); tiles / 4, rounded up
    int64_t quads;      // the same with every group's tiles rounded up to fours: workgroups of the chunk-state launch
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

// The same where a group's tiles are no multiple of four: the chunk-state launch takes 7.1 us a workgroup's chunk (the
// four-tile kernel's time on a full device) also for workgroups that are not full, and is followed by the recurrence.
inline double ragged_pair_us(const Problem &q)
{
    const double x_bytes = (double)q.units * q.chunks * 256.0 * q.chunk_size, s_bytes = (double)q.units * q.chunks * 512.0 * q.dstate;
    const double states = (double)q.quads * q.chunks * 7.1 * work(q) / q.n_cu, bytes = (x_bytes + s_bytes) / 5.0e6 * (256.0 / q.n_cu);
    return 6.0 + (states > bytes ? states : bytes) + 2.0 * s_bytes / 5.0e6 * (256.0 / q.n_cu);
}

// ... against the walk of one workgroup per tile, whose chunks take a third longer in rows of more than 32.  On 110 random shapes
// the pair was ahead wherever its estimate is a tenth lower, by 1.3 to 3.4 times; between that and the other side of the line it
// lost up to a third.  Walk / pair, us (tiles of a group): 4 x 8448 tokens x 30 heads x 32 in 2 groups (15) 97.9 / 58.3;
// 8 x 22528 x 8 x 64 in 8 groups (2) 288 / 216; 2 x 20480 x 40 in 8 groups (10) 259 / 187; on the other side 8 x 31195 x 16 x 32 in 16 groups (1),
// bf16 out, 387 / 390; 8 x 8923 x 28 in 4 groups (14), dstate 64, bf16 out, 122 / 144.
inline bool ragged_pair_ahead(const Problem &q)
{
    return ragged_pair_us(q) < 0.9 * token_split_us(q) * (q.chunks > 32 ? 4.0 / 3.0 : 1.0);
}

// Chunk states: whether workgroups of four tiles, the last of each group partly filled, are ahead of one workgroup per tile.  A wave
// without a tile of its own multiplies all the same, so four fifths of them have to have one, and at dstate 64 with chunks of 128 a
// workgroup's start is too much for what it does.  One per tile / four-tile, us (tiles of a group, dstate, chunk): 7, 128, 256 22.9 / 18.8;
// 13 22.5 / 18.7; 50, 128, 128 116 / 97; 6 23.0 / 23.4; 9 161 / 163; 3 183 / 193; 2 57.7 / 66.7; 1 84 / 104; 7, 64, 256 33.6 / 29.7;
// 9 110 / 122; 7, 64, 128 10.1 / 11.1; 50 20.2 / 23.5; 1 27 / 48.
inline bool quads_filled(int64_t tiles, int dstate, int chunk_size)
{
    if (tiles % 4 == 0) return true;
    return 5 * tiles >= 16 * ceil_div(tiles, 4) && (dstate > 64 || chunk_size > 128);
}

// Row kernel (ssd_rows.hip): workgroups of kr slices of 16 state rows, one per compute unit, each walking its whole sequence.
// Per chunk and relative to dstate 128, chunk 256 (measured 0.61 at chunk 128, 0.75 at dstate 64, 0.45 at both):
inline double rows_us(const Problem &q, int kr)
{
    static const double t_chunk[6] = {0., 1.5, 1.85, 3.0, 3.75, 5.2};
    const double k = q.chunk_size / 256.0, n = q.dstate / 128.0;
    return 5.5 + q.chunks * t_chunk[kr] * (0.08 + 0.42 * k + 0.14 * n + 0.36 * k * n);
}

// Slices per workgroup of the row kernel, 0 where it is no candidate.  slices: 16-row slices of a (batch, group); groups:
// (batch, group) pairs.  There is a workgroup per compute unit at most: a second round of workgroups costs as much as the
// first (8 x 2048 x 48 heads: 66 us, the others 57).  A workgroup reads the same few columns of x to the end, so long rows
// depend on how those columns fall on the memory channels, and a third of the workgroups finish up to a fifth late.  Up to 5120
// tokens the kernel is ahead wherever its estimate is (rows_margin), beyond that only with four slices at dstate 128 or with chunks
// of 128, and there in groups of 16 slices and more: below, too few workgroups share a group's B (12 x 10730).  Inputs from
// memory, the faster of the others against this kernel, us (slices):
//     8 x 2048 x 24 heads       48.4 /  35.9 (3)      4 x 8192 x 64                   143.5 / 132.7 (4)
//     2 x 2048 x 80             49.0 /  34.9 (3)      4 x 8192 x 80                   175.7 / 177.1 (5)   (not taken)
//     1 x 4096 x 80             53.9 /  46.3 (2)      1 x 8192 x 80                    70.9 /  85.9 (2)   (not taken)
//     4 x 4096 x 48             67.4 /  60.0 (4)      8 x 8192 x 24                   117.2 / 123.6 (3)   (not taken)
//     4 x 2048 x 80             56.3 /  48.5 (5)      4 x 8192 x 80, chunk 128        249.2 / 228.5 (5)
//     8 x 2048 x 24, chunk 128  64.9 /  42.7 (3)      4 x 8192 x 80, dstate 64        130.2 / 137.0 (5)   (not taken)
//     8 x 2048 x 24, dstate 64  34.7 /  28.9 (3)      8 x 3729 x 24, 8 groups, dstate 64, chunk 128   75.7 / 54.7 (3)
//     2 x 4608 x 52             53.8 /  47.4 (2)      12 x 10730 x 32 x 32, 8 groups, chunk 128      238.8 / 248.0 (4)   (not taken)
//     1 x 5120 x 64             52.5 /  43.0 (1)      1 x 5120 x 80                    53.1 /  56.2 (2)   (not taken)
inline int rows_slices(const Problem &q, int64_t slices, int64_t groups, int most, double *us)
{
    int best = 0;
    const int64_t tokens = (int64_t)q.chunks * q.chunk_size;
    for (int kr = 1; kr <= most && kr <= slices; ++kr) {
        if (groups * ceil_div(slices, kr) > q.n_cu) continue;
        if (tokens > 5120 && !(slices >= 16 && kr >= 4 && (q.chunk_size == 128 || (kr == 4 && q.dstate == 128)))) continue;
        const double t = rows_us(q, kr);
        if (!best || t < *us) { best = kr; *us = t; }
    }
    return best;
}

// How far below the other families' the row kernel's estimate has to be.  With dstate 64 and few chunks theirs are up to a fifth
// too high, and four and five slices pay their start (other family / row kernel, us: 4 x 512 x 51 heads, chunk 128, 12.8 / 14.1;
// 1338 x 113 x 128 22.6 / 23.6; 3 x 486 x 66, 2 groups, chunk 128, 12.9 / 13.3); two slices of long rows take longer than their
// estimate (1 x 5120 x 80, 0.90 of the chain kernel's, 53.1 / 56.2; 1 x 5120 x 128, 0.84, 66.7 / 55.9).
inline double rows_margin(const Problem &q, int kr)
{
    if (q.dstate == 64) return q.chunks <= 6 && kr >= 4 ? 0.9 : 1.0;
    return kr == 2 && q.chunk_size > 128 && (int64_t)q.chunks * q.chunk_size > 4608 ? 0.88 : 1.0;
}

// Packed sequences (seq_idx) where the chain kernel would have the call: the estimate knows nothing of its chains being cut, so
// with a sequence start in every chunk it is ahead of narrow workgroups, which walk the whole row all the same.  Chain / row
// kernel (slices), us, a start in every chunk:
//     1 x 5120 x 64, fp32 out    37.3 / 44.1 (1)      8 x 4352 x 10, bf16 out         38.7 /  41.9 (2)      (neither taken)
//     2 x 3840 x 28, 2 groups    24.5 / 34.3 (1)      6 x 4608 x 12 x 128             56.2 /  66.3 (3)      (neither taken)
//     12 x 3340 x 12 x 32, dstate 64, chunk 128   27.0 / 30.7 (2)      4 x 4096 x 48     58.1 /  62.7 (3)      (neither taken)
//     6 x 2560 x 28              53.4 / 40.0 (3)      12 x 2329 x 12, 2 groups        41.4 /  39.4 (3)
//     4 x 4608 x 44, chunk 128   91.2 / 86.3 (3)      8 x 4449 x 22, bf16 out         69.0 /  62.0 (3)
//     4 x 8192 x 64             134.2 / 129.6 (4)     12 x 3307 x 16, 2 groups, chunk 128   78.9 / 63.0 (4)
inline bool rows_packed(const Problem &q, int kr, bool out_f32)
{
    return kr >= 4 || (kr == 3 && (q.chunk_size == 128 || !out_f32 || (int64_t)q.chunks * q.chunk_size <= 3072));
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
// long those are only the device knows.  The pair goes in front where it loses next to nothing (a twentieth at most) with a
// sequence start in every second chunk; it is then ahead by up to threefold with a few long sequences a row and loses up to
// a fifth with a start in every chunk.  The chain kernel's time hardly depends on the size there (38 - 42 us for a
// unit-chunk of work 1; beyond 512 unit-chunks 80 us and more with the scan's state half, which runs items of two chunks),
// the pair's grows with the chunks of a row and with all unit-chunks.  Around the lines, two sequences a row / a start in
// every fourth chunk / second / every one, chain kernel against pair, us:
//     dstate, chunk   heads x chunks
//     128, 256, fp32 out      4 x 89        94.5 / 33.7   47.6 / 33.7   39.6 / 33.7   35.9 / 33.8
//                             8 x 110      109.5 / 43.8   46.2 / 43.4   41.3 / 43.6   37.7 / 43.3      (beyond)
//                            16 x 50        73.1 / 34.0   46.6 / 34.0   39.8 / 33.4   38.0 / 33.3
//                            16 x 69        87.5 / 41.2   44.7 / 41.1   40.3 / 41.2   37.8 / 41.1
//                            32 x 47        63.9 / 42.8   46.1 / 43.2   42.2 / 43.1   38.6 / 43.2
//                             4 x 512 in 4, 16 and 64 sequences: 260 / 127, 121 / 127, 69 / 126               (beyond)
//     128, 256, bf16 out      4 x 89       106.6 / 41.0   50.7 / 41.1   41.1 / 41.1   36.7 / 41.1
//                            12 x 63        84.7 / 39.3   48.3 / 39.3   41.3 / 39.2   38.4 / 39.2
//                            20 x 64        81.6 / 45.5   51.3 / 46.9   45.2 / 45.6   39.0 / 45.7      (beyond)
//                            40 x 38        66.0 / 46.4   49.6 / 44.0   43.5 / 44.1   40.8 / 43.4
//     128, 256, scan          4 x 89       135.0 / 43.6   62.5 / 43.4   52.4 / 43.5   47.0 / 43.4
//                            12 x 63       103.5 / 54.7   60.6 / 54.7   51.8 / 54.5   47.6 / 54.2      (beyond)
//                            24 x 35        77.1 / 53.8   60.9 / 53.6   55.6 / 53.2   47.1 / 53.2
//                            48 x 18        63.2 / 52.0   54.8 / 52.1   51.4 / 52.2   46.1 / 51.8
//     128, 128, fp32 out      8 x 59        69.0 / 28.8   36.2 / 28.7   31.3 / 28.3   27.4 / 28.7
//     64, 128, fp32 out      24 x 35        36.5 / 23.7   26.2 / 23.5   24.1 / 23.5   22.9 / 23.8
enum PackedForm { PACKED_OUT_F32, PACKED_OUT_16BIT, PACKED_SCAN };      // scan: no passed states, the scan's state half instead
inline bool few_units_packed(const Problem &q, PackedForm form)
{
    if (!few_units(q)) return false;
    const double chunks = q.chunks, per_cu = (double)(q.units * q.chunks) / q.n_cu;
    if (form == PACKED_OUT_16BIT) return chunks / 100.0 + per_cu / 6.0 <= work(q);
    if (form == PACKED_SCAN && chunks / 260.0 + per_cu / 1.8 > work(q)) return false;       // and the fused part's own
    return chunks / 160.0 + per_cu / 4.6 <= work(q);
}

// The scan's state half without passed states: the chain kernel multiplies each entering state by its chunk's C rows, one launch
// that keeps the states on chip but does everything in one instruction stream per SIMD; with room for the states the fused
// call and the scan's own kernel run one after the other, each on the kernel that suits it.  One launch / two, bf16 y, us:
//     units x chunks (dstate 128, chunk 256)     8 x 1 (64, 128)   23.0 /  11.1        80 x  8    76.7 /  61.0
//                                               40 x 2             37.3 /  18.4       160 x  8   107.3 /  95.7
//                                               20 x 3             38.1 /  18.0        40 x 16    76.9 /  70.4
//                                              192 x 2             42.0 /  37.5        96 x 16   115.9 / 122.0   (not taken)
//                                              320 x 3             90.8 /  81.2        80 x 32   198.2 / 229.0   (not taken)
//                                               40 x 8             52.2 /  40.5       160 x 32   342.7 / 358.8   (not taken)
//     dstate 64:  48 x 16   64.1 / 55.2     chunk 128:  96 x 8   54.8 / 45.3     four sequences a row:  160 x 8   109.3 / 98.8
// and level from there on: 320 x 4 105.7 / 107.3, 960 x 1 82.6 / 78.7 (fp32 y: 85.4 / 87.0; elsewhere two are ahead by a little more
// with it).  The line: up to eight chunks while units or units x chunks stay within what was measured, sixteen up to 48 units; the
// room is then 84 MB at most for dstate 128.
// Packed sequences cut the one launch's chains: where its items of two chunks are one round of workgroups it then takes the
// same time whatever the work, and two launches are ahead only up to one and a half unit-chunks a compute unit (a start in every
// chunk, inputs from memory: 40 x 8 46.4 / 44.2, 192 x 2 42.9 / 39.6, 80 x 5 45.8 / 47.2, 40 x 10 47.7 / 54.0, 72 x 6 44.7 / 50.5,
// 40 x 12 48.5 / 60.0; dstate 64 40 x 10 37.9 / 40.3; two rounds: 160 x 3 55.0 / 46.4, 80 x 8 74.8 / 62.6, 160 x 6 76.7 / 77.7).
inline bool scan_in_two(const Problem &q, bool packed)
{
    if (packed && q.units * ceil_div(q.chunks, 2) <= q.n_cu && 2 * q.units * q.chunks > 3 * (int64_t)q.n_cu) return false;
    if (q.chunks > 8) return q.chunks <= 16 && q.units <= 48;
    return q.units <= 160 || (q.units <= 320 && q.units * q.chunks <= 960);
}

// Chunk states of the sizes and types that the bf16 kernels do not take (ssd_generic.hip): a wave per tile or a quarter of a chunk per
// wave, and whether the operands enter as bf16 parts.  a x sv: elements per lane of the largest tile (of 16 a x 16 sv); b_parts: of an
// element of B (fp32 3, f16 2, bf16 1); tiles: 64 x 64 tiles per compute unit, all chunks counted.
// Without parts: a wave per tile in chunks up to 64 and from 24 tiles on.  Parts are ahead as a wave per tile where tiles are plenty --
// the earlier the larger the tile, which splits fewer operands per product, and the fewer parts B has --, and in quarters where a
// chunk is long or tiles are few.  Lines through 3400 timings (18 tiles, 3 types, chunks of 64 to 256, 1/4 to 40 tiles); fp32
// instructions / a wave per tile / quarters, us (type, headdim x dstate, chunk, tiles):
//     fp16 64 x 64, 64, 4      16.5 / 13.9 / 20.1      bf16 48 x 96, 64, 6       13.6 / 12.8 / 19.1      fp32 64 x 64, 64, 12     28.8 / 30.0 / 51.2
//     fp16 64 x 64, 128, 3     15.6 / 14.4 / 15.5      fp16 64 x 64, 128, 1      10.4 / 12.9 / 9.4       fp32 64 x 128, 128, 4    20.1 / 16.7 / 19.5
//     fp16 48 x 48, 128, 4     16.4 / 16.7 / 17.0      fp16 48 x 48, 128, 8      25.3 / 20.9 / 28.9      fp32 48 x 48, 128, 8     23.3 / 23.3 / 31.9
//     fp32 64 x 128, 256, 2    20.0 / 21.2 / 18.8      fp16 64 x 32, 256, 4      22.2 / 24.3 / 19.4      fp32 64 x 32, 128, 24    56.5 / 59.3 / 84.0
// Of those 3400 calls 10 run more than 3 % longer than with fp32 instructions throughout, by 10 % at most (6 us at 1/4 tile).
struct GenericWay { bool quarters, parts; };

inline GenericWay generic_way(int Q, int a, int sv, int b_parts, int dstate, double tiles)
{
    const int m = a * sv;
    const bool bf16 = b_parts == 1, two_bytes = b_parts < 3, largest = m == 16, longer = Q > 160;
    const GenericWay fp32 = {Q > 64 && tiles < 24, false}, wave = {false, true}, quarters = {true, true};
    // one row or column block splits as many operands as it has products; fp32 splits both in three
    if (a == 1 || sv == 1 || (!two_bytes && sv == 2)) return fp32;
    if (Q <= 64) {
        if (Q < 64) return bf16 && largest && Q >= 32 ? wave : fp32;
        if (bf16) return m != 6 || tiles < 16 ? wave : fp32;
        if (two_bytes) return m >= 8 && (m != 9 || tiles < 16) ? wave : fp32;
        return (largest && tiles >= 3.5 && tiles < 7) || (m == 9 && dstate > 64 && tiles >= 5.5 && tiles < 16) ? wave : fp32;
    }
    if (tiles >= 24) {      // the fp32 instructions go a wave per tile too
        const int shortest = two_bytes && m >= 8 && m != 9 ? 65 : largest ? 100 : two_bytes || m >= 8 ? 128 : 256;
        return Q >= shortest ? wave : fp32;
    }
    double first = 7;
    if (two_bytes) first = m >= 12 ? (longer ? 5 : 2.5) : m >= 8 ? (longer ? 7 : 5) : bf16 && m == 4 && !longer ? 5.5 : 7;
    else if (largest) first = longer ? 5.5 : 3.5;
    else if (m == 12 || (m == 9 && Q <= 128)) first = 5.5;
    if (tiles >= first) return wave;
    if (!two_bytes) return largest && longer && (dstate > 64 || tiles < 2.5) ? quarters : fp32;
    if (longer) return m >= 8 || bf16 ? quarters : fp32;
    if (largest) return tiles >= (bf16 ? 0.75 : 1) ? quarters : fp32;
    // a quarter of one whole step of 32 tokens
    return Q >= 96 && Q <= 128 && tiles >= 1 && (m == 12 || (m == 8 && (bf16 || tiles < 3.5))) ? quarters : fp32;
}

}  // namespace cost
}  // namespace ssd
