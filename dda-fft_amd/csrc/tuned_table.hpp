// Launch schedule per (lattice, right-hand sides): written by
// dda-fft_amd/tune.py from measurements on an MI355X.  x_rb: right-hand
// sides per X-pass tile; x_blocks: X-pass launch size up to which groups of
// right-hand sides are spread over blocks (1 << 30: each group its own
// block); graph: iterations replayed as captured HIP graphs; fuse: z- and
// y-forward transforms of an i-plane in one kernel (always, whatever stands
// here, where the plane has at most 2^11 cells).
#pragma once

namespace ddafft {

struct TunedEntry {
    int ni, nj, nl, nrhs, x_rb, x_blocks, graph, fuse;
};

// realizations in flight in ddafft_solve_batch for the batched Monte-Carlo
// workload (the call's width argument 0 stands for it)
constexpr int kTunedBatchWidth = 12;

constexpr TunedEntry kTuned[] = {
    {32, 32, 32, 2, 1, 2048, 0, 1},   // X pass 11.7 us, solve 0.695 ms
    {64, 64, 64, 2, 2, 1 << 30, 0, 0},   // X pass 41.4 us, solve 2.225 ms
    {128, 128, 128, 2, 2, 1 << 30, 1, 0},   // X pass 371.4 us, solve 7.908 ms
    {256, 256, 256, 2, 2, 1 << 30, 1, 0},   // X pass 3262.3 us, solve 66.691 ms
    {32, 32, 32, 16, 2, 1 << 30, 0, 1},   // X pass 33.5 us, solve 1.817 ms
    {32, 32, 64, 16, 2, 1 << 30, 0, 1},   // X pass 59.6 us, solve 2.978 ms
    {64, 64, 64, 16, 2, 1 << 30, 1, 1},   // X pass 292.8 us, solve 14.756 ms
    {32, 32, 64, 2, 2, 1 << 30, 0, 1},   // X pass 15.7 us, solve 0.934 ms
    {64, 64, 64, 4, 2, 1 << 30, 0, 0},   // X pass 83.7 us, solve 4.115 ms
    {128, 128, 128, 4, 2, 1 << 30, 0, 0},   // X pass 692.1 us, solve 15.295 ms
};

}  // namespace ddafft
