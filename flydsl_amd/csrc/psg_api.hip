// C ABI of libpsgemm.so: argument validation, regime selection and launch on the caller's stream.
// Nothing here allocates, synchronises or touches any stream but the caller's.
#include "../../include/psgemm.h"

#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <mutex>

#include "psg_common.h"
#include "moe_gating.h"
#include "moe_rows.h"
#include "tile_order.h"

hipError_t psg_launch_a8w8_tiled(const A8W8Params& p, int kind, int store, int tile_m, int tile_n, hipStream_t stream);
hipError_t psg_launch_a8w8_stream(const A8W8Params& p, int kind, int store, hipStream_t stream);
hipError_t psg_launch_moe_reads_once(const int32_t* expert_ids, int blocks, int used, int per_tile, int experts, int cached, int32_t* out, hipStream_t stream);
hipError_t psg_launch_moe_gemm(const MoeParams& p, const MoeRowsParams& rows, int kind, int stage, int block_m, int blocks, hipStream_t stream);
hipError_t psg_launch_moe_mx_gemm(const MoeMxParams& p, const MoeRowsParams& rows, int a_format, int stage, int block_m, int blocks, hipStream_t stream);
hipError_t psg_launch_moe_mx_scale_sort(const void* scale, const int32_t* sorted_ids, const int32_t* num_valid, void* out, int tokens, int topk, int cols,
                                        int sorted_size, hipStream_t stream);
hipError_t psg_launch_moe_sort(const MoeSortParams& p, void* workspace, uint64_t workspace_bytes, hipStream_t stream);
uint64_t psg_moe_sort_workspace(int64_t pairs, int experts);
int psg_moe_sort_max_experts();
hipError_t psg_launch_moe_gating(MoeGatingParams p, int dtype, hipStream_t stream);
hipError_t psg_launch_moe_gate_sort(const MoeSortParams& p, MoeGatingParams g, int dtype, hipStream_t stream);
hipError_t psg_launch_moe_gate_then_sort(const MoeSortParams& p, MoeGatingParams g, int dtype, void* workspace, uint64_t workspace_bytes, hipStream_t stream);
bool psg_moe_gate_sort_fuses(int tokens, int topk, int experts);
hipError_t psg_launch_moe_reduce(const void* x, void* y, int tokens, int topk, int dim, int out_dtype, const int32_t* mask,
                                 const int32_t* ids, int experts, hipStream_t stream);
hipError_t psg_launch_mx_generic(const MxGenParams& p, int af, int bf, int store, int batch, hipStream_t stream);
hipError_t psg_launch_tiled_mxw4(const A8W8Params& p, bool fp6, int tile_m, int tile_n, hipStream_t stream);
hipError_t psg_launch_mx_smallm(const MxGenParams& p, int af, int bf, int batch, hipStream_t stream);
hipError_t psg_launch_mxfp4_smallm(const MxParams& p, int store, int nw, hipStream_t stream);
hipError_t psg_launch_splitk_finalize(const A8W8Params& p, const void* partial, int is_int, int scaled, hipStream_t stream);
hipError_t psg_launch_tile_order(int tiles_m, int tiles_n, int group_m, int32_t* out, hipStream_t stream);
hipError_t psg_launch_quant_pertoken(const void* x, int x_dtype, void* y, float* scale, int M, int K, int out_fp8, hipStream_t stream);
hipError_t psg_launch_quant_mxfp4(const void* x, int x_dtype, void* packed, void* scales, int M, int R, int K, int shuffled,
                                  hipStream_t stream);

// Scratch of the entry point that allocates nothing (psg_gemm_a8w8_static): the split-K partial sums of the tiled
// path live here instead of in a caller-supplied workspace.  Every GPU the library runs on holds its own copy of the
// array at its own address until the process ends.  In host code the name below is only a stand-in for the symbol:
// the device address is looked up once per device with hipGetSymbolAddress and that pointer is what kernels get.
#define PSG_STATIC_SCRATCH_BYTES (32u << 20)
static __device__ __align__(256) unsigned char scratch[PSG_STATIC_SCRATCH_BYTES];

// Compute units of the current device, read once (the planners deal workgroups out per CU).  Without a device (host-only use of
// the planning entry points) the MI355X's 256.
int psg_cu_count() {
    static const int n = [] {
        int dev = 0, cus = 0;
        if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus < 1) {
            (void)hipGetLastError();
            cus = 256;
        }
        return cus;
    }();
    return n;
}

namespace {

thread_local char g_err[512] = "";

constexpr int kMaxDevices = 64;
void* g_scratch_ptr[kMaxDevices] = {};  // device address of `scratch` on each device, filled on first use
std::mutex g_scratch_mu;

int fail(int code, const char* fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof(g_err), fmt, ap);
    va_end(ap);
    return code;
}

int hip_fail(hipError_t e, const char* what) {
    snprintf(g_err, sizeof(g_err), "%s: %s", what, hipGetErrorString(e));
    return (int)e;
}

bool aligned(const void* p, uintptr_t a) { return (reinterpret_cast<uintptr_t>(p) & (a - 1)) == 0; }

constexpr int kSmallM = 32;      // rows the split-K path covers
constexpr int kStreamMaxM = 64;  // rows the small-M kernels can hold (four 16-row blocks)

// Which regime an fp4 x fp4 problem takes: the small-M kernel up to 32 rows; up to 64 rows while the weight is at most 40 MB, K at least
// 2048 and its workgroups of 32 columns come one to a CU (measured, us small-M / tiled plan: M=33 7168x2048 4.9 / 6.5, 8192x8192 10.9 / 14.6,
// 1024x2048 4.3 / 5.3, 4096x1024 4.8 / 4.1; M=64 5.9 / 6.7, 13.2 / 15.8, 5.4 / 5.3, 5.8 / 4.2).  With more columns a few CUs work a second round
// while the others wait, and 32x128 tiles, two or three to a CU, take over at once: M=33 8960x8704 16.7 / 13.5, 12288x4096 9.4 / 8.0,
// 16384x2048 6.5 / 5.8, 24576x2048 8.2 / 7.8; M=64 8224x2048 7.1 / 5.2, 16384x2048 8.3 / 6.2, 20480x4096 17.2 / 10.7, with the weights in the last-level cache.  From
// memory the tiles are 9 % faster from 49 rows on, level from 40, and 8 to 16 % slower below that, where from the cache they are as much faster (34x15552x3840
// 10.5 / 12.7; 10.0 / 8.8, 44 to 48 rows 1.0 to 1.05; 0.80 to 0.82, 62x9920x4608 13.9 / 12.0; 13.9 / 9.0).  Up to 32 rows the two are
// too close to draw a line by (32x10240x4096 8.7 / 8.0, 17x8224x4096 7.0 / 7.8, 32x16384x14336 25.8 / 33.1).
bool mx_small_holds(int M, int N, int K) { return M > kSmallM && M <= kStreamMaxM && K >= 2048 && (long)N * (K / 2) <= (40L << 20); }
bool mx_takes_small(int M, int N, int K) { return M <= kSmallM || (mx_small_holds(M, N, K) && N <= 32 * psg_cu_count()); }

// Which regime an 8- / 16-bit problem takes when the caller does not force one.  Up to 32 rows always the streaming
// kernel.  Above that every workgroup of the streaming kernel still reads all of A (M x K bytes through its texture
// path), so it only wins while the weight is small enough that the split-K pair of the tiled kernel is bound by its
// two launches and its partial sums rather than by bandwidth (measured, fp8, us streaming / tiled+split-K: M=33 1024x2048
// 4.3 / 8.0, 6144x4096 9.2 / 14.1, 8192x8192 15.3 / 19.6, 2048x16384 15.5 / 16.0; M=48 9.7 / 14.4, 16.5 / 20.4, 17.3 / 16.3; M=64
// 1024x2048 5.5 / 8.2, 6144x4096 11.3 / 15.0, 8192x8192 18.3 / 22.2, 5120x8192 15.8 / 19.0, 2048x16384 20.0 / 15.6), and while 32
// columns for each CU are all there are.  With more columns the CUs go round again, and 64x64 tiles, several to a CU and without a split,
// are better from the first column on (us streaming / 64x64 tiles, weights in the last-level cache: fp8 33x8208x1024 8.6 / 5.0, 33x9216x8064 23.2 / 20.5, 64x8208x4096
// 16.0 / 11.7, 48x10240x6144 20.6 / 16.5, 33x16384x4096 17.3 / 13.7, 64x28672x2048 23.8 / 12.6, 33x65536x1024 35.6 / 13.7; fp16
// 33x16384x2048 17.4 / 14.4, 40x12288x3328 23.4 / 18.5; just below the line 60x8192x4096 10.7 / 14).  With the weights in memory too, at 102 of 120 drawn
// problems by more than 5 % (fp8 44x40512x1024 24.1 / 12.1, 51x13744x4032 20.4 / 20.1); at ten, rows of 5 KB and more just past the line, the streaming
// kernel is up to 15 % faster there and as much slower from the cache (int8 36x9472x6080 21.5 / 24.4; 20.7 / 18.4, fp8 42x8512x5888 20.0 / 22.8; 18.8 / 17.2).
// Beyond 64 rows a workgroup takes 64 of them, and the kernel is the better one while 32 columns a workgroup make one round of the CUs (N
// times the 64-row groups up to 8192) on rows of 2 to 4 KB (us streaming / tiled plan: fp8 80x1024x4096 6.6 / 9.5, 256x1024x4096 7.2 /
// 10.1, 128x2048x2048 4.8 / 7.3, 128x4096x4096 9.9 / 11.9, 192x2048x2048 7.2 / 7.4; bf16 256x1024x1024 4.8 / 6.8, 128x2048x2048 7.4 /
// 10.4; but fp8 128x4096x1024 6.2 / 5.5, 192x4096x4096, one and a half rounds, 19.2 / 11.9).  On rows of 4 to 8 KB it is while they fill half of
// the CUs (fp8 65x1024x4224 7.1 / 9.1, 80x2048x8128 11.4 / 13.7, 128x2048x6144 9.2 / 12.9, 256x1024x8128 12.2 / 15.7; int8 256x1024x4224 7.9 /
// 11.0; bf16 66x2048x2112 7.0 / 9.8; fp16 128x2048x4032 11.2 / 14.1); between a half and one round it depends on the columns (256x2048x5120 11.0 /
// 12.7, but 192x2048x4160 11.8 / 11.4, 128x4096x7168 14.2 / 13.6, 192x2720x6144 15.1 / 13.9) and the tiles stay.  On rows of 8 KB and more they are the better
// ones from the first (165x1056x8576 15.0 / 15.2, 65x1968x10880 17.2 / 14.9, 163x2128x9216 19.8 / 16.6, 89x320x10752 14.7 / 11.9).  With fewer than 1024 columns, 32
// workgroups of the streaming kernel, rows of 4 to 8 KB go either way too (fp8 202x368x5440 10.4 / 11.5, int8 221x336x4864 9.7 / 11.0, but fp8 93x368x8128 12.7 /
// 10.7, bf16 109x880x3456 11.9 / 11.3), and the tiles stay; on 2 to 4 KB it is better with any number of columns (86x288x2688 6.4 / 10.8).
bool stream_holds(int M, int N, int kbytes) {
    const long w = (long)N * kbytes, a = (long)M * kbytes;
    return M > kSmallM && M <= kStreamMaxM && a <= (512L << 10) && w <= (80L << 20);
}
bool takes_stream(int M, int N, int kbytes) {
    if (M <= kSmallM) return true;
    if (M > kStreamMaxM) {
        const long columns = (long)N * ((M + 63) / 64);
        const long round = 32L * psg_cu_count();
        return M <= 256 && (kbytes >= 2048 && kbytes <= 4096 ? columns <= round : kbytes > 4096 && kbytes < 8192 && N >= 1024 && columns <= round / 2);
    }
    return stream_holds(M, N, kbytes) && N <= 32 * psg_cu_count();
}
constexpr int kTargetWaves = 1536;  // wavefronts wanted in flight for the streaming path (6 per CU)

int pick_ksplit(int units, int steps) {
    int ks = 1;
    while (ks < 8 && units * ks < kTargetWaves && ks * 2 <= steps) ks *= 2;
    return ks;
}

struct Tile {
    int m, n;
    int waves;  // wavefronts per workgroup: 4 (side by side along N, or 2x2) or 8 (side by side along N)
};

// Tile by score: what the split rules below start from (the MX table's 256x256 stands for two of the 128x256 tiles that fp4 runs), and the tile of an fp8 x fp8 problem unless an estimate is better (other problems whose K isn't split take
// the smallest estimate).  Each shape has a measured relative efficiency at full occupancy; the score multiplies it by how evenly the tiles fill the CUs'
// workgroup slots and by the fraction of each tile that is not padding.
Tile pick_tile(int M, int N, bool mx, int hint_m, int hint_n) {
    struct Shape {
        int m, n, waves, per_cu;
        double eff;
    };
    static const Shape shapes8[] = {{256, 256, 8, 1, 1.17}, {128, 256, 4, 2, 1.00}, {64, 256, 4, 2, 0.62}, {32, 256, 4, 3, 0.36},
                                    {128, 128, 4, 2, 0.70}, {64, 64, 4, 5, 0.25}};
    static const Shape shapesx[] = {{256, 256, 8, 1, 1.00}, {128, 256, 4, 1, 0.80}, {64, 256, 4, 2, 0.75}, {32, 256, 4, 3, 0.40},
                                    {64, 128, 4, 3, 0.60}, {32, 128, 4, 4, 0.34}};
    const Shape* shapes = mx ? shapesx : shapes8;
    if (hint_m > 0 && hint_n > 0) return {hint_m, hint_n, 4};  // forced by the caller; the launcher rejects unknown shapes
    double best = -1.0;
    Tile t = {shapes[0].m, shapes[0].n, shapes[0].waves};
    for (int i = 0; i < 6; i++) {
        const int tm = shapes[i].m, tn = shapes[i].n;
        const long tiles_m = (M + tm - 1) / tm, tiles_n = (N + tn - 1) / tn;
        const long tiles = tiles_m * tiles_n;
        const long cus = psg_cu_count();
        const long slots = cus * shapes[i].per_cu;
        const long rounds = (tiles + slots - 1) / slots;
        // a partly filled last round still costs a full tile time on the CUs it touches
        const double fill = (double)tiles / (double)(rounds * slots);
        // between one workgroup per CU and a full set of slots the CUs that hold one more than the others finish last (scored
        // for the MX kinds, whose 64x128 and 64x256 tiles meet that case: 1024x5120x5120 24.7 us with 640 tiles of 64x128
        // against 27.7 with 320 of 64x256; the 8- and 16-bit kinds have the rule behind the loop instead)
        const double between = (double)tiles / (double)(((tiles + cus - 1) / cus) * cus);
        const double busy = tiles >= slots ? fill : (tiles <= cus ? (double)tiles / (double)cus : (mx ? between : 1.0));
        const double pad = ((double)M / (double)(tiles_m * tm)) * ((double)N / (double)(tiles_n * tn));
        const double score = busy * pad * shapes[i].eff;
        if (score > best) {
            best = score;
            t = {tm, tn, shapes[i].waves};
        }
    }
    // The score counts workgroup slots, two per CU for 128x256, so between one and two such tiles per CU it sees one round where
    // the CUs that hold two take twice as long.  When the 256x256 tiles of the same problem make one round that fills more
    // than half of the CUs, they are faster (fp8, us 256x256 / 128x256: 5120x2048x8320 86 / 96; 1536x8192x8192 89 / 103;
    // 2048x5120x5120 60 / 71; 3072x4096x4096 52 / 56; with only half of the CUs filled they are not: 2048x4096x4096 47 / 38).
    if (!mx && t.m == 128 && t.n == 256) {
        const long cus = psg_cu_count();
        const long t256 = (long)((M + 255) / 256) * (long)((N + 255) / 256), t128 = (long)((M + 127) / 128) * (long)((N + 255) / 256);
        if (t128 > cus && t256 <= cus && t256 * 20 > cus * 11) t = {256, 256, 8};
    }
    return t;
}

// A tile's estimated time on a problem whose K isn't split: a start, one `round` per set of tiles that the CUs hold together and, per K step of 128
// bytes, what a CU takes for the 1 .. per_cu tiles it works on at once.  It knows what the score above doesn't: a second tile on a CU costs little
// while a step is bound by its loads, short rows are bound by the rounds' ends, and a last round with few tiles is shorter.  The constants are
// least-squares fits to problems of 65 to 8192 rows, 1024 to 16384 columns (8 and 16 bits: 28672) and K 1024 to 14336, every tile timed on each, most weights in the
// last-level cache.
struct TileCost {
    int m, n, waves, per_cu;
    double start, round, step[6];  // us; step[r]: r tiles on a CU
};

// mem: us of the memory bus; near that bound a launch takes longer than either estimate
double tile_us(const TileCost& c, int M, int N, double steps, double mem) {
    const double cus = psg_cu_count(), tiles = (double)((M + c.m - 1) / c.m) * (double)((N + c.n - 1) / c.n), slots = cus * c.per_cu;
    const double full = std::floor(tiles / slots), rest = (tiles - full * slots) / cus;
    double us = full * (c.round + steps * c.step[c.per_cu]);
    if (rest > 0) {
        // the last round: CUs with one tile more than others finish last, but those with fewer are done sooner and leave them the bus
        const double r = rest > 1 ? 0.25 * rest + 0.75 * std::ceil(rest) : 1;
        const int lo = (int)r;
        double step = c.step[lo] + (lo < c.per_cu ? (r - lo) * (c.step[lo + 1] - c.step[lo]) : 0);
        if (full == 0 && tiles < cus) step *= std::sqrt(std::sqrt(std::sqrt(std::sqrt(tiles / cus))));  // fewer CUs at work clock higher
        us += c.round + steps * step;
    }
    return c.start + std::sqrt(std::sqrt(us * us * us * us + mem * mem * mem * mem));
}

// Whether 256x256 tiles are kept although the estimate of the 128x256 tile is the smallest: the estimates don't see W read from memory by few rows of tiles, for which the 128x256 tile has too few bytes on their way.
// One round: where 256x256 tiles make one round of the CUs, more than half full, and 128x256 tiles would come two to some CUs (up to 768 rows from 136 tiles on: with 136 to 140 of them 128x256 takes 1.13 of the time from memory and
// 0.98 from the cache in int8, 1.14 and 0.97 in 16 bits, us 256x256 / 128x256 from memory int8 463x17184x4800 54.1 / 63.9).  How much the estimates
// have to say then depends on the rows that share W (524 problems, both tiles timed with W in memory and in the cache; time of 128x256 over that of 256x256 where the estimates are at most 12 % apart, memory; cache: int8 up to
// 768 rows 1.16; 1.00, up to 1536 1.13; 0.98, beyond 0.99; 0.98, but at less than one and a half of the smaller tiles a CU 1.01; 1.02; 16 bits 1.14; 0.98, 1.08; 0.98, 0.97; 0.96, 0.98; 1.00). Further apart 128x256 is the better one
// from some 14 to 18 % on (int8 650x11920x832 17.5 / 16.9; but 1261x8480x1856, 14 % apart, 27.5 / 31.1 from memory, 26.5 / 25.9 from the cache), and on rows of up to 1 KB always (bf16 2863x4096x192 11.8 / 10.9).  Of the 524 the tile so chosen takes 0.1 % longer than the better of the two, none is slower both ways.
// The other tiles, where one of them has the smallest estimate, stay (256x256 / the smallest estimate's, memory; cache: int8 838x9248x7296 71.4 / 63.9; 68.5 / 58.6 on 128x128, bf16 826x9360x1088 27.2 / 26.4; 26.3 / 22.4 on
// 64x256; 64 problems 1.01; 1.19).
// W beyond the last-level cache (256 MB, of which A and C take some): W comes from memory then in every pass.  Where the estimates are at most 7 % apart 128x256 takes 1.03 of the time in int8, 1.06 in 16 bits up to 2048 rows
// (102 problems; 76 drawn afterwards 1.02 and 1.04; us 256x256 / 128x256: int8 3337x21488x13248 771 / 817, 2985x23344x13632 777 / 832, bf16 1113x23744x8320 363 / 408, 1270x22928x7552 343 / 391); with more rows 16 bits are level (16 problems 0.97 to 1.07). With 200 to
// 240 MB of W there is no difference (0.99), further apart 128x256 is the better one (int8 2624x25376x8384 491 / 482, bf16 1953x27936x4032 368 / 338).
bool keeps_256(int M, int N, int kbytes, bool wide, double us256, double us128) {
    const long cus = psg_cu_count(), t256 = (long)((M + 255) / 256) * (long)((N + 255) / 256), t128 = (long)((M + 127) / 128) * (long)((N + 255) / 256);
    if ((double)N * kbytes > 240e6 && (!wide || M <= 2048) && us128 > 0.93 * us256) return true;
    const bool one_round = t256 <= cus && t256 * 100 > cus * (M <= 768 ? 53 : 55) && t128 > cus;
    if (!one_round || kbytes <= 1024 || (M > 1536 && (wide || t128 * 2 >= cus * 3))) return false;
    return us128 > (wide ? 0.86 : M <= 1536 ? 0.82 : 0.92) * us256;
}

// Tile of an 8- or 16-bit problem whose K isn't split: the one with the smallest estimate.  On 310 drawn problems (weights in memory and in the
// last-level cache, profiles/tile_times.csv) the estimates are 9 to 16 % off (r.m.s.) and the chosen tile takes 0.2 to 1 % longer than the best of the five; the 128x256 tile, which reads W from the
// cache fastest, waits for it from memory (fp8 4197x1088x11904 64 on 128x256, 71 on 128x128 from the cache, 76 and 71 from memory).  us by the tiles' scores, with the 128x256 tile of that time / by estimate: int8 813x7600x3136
// 30.1 / 22.4, 1416x3136x5568 41.8 / 31.2; fp8 137x16656x1152 13.5 / 10.8; bf16 3156x1536x2752 39.1 / 28.7, 643x9088x1344 25.0 / 18.4.
// Two tiles are left out where they read W from memory more often than the estimate sees (us, W in memory): 64x256 up to 128 rows, where one row of 128x128 tiles does
// (64x256 / 128x128: fp8 96x28672x4096 33.0 / 31.4, bf16 80x26624x1280 20.7 / 19.8, 128x28672x4096 59.5 / 54.1), and with nine rows of tiles where tile_group makes groups of eight, the ninth with all of W to itself (64x256 /
// 128x256: int8 550x14144x13312 161 / 125, 528x26176x8128 184 / 138, bf16 556x26928x4480 215 / 153, fp8 540x26688x11648 275 / 200; the 256x256 tile is faster too), and 64x64 on long rows (64x64 / 128x128: fp8
// 302x5872x9920 43.4 / 38.6, bf16 302x5872x6208 50.6 / 45.7).  Up to a 128x128 tile a CU the 256 columns wide ones don't come into question either: on the short rows that are left there (longer ones
// are split or have fixed tiles) their estimates lie beside that of 128x128, but not their times (us chosen before / 128x128, W in memory: bf16 1182x3200x960 14.4 / 12.6, 2557x1248x1088 15.2 / 13.7,
// 915x3872x704 11.7 / 10.7; of 190 drawn problems this changes 12, by 0.85 to 1.01).
// int8 and the 16-bit kinds have fits of their own for the two large tiles since these share operands between MFMAs, which the 128x256 tile gains more from (us 256x256 / 128x256: bf16
// 5133x5120x8320 359 / 352, 8192x8192x1024 124 / 113, 5817x21104x1792 370 / 337, int8 8192x4096x4096 110 / 104, 4693x22320x3840 346 / 311).  What these don't see: keeps_256.  Over the 1800 problems of profiles/large_tile_times.csv, most of them drawn on the lines of the rules here and there, the chosen tile takes 1 % longer than the best.
// Up to a 128x256 tile a CU the 16-bit fit, made where they come in rounds, has their start 1.4 us too early, so that they replaced 64x256 tiles on short rows (us 64x256 / 128x256, memory; cache: fp16 264x11872x1152
// 17.0 / 18.2; 13.6 / 14.6, 161x20640x1152 18.6 / 19.4; 14.2 / 15.3; 46 problems 1.03; 1.03).
Tile pick_plain_tile(int M, int N, int kbytes, int kind, bool long_rows) {
    static const TileCost costs8[] = {{256, 256, 8, 1, 0.0, 6.7, {0, 1.25}}, {128, 256, 4, 2, 4.8, 0.2, {0, 0.75, 1.60}}, {128, 128, 4, 2, 5.7, 0.0, {0, 0.47, 0.99}},
                                      {64, 64, 4, 5, 3.2, 0.0, {0, 0.30, 0.45, 0.67, 0.95, 1.06}}, {64, 256, 4, 2, 4.6, 0.9, {0, 0.55, 1.10}}};
    static const TileCost costsi[] = {{256, 256, 8, 1, 1.6, 7.7, {0, 1.38}}, {128, 256, 4, 2, 4.2, 0.3, {0, 0.70, 1.53}}, {128, 128, 4, 2, 5.7, 0.0, {0, 0.47, 0.99}},
                                      {64, 64, 4, 5, 3.2, 0.0, {0, 0.30, 0.45, 0.67, 0.95, 1.06}}, {64, 256, 4, 2, 4.6, 0.9, {0, 0.55, 1.10}}};
    static const TileCost costs16[] = {{256, 256, 8, 1, 0.0, 3.6, {0, 1.39}}, {128, 256, 4, 2, 1.3, 0.1, {0, 0.70, 1.46}}, {128, 128, 4, 2, 4.8, 0.0, {0, 0.51, 0.94}},
                                       {64, 64, 4, 5, 2.4, 0.0, {0, 0.33, 0.43, 0.64, 0.91, 0.99}}, {64, 256, 4, 2, 3.3, 0.0, {0, 0.60, 1.08}}};
    const double mem = ((double)(M + N) * kbytes + 2.0 * M * N) / 4.3e6;
    const bool one_each = (long)((M + 127) / 128) * (long)((N + 127) / 128) <= psg_cu_count();
    const bool few = kind != KIND_FP8 && kind != KIND_INT8 && (long)((M + 127) / 128) * (long)((N + 255) / 256) <= psg_cu_count();
    const bool ninth = M > 512 && M <= 576 && (double)(M + (double)N) * kbytes + 2.0 * M * N > 200e6;
    double best = 1e30, us256 = 0;
    Tile t{};
    for (const TileCost& c : kind == KIND_FP8 ? costs8 : kind == KIND_INT8 ? costsi : costs16) {
        if ((c.m == 64 && c.n == 256 && (M <= 128 || ninth)) || (c.n == 64 && long_rows) || (c.n == 256 && one_each)) continue;
        const double us = tile_us(c, M, N, (kbytes + 127) / 128, mem) + (few && c.m == 128 && c.n == 256 ? 1.4 : 0);
        if (c.m == 256) us256 = us;
        if (us < best) {
            best = us;
            t = {c.m, c.n, c.waves};
        }
    }
    if (kind != KIND_FP8 && t.m == 128 && t.n == 256 && keeps_256(M, N, kbytes, kind != KIND_INT8, us256, best)) t = {256, 256, 8};
    return t;
}

// Tile of an MX problem whose K isn't split (kbytes: of a row of A): of an fp4 x fp4 or fp8 / fp6 x fp4 problem the one with the smallest estimated time; of
// fp8 x fp8 the score's unless an estimate is 6 % below that of the score's tile.
// fp4: on 260 drawn problems, weights in memory and in the last-level cache (profiles/tile_times.csv), the estimates are 8 to 11 % off (r.m.s.) and the tile they choose takes 0.3 % longer
// than the best of the five, at worst 8 %.
// Where 64x128 tiles come one to a CU and 32x128 tiles would come two to some, the latter are left out, because reading W once more costs more than the estimate sees (us 32x128 / 64x128, W in
// memory; in the cache: 113x10720x1792 8.5 / 7.7; 6.9 / 6.6, 187x7360x1536 7.3 / 6.8; 6.0 / 5.9, 539x3328x1280 6.9 / 6.5; 6.1 / 6.0, 40x20480x2048 8.7 / 8.0; 6.8 / 6.5; fifteen of 260 drawn problems,
// 3.3 and 2.3 % faster), but for rows of up to 1024 elements and few tiles above the CUs (315x3264x1024, 260 tiles, 5.2 / 5.5; with 320 40x20480x1024 6.1 / 5.8).
// fp8: with most weights in memory the estimates are 10 to 13 % off, so the score's tile stays where they are close: at 3 % twelve of 115 drawn
// problems, those between the two lines, took 2 % longer on average (590x14048x10496 154 instead of 126); of the 115 34 take another tile, 10 % faster and three
// 4 to 7 % slower (us score / estimate 600x7680x3840 35.8 / 38.2).
enum { MX_FP4, MX_FP8, MX_W4 };
Tile pick_mx_tile(int M, int N, int kbytes, int formats) {
    static const TileCost costs4[] = {{128, 256, 4, 2, 1.3, 4.3, {0, 0.65, 1.66}},
                                      {64, 256, 4, 2, 1.8, 3.6, {0, 0.61, 1.17}},      {32, 256, 4, 3, 2.3, 1.9, {0, 0.51, 0.96, 1.35}},
                                      {64, 128, 4, 3, 2.7, 1.5, {0, 0.39, 0.68, 0.98}}, {32, 128, 4, 4, 2.4, 1.0, {0, 0.32, 0.52, 0.77, 0.96}}};
    // (the fp8 launcher runs its 256x256 tile on four wavefronts whatever `waves` says)
    static const TileCost costs8[] = {{256, 256, 8, 1, 2.3, 9.5, {0, 1.45}},           {128, 256, 4, 1, 2.3, 5.7, {0, 0.85}},
                                      {64, 256, 4, 2, 3.9, 1.9, {0, 0.58, 1.02}},      {32, 256, 4, 3, 4.6, 0.0, {0, 0.50, 0.90, 1.21}},
                                      {64, 128, 4, 3, 4.1, 0.5, {0, 0.37, 0.60, 0.88}}, {32, 128, 4, 4, 3.6, 0.2, {0, 0.31, 0.48, 0.73, 0.87}}};
    static const TileCost costs48[] = {{256, 256, 8, 1, 0.0, 7.1, {0, 1.14}},               {128, 256, 4, 2, 4.0, 3.5, {0, 0.77, 1.36}},
                                       {64, 256, 4, 3, 3.4, 2.2, {0, 0.48, 0.77, 1.13}},    {32, 256, 4, 3, 3.6, 0.8, {0, 0.37, 0.58, 0.76}},
                                       {64, 128, 4, 3, 3.4, 1.0, {0, 0.34, 0.49, 0.68}},    {32, 128, 4, 4, 3.1, 0.5, {0, 0.28, 0.35, 0.49, 0.60}}};
    const double mem = ((double)M * kbytes + (double)N * (formats == MX_W4 ? kbytes / 2 : kbytes) + 2.0 * M * N) / 4.3e6;
    const Tile scored = formats == MX_FP8 ? pick_tile(M, N, true, 0, 0) : Tile{};
    const long cus = psg_cu_count(), n128 = (N + 127) / 128, tiles32 = (M + 31) / 32 * n128;
    const bool no32 = formats == MX_FP4 && (M + 63) / 64 * n128 <= cus && tiles32 > cus && (kbytes > 512 || tiles32 * 5 > cus * 6);
    double best = 1e30, kept = 1e30;
    Tile t = scored;
    auto consider = [&](const auto& costs) {
        for (const TileCost& c : costs) {
            if (no32 && c.m == 32 && c.n == 128) continue;
            const double us = tile_us(c, M, N, (kbytes + 127) / 128, mem);
            if (formats == MX_FP8 && c.m == scored.m && c.n == scored.n) kept = us;
            if (us < best) {
                best = us;
                t = {c.m, c.n, c.waves};
            }
        }
    };
    if (formats == MX_FP4) consider(costs4);
    else if (formats == MX_FP8) consider(costs8);
    else consider(costs48);
    return best < 0.94 * kept ? t : scored;
}

// Where the eight XCDs' ranges of an order in groups of `g` M-tiles start: the longest stretch of column tiles without a start, as a share of all
double widest_gap(int tiles_m, int tiles_n, int g) {
    const int num = tiles_m * tiles_n, q = num >> 3, r = num & 7;
    int at[8];
    for (int x = 0; x < 8; x++) {
        const int wg = x * q + (x < r ? x : r), grp = wg / (g * tiles_n), rows = tiles_m - grp * g < g ? tiles_m - grp * g : g;
        const int tn = (wg - grp * g * tiles_n) / rows;
        int i = x;
        for (; i > 0 && at[i - 1] > tn; i--) at[i] = at[i - 1];
        at[i] = tn;
    }
    int gap = at[0] + tiles_n - at[7];
    for (int x = 1; x < 8; x++) gap = at[x] - at[x - 1] > gap ? at[x] - at[x - 1] : gap;
    return (double)gap / tiles_n;
}

// M-tiles per group of the XCD-aware tile order.  Eight make the set of tiles that an XCD works on at a time roughly square in bytes, which
// is the least for its L2 to fetch.  But where its range starts, every XCD asks for one panel of W and stores to one range of columns, and with eight many
// problems have all of them start at the same column tile or at two (whenever num / 8 is a multiple of half a group): they then walk
// the columns side by side, and the rows of C, a power of two apart, meet in a few memory channels.  So the group of about that size is taken
// whose starts lie apart (us in groups of 8 / as chosen here: fp8 8192x4096x4096 111.2 / 107.8, 8192x8192x1024 87.2 / 79.0, 4096x7168x2048 58.8 / 56.0, 4096x6144x4096 93.9 / 89.9; int8 8192x8192x1024 92.1 / 82.7; bf16
// 8192x4096x2048 111.5 / 108.6; fp4 8192x8192x1024 65.4 / 58.1, 4221x7744x1536 49.9 / 45.7; over 40 drawn sizes, few of which are aligned like that,
// 0.98 to 1.10 and 1.004 on average).
// Only where A, W and C fit the last-level cache together: beyond, XCDs that walk side by side read a panel of W from memory once (int8
// 4096x28672x8192 714 in groups of 8 or 6, four or three starts, 728 to 732 with 7, 9 or 11, eight).  A last group of one M-tile
// reads all of W for it (fp8 4096x8192x2048, 16 M-tiles, 64 / 71 in groups of 8 / 5), and so does one of less than half the size behind a single whole one, with W in memory (12 to 14
// M-tiles, us in groups of 8 / 9 to 11, from memory: fp8 1506x12800x2432 48.8 / 52.1, 1460x13696x2176 46.1 / 49.5, fp4 1532x12736x1280 24.3 / 26.4, bf16 1536x6656x1280 31.1 / 34.4; 2 % over 40
// such problems, 1 % from the cache).  Behind two whole ones it does not (fp4 2048x9728x3072, 16 M-tiles, 42.2 / 37.4 in groups of 8 / 7).  Up to a tile a CU all of them are at work at once in any order (fp8
// 4096x4096x7168, 256 tiles, 87 / 89).
int tile_group(int hint, int M, int N, Tile t, double bytes) {
    if (hint > 0) return hint;
    const int tiles_m = (M + t.m - 1) / t.m, tiles_n = (N + t.n - 1) / t.n;
    if ((long)tiles_m * tiles_n <= psg_cu_count() || bytes > 200e6) return 8;
    int best = 8;
    double gap = 2;
    for (const int g : {8, 7, 9, 6, 10, 11, 5}) {
        const int last = tiles_m % g;
        if (tiles_m > g && (last == 1 || (g != 8 && tiles_m < 2 * g && 2 * last < g))) continue;
        const double d = widest_gap(tiles_m, tiles_n, g);
        if (d < gap - 0.02) {
            gap = d;
            best = g;
        }
        if (gap <= 0.16) break;
    }
    return best;
}

// Split-K for the regime between the streaming kernel (takes_stream) and problems with enough tiles to fill the GPU:
// with few tiles every workgroup walks all of K behind a one-step prefetch and the launch is latency-bound.
// Splitting K over `splits` workgroups per tile multiplies the loads in flight; the price is one fp32 slice of
// [M,N] per split written and read back, so the split count is capped where that traffic reaches 1.25 W, and where the
// workgroups would no longer all be resident at once.
// Returns 1 when splitting does not pay.  kbytes = bytes of one operand row.
int pick_splits(int M, int N, int kbytes, Tile t) {
    const long tiles = (long)((M + t.m - 1) / t.m) * (long)((N + t.n - 1) / t.n);
    const int steps = (kbytes + 127) / 128;
    const long cus = psg_cu_count();
    // a CU holds one workgroup of a 128x128 tile (or larger), two of a 64x64 tile on long rows
    const bool pairs = t.m == 64 && t.n == 64 && steps >= 48;
    if (tiles >= (pairs ? 2 * cus : cus) * 3 / 4 || steps < 32) return 1;
    // Measured on operands that do not fit the last-level cache (fp8, 128x128 tiles): the best split count is the largest one
    // that still gives every workgroup a CU of its own, powers of two or not (us for 2/3/4/5/6/7/8 splits: 256x2304x14336,
    // 36 tiles, 40/32/27/25/24/23.5/30; 384x1664x10240, 39 tiles, 32/26/23/22/21.7/24.5/27; 256x3072x14336, 48 tiles,
    // 43/34/30/27.6/35/35/33; 512x2112x7168, 68 tiles, 24.8/22.1 for 2/3; one workgroup more than there are CUs costs a second
    // round).  64x64 tiles on long rows may also come two to a CU, but then (nearly) all CUs should have two: between one and one
    // and a half workgroups per CU the doubled CUs finish last (64x6144x16384, 96 tiles, us for 2/3/4/5/8 splits: 34/35/31/29/29;
    // 48x5120x13824, 80 tiles, 3/6/8 splits: 23.3/21.4/22.7; 48x2304x14336, 36 tiles, 7/8 splits: 14.9/16.6).  Bounds: at least
    // 8 K steps per workgroup (12 on rows shorter than 48 steps), partial sums at most 1.25 W.
    const int min_steps = steps >= 48 ? 8 : 12;
    int s = 1;
    for (int c = 2; c <= 8; c++) {
        const long wgs = tiles * c;
        const bool fits = wgs <= cus || (pairs && 2 * wgs >= 3 * cus && wgs <= 2 * cus);
        if (fits && steps / c >= min_steps && (long)c * M * 16 <= (long)kbytes * 5) s = c;
    }
    return s;
}

// Whether a batch of several dense MX products runs on the tiles of the dense kernels, a launch each: where 128x256 tiles of one product would
// give every CU one, since the general kernel takes all batches in one launch (us tiles / general: fp8 x fp8 2 x 1024x8192x4096 78 / 104, 8 324 /
// 497, 12 473 / 744, 4 x 1280x8192x2048 139 / 139; fp4 x fp4 2 x 512x16384x2048 34.8 / 45.7, 8 x 2048x4096x4096 194 / 277; fp8 x fp4 2 x 2048x4096x4096
// 88 / 93, 8 327 / 371; fp6 x fp4 2 x 512x16384x2048 53.6 / 52.6, 8 205 / 216; with half as many tiles fp8 x fp4 8 x 512x8192x2048 183 / 104).
// More batches gain as much; the limit of eight (mx_common) is what one call may queue as launches of its own.
bool mx_fills_tiles(int M, int N) {
    return M > kStreamMaxM && (long)((M + 127) / 128) * (long)((N + 255) / 256) >= psg_cu_count();
}

// Which calls of the general MX path the small-M kernel takes (the others: gemm_mx_generic.hip).
// Up to 64 rows, while what its N / 32 workgroups read of A together stays below 160 MB with fp4 weights and 320 MB with fp8 weights (N K M
// / 32, M in whole register tiles of 16, 32 or 64 rows), and from 1024 columns on (32 workgroups).  Measured, us small-M / general:
// fp8 x fp4 1 x 8192 x 8192 7.7 / 12.2, 64 x 8192 x 8192 12.3 / 20.2, 64 x 4096 x 4096 6.9 / 16.0, 16 x 1024 x 2048 3.1 / 6.8, 64 x 1024 x
// 14336 15.7 / 27.3, 64 x 16384 x 4096 (134 MB) 14.5 / 17.7, 16 x 16384 x 14336 (117 MB) 22.6 / 23.2, but 24 rows of it (235 MB) 25.9 / 24.1
// and 64 (470 MB) 37.5 / 32.0; fp8 x fp8 32 x 16384 x 14336 (235 MB) 40.9 / 46.8, 64 rows 51.1 / 48.8; fp6 x fp4 as fp8 x fp4.
// Beyond 64 rows a workgroup takes 64 of them, and the kernel is the better one while its workgroups make one round of one per CU, or two on
// rows of up to 8192 elements (fp8 x fp4, 128 x 2048 x 4096 6.7 / 16.1, 256 x 1024 x 14336 16.6 / 46.8, 128 x 4096 x 4096 7.2 / 16.2; two
// rounds 256 x 4096 x 4096 12.8 / 16.5, 128 x 8192 x 8192 22.8 / 29.0; three 192 x 8192 x 8192 32.8 / 29.1, four 128 x 16384 x 4096 26 / 18).
// Batches multiply the workgroups, and the general kernel, which cannot split K over them, gets the workgroups it lacked.  So up to 64 rows
// batches also have to make at most two rounds of 64-row workgroups (one with fp4 activations, which are read in fragment order), fewer
// rows counting for as much less (768 points of 2 to 8 batches: the other kernel more than 5 % faster at 53 of them, at 198 without this
// bound; us small-M / general: fp8 x fp4 64 x 4096 x 4096 2 batches 7.6 / 16.4, 4 (two rounds) 13.8 / 17.3, 8 27.1 / 21.8; 64 x 16384 x 4096 2
// batches 27.3 / 21.5; fp4 x fp4 64 x 4096 x 4096 2 (one round) 8.0 / 11.7, 4 14.3 / 13.4, 8 27.6 / 19.1; 16 x 4096 x 4096 8 14.0 / 15.7; fp8 x
// fp8 64 x 8192 x 8192 2 (two rounds) 32.0 / 33.0, 4 65.0 / 47.8).
bool mx_general_small(int M, int N, int K, bool fp4_acts, bool fp8_weights, int batch) {
    if (M > kStreamMaxM) {
        const long wgs = (long)(N / 32) * ((M + 63) / 64) * batch, cus = psg_cu_count();
        return N >= 1024 && wgs <= (K <= 8192 ? 2 : 1) * cus;
    }
    const long rows = M <= 16 ? 16 : M <= 32 ? 32 : 64;
    if (batch > 1 && (long)(N / 32) * batch * rows > (fp4_acts ? 1 : 2) * 64L * psg_cu_count()) return false;
    return N >= 1024 && (long)(N / 32) * rows * K <= (fp8_weights ? 320L : 160L) * 1000000L;
}

// Split-K for the general MX kernel: its tiles are 64x128 (32x128 for M <= 32), so decode-like shapes launch few
// workgroups; K is split until about two workgroups per CU exist, every split keeps at least eight 128-element steps
// and the fp32 partials (written and read back once) stay below a quarter of the bytes of an fp4 W.
int mx_general_splits(int M, int N, int K) {
    const uint64_t w_bytes = (uint64_t)N * (uint64_t)K / 2;  // of fp4 W; fp8 W gets the same plan
    const long tiles = (long)((M + (M <= 32 ? 31 : 63)) / (M <= 32 ? 32 : 64)) * (long)((N + 127) / 128);
    const int steps = K / 128;
    int s = 1;
    while (s < 8 && tiles * (s * 2) <= 2L * psg_cu_count() && steps / (s * 2) >= 8 && (uint64_t)(s * 2) * (uint64_t)M * (uint64_t)N * 8ull <= w_bytes / 4) s *= 2;
    return s;
}

// Where a dense, unbatched fp8 x fp8 or fp8 / fp6 x fp4 problem runs: on the small-M kernel, on the general kernel with its K splits (`room`: the caller
// brought their workspace), or on the tiles of the dense kernels.  Up to 32 rows on the first two (fp8 x fp8 32x12288x4096 13.6 / 14.2 on tiles).
// Beyond that the small-M kernel, whose N / 32 workgroups for every 64 rows stream W best, while they make one round of the CUs; the tiles read W
// from the last-level cache faster than that, but from memory slower, so in the second round it depends.  The lines are from 900 problems of 33 to 400 rows,
// 200 to 1100 such workgroups and K 1024 to 14336, each with W in memory and with W in that cache (us small-M / splits / tiles, memory; cache):
//   rows below 1536 elements: an eighth of a round more than one; below 2048 and with fp4 weights two rounds, up to 320 rows (68x5120x1280 5.4 / 8.3 / 6.8; 5.2 /
//     8.1 / 5.5, 106x6432x1792 7.3 / 10.1 / 8.5; 6.7 / 9.9 / 7.0; but 389x1248x1536 8.4 / 10.0 / 7.3)
//   splits, up to 64 rows while they make at most two workgroups a CU, beyond at most one: fp8 x fp8 42x8544x10240 33.0 / 30.5 / 40.0;
//     31.5 / 24.5 / 29.1, 48x10400x13312 43.3 / 40.6 / 52.6; 40.8 / 32.1 / 36.2, 75x5216x10752 33.7 / 30.5 / 40.0; 32.3 / 26.3 / 29.2; fp8 x fp4 38x10112x9984
//     24.7 / 21.2 / 33.2; 23.7 / 18.6 / 24.2; but more of them fp8 x fp8 67x9568x8960 - / 36.6 / 36.3; - / 36.0 / 25.7.
//     With fp4 weights and at most one workgroup a CU, or without the workspace, the small-M kernel is as good or better: 38x12992x6912 19.4 / 20.6 / 24.5;
//     18.6 / 18.6 / 18.3, 47x11456x8448 23.0 / 24.1 / 29.3; 22.2 / 21.0 / 21.4
//   long rows of fp4 weights in the second round up to 192 rows: 94x6400x7424 20.5 / 30.4 / 25.3; 17.1 / 26.7 / 18.4, 149x3040x6912 17.6 / 27.4 / 23.6; 17.3 / 26.1 / 17.0, 140x4480x7680
//     23.2 / 31.4 / 25.9; 21.1 / 27.5 / 18.5; beyond, 345x1472x6144 17.9 / 26.6 / 20.6; 16.1 / 22.8 / 15.0, the cache loses as much as the memory gains
//   everything else on tiles (33x9184x3072 10.7 / 13.9 / 12.3; 9.7 / 13.3 / 9.4, 40x15456x3840 18.7 / 23.2 / 21.4; 16.7 / 17.4 / 13.7, 65x13664x12032 56 / 38 /
//     43.6; 55 / 36 / 31.5; three rounds or more always, where against the general kernel, from memory, fp8 x fp8 1164x2880x4096 takes 24.6 / 36.8, fp8 x fp4 591x8032x5632 37 / 55)
enum MxRoute { MX_SMALL, MX_GENERAL, MX_TILES };
MxRoute mx_route(int M, int N, int K, bool fp8_weights, bool room) {
    const bool holds = mx_general_small(M, N, K, false, fp8_weights, 1);
    if (M <= kSmallM) return holds ? MX_SMALL : MX_GENERAL;
    const long cus = psg_cu_count(), groups = (M + 63) / 64, wgs = (long)(N / 32) * groups;
    const bool small = holds && wgs <= 2 * cus;
    if (small && (wgs <= cus || (K < 1536 && wgs * 8 <= cus * 9) || (K < 2048 && !fp8_weights && M <= 320))) return MX_SMALL;
    const int splits = mx_general_splits(M, N, K);
    const long split_wgs = groups * ((N + 127) / 128) * splits;
    if (splits > 1 && split_wgs <= (M <= kStreamMaxM ? 2 : 1) * cus) {
        if (small && (!room || (!fp8_weights && split_wgs <= cus))) return MX_SMALL;
        return room ? MX_GENERAL : MX_TILES;
    }
    return small && !fp8_weights && K >= 6144 && M <= 192 ? MX_SMALL : MX_TILES;
}

// Tile + split plan of the tiled path.  With few tiles and a long K (the regime between the streaming kernel and
// GPU-filling problems) small square-ish tiles with split-K measured best: 64x64 up to M=64, 128x128 above.
struct Plan {
    Tile t;
    int splits;
};
// kind: of the operands, for the tile where K isn't split (mx: of no account; the splits are the same for all)
Plan plan_tiled(int M, int N, int kbytes, bool mx, int kind) {
    // more columns than the streaming kernel takes in one round: 64x64 tiles, unsplit (these problems have no workspace)
    if (!mx && stream_holds(M, N, kbytes) && N > 32 * psg_cu_count()) return {Tile{64, 64, 4}, 1};
    Tile t = pick_tile(M, N, mx, 0, 0);
    const long tiles_big = (long)((M + 127) / 128) * (long)((N + 255) / 256);
    const int steps = (kbytes + 127) / 128;
    const long tiles64 = (long)((M + 63) / 64) * (long)((N + 63) / 64);
    // long rows, few tiles: 128x128 tiles with split-K; 64x64 tiles up to 64 rows, and above that while the whole problem is small
    // (tiles x steps, i.e. M N K / 2^19, up to 11,000: then twice as many workgroups count for more than the W fragments that are
    // loaded twice; fp8, us, 64x64 plan against 128x128 plan: 256x2112x7168 14.8 / 16.8; 320x2112x7168 15.6 / 18.4; 320x1664x10240
    // 18.3 / 20.2; 128x2048x16384 19.2 / 21.2; but 256x2304x14336 27.1 / 23.9; 320x2048x16384 30.0 / 26.3; 65x5120x13824 25.8 / 23.4)
    const bool long_rows = !mx && tiles_big < psg_cu_count() * 3L / 4 && steps >= 48;
    bool fixed = long_rows && (M <= 64 || tiles64 * steps <= 11000);
    if (long_rows) t = fixed ? Tile{64, 64, 4} : Tile{128, 128, 4};
    // Shorter rows (8..47 steps; K = 4096 one-byte elements is 32): while at most about 600 of them exist, 64x64 tiles beat
    // every larger shape, with or without split-K: many small workgroups keep more bytes of W in flight than a few large ones
    // (fp8, weights not cache-resident: M=128, N=K=4096 14.0 us against 19.4 with 128x128 tiles and two K splits; M=256,
    // N=8192 22.0 against 23.7; M=384, N=8192, 768 tiles: 28.0 against 26.5, so the larger tile is kept there)
    if (!mx && steps >= 8 && steps < 48 && tiles64 <= 600) t = Tile{64, 64, 4}, fixed = true;
    const int splits = mx && mx_small_holds(M, N, kbytes * 2) ? 1 : pick_splits(M, N, kbytes, t);
    if (splits == 1 && !fixed) t = mx ? pick_mx_tile(M, N, kbytes, MX_FP4) : pick_plain_tile(M, N, kbytes, kind, long_rows);
    return {t, splits};
}

uint64_t splitk_bytes(int M, int N, int splits) { return splits > 1 ? (uint64_t)splits * M * N * 4ull : 0; }

int validate_a8w8(const psg_a8w8_args* a, bool acc_only, const void* acc) {
    if (!a) return fail(PSG_E_NULL, "args is NULL");
    if (!a->a || !a->b) return fail(PSG_E_NULL, "a and b must be non-NULL");
    const bool is16 = a->in_dtype == PSG_IN_FP16 || a->in_dtype == PSG_IN_BF16;
    const int64_t eb = is16 ? 2 : 1;
    if (acc_only) {
        if (!acc) return fail(PSG_E_NULL, "acc must be non-NULL");
    } else {
        if (!a->c) return fail(PSG_E_NULL, "c must be non-NULL");
        if (!is16 && (!a->scale_a || !a->scale_b)) return fail(PSG_E_NULL, "scale_a and scale_b must be non-NULL for 8-bit inputs");
        if (a->epilogue != PSG_EPI_NONE && !a->bias) return fail(PSG_E_NULL, "bias must be non-NULL when epilogue != none");
    }
    if (a->in_dtype < PSG_IN_INT8 || a->in_dtype > PSG_IN_BF16) return fail(PSG_E_DTYPE, "in_dtype %d unknown", a->in_dtype);
    if (a->out_dtype != PSG_OUT_BF16 && a->out_dtype != PSG_OUT_FP16) return fail(PSG_E_DTYPE, "out_dtype %d unknown", a->out_dtype);
    if (a->epilogue < PSG_EPI_NONE || a->epilogue > PSG_EPI_BIAS_GELU) return fail(PSG_E_DTYPE, "epilogue %d unknown", a->epilogue);
    if (a->M < 1 || a->M > 65536) return fail(PSG_E_SHAPE, "M=%d outside [1, 65536]", a->M);
    if (a->N < 16 || a->N % 16) return fail(PSG_E_SHAPE, "N=%d must be a positive multiple of 16", a->N);
    if (a->K < 64 / eb || (a->K * eb) % 64) return fail(PSG_E_SHAPE, "K=%d must be a positive multiple of %d", a->K, (int)(64 / eb));
    if ((uint64_t)a->N * (uint64_t)a->K * (uint64_t)eb > 0xFFFFFFFFull) return fail(PSG_E_SHAPE, "N*K bytes exceed the 4 GiB descriptor range");
    if (!aligned(a->a, 16) || !aligned(a->b, 16)) return fail(PSG_E_ALIGN, "a and b must be 16-byte aligned");
    if (acc_only) {
        if (!aligned(acc, 16)) return fail(PSG_E_ALIGN, "acc must be 16-byte aligned");
    } else {
        if (!aligned(a->c, 16)) return fail(PSG_E_ALIGN, "c must be 16-byte aligned");
        if (!is16 && !aligned(a->scale_b, 16)) return fail(PSG_E_ALIGN, "scale_b must be 16-byte aligned");
        if (!is16 && !aligned(a->scale_a, 4)) return fail(PSG_E_ALIGN, "scale_a must be 4-byte aligned");
        if (a->epilogue != PSG_EPI_NONE && !aligned(a->bias, 8)) return fail(PSG_E_ALIGN, "bias must be 8-byte aligned");
    }
    if (a->workspace && !aligned(a->workspace, 16)) return fail(PSG_E_ALIGN, "workspace must be 16-byte aligned");
    if (a->b_layout != 0 && a->b_layout != 1) return fail(PSG_E_DTYPE, "b_layout=%d unknown (0 preshuffled, 1 row-major)", a->b_layout);
    if (a->force_path < 0 || a->force_path > 2) return fail(PSG_E_SHAPE, "force_path=%d unknown", a->force_path);
    if (a->force_path == 2 && a->M > kStreamMaxM) return fail(PSG_E_SHAPE, "small-M path needs M <= %d, got %d", kStreamMaxM, a->M);
    return 0;
}

// Device address of `scratch` on the current device (looked up once per device, then cached).
int static_scratch(void** out) {
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return hip_fail(e, "hipGetDevice");
    if (dev < 0 || dev >= kMaxDevices) return fail(PSG_E_UNSUPPORTED, "device index %d outside [0, %d)", dev, kMaxDevices);
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void* ptr = nullptr;
        e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return hip_fail(e, "hipGetSymbolAddress(scratch)");
        if (!ptr) return fail(PSG_E_WORKSPACE, "hipGetSymbolAddress returned a null address for the static scratch");
        g_scratch_ptr[dev] = ptr;
    }
    *out = g_scratch_ptr[dev];
    return 0;
}

// Argument checks of the expert sorter; `need_routing`: topk_ids / topk_weights are read (not with the fused gating).
int check_moe_sort(const psg_moe_sort_args* a, bool need_routing, MoeSortParams* out) {
    if (!a) return fail(PSG_E_NULL, "args is NULL");
    if ((need_routing && (!a->topk_ids || !a->topk_weights)) || !a->sorted_ids || !a->sorted_weights || !a->sorted_expert_ids || !a->num_valid_ids)
        return fail(PSG_E_NULL, "topk_ids, topk_weights, sorted_ids, sorted_weights, sorted_expert_ids, num_valid_ids must be non-NULL");
    if (a->tokens < 1 || a->tokens >= (1 << 24)) return fail(PSG_E_SHAPE, "tokens=%d outside [1, 2^24)", a->tokens);
    if (a->topk < 1 || a->topk > 255) return fail(PSG_E_SHAPE, "topk=%d outside [1, 255]", a->topk);
    if (a->experts < 1 || a->experts > psg_moe_sort_max_experts()) return fail(PSG_E_SHAPE, "experts=%d outside [1, %d]", a->experts, psg_moe_sort_max_experts());
    if (a->block_m < 1 || a->block_m > 4096) return fail(PSG_E_SHAPE, "block_m=%d outside [1, 4096]", a->block_m);
    // the bound below (the reference's) counts at most one partly filled block per expert and at least topk rows routed: with
    // more slots than experts a token repeats an expert and the padded total can exceed it
    if (a->topk > a->experts) return fail(PSG_E_SHAPE, "topk=%d exceeds experts=%d", a->topk, a->experts);
    const int64_t pairs = (int64_t)a->tokens * a->topk;
    const int64_t need = pairs + (int64_t)a->experts * a->block_m - a->topk;
    if (need > 0x7FFFFFFF) return fail(PSG_E_SHAPE, "tokens*topk + experts*block_m must stay below 2^31");
    if (a->sorted_size < need) return fail(PSG_E_SHAPE, "sorted_size=%d is below tokens*topk + experts*block_m - topk = %lld", a->sorted_size, (long long)need);
    if ((int64_t)a->blocks * a->block_m < a->sorted_size)
        return fail(PSG_E_SHAPE, "blocks=%d must cover sorted_size=%d rows in blocks of %d", a->blocks, a->sorted_size, a->block_m);
    if (a->zero_buf && (a->zero_bytes < 0 || a->zero_bytes % 16 || !aligned(a->zero_buf, 16)))
        return fail(PSG_E_ALIGN, "zero_buf must be 16-byte aligned and zero_bytes a multiple of 16");
    if (a->workspace && !aligned(a->workspace, 4)) return fail(PSG_E_ALIGN, "workspace must be 4-byte aligned");
    MoeSortParams p;
    p.topk_ids = a->topk_ids;
    p.topk_weights = a->topk_weights;
    p.expert_mask = a->expert_mask;
    p.sorted_ids = a->sorted_ids;
    p.sorted_weights = a->sorted_weights;
    p.sorted_expert_ids = a->sorted_expert_ids;
    p.num_valid = a->num_valid_ids;
    p.zero_buf = a->zero_bytes > 0 ? static_cast<v4i*>(a->zero_buf) : nullptr;
    p.zero_vec = a->zero_buf ? a->zero_bytes / 16 : 0;
    p.tokens = a->tokens;
    p.topk = a->topk;
    p.experts = a->experts;
    p.block_m = a->block_m;
    p.sorted_size = a->sorted_size;
    p.blocks = a->blocks;
    *out = p;
    return 0;
}

// Argument checks of the router gating; `need_outputs`: weights / indices must be given (optional with the fused sorting).
int check_moe_gating(const psg_moe_gating_args* a, bool need_outputs, MoeGatingParams* out) {
    if (!a) return fail(PSG_E_NULL, "args is NULL");
    if (!a->gating) return fail(PSG_E_NULL, "gating must be non-NULL");
    if (need_outputs && (!a->weights || !a->indices)) return fail(PSG_E_NULL, "weights and indices must be non-NULL");
    if (a->dtype < 0 || a->dtype > 2) return fail(PSG_E_DTYPE, "dtype %d unknown (0 fp32, 1 bf16, 2 fp16)", a->dtype);
    if (a->tokens < 1 || a->tokens >= (1 << 24)) return fail(PSG_E_SHAPE, "tokens=%d outside [1, 2^24)", a->tokens);
    if (a->experts < 1 || a->experts > GATE_MAX_EXPERTS) return fail(PSG_E_SHAPE, "experts=%d outside [1, %d]", a->experts, GATE_MAX_EXPERTS);
    if (a->topk < 1 || a->topk > GATE_MAX_TOPK || a->topk > a->experts)
        return fail(PSG_E_SHAPE, "topk=%d outside [1, min(%d, experts=%d)]", a->topk, GATE_MAX_TOPK, a->experts);
    if (a->renormalize != 0 && a->renormalize != 1) return fail(PSG_E_SHAPE, "renormalize=%d must be 0 or 1", a->renormalize);
    if (!aligned(a->gating, a->dtype == 0 ? 4 : 2) || (a->weights && !aligned(a->weights, 4)) || (a->indices && !aligned(a->indices, 4)) ||
        (a->token_expert_indices && !aligned(a->token_expert_indices, 4)))
        return fail(PSG_E_ALIGN, "gating must be aligned to its element size, the outputs to 4 bytes");
    MoeGatingParams g;
    g.gating = a->gating;
    g.weights = a->weights;
    g.indices = a->indices;
    g.tei = a->token_expert_indices;
    g.tokens = a->tokens;
    g.experts = a->experts;
    g.topk = a->topk;
    g.renorm = a->renormalize;
    g.lanes = 1;
    g.vec = 0;
    *out = g;
    return 0;
}

constexpr int kKinds[4] = {KIND_INT8, KIND_FP8, KIND_FP16, KIND_BF16};  // by PSG_IN_*

int run_a8w8(const psg_a8w8_args* a, void* out, int store, void* stream) {
    A8W8Params p{};
    p.c = out;
    p.a = static_cast<const uint8_t*>(a->a);
    p.b = static_cast<const uint8_t*>(a->b);
    p.sa = a->scale_a;
    p.sb = a->scale_b;
    p.bias = static_cast<const uint16_t*>(a->bias);
    p.M = a->M;
    p.N = a->N;
    p.K = a->K;
    p.epi = a->epilogue;
    p.out = a->out_dtype;
    p.b_rowmajor = a->b_layout;
    const int kind = kKinds[a->in_dtype];
    const int kbytes = (kind == KIND_FP16 || kind == KIND_BF16) ? a->K * 2 : a->K;
    const bool small = a->force_path == 2 || (a->force_path == 0 && takes_stream(a->M, a->N, kbytes));
    hipError_t e;
    if (small) {
        e = psg_launch_a8w8_stream(p, kind, store, static_cast<hipStream_t>(stream));
    } else {
        const bool forced = a->force_path == 1 && a->tile_m > 0 && a->tile_n > 0;
        const Plan plan = plan_tiled(a->M, a->N, kbytes, false, kind);
        const Tile t = forced ? Tile{a->tile_m, a->tile_n, 4} : plan.t;
        p.ksplit = 1;
        // wavefront layout of the 256x256 tile: the planner's choice, or forced (2 = 2x2, 8 = 1x8) by tests / tuning
        p.wave_layout = a->reserved >= 2 ? a->reserved : (!forced && t.waves == 8 ? 8 : 1);
        // forced launches take the split count from tile_k (1..16); otherwise the planner decides
        int splits = forced ? (a->tile_k >= 1 && a->tile_k <= 16 ? a->tile_k : 1) : plan.splits;
        if (store != STORE_C || !a->workspace || a->workspace_bytes < splitk_bytes(a->M, a->N, splits)) splits = 1;
        p.splits = splits;
        p.group_m = tile_group(a->xcd_swizzle, a->M, a->N, t, splits > 1 ? 1e30 : (double)(a->M + (double)a->N) * kbytes + 2.0 * a->M * a->N);
        // at most two workgroups per CU: the launch is bound by the bytes of W in flight, so the builds that fetch W three
        // steps ahead run (ksplit doubles as that mark for the tiled kernel); reserved = 7 keeps the one-step builds (tests)
        const long wgs = (long)((a->M + t.m - 1) / t.m) * (long)((a->N + t.n - 1) / t.n) * splits;
        const int steps_per_wg = ((kbytes + 127) / 128 + splits - 1) / splits;
        // Not so one row of 64x64 tiles, more than one to a CU: from memory both builds are as fast, from the last-level cache the one-step build is (us three steps / one, memory; cache: int8
        // 35x17056x12096 60.3 / 58.5; 46.4 / 37.3, 64x24576x4096 24.5 / 25.0; 19.3 / 18.0, fp8 46x19456x7424 38.5 / 38.7; 28.9 / 24.9, bf16 44x17632x1472 16.6 / 16.8; 13.3 / 11.6; but with four rows
        // of tiles 200x8192x8192 32.9 / 38.0; 28.3 / 26.8).
        const bool one_row = t.m == 64 && t.n == 64 && a->M <= 64 && splits == 1 && wgs > psg_cu_count();
        if (wgs <= 512 && steps_per_wg >= 6 && a->reserved != 7 && (forced || !one_row)) p.ksplit = 3;
        if (splits > 1) {
            A8W8Params part = p;
            part.c = a->workspace;
            e = psg_launch_a8w8_tiled(part, kind, STORE_ACC, t.m, t.n, static_cast<hipStream_t>(stream));
            if (e == hipSuccess)
                e = psg_launch_splitk_finalize(p, a->workspace, kind == KIND_INT8, kind == KIND_INT8 || kind == KIND_FP8,
                                               static_cast<hipStream_t>(stream));
        } else {
            e = psg_launch_a8w8_tiled(p, kind, store, t.m, t.n, static_cast<hipStream_t>(stream));
        }
    }
    if (e != hipSuccess) return hip_fail(e, "psg_gemm_a8w8 launch");
    g_err[0] = 0;
    return 0;
}

}  // namespace

extern "C" {

int psg_abi_version(void) { return PSG_ABI_VERSION; }

const char* psg_last_error(void) { return g_err; }

uint64_t psg_workspace_bytes(int32_t M, int32_t N, int32_t K, int32_t in_dtype) {
    // Only the split-K variant of the tiled path (few tiles, long K) uses global scratch: one fp32 / int32 slice of
    // [M,N] per split.  Without it (NULL or too small) the library runs the same problem unsplit.
    if (in_dtype >= 16) {  // psg_gemm_mxfp4, whichever kernel takes the pair of formats
        const int fa = (in_dtype - 16) >> 2, fb = (in_dtype - 16) & 3;
        if (M < 1 || N < 32 || K < 256 || fa > PSG_MX_FP8 || (fb != PSG_MX_FP4 && fb != PSG_MX_FP8)) return 0;
        if (fa == PSG_MX_FP4 && fb == PSG_MX_FP4) return psg_workspace_bytes(M, N, K, 4);
        const bool planned = fb == PSG_MX_FP4 || fa == PSG_MX_FP8;
        if (planned ? mx_route(M, N, K, fb == PSG_MX_FP8, true) != MX_GENERAL : mx_general_small(M, N, K, fa == PSG_MX_FP4, fb == PSG_MX_FP8, 1)) return 0;
        return splitk_bytes(M, N, mx_general_splits(M, N, K));
    }
    if (in_dtype == 5) return M >= 1 && N >= 32 && K >= 256 ? splitk_bytes(M, N, mx_general_splits(M, N, K)) : 0;  // general MX kernel
    if (M <= kSmallM || M < 1 || N < 16 || K < 64) return 0;
    const bool mx = in_dtype == 4;  // MXFP4 (psg_gemm_mxfp4)
    const int kbytes = mx ? K / 2 : ((in_dtype == PSG_IN_FP16 || in_dtype == PSG_IN_BF16) ? K * 2 : K);
    if (mx ? mx_takes_small(M, N, K) : takes_stream(M, N, kbytes)) return 0;  // the small-M kernels reduce inside their workgroups
    return splitk_bytes(M, N, plan_tiled(M, N, kbytes, mx, KIND_FP8).splits);
}

int psg_gemm_a8w8(const psg_a8w8_args* args, void* stream) {
    if (int rc = validate_a8w8(args, false, nullptr)) return rc;
    return run_a8w8(args, args->c, STORE_C, stream);
}

int psg_init(void) {
    (void)psg_cu_count();
    void* ptr = nullptr;
    if (int rc = static_scratch(&ptr)) return rc;
    g_err[0] = 0;
    return 0;
}

uint64_t psg_static_scratch_bytes(void) { return PSG_STATIC_SCRATCH_BYTES; }

int psg_gemm_a8w8_static(const psg_a8w8_args* args, void* stream) {
    if (int rc = validate_a8w8(args, false, nullptr)) return rc;
    // what the same problem's plan would want as workspace; forced tiles take their split count from tile_k
    uint64_t need = psg_workspace_bytes(args->M, args->N, args->K, args->in_dtype);
    if (args->force_path == 1 && args->tile_m > 0 && args->tile_n > 0)
        need = splitk_bytes(args->M, args->N, args->tile_k >= 1 && args->tile_k <= 16 ? args->tile_k : 1);
    if (args->force_path == 2) need = 0;  // (psg_workspace_bytes is already 0 for what the streaming kernel takes by itself)
    if (need > PSG_STATIC_SCRATCH_BYTES)
        return fail(PSG_E_WORKSPACE, "this problem's split-K plan needs %llu bytes of scratch, the static scratch holds %u; use "
                    "psg_gemm_a8w8 with a caller workspace", (unsigned long long)need, PSG_STATIC_SCRATCH_BYTES);
    psg_a8w8_args local = *args;
    local.workspace = nullptr;
    local.workspace_bytes = 0;
    if (need) {
        void* ptr = nullptr;
        if (int rc = static_scratch(&ptr)) return rc;
        local.workspace = ptr;  // the per-device address, never the symbol's host-side name
        local.workspace_bytes = PSG_STATIC_SCRATCH_BYTES;
    }
    return run_a8w8(&local, local.c, STORE_C, stream);
}

void psg_tile_coords(int32_t id, int32_t tiles_m, int32_t tiles_n, int32_t group_m, int32_t* tm, int32_t* tn) {
    int a = 0, b = 0;
    psg_tile_order(id, tiles_m, tiles_n, group_m, &a, &b);
    *tm = a;
    *tn = b;
}

int psg_debug_tile_order(int32_t tiles_m, int32_t tiles_n, int32_t group_m, int32_t* out, void* stream) {
    if (!out) return fail(PSG_E_NULL, "out must be non-NULL");
    if (tiles_m < 1 || tiles_n < 1 || group_m < 1 || (int64_t)tiles_m * tiles_n > (1 << 24))
        return fail(PSG_E_SHAPE, "need tiles_m, tiles_n, group_m >= 1 and at most 2^24 tiles");
    const hipError_t e = psg_launch_tile_order(tiles_m, tiles_n, group_m, out, static_cast<hipStream_t>(stream));
    if (e != hipSuccess) return hip_fail(e, "psg_debug_tile_order launch");
    g_err[0] = 0;
    return 0;
}

int psg_debug_plan(int32_t M, int32_t N, int32_t K, int32_t in_dtype, int32_t* tile_m, int32_t* tile_n, int32_t* splits) {
    if (!tile_m || !tile_n || !splits) return fail(PSG_E_NULL, "tile_m, tile_n and splits must be non-NULL");
    if (in_dtype < PSG_IN_INT8 || in_dtype > PSG_IN_BF16) return fail(PSG_E_DTYPE, "in_dtype %d unknown", in_dtype);
    const int kind = kKinds[in_dtype], eb = kind == KIND_FP16 || kind == KIND_BF16 ? 2 : 1;
    if (M < 1 || M > 65536 || N < 16 || K < 1 || (uint64_t)N * (uint64_t)K * eb > 0xFFFFFFFFull)
        return fail(PSG_E_SHAPE, "M=%d outside [1, 65536], N=%d below 16, K=%d below 1 or W above 4 GiB", M, N, K);
    const int kbytes = K * eb;
    const bool small = takes_stream(M, N, kbytes);
    const Plan plan = small ? Plan{Tile{0, 0, 0}, 1} : plan_tiled(M, N, kbytes, false, kind);
    *tile_m = plan.t.m;
    *tile_n = plan.t.n;
    *splits = plan.splits;
    g_err[0] = 0;
    return 0;
}

int psg_debug_moe_reads_once(const int32_t* expert_ids, int32_t blocks, int32_t used, int32_t per_tile, int32_t experts, int32_t cached, int32_t* out, void* stream) {
    if (!expert_ids || !out) return fail(PSG_E_NULL, "expert_ids and out must be non-NULL");
    if (blocks < 1 || blocks > (1 << 20) || used < 0 || used > blocks || (per_tile != 1 && per_tile != 2) || experts < 1 || cached < 0)
        return fail(PSG_E_SHAPE, "need 1 <= blocks <= 2^20, 0 <= used <= blocks, per_tile 1 or 2, experts >= 1, cached >= 0");
    const hipError_t e = psg_launch_moe_reads_once(expert_ids, blocks, used, per_tile, experts, cached, out, static_cast<hipStream_t>(stream));
    if (e != hipSuccess) return hip_fail(e, "psg_debug_moe_reads_once launch");
    g_err[0] = 0;
    return 0;
}

int psg_gemm_a8w8_acc(const psg_a8w8_args* args, void* acc, void* stream) {
    if (int rc = validate_a8w8(args, true, acc)) return rc;
    return run_a8w8(args, acc, STORE_ACC, stream);
}

static int mx_common(const psg_mxfp4_args* a, void* out, int store, void* stream) {
    if (!a) return fail(PSG_E_NULL, "args is NULL");
    if (!out || !a->a || !a->b || !a->scale_a || !a->scale_b) return fail(PSG_E_NULL, "c, a, b, scale_a, scale_b must be non-NULL");
    if (a->out_dtype != PSG_OUT_BF16 && a->out_dtype != PSG_OUT_FP16) return fail(PSG_E_DTYPE, "out_dtype %d unknown", a->out_dtype);
    if (a->a_dtype < PSG_MX_FP4 || a->a_dtype > PSG_MX_FP8) return fail(PSG_E_DTYPE, "a_dtype %d unknown (0 fp4, 1 fp6, 2 fp8)", a->a_dtype);
    if (a->b_dtype != PSG_MX_FP4 && a->b_dtype != PSG_MX_FP8) return fail(PSG_E_DTYPE, "b_dtype %d must be 0 (fp4) or 2 (fp8)", a->b_dtype);
    if (a->M < 1 || a->M > 65536) return fail(PSG_E_SHAPE, "M=%d outside [1, 65536]", a->M);
    if (a->N < 32 || a->N % 32) return fail(PSG_E_SHAPE, "N=%d must be a positive multiple of 32", a->N);
    if (a->K < 256 || a->K % 256) return fail(PSG_E_SHAPE, "K=%d must be a positive multiple of 256", a->K);
    if (a->batch < 0 || a->batch > 65535) return fail(PSG_E_SHAPE, "batch=%d outside [0, 65535]", a->batch);
    if (a->pad0 != 0) return fail(PSG_E_SHAPE, "pad0 must be 0");
    const int batch = a->batch > 1 ? a->batch : 1;
    const uint64_t a_row = a->a_dtype == PSG_MX_FP4 ? (uint64_t)a->K / 2 : (uint64_t)a->K;
    const uint64_t b_row = a->b_dtype == PSG_MX_FP4 ? (uint64_t)a->K / 2 : (uint64_t)a->K;
    const uint64_t chunk = (uint64_t)(a->K / 256) * 256;
    if ((uint64_t)a->N * b_row > 0xFFFFFFFFull) return fail(PSG_E_SHAPE, "one batch of W exceeds the 4 GiB descriptor range");
    if (a->a_row_stride < 0 || a->c_row_stride < 0 || a->scale_a_chunk_stride < 0 || a->a_batch_stride < 0 || a->c_batch_stride < 0 ||
        a->scale_a_batch_stride < 0)
        return fail(PSG_E_SHAPE, "strides must be >= 0 (0 = dense)");
    const uint64_t a_rs = a->a_row_stride ? (uint64_t)a->a_row_stride : a_row;
    const uint64_t c_rs = a->c_row_stride ? (uint64_t)a->c_row_stride : (uint64_t)a->N;
    const uint64_t sa_cs = a->scale_a_chunk_stride ? (uint64_t)a->scale_a_chunk_stride : chunk;
    if (a_rs < a_row || a_rs % 16) return fail(PSG_E_SHAPE, "a_row_stride=%lld must be a multiple of 16 and at least the %llu bytes of a row",
                                               (long long)a_rs, (unsigned long long)a_row);
    if (c_rs < (uint64_t)a->N || c_rs % 4) return fail(PSG_E_SHAPE, "c_row_stride=%lld must be a multiple of 4 elements and at least N", (long long)c_rs);
    if (sa_cs < chunk || sa_cs % 4) return fail(PSG_E_SHAPE, "scale_a_chunk_stride=%lld must be a multiple of 4 and at least %llu", (long long)sa_cs,
                                                (unsigned long long)chunk);
    if ((uint64_t)a->M * a_rs > 0xFFFFFFFFull || (uint64_t)((a->M + 31) / 32) * sa_cs > 0xFFFFFFFFull)
        return fail(PSG_E_SHAPE, "one batch of A or scale_a exceeds the 4 GiB descriptor range");
    if (a->a_batch_stride % 16 || a->c_batch_stride % 8 || a->scale_a_batch_stride % 4)
        return fail(PSG_E_ALIGN, "batch strides must keep a 16-byte, c 8-byte and scale_a 4-byte aligned");
    if (!aligned(a->a, 16) || !aligned(a->b, 16)) return fail(PSG_E_ALIGN, "a and b must be 16-byte aligned");
    if (!aligned(a->scale_a, 4) || !aligned(a->scale_b, 4)) return fail(PSG_E_ALIGN, "scales must be 4-byte aligned");
    if (!aligned(out, 16)) return fail(PSG_E_ALIGN, "output must be 16-byte aligned");
    if (a->force_path < 0 || a->force_path > 3) return fail(PSG_E_SHAPE, "force_path=%d unknown", a->force_path);
    const bool dense = a_rs == a_row && c_rs == (uint64_t)a->N && sa_cs == chunk;
    const bool fp4_fast = a->a_dtype == PSG_MX_FP4 && a->b_dtype == PSG_MX_FP4 && batch == 1 && dense;
    const bool fp8_pair = a->a_dtype == PSG_MX_FP8 && a->b_dtype == PSG_MX_FP8 && batch == 1 && dense;
    const bool w4 = a->b_dtype == PSG_MX_FP4 && a->a_dtype != PSG_MX_FP4;
    // what the general kernel's split-K plan needs is there
    const bool room = store == STORE_C && a->workspace && aligned(a->workspace, 16) && a->workspace_bytes >= splitk_bytes(a->M, a->N, mx_general_splits(a->M, a->N, a->K));
    const bool routed = a->force_path == 0 && (fp8_pair || (w4 && batch == 1 && dense && store == STORE_C));
    const MxRoute route = routed ? mx_route(a->M, a->N, a->K, fp8_pair, room) : MX_GENERAL;
    if (a->force_path == 2 && !fp4_fast) return fail(PSG_E_SHAPE, "force_path=2 is for dense, unbatched fp4 x fp4 only");
    if (a->force_path == 1 && !fp4_fast && !fp8_pair)
        return fail(PSG_E_SHAPE, "force_path=1 is for dense, unbatched fp4 x fp4 or fp8 x fp8 only");
    if (a->force_path == 2 && a->M > kStreamMaxM) return fail(PSG_E_SHAPE, "small-M path needs M <= %d, got %d", kStreamMaxM, a->M);
    // batches of the fp4 and fp8 pairs and of fp8 / fp6 x fp4: a launch of the dense tiles per batch
    const int64_t a_bs = a->a_batch_stride ? a->a_batch_stride : (int64_t)((uint64_t)a->M * a_rs);
    const int64_t c_bs = a->c_batch_stride ? a->c_batch_stride : (int64_t)((uint64_t)a->M * c_rs * 2);
    const int64_t sa_bs = a->scale_a_batch_stride ? a->scale_a_batch_stride : (int64_t)((uint64_t)((a->M + 31) / 32) * sa_cs);
    const bool per_batch = (w4 || a->b_dtype == a->a_dtype) && batch > 1 && dense && store == STORE_C && a->force_path == 0 && batch <= 8 && mx_fills_tiles(a->M, a->N) &&
                           a_bs % 16 == 0 && c_bs % 16 == 0 && sa_bs % 4 == 0;
    if (route == MX_TILES || per_batch || (fp8_pair && a->force_path == 1)) {
        const bool forced = a->force_path == 1 && a->tile_m > 0 && a->tile_n > 0;
        const bool fp4 = a->a_dtype == PSG_MX_FP4;
        const Tile t = forced ? Tile{a->tile_m, a->tile_n, 4} : pick_mx_tile(a->M, a->N, fp4 ? a->K / 2 : a->K, fp4 ? MX_FP4 : w4 ? MX_W4 : MX_FP8);
        A8W8Params q{};
        q.c = out;
        q.a = static_cast<const uint8_t*>(a->a);
        q.b = static_cast<const uint8_t*>(a->b);
        q.mx_sa = static_cast<const uint8_t*>(a->scale_a);
        q.mx_sb = static_cast<const uint8_t*>(a->scale_b);
        q.M = a->M;
        q.N = a->N;
        q.K = a->K;
        q.group_m = tile_group(a->xcd_swizzle, a->M, a->N, t, (double)a->M * a_row + (double)a->N * b_row + 2.0 * a->M * a->N);
        q.ksplit = 1;
        q.wave_layout = a->reserved >= 2 ? a->reserved : 1;  // four wavefronts: 8192x4096x4096 117 us against 130 with eight
        q.splits = 1;
        q.epi = EPI_NONE;
        q.out = a->out_dtype;
        if (fp4) q.wave_layout = t.waves == 8 ? 8 : 1;
        for (int z = 0; z < batch; z++) {
            const hipError_t te = w4 ? psg_launch_tiled_mxw4(q, a->a_dtype == PSG_MX_FP6, t.m, t.n, static_cast<hipStream_t>(stream))
                                     : psg_launch_a8w8_tiled(q, fp4 ? KIND_MXFP4 : KIND_MXFP8, store, t.m, t.n, static_cast<hipStream_t>(stream));
            if (te != hipSuccess) return hip_fail(te, "psg_gemm_mxfp4 launch");
            q.c = static_cast<uint8_t*>(q.c) + c_bs;
            q.a += a_bs;
            q.b += (uint64_t)a->N * b_row;
            q.mx_sa += sa_bs;
            q.mx_sb += (uint64_t)(a->N / 32) * chunk;
        }
        g_err[0] = 0;
        return 0;
    }
    if (a->force_path == 3 || !fp4_fast) {
        MxGenParams g;
        g.c = out;
        g.a = static_cast<const uint8_t*>(a->a);
        g.b = static_cast<const uint8_t*>(a->b);
        g.sa = static_cast<const uint8_t*>(a->scale_a);
        g.sb = static_cast<const uint8_t*>(a->scale_b);
        g.M = a->M;
        g.N = a->N;
        g.K = a->K;
        g.out = a->out_dtype;
        g.splits = 1;
        g.a_row_stride = (int64_t)a_rs;
        g.c_row_stride = (int64_t)c_rs;
        g.sa_chunk_stride = (int64_t)sa_cs;
        g.a_batch = a_bs;
        g.b_batch = (int64_t)((uint64_t)a->N * b_row);
        g.c_batch = store == STORE_ACC ? (int64_t)a->M * a->N * 4 : c_bs;
        g.sa_batch = sa_bs;
        g.sb_batch = (int64_t)((uint64_t)(a->N / 32) * chunk);
        hipError_t ge;
        const bool small = store == STORE_C && a->force_path == 0 &&
                           (routed ? route == MX_SMALL : mx_general_small(a->M, a->N, a->K, a->a_dtype == PSG_MX_FP4, a->b_dtype == PSG_MX_FP8, batch));
        const int splits = !small && batch == 1 && c_rs == (uint64_t)a->N && store == STORE_C ? mx_general_splits(a->M, a->N, a->K) : 1;
        if (small) {
            ge = psg_launch_mx_smallm(g, a->a_dtype, a->b_dtype, batch, static_cast<hipStream_t>(stream));
        } else if (splits > 1 && a->workspace && aligned(a->workspace, 16) && a->workspace_bytes >= splitk_bytes(a->M, a->N, splits)) {
            MxGenParams part = g;
            part.c = a->workspace;
            part.splits = splits;
            ge = psg_launch_mx_generic(part, a->a_dtype, a->b_dtype, STORE_ACC, 1, static_cast<hipStream_t>(stream));
            A8W8Params q{};
            q.c = out;
            q.M = a->M;
            q.N = a->N;
            q.K = a->K;
            q.splits = splits;
            q.epi = EPI_NONE;
            q.out = a->out_dtype;
            if (ge == hipSuccess) ge = psg_launch_splitk_finalize(q, a->workspace, 0, 0, static_cast<hipStream_t>(stream));
        } else {
            ge = psg_launch_mx_generic(g, a->a_dtype, a->b_dtype, store, batch, static_cast<hipStream_t>(stream));
        }
        if (ge != hipSuccess) return hip_fail(ge, "psg_gemm_mxfp4 launch");
        g_err[0] = 0;
        return 0;
    }
    MxParams p;
    p.c = out;
    p.a = static_cast<const uint8_t*>(a->a);
    p.b = static_cast<const uint8_t*>(a->b);
    p.sa = static_cast<const uint8_t*>(a->scale_a);
    p.sb = static_cast<const uint8_t*>(a->scale_b);
    p.M = a->M;
    p.N = a->N;
    p.K = a->K;
    p.out = a->out_dtype;
    p.group_m = 8;
    const bool small = a->force_path == 2 || (a->force_path == 0 && mx_takes_small(a->M, a->N, a->K));
    hipError_t e;
    if (small) {
        // four wavefronts x four K slices per workgroup when every slice still holds two 256-K steps, else eight
        const int kt = a->K / 256;
        const int nw = kt >= 8 ? 4 : 8;
        p.ksplit = pick_ksplit(a->N / 32, kt);
        if (p.ksplit > nw) p.ksplit = nw;
        if (nw == 4 && p.ksplit < 4) p.ksplit = 4;
        e = psg_launch_mxfp4_smallm(p, store, nw, static_cast<hipStream_t>(stream));
    } else {
        const bool forced = a->force_path == 1 && a->tile_m > 0 && a->tile_n > 0;
        const Plan plan = plan_tiled(a->M, a->N, a->K / 2, true, KIND_MXFP4);
        const Tile t = forced ? Tile{a->tile_m, a->tile_n, 4} : plan.t;
        int splits = forced ? (a->tile_k >= 1 && a->tile_k <= 16 ? a->tile_k : 1) : plan.splits;
        if (store != STORE_C || !a->workspace || !aligned(a->workspace, 16) || a->workspace_bytes < splitk_bytes(a->M, a->N, splits)) splits = 1;
        A8W8Params q{};
        q.c = p.c;
        q.a = p.a;
        q.b = p.b;
        q.mx_sa = p.sa;
        q.mx_sb = p.sb;
        q.M = p.M;
        q.N = p.N;
        q.K = p.K;
        q.group_m = tile_group(a->xcd_swizzle, a->M, a->N, t, splits > 1 ? 1e30 : (double)(a->M + (double)a->N) * (a->K / 2) + 2.0 * a->M * a->N);
        q.ksplit = 1;
        q.wave_layout = a->reserved >= 2 ? a->reserved : (!forced && t.waves == 8 ? 8 : 1);
        q.splits = splits;
        q.epi = EPI_NONE;
        q.out = p.out;
        if (splits > 1) {
            A8W8Params part = q;
            part.c = a->workspace;
            e = psg_launch_a8w8_tiled(part, KIND_MXFP4, STORE_ACC, t.m, t.n, static_cast<hipStream_t>(stream));
            if (e == hipSuccess) e = psg_launch_splitk_finalize(q, a->workspace, 0, 0, static_cast<hipStream_t>(stream));
        } else {
            e = psg_launch_a8w8_tiled(q, KIND_MXFP4, store, t.m, t.n, static_cast<hipStream_t>(stream));
        }
    }
    if (e != hipSuccess) return hip_fail(e, "psg_gemm_mxfp4 launch");
    g_err[0] = 0;
    return 0;
}

int psg_gemm_mxfp4(const psg_mxfp4_args* args, void* stream) { return mx_common(args, args ? args->c : nullptr, STORE_C, stream); }

int psg_gemm_mxfp4_acc(const psg_mxfp4_args* args, void* acc, void* stream) { return mx_common(args, acc, STORE_ACC, stream); }

// Workspace of a stage 2 that accumulates by way of rows (moe_rows.hip), or 0 where adding directly is faster.
// The MX pair goes by rows from 12 MB of additions (tokens x topk x model_dim) on (us by rows / atomics, model 4096, inter 1536, top-8:
// 64 tokens 28.4 / 24.2, 128 34.4 / 33.4, 256 42.7 / 53.4, 512 53.5 / 74.3, 1024 79.8 / 119.6, 4096 297 / 392; top-1 4096 x 4096 58.6 /
// 63.1, 4096 x 1024 23.4 / 21.0; top-6 512 x 2048 26.5 / 28.2, 4096 x 1024 42.6 / 75.4).  The stages with one scale per row go by rows from
// 24 MB and four slots on (fp8: 333 tokens x top-9 72 / 75, 512 x top-8 70 / 72, 1024 105 / 118, 4096 330 / 371; 4096 x top-6 x 1024 53 / 60;
// but 1024 x top-2 x 4096 41 / 35, 4096 x top-1 75 / 64).
// The scratch is bounded: 1 GiB with one scale per row, where it stops being faster anyway (fp8, model 7168, inter 2048, top-8 on 32
// experts: 8192 tokens, 0.95 GB, 1355 / 1412; 16384 tokens, 1.85 GB, 2791 / 2768; 32768 tokens, 3.6 GB, 6046 / 5882), and 4 GiB, one and a
// half per cent of the device, for the MX pair, which still gains there (1042 / 1395, 2040 / 2947, 4013 / 6383).  With int4 weights, whose
// tiles run two workgroups a CU and hide more of the additions, 256 MB, what the last-level cache holds of the rows (model 4096, inter 1536,
// top-8 on 32 experts: 1024 tokens 120 / 134, 2048, 160 MB, 213 / 224, but 4096, 288 MB, 446 / 402; 2048 x 7168 x 2048, 280 MB, 461 / 442).
uint64_t psg_moe_rows_workspace_bytes(int32_t tokens, int32_t topk, int32_t sorted_size, int32_t model_dim, int32_t out_dtype, int32_t kind) {
    if (tokens < 1 || topk < 1 || sorted_size < 1 || model_dim < 2 || (out_dtype != PSG_OUT_BF16 && out_dtype != PSG_OUT_FP16)) return 0;
    const int64_t bytes = (int64_t)tokens * topk * model_dim * 2;
    const bool mx = kind == 1;
    if (bytes < (mx ? 12ll << 20 : 24ll << 20) || (!mx && topk < 4)) return 0;
    const uint64_t need = psg_moe_rows_bytes(tokens, topk, sorted_size, model_dim);
    return need <= (mx ? 4ull << 30 : kind == 2 ? 256ull << 20 : 1ull << 30) ? need : 0;
}

static int moe_gemm_common(const psg_moe_args* a, void* workspace, uint64_t workspace_bytes, void* stream) {
    if (!a) return fail(PSG_E_NULL, "args is NULL");
    if (!a->out || !a->x || !a->w || !a->scale_x || !a->scale_w || !a->sorted_token_ids || !a->sorted_expert_ids || !a->num_valid_ids)
        return fail(PSG_E_NULL, "out, x, w, scale_x, scale_w, sorted_token_ids, sorted_expert_ids, num_valid_ids must be non-NULL");
    if (a->doweight && !a->sorted_weights) return fail(PSG_E_NULL, "sorted_weights must be non-NULL when doweight is set");
    if (a->stage != 1 && a->stage != 2) return fail(PSG_E_SHAPE, "stage=%d must be 1 or 2", a->stage);
    if (a->in_dtype != PSG_IN_INT8 && a->in_dtype != PSG_IN_FP8_E4M3FN && a->in_dtype != PSG_IN_INT8_W4)
        return fail(PSG_E_DTYPE, "in_dtype %d must be int8, fp8 or int8 with int4 weights", a->in_dtype);
    if (a->out_dtype < PSG_OUT_BF16 || a->out_dtype > PSG_OUT_F32) return fail(PSG_E_DTYPE, "out_dtype %d unknown", a->out_dtype);
    if (a->out_dtype == PSG_OUT_F32 && !(a->stage == 2 && a->accumulate))
        return fail(PSG_E_DTYPE, "fp32 output exists only for stage 2 with accumulate (kernels/moe/moe_gemm_2stage/gemm2.py:629)");
    if (a->x_slot_major != 0 && !(a->x_slot_major == 1 && a->stage == 1))
        return fail(PSG_E_SHAPE, "x_slot_major=%d must be 0, or 1 for stage 1", a->x_slot_major);
    if ((a->no_pairing != 0 && a->no_pairing != 1) || a->pad0 != 0) return fail(PSG_E_SHAPE, "no_pairing must be 0 or 1 and pad0 0");
    if (a->tokens < 1 || a->tokens >= (1 << 24)) return fail(PSG_E_SHAPE, "tokens=%d outside [1, 2^24)", a->tokens);
    if (a->topk < 1 || a->topk > 255) return fail(PSG_E_SHAPE, "topk=%d outside [1, 255]", a->topk);
    if (a->experts < 1) return fail(PSG_E_SHAPE, "experts=%d must be positive", a->experts);
    if (a->block_m != 16 && a->block_m != 32 && a->block_m != 64 && a->block_m != 128) return fail(PSG_E_SHAPE, "block_m=%d must be 16, 32, 64 or 128", a->block_m);
    if (a->blocks < 1 || a->blocks > 65535) return fail(PSG_E_SHAPE, "blocks=%d outside [1, 65535]", a->blocks);
    if (a->sorted_size < 1) return fail(PSG_E_SHAPE, "sorted_size=%d must be positive", a->sorted_size);
    const int K = a->stage == 1 ? a->model_dim : a->inter_dim, n_out = a->stage == 1 ? a->inter_dim : a->model_dim;
    if (K < 128 || K % 128) return fail(PSG_E_SHAPE, "K=%d of stage %d must be a positive multiple of 128", K, a->stage);
    if (n_out < 16 || n_out % 16) return fail(PSG_E_SHAPE, "output width %d of stage %d must be a positive multiple of 16", n_out, a->stage);
    const uint64_t rows_x = (a->stage == 1 && !a->x_slot_major) ? (uint64_t)a->tokens : (uint64_t)a->tokens * (uint64_t)a->topk;
    const uint64_t rows_e = a->stage == 1 ? 2ull * (uint64_t)n_out : (uint64_t)n_out;
    if (rows_x * (uint64_t)K > 0xFFFFFFF0ull) return fail(PSG_E_SHAPE, "x exceeds the 4 GiB descriptor range");
    if (rows_e * (uint64_t)K > 0xFFFFFFF0ull) return fail(PSG_E_SHAPE, "one expert's weights exceed the 4 GiB descriptor range");
    if (!aligned(a->x, 16) || !aligned(a->w, 16) || !aligned(a->scale_w, 16) || !aligned(a->out, 16))
        return fail(PSG_E_ALIGN, "x, w, scale_w and out must be 16-byte aligned");
    MoeParams p;
    p.out = a->out;
    p.x = static_cast<const uint8_t*>(a->x);
    p.w = static_cast<const uint8_t*>(a->w);
    p.sx = a->scale_x;
    p.sw = a->scale_w;
    p.sorted_ids = a->sorted_token_ids;
    p.expert_ids = a->sorted_expert_ids;
    p.sorted_w = a->sorted_weights;
    p.num_valid = a->num_valid_ids;
    p.x_slot_major = a->x_slot_major;
    p.pair_blocks = a->no_pairing ? 0 : 1;
    p.tokens = a->tokens;
    p.topk = a->topk;
    p.experts = a->experts;
    p.n_out = n_out;
    p.K = K;
    p.sorted_size = a->sorted_size;
    p.out_dtype = a->out_dtype;
    p.doweight = a->doweight ? 1 : 0;
    p.accumulate = a->stage == 2 && a->accumulate ? 1 : 0;
    p.by_position = 0;
    p.blocks = 0;
    hipError_t e = hipSuccess;
    const bool rows = workspace && p.accumulate && a->out_dtype != PSG_OUT_F32 && workspace_bytes >= psg_moe_rows_bytes(a->tokens, a->topk, a->sorted_size, n_out);
    MoeRowsParams r{};
    if (rows) {
        r.out = static_cast<uint16_t*>(a->out);
        r.sorted_ids = p.sorted_ids;
        r.expert_ids = p.expert_ids;
        r.num_valid = p.num_valid;
        r.tokens = p.tokens;
        r.topk = p.topk;
        r.experts = p.experts;
        r.dim = n_out;
        r.sorted_size = p.sorted_size;
        r.blocks = a->blocks;
        r.block_m = r.granule = a->block_m;
        r.slots = p.topk;
        r.out_dtype = p.out_dtype;
        psg_moe_rows_carve(r, workspace);
        p.out = r.rows;
        p.accumulate = 0;
        p.by_position = 1;
    }
    e = psg_launch_moe_gemm(p, r, a->in_dtype == PSG_IN_INT8 ? KIND_INT8 : a->in_dtype == PSG_IN_INT8_W4 ? KIND_INT8W4 : KIND_FP8, a->stage, a->block_m, a->blocks, static_cast<hipStream_t>(stream));
    if (e == hipSuccess && rows) e = psg_launch_moe_rows_add(r, static_cast<hipStream_t>(stream));
    if (e != hipSuccess) return hip_fail(e, "psg_moe_gemm launch");
    g_err[0] = 0;
    return 0;
}

int psg_moe_gemm(const psg_moe_args* a, void* stream) { return moe_gemm_common(a, nullptr, 0, stream); }

int psg_moe_gemm_rows(const psg_moe_args* a, void* workspace, uint64_t workspace_bytes, void* stream) {
    if (workspace && !aligned(workspace, 16)) return fail(PSG_E_ALIGN, "workspace must be 16-byte aligned");
    return moe_gemm_common(a, workspace, workspace_bytes, stream);
}

namespace {
int moe_reduce_common(const void* x, void* y, const int32_t* mask, const int32_t* ids, int32_t tokens, int32_t topk, int32_t model_dim,
                      int32_t experts, int32_t dtype, void* stream) {
    if (!x || !y) return fail(PSG_E_NULL, "x and y must be non-NULL");
    if (dtype != PSG_OUT_BF16 && dtype != PSG_OUT_FP16 && dtype != PSG_OUT_F32) return fail(PSG_E_DTYPE, "dtype %d must be bf16, fp16 or fp32", dtype);
    if (tokens < 1 || topk < 1 || model_dim < 4 || model_dim % 4) return fail(PSG_E_SHAPE, "need tokens, topk >= 1 and model_dim a positive multiple of 4");
    const int al = dtype == PSG_OUT_F32 ? 16 : 8;
    if (!aligned(x, al) || !aligned(y, al)) return fail(PSG_E_ALIGN, "x and y must be %d-byte aligned", al);
    if (mask && (!ids || experts < 1)) return fail(PSG_E_NULL, "an expert mask needs topk_ids and experts >= 1");
    const hipError_t e = psg_launch_moe_reduce(x, y, tokens, topk, model_dim, dtype, mask, ids, experts, static_cast<hipStream_t>(stream));
    if (e != hipSuccess) return hip_fail(e, "psg_moe_reduce launch");
    g_err[0] = 0;
    return 0;
}
}  // namespace

int psg_moe_mx_scale_sort(const void* scale, const int32_t* sorted_token_ids, const int32_t* num_valid_ids, void* out, int32_t tokens, int32_t topk,
                          int32_t cols, int32_t sorted_size, void* stream) {
    if (!scale || !sorted_token_ids || !num_valid_ids || !out) return fail(PSG_E_NULL, "scale, sorted_token_ids, num_valid_ids and out must be non-NULL");
    if (tokens < 1 || tokens >= (1 << 24)) return fail(PSG_E_SHAPE, "tokens=%d outside [1, 2^24)", tokens);
    if (topk < 1 || topk > 255) return fail(PSG_E_SHAPE, "topk=%d outside [1, 255]", topk);
    if (cols < 8 || cols % 8) return fail(PSG_E_SHAPE, "cols=%d must be a positive multiple of 8", cols);
    if (sorted_size < 1) return fail(PSG_E_SHAPE, "sorted_size=%d must be positive", sorted_size);
    if (((int64_t)sorted_size + 31) / 32 * 8 * (int64_t)cols > 0x7FFFFFFFll) return fail(PSG_E_SHAPE, "sorted_size * cols exceeds 2^33 bytes");
    if (!aligned(out, 4)) return fail(PSG_E_ALIGN, "out must be 4-byte aligned");
    const hipError_t e = psg_launch_moe_mx_scale_sort(scale, sorted_token_ids, num_valid_ids, out, tokens, topk, cols, sorted_size, static_cast<hipStream_t>(stream));
    if (e != hipSuccess) return hip_fail(e, "psg_moe_mx_scale_sort launch");
    g_err[0] = 0;
    return 0;
}

static int moe_mx_gemm_common(const psg_moe_mx_args* a, int32_t topk, void* workspace, uint64_t workspace_bytes, void* stream) {
    if (!a) return fail(PSG_E_NULL, "args is NULL");
    const bool inline_quant = a->stage == 1 && a->a_dtype == PSG_MX_BF16_QUANT;
    if (!a->out || !a->a || (!a->a_scale && !inline_quant) || !a->w || !a->w_scale || !a->sorted_token_ids || !a->sorted_expert_ids || !a->num_valid_ids)
        return fail(PSG_E_NULL, "out, a, a_scale, w, w_scale, sorted_token_ids, sorted_expert_ids and num_valid_ids must be non-NULL");
    if (a->stage != 1 && a->stage != 2) return fail(PSG_E_SHAPE, "stage=%d must be 1 or 2", a->stage);
    if (a->stage == 1 && !a->out_scale) return fail(PSG_E_NULL, "out_scale must be non-NULL in stage 1");
    if (a->stage == 2 && a->atomic && !a->sorted_weights) return fail(PSG_E_NULL, "sorted_weights must be non-NULL for the atomic epilogue");
    if (a->pad0 != 0) return fail(PSG_E_SHAPE, "pad0 must be 0");
    if (a->stage == 1 ? (a->a_dtype != PSG_MX_FP4 && a->a_dtype != PSG_MX_FP8 && a->a_dtype != PSG_MX_BF16_QUANT) : a->a_dtype != PSG_MX_FP4)
        return fail(PSG_E_DTYPE, "a_dtype %d: stage 1 takes 0 (fp4), 2 (fp8) or 3 (bf16, quantised by the kernel), stage 2 takes 0 (fp4)", a->a_dtype);
    if (a->stage == 2 && a->out_dtype != PSG_OUT_BF16 && a->out_dtype != PSG_OUT_FP16) return fail(PSG_E_DTYPE, "out_dtype %d unknown", a->out_dtype);
    if (a->block_m != 16 && a->block_m != 32 && a->block_m != 64 && a->block_m != 128) return fail(PSG_E_SHAPE, "block_m=%d must be 16, 32, 64 or 128", a->block_m);
    if (a->stage == 1 && (a->block_m == 16) != inline_quant)
        return fail(PSG_E_SHAPE, "stage 1: blocks of 16 rows go with a_dtype 3 (bf16 activations quantised by the kernel) and only with it, got block_m=%d a_dtype=%d", a->block_m, a->a_dtype);
    if (a->tokens < 1 || a->tokens >= (1 << 24)) return fail(PSG_E_SHAPE, "tokens=%d outside [1, 2^24)", a->tokens);
    if (a->experts < 1) return fail(PSG_E_SHAPE, "experts=%d must be positive", a->experts);
    if (a->model_dim < 256 || a->model_dim % 256) return fail(PSG_E_SHAPE, "model_dim=%d must be a positive multiple of 256", a->model_dim);
    if (a->inter_dim < 256 || a->inter_dim % 256) return fail(PSG_E_SHAPE, "inter_dim=%d must be a positive multiple of 256", a->inter_dim);
    if (a->sorted_size < a->block_m) return fail(PSG_E_SHAPE, "sorted_size=%d is below one block of %d rows", a->sorted_size, a->block_m);
    if (a->blocks < 1) return fail(PSG_E_SHAPE, "blocks=%d must be positive", a->blocks);
    if ((int64_t)a->blocks * a->block_m > (int64_t)a->sorted_size)
        return fail(PSG_E_SHAPE, "blocks=%d of %d rows exceed sorted_size=%d", a->blocks, a->block_m, a->sorted_size);
    const int K = a->stage == 1 ? a->model_dim : a->inter_dim;
    const int n_out = a->stage == 1 ? a->inter_dim : a->model_dim;
    const uint64_t a_row = inline_quant ? 2ull * (uint64_t)K : a->a_dtype == PSG_MX_FP8 ? (uint64_t)K : (uint64_t)K / 2;
    const uint64_t a_rows = a->stage == 1 ? (uint64_t)a->tokens : (uint64_t)a->sorted_size;
    const uint64_t rows_e = a->stage == 1 ? 2ull * (uint64_t)n_out : (uint64_t)n_out;
    if (a_rows * a_row > 0xFFFFFFF0ull) return fail(PSG_E_SHAPE, "a exceeds the 4 GiB descriptor range");
    if (rows_e * (uint64_t)(K / 2) > 0xFFFFFFF0ull) return fail(PSG_E_SHAPE, "one expert's weights exceed the 4 GiB descriptor range");
    if (!aligned(a->a, 16) || !aligned(a->w, 16) || (!inline_quant && !aligned(a->a_scale, 4)) || !aligned(a->w_scale, 4) || !aligned(a->out, 16))
        return fail(PSG_E_ALIGN, "a, w and out must be 16-byte aligned, a_scale and w_scale 4-byte aligned");
    MoeMxParams p;
    p.out = a->out;
    p.out_scale = static_cast<uint8_t*>(a->out_scale);
    p.a = static_cast<const uint8_t*>(a->a);
    p.a_scale = static_cast<const uint8_t*>(a->a_scale);
    p.w = static_cast<const uint8_t*>(a->w);
    p.w_scale = static_cast<const uint8_t*>(a->w_scale);
    p.sorted_ids = a->sorted_token_ids;
    p.expert_ids = a->sorted_expert_ids;
    p.sorted_w = a->sorted_weights;
    p.num_valid = a->num_valid_ids;
    p.tokens = a->tokens;
    p.experts = a->experts;
    p.n_out = n_out;
    p.K = K;
    p.sorted_size = a->sorted_size;
    p.out_dtype = a->out_dtype;
    p.atomic = a->stage == 2 && a->atomic ? 1 : 0;
    p.eshift = 0;
    p.n_tiles = p.n_groups = p.by_expert = p.quad_tiles = 0;
    if (((int64_t)a->blocks << 1) * (int64_t)((n_out / 128 + 7) / 8 * 8) > 0x7FFFFFFFll - ROWS_INDEX_WGS) return fail(PSG_E_SHAPE, "blocks=%d times the column tiles exceed the grid", a->blocks);
    hipError_t e = hipSuccess;
    const bool rows = workspace && p.atomic && topk >= 1 && topk <= 255 && workspace_bytes >= psg_moe_rows_bytes(a->tokens, topk, a->sorted_size, n_out);
    MoeRowsParams r{};
    if (rows) {
        r.out = static_cast<uint16_t*>(a->out);
        r.sorted_ids = p.sorted_ids;
        r.expert_ids = p.expert_ids;
        r.num_valid = p.num_valid;
        r.tokens = p.tokens;
        r.topk = topk;
        r.experts = p.experts;
        r.dim = n_out;
        r.sorted_size = p.sorted_size;
        r.blocks = a->blocks;
        r.block_m = a->block_m;
        r.granule = a->block_m == 128 ? 64 : a->block_m;
        r.slots = 256;  // this pair of stages reads the token of an id only
        r.out_dtype = p.out_dtype;
        psg_moe_rows_carve(r, workspace);
        p.out = r.rows;
        p.atomic = 2;
    }
    e = psg_launch_moe_mx_gemm(p, r, a->a_dtype == PSG_MX_FP8 ? MXF_FP8 : MXF_FP4, a->stage, a->block_m, a->blocks, static_cast<hipStream_t>(stream));
    if (e == hipSuccess && rows) e = psg_launch_moe_rows_add(r, static_cast<hipStream_t>(stream));
    if (e != hipSuccess) return hip_fail(e, "psg_moe_mx_gemm launch");
    g_err[0] = 0;
    return 0;
}

int psg_moe_mx_gemm(const psg_moe_mx_args* a, void* stream) { return moe_mx_gemm_common(a, 0, nullptr, 0, stream); }

int psg_moe_mx_gemm_rows(const psg_moe_mx_args* a, int32_t topk, void* workspace, uint64_t workspace_bytes, void* stream) {
    if (workspace && !aligned(workspace, 16)) return fail(PSG_E_ALIGN, "workspace must be 16-byte aligned");
    return moe_mx_gemm_common(a, topk, workspace, workspace_bytes, stream);
}

int psg_moe_reduce(const void* x, void* y, int32_t tokens, int32_t topk, int32_t model_dim, int32_t dtype, void* stream) {
    return moe_reduce_common(x, y, nullptr, nullptr, tokens, topk, model_dim, 0, dtype, stream);
}

int psg_moe_reduce_masked(const void* x, void* y, const int32_t* expert_mask, const int32_t* topk_ids, int32_t tokens, int32_t topk,
                          int32_t model_dim, int32_t experts, int32_t dtype, void* stream) {
    if (!expert_mask || !topk_ids) return fail(PSG_E_NULL, "expert_mask and topk_ids must be non-NULL");
    return moe_reduce_common(x, y, expert_mask, topk_ids, tokens, topk, model_dim, experts, dtype, stream);
}

uint64_t psg_moe_sorting_workspace_bytes(int32_t tokens, int32_t topk, int32_t experts) {
    if (tokens < 1 || topk < 1 || experts < 1) return 0;
    return psg_moe_sort_workspace((int64_t)tokens * topk, experts);
}

int psg_moe_sorting(const psg_moe_sort_args* a, void* stream) {
    MoeSortParams p;
    if (int rc = check_moe_sort(a, true, &p)) return rc;
    const hipError_t e = psg_launch_moe_sort(p, a->workspace, a->workspace ? a->workspace_bytes : 0, static_cast<hipStream_t>(stream));
    if (e != hipSuccess) return hip_fail(e, "psg_moe_sorting launch");
    g_err[0] = 0;
    return 0;
}

int psg_moe_topk_gating(const psg_moe_gating_args* a, void* stream) {
    MoeGatingParams g;
    if (int rc = check_moe_gating(a, true, &g)) return rc;
    const hipError_t e = psg_launch_moe_gating(g, a->dtype, static_cast<hipStream_t>(stream));
    if (e != hipSuccess) return hip_fail(e, "psg_moe_topk_gating launch");
    g_err[0] = 0;
    return 0;
}

int psg_moe_softmax_sorting_fused(int32_t tokens, int32_t topk, int32_t experts) {
    return tokens >= 1 && topk >= 1 && experts >= 1 && psg_moe_gate_sort_fuses(tokens, topk, experts) ? 1 : 0;
}

int psg_moe_softmax_sorting(const psg_moe_gating_args* ga, const psg_moe_sort_args* sa, void* stream) {
    if (!ga || !sa) return fail(PSG_E_NULL, "args is NULL");
    if (ga->tokens != sa->tokens || ga->topk != sa->topk || ga->experts != sa->experts)
        return fail(PSG_E_SHAPE, "gating (tokens=%d topk=%d experts=%d) and sorting (tokens=%d topk=%d experts=%d) disagree", ga->tokens,
                    ga->topk, ga->experts, sa->tokens, sa->topk, sa->experts);
    const bool fused = ga->tokens >= 1 && ga->topk >= 1 && ga->experts >= 1 && psg_moe_gate_sort_fuses(ga->tokens, ga->topk, ga->experts);
    MoeGatingParams g;
    MoeSortParams p;
    if (int rc = check_moe_gating(ga, !fused, &g)) return rc;
    if (int rc = check_moe_sort(sa, false, &p)) return rc;
    hipError_t e;
    if (fused) {
        e = psg_launch_moe_gate_sort(p, g, ga->dtype, static_cast<hipStream_t>(stream));
    } else {
        // two steps: the sorter reads what the gating kernel wrote
        if ((const void*)sa->topk_ids != (const void*)ga->indices || (const void*)sa->topk_weights != (const void*)ga->weights)
            return fail(PSG_E_NULL, "beyond the fused range the sorter's topk_ids / topk_weights must be the gating's indices / weights");
        e = psg_launch_moe_gate_then_sort(p, g, ga->dtype, sa->workspace, sa->workspace ? sa->workspace_bytes : 0, static_cast<hipStream_t>(stream));
    }
    if (e != hipSuccess) return hip_fail(e, "psg_moe_softmax_sorting launch");
    g_err[0] = 0;
    return 0;
}

int psg_quant_pertoken(const void* x, int32_t x_dtype, void* y, float* scale, int32_t M, int32_t K, int32_t out_dtype, void* stream) {
    if (!x || !y || !scale) return fail(PSG_E_NULL, "x, y and scale must be non-NULL");
    if (x_dtype < 0 || x_dtype > 2) return fail(PSG_E_DTYPE, "x_dtype %d unknown (0 fp32, 1 bf16, 2 fp16)", x_dtype);
    if (out_dtype != PSG_IN_INT8 && out_dtype != PSG_IN_FP8_E4M3FN) return fail(PSG_E_DTYPE, "out_dtype must be int8 or fp8");
    if (M < 1 || K < 8 || K % 8) return fail(PSG_E_SHAPE, "need M >= 1 and K a positive multiple of 8 (got M=%d K=%d)", M, K);
    if (!aligned(x, 16) || !aligned(y, 8)) return fail(PSG_E_ALIGN, "x must be 16-byte and y 8-byte aligned");
    const hipError_t e = psg_launch_quant_pertoken(x, x_dtype, y, scale, M, K, out_dtype == PSG_IN_FP8_E4M3FN, static_cast<hipStream_t>(stream));
    if (e != hipSuccess) return hip_fail(e, "psg_quant_pertoken launch");
    g_err[0] = 0;
    return 0;
}

int psg_quant_mxfp4(const void* x, int32_t x_dtype, void* packed, void* scales, int32_t M, int32_t K, int32_t shuffled, void* stream) {
    if (!x || !packed || !scales) return fail(PSG_E_NULL, "x, packed and scales must be non-NULL");
    if (x_dtype < 0 || x_dtype > 2) return fail(PSG_E_DTYPE, "x_dtype %d unknown (0 fp32, 1 bf16, 2 fp16)", x_dtype);
    if (M < 1 || K < 32 || K % 32) return fail(PSG_E_SHAPE, "need M >= 1 and K a positive multiple of 32 (got M=%d K=%d)", M, K);
    if (shuffled && K % 256) return fail(PSG_E_SHAPE, "the shuffled scale layout needs K %% 256 == 0 (got K=%d)", K);
    if (!aligned(x, 16) || !aligned(packed, 16)) return fail(PSG_E_ALIGN, "x and packed must be 16-byte aligned");
    const int R = (M + 31) / 32 * 32;  // scales cover whole 32-row chunks; the padding rows get scale byte 0
    const hipError_t e = psg_launch_quant_mxfp4(x, x_dtype, packed, scales, M, R, K, shuffled, static_cast<hipStream_t>(stream));
    if (e != hipSuccess) return hip_fail(e, "psg_quant_mxfp4 launch");
    g_err[0] = 0;
    return 0;
}

}  // extern "C"
