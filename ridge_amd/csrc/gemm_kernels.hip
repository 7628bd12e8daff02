// gemm_kernels.hip -- instantiates the gfx950 GEMM template over the registered
// variant table and exports the table through the C ABI in include/ridge_gemm.h.
//
// Counterpart of bench/kernels/gemm-mma.cu (launchVariant :19-43, kVariants
// :55-117, numVariants/variant/printVariantTable :121-141).

#include "gemm_mfma.hpp"
#include "gemm_resources.h"
#include "ridge_gemm.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstdio>
#include <cstring>
#include <string>

namespace {

// How a launch runs a row's output tiles: ownTiles of them in the row's own tile and the
// others in partWorkgroups blocks of `part`, as parts of tiles (a ping-pong row's last
// round) or as the whole grid's blocks (smallGrid, a number of ridge::SmallGridPart).
struct Form {
    int ownTiles = 0, parts = 1, smallGrid = 0, partWorkgroups = 0;
    ridge::BlockShape part = {};
};

// With ownTile the row's tile runs everywhere, whatever the grid.
typedef hipError_t (*LaunchFn)(const void*, const void*, void*, int, int, int, bool ownTile, hipStream_t);
typedef Form (*FormFn)(int M, int N, int K, int cus);

// Schedules (ridge_gemm_variant_t.schedule). Rows written RIDGE_VARIANT take
// theirs from the tile config: eight wavefronts (two per SIMD) with a ring of
// three or more stages run the ping-pong schedule, every other row the uniform
// one. Rows written RIDGE_VARIANT_PERSISTENT run the persistent store-behind
// schedule.
enum Schedule { kUniform = 0, kPingPong = 1, kPersistent = 2 };
constexpr bool usesPingPong(int waves, int stages) { return waves == 8 && stages >= 3; }

// Workgroups of `kernel` resident on the current device at once (CUs x
// workgroups per CU), cached per device: the persistent grid. Launches from
// several host threads may fill the cache concurrently; they compute the same
// value, and the atomic makes the store and the loads well defined.
int residentSlots(const void* kernel, int threads, std::atomic<int>& cache) {
    const int cached = cache.load(std::memory_order_relaxed);
    if (cached > 0) return cached;
    int dev = 0, cus = 0, perCu = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&perCu, kernel, threads, 0) != hipSuccess) return 0;
    const int slots = cus * (perCu > 0 ? perCu : 1);
    cache.store(slots, std::memory_order_relaxed);
    return slots;
}

constexpr int kMaxDevices = 64;

// Resident workgroups of a kernel on the current device; 0 with *err set when the
// device cannot be asked.
struct SlotCache {
    std::atomic<int> slots[kMaxDevices];
    int of(const void* kernel, int threads, hipError_t* err) {
        int dev = 0;
        *err = hipGetDevice(&dev);
        if (*err != hipSuccess) return 0;
        if (dev < 0 || dev >= kMaxDevices) {
            *err = hipErrorInvalidDevice;
            return 0;
        }
        const int n = residentSlots(kernel, threads, slots[dev]);
        if (n <= 0) *err = hipErrorInvalidConfiguration;
        return n > 0 ? n : 0;
    }
};

// CUs of the current device, cached per device; 0 when it cannot be asked. Its callers
// then run the row's own tiles, so the query's error is dropped: the launch reports its
// own by hipGetLastError.
int deviceCus() {
    static std::atomic<int> cache[kMaxDevices];
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess) {
        (void)hipGetLastError();
        return 0;
    }
    if (dev < 0 || dev >= kMaxDevices) return 0;
    const int cached = cache[dev].load(std::memory_order_relaxed);
    if (cached > 0) return cached;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) {
        (void)hipGetLastError();
        return 0;
    }
    cache[dev].store(cus, std::memory_order_relaxed);
    return cus;
}

// The block (ridge::SmallGridPart) in which a uniform or persistent row runs a grid of
// at most half as many of its tiles as the device has CUs, 0 for the row's own tile:
// the smallest whose workgroups still fit one round. Own tile -> parts, operands cold:
// 128x128x64 s4 persistent 1024^3 9.1 -> 5.6 us, 2048 x 1024 x 1024 9.1 -> 7.5, 1024 x
// 1024 x 4096 25.4 -> 15.9; 128x128x64 s2 1024^3 11.7 -> 5.6; 128x64x64 s3 512^3 4.9 ->
// 3.8; 64x128x128 s3 persistent 8192 x 128 x 4096 (128 tiles) 19.7 -> 15.3; 256x256x64
// s2 1024 x 2048 x 1024 24.9 -> 7.7.
int smallGridPart(int BM, int BN, int M, int N, int K, int cus) {
    if (BM * BN <= 64 * 64 || !ridge::partsFit(N, K)) return 0;
    if ((M / BM) * (N / BN) > cus / 2) return 0;
    if ((M / 64) * (N / 64) <= cus) return 1;
    if (BN >= 128 && (M / 64) * (N / 128) <= cus) return 2;
    if (BM >= 128 && BN >= 128 && (M / 128) * (N / 128) <= cus) return 3;
    return 0;
}

template <int PART>
void enqueuePart(const _Float16* A, const _Float16* B, _Float16* C, int M, int N, int K, hipStream_t stream) {
    using P = typename ridge::SmallGridPart<PART>::Part;
    const ridge::TileOrder order = ridge::tileOrder<P::kBM, P::kBN, ridge::kPartGroupM>(M, N);
    hipLaunchKernelGGL((ridge::gemmMfmaSmallGridKernel<PART>), dim3((unsigned)((M / P::kBM) * (N / P::kBN))),
                       dim3(ridge::kPartThreads), 0, stream, A, B, C, M, N, K, order.group, order.lastRows);
}

// Enqueues a small grid of a row's BM x BN tiles in its blocks; false where the row
// runs its own tile.
bool enqueueSmallGrid(int BM, int BN, const _Float16* A, const _Float16* B, _Float16* C, int M, int N, int K,
                      hipStream_t stream) {
    if (BM * BN <= 64 * 64) return false;
    switch (smallGridPart(BM, BN, M, N, K, deviceCus())) {
        case 1: enqueuePart<1>(A, B, C, M, N, K, stream); return true;
        case 2: enqueuePart<2>(A, B, C, M, N, K, stream); return true;
        case 3: enqueuePart<3>(A, B, C, M, N, K, stream); return true;
        default: return false;
    }
}

Form smallGridForm(int BM, int BN, int M, int N, int K, int cus) {
    Form f;
    f.smallGrid = smallGridPart(BM, BN, M, N, K, cus);
    if (f.smallGrid == 0) {
        f.ownTiles = (M / BM) * (N / BN);
        return f;
    }
    f.part = f.smallGrid == 1   ? ridge::SmallGridPart<1>::Part::kShape
             : f.smallGrid == 2 ? ridge::SmallGridPart<2>::Part::kShape
                                : ridge::SmallGridPart<3>::Part::kShape;
    f.partWorkgroups = (M / f.part.BM) * (N / f.part.BN);
    return f;
}

template <int BM, int BN, int BK, int WM, int WN, int S, int G>
hipError_t launchPersistent(const void* A, const void* B, void* C, int M, int N, int K, bool ownTile,
                            hipStream_t stream) {
    using P = ridge::PersistentTraits<BM, BN, BK, WM, WN, S, G>;
    const auto* a = static_cast<const _Float16*>(A);
    const auto* b = static_cast<const _Float16*>(B);
    auto* c = static_cast<_Float16*>(C);
    if (!ownTile && enqueueSmallGrid(BM, BN, a, b, c, M, N, K, stream)) return hipGetLastError();
    static SlotCache cache;
    hipError_t err;
    const int resident = cache.of(
        reinterpret_cast<const void*>(&ridge::gemmMfmaPersistentKernel<BM, BN, BK, WM, WN, S, G>), P::kThreads,
        &err);
    if (resident <= 0) return err;
    // Every workgroup must own at least one tile (the kernel's tile count per
    // workgroup assumes it).
    const int tiles = (M / BM) * (N / BN);
    const int grid = tiles < resident ? tiles : resident;
    const ridge::TileOrder order = ridge::tileOrder<BM, BN, G>(M, N);
    hipLaunchKernelGGL((ridge::gemmMfmaPersistentKernel<BM, BN, BK, WM, WN, S, G>), dim3((unsigned)grid),
                       dim3(P::kThreads), 0, stream, a, b, c, M, N, K, order.group,
                       order.lastRows, ridge::reciprocalOf(K / BK), grid, tiles / grid, tiles % grid);
    return hipGetLastError();
}

// Parts per output tile of the last round of a ping-pong grid: `rem` tiles on
// `slots` CUs, one workgroup each. Whole, they hold rem CUs for the time of a tile
// while the others idle. The line is where the parts still fit one round; a second
// round of parts costs more than the whole tile. 256x256x32 s3, whole -> cut:
//   quarters   5888 x 5888 x 1664 (2 rounds and 17 tiles)  112.8 -> 97.2 us
//              4352 x 4096 x 1024 (1 round and 16)          46.7 -> 36.2
//              2048^3 (64 tiles)                            35.0 -> 18.8
//   sixteenths, against eighths: 1024^3 (16 tiles) 6.9 -> 5.7, x 4096 19.8 -> 15.5,
//              4352 x 4096 x 1024 33.6 -> 33.1
//   eighths, against quarters: 5888 x 5888 x 1664 92.7 -> 90.6, 4352 x 4096 x 1024
//              34.4 -> 32.8, 1024 x 2048 x 1024 (32 tiles) 9.3 -> 7.7, 256 x 256 x
//              1024 8.1 -> 6.2
//   halves     2560^3 (100 tiles)                           44.2 -> 34.6
//              4864 x 4864 x 1024 (1 round and 105)         48.4 -> 45.0
//   K no multiple of the smaller parts' 64: halves, 5888 x 5888 x 1632 107.6 -> 100.3
// The halves of the 256x256x32 rows keep the row's BK and with it the row's offset
// bound; those of 256x128x64 are of the smaller parts' BK, which is also the row's.
// 256x128x64 s3 (its parts are the same blocks): halves at 2048^3 (128
// tiles) 23.2 -> 19.6; quarters against halves at 2304 x 4096 x 2048 (1 round and 32)
// 41.0 -> 38.1, whole 50.2.
int tailParts(int rem, int slots, int N, int K, int most) {
    if (rem == 0) return 1;
    if (ridge::partsFit(N, K))
        for (int parts = most; parts >= 4; parts /= 2)
            if (parts * rem <= slots) return parts;
    if (most >= 2 && 2 * rem <= slots) return 2;
    return 1;
}

// Workgroups per step of the first round's phased start, 0 for none: grids of three
// whole rounds and more whose K loop is short enough that the shared drains of C count
// for more than the last step's 7168 cycles. 256x256x32 s3, together -> phased (two
// devices): 8192 x 8192 x 256 47.6 -> 45.4, 58.0 -> 46.3 us; x 1024 114.4 -> 112.6,
// 117.8 -> 111.7; x 2048 198.7 -> 197.6, 203.4 -> 201.0; x 3072 304.0 -> 303.3; 9728 x
// 6400 x 768 88.3 -> 86.0, 93.0 -> 85.2; 15104 x 15104 x 512 219.5 -> 216.5, 232.9 ->
// 224.4; 256x128x64 s3 at 8192 x 4096 x 512 41.6 -> 39.8, 49.8 -> 46.6. Two rounds
// gained up to 20% on one device and lost up to 2% on another (8192 x 4096 x 512 40.2
// -> 36.9, 34.8 -> 34.9; 6144 x 6144 x 512 41.5 -> 42.3). The shortest K loops gain the
// most, the mean of the eight 256x256x32 rows: 8192 x 8192 x 32 29.3 -> 24.7, x 64 33.9
// -> 30.8, x 128 39.6 -> 34.5, x 192 47.2 -> 44.0; 12288 x 4096 (three rounds) x 32 21.9
// -> 19.7, x 64 24.3 -> 21.2; the least 8192 x 6144 x 32 21.3 -> 19.1, x 64 24.2 -> 24.7
// (four of the rows 2-8% slower), x 96 25.7 -> 25.0, x 128 27.5 -> 25.5.
int phaseWidth(int wholeTiles, int slots, int K) {
    return slots >= ridge::kPhases && wholeTiles / slots >= 3 && K <= 2048 ? slots / ridge::kPhases : 0;
}

template <int BM, int BN, int BK>
Form pingPongForm(int M, int N, int K, int cus) {
    using Tail = ridge::TailTiles<BM, BN, BK>;
    const int tiles = (M / BM) * (N / BN);
    // A device that does not say its CUs runs every tile whole.
    const int rem = cus > 0 ? tiles % cus : 0;
    Form f;
    f.parts = tailParts(rem, cus, N, K, Tail::kParts);
    f.ownTiles = f.parts > 1 ? tiles - rem : tiles;
    f.partWorkgroups = (tiles - f.ownTiles) * f.parts;
    if (f.parts > 1) f.part = Tail::shapeOf(f.parts);
    return f;
}

template <int BM, int BN, int BK, int WM, int WN, int S, int G, bool NT>
hipError_t enqueueTiles(const _Float16* A, const _Float16* B, _Float16* C, int M, int N, int K, bool ownTile,
                        hipStream_t stream) {
    using T = ridge::GemmTraits<BM, BN, BK, WM, WN, S, G>;
    const int tiles = (M / BM) * (N / BN);
    const dim3 block(T::kThreads);
    const ridge::TileOrder order = ridge::tileOrder<BM, BN, G>(M, N);
    if constexpr (usesPingPong(T::kWaves, S)) {
        static_assert(2 * T::kLdsBytes > 163840, "a ping-pong row has one workgroup per CU");
        const int cus = deviceCus();
        const Form f = pingPongForm<BM, BN, BK>(M, N, K, ownTile ? 0 : cus);
        hipLaunchKernelGGL((ridge::gemmMfmaPingPongKernel<BM, BN, BK, WM, WN, S, G, NT>),
                           dim3((unsigned)(f.ownTiles + f.partWorkgroups)), block, 0, stream, A, B, C, M, N, K,
                           order.group, order.lastRows, f.ownTiles, f.partWorkgroups,
                           f.parts | phaseWidth(f.ownTiles, cus, K) << 8);
    } else {
        hipLaunchKernelGGL((ridge::gemmMfmaKernel<BM, BN, BK, WM, WN, S, G, NT>), dim3((unsigned)tiles), block, 0,
                           stream, A, B, C, M, N, K, order.group, order.lastRows, ridge::reciprocalOf(K / BK));
    }
    return hipGetLastError();
}

template <int BM, int BN, int BK, int WM, int WN, int S, int G>
hipError_t launchVariant(const void* A, const void* B, void* C, int M, int N, int K, bool ownTile,
                         hipStream_t stream) {
    const auto* a = static_cast<const _Float16*>(A);
    const auto* b = static_cast<const _Float16*>(B);
    auto* c = static_cast<_Float16*>(C);
    constexpr bool pingPong = usesPingPong(ridge::GemmTraits<BM, BN, BK, WM, WN, S, G>::kWaves, S);
    if (!pingPong && !ownTile && enqueueSmallGrid(BM, BN, a, b, c, M, N, K, stream)) return hipGetLastError();
    if ((size_t)M * N * 2 > ridge::kNonTemporalBytes && !(pingPong && K < ridge::kNonTemporalPingPongK))
        return enqueueTiles<BM, BN, BK, WM, WN, S, G, true>(a, b, c, M, N, K, ownTile, stream);
    return enqueueTiles<BM, BN, BK, WM, WN, S, G, false>(a, b, c, M, N, K, ownTile, stream);
}

template <int BM, int BN, int BK, int WM, int WN, int S>
Form formOf(int M, int N, int K, int cus) {
    if constexpr (usesPingPong((BM / WM) * (BN / WN), S)) return pingPongForm<BM, BN, BK>(M, N, K, cus);
    return smallGridForm(BM, BN, M, N, K, cus);
}

template <int BM, int BN>
Form formOfPersistent(int M, int N, int K, int cus) {
    return smallGridForm(BM, BN, M, N, K, cus);
}

struct Entry {
    int BM, BN, BK, WM, WN, stages, groupM;
    int ldsBytes;
    int threads;
    int waves;
    int schedule;
    LaunchFn launch;
    FormFn form;
};

#define RIDGE_VARIANT(BM, BN, BK, WM, WN, S, G)                                              \
    Entry{BM, BN, BK, WM, WN, S, G,                                                          \
          ridge::GemmTraits<BM, BN, BK, WM, WN, S, G>::kLdsBytes,                            \
          ridge::GemmTraits<BM, BN, BK, WM, WN, S, G>::kThreads,                             \
          ridge::GemmTraits<BM, BN, BK, WM, WN, S, G>::kWaves,                               \
          usesPingPong(ridge::GemmTraits<BM, BN, BK, WM, WN, S, G>::kWaves, S) ? kPingPong : kUniform, \
          &launchVariant<BM, BN, BK, WM, WN, S, G>,                                          \
          &formOf<BM, BN, BK, WM, WN, S>},

// ldsBytes includes the epilogue staging; threads and waves include the two
// loader wavefronts.
#define RIDGE_VARIANT_PERSISTENT(BM, BN, BK, WM, WN, S, G)                                   \
    Entry{BM, BN, BK, WM, WN, S, G,                                                          \
          ridge::PersistentTraits<BM, BN, BK, WM, WN, S, G>::kLdsBytes,                      \
          ridge::PersistentTraits<BM, BN, BK, WM, WN, S, G>::kThreads,                       \
          ridge::PersistentTraits<BM, BN, BK, WM, WN, S, G>::kWaves,                         \
          kPersistent,                                                                       \
          &launchPersistent<BM, BN, BK, WM, WN, S, G>,                                       \
          &formOfPersistent<BM, BN>},

const Entry kTable[] = {
#include "gemm_variants.def"
};
#undef RIDGE_VARIANT
#undef RIDGE_VARIANT_PERSISTENT

constexpr int kNumVariants = int(sizeof(kTable) / sizeof(kTable[0]));

bool validIndex(int i) { return i >= 0 && i < kNumVariants; }

}  // namespace

extern "C" {

int ridge_gemm_num_variants(void) { return kNumVariants; }

int ridge_gemm_get_variant(int i, ridge_gemm_variant_t* out) {
    if (!validIndex(i) || out == nullptr) return (int)hipErrorInvalidValue;
    const Entry& e = kTable[i];
    ridge_gemm_variant_t v;
    std::memset(&v, 0, sizeof(v));
    v.BM = e.BM; v.BN = e.BN; v.BK = e.BK; v.WM = e.WM; v.WN = e.WN;
    v.stages = e.stages; v.groupM = e.groupM;
    v.ldsBytes = e.ldsBytes; v.threads = e.threads; v.waves = e.waves;
    v.pingPong = e.schedule == kPingPong ? 1 : 0;
    v.schedule = e.schedule;
    if (i < ridge_gemm_resource_count) {
        const ridge_gemm_resources_t& r = ridge_gemm_resource_table[i];
        v.vgprs = r.vgprs; v.agprs = r.agprs; v.sgprs = r.sgprs;
        v.scratchBytes = r.scratchBytes; v.occupancy = r.occupancy;
        v.regsPerThread = r.vgprs + r.agprs;
    } else {
        v.regsPerThread = -1;
        v.vgprs = v.agprs = v.sgprs = v.scratchBytes = v.occupancy = -1;
    }
    *out = v;
    return 0;
}

int ridge_gemm_find_variant(int BM, int BN, int BK, int WM, int WN, int stages, int groupM) {
    for (int i = 0; i < kNumVariants; ++i) {
        const Entry& e = kTable[i];
        if (e.BM == BM && e.BN == BN && e.BK == BK && e.WM == WM && e.WN == WN && e.stages == stages &&
            e.groupM == groupM)
            return i;
    }
    return -1;
}

int ridge_gemm_divides(int i, int M, int N, int K) {
    if (!validIndex(i)) return 0;
    const Entry& e = kTable[i];
    if (M <= 0 || N <= 0 || K <= 0) return 0;
    if (M % e.BM || N % e.BN || K % e.BK) return 0;
    // The grid is one-dimensional and offsets inside the kernel are 32-bit.
    if ((long long)(M / e.BM) * (N / e.BN) > 0x7fffffffLL) return 0;
    return ridge::tileOffsetsFit(e.BM, e.BK, N, K) ? 1 : 0;
}

static int launchRow(int i, const void* A, const void* B, void* C, int M, int N, int K, bool ownTile,
                     void* stream) {
    if (!ridge_gemm_divides(i, M, N, K)) return (int)hipErrorInvalidValue;
    if (A == nullptr || B == nullptr || C == nullptr) return (int)hipErrorInvalidValue;
    if (((uintptr_t)A | (uintptr_t)B | (uintptr_t)C) & 15u) return (int)hipErrorInvalidValue;
    return (int)kTable[i].launch(A, B, C, M, N, K, ownTile, static_cast<hipStream_t>(stream));
}

int ridge_gemm_launch(int i, const void* A, const void* B, void* C, int M, int N, int K, void* stream) {
    return launchRow(i, A, B, C, M, N, K, false, stream);
}

int ridge_gemm_launch_own_tile(int i, const void* A, const void* B, void* C, int M, int N, int K, void* stream) {
    return launchRow(i, A, B, C, M, N, K, true, stream);
}

int ridge_gemm_launch_form(int i, int M, int N, int K, int numCUs, ridge_gemm_form_t* out) {
    if (out == nullptr || numCUs <= 0 || !ridge_gemm_divides(i, M, N, K)) return (int)hipErrorInvalidValue;
    const Form f = kTable[i].form(M, N, K, numCUs);
    out->ownTiles = f.ownTiles;
    out->partWorkgroups = f.partWorkgroups;
    out->partBM = f.part.BM; out->partBN = f.part.BN; out->partBK = f.part.BK;
    out->partWM = f.part.WM; out->partWN = f.part.WN; out->partStages = f.part.stages;
    return 0;
}

int ridge_gemm_split_rows(int body, int M, int N, int K, int numCUs) {
    if (!validIndex(body) || numCUs <= 0 || !ridge_gemm_divides(body, M, N, K)) return -1;
    ridge_gemm_variant_t v;
    ridge_gemm_get_variant(body, &v);
    // Resident workgroups per CU: LDS, wave slots, and the register file (the
    // compiler's waves per SIMD; a workgroup's waves spread over the 4 SIMDs).
    int perCU = 163840 / v.ldsBytes;
    perCU = std::min(perCU, 32 / v.waves);
    if (v.occupancy > 0) perCU = std::min(perCU, v.occupancy / ((v.waves + 3) / 4));
    if (perCU < 1) return -1;
    const long long slots = (long long)perCU * numCUs;
    const long long perPanel = N / v.BN, panels = M / v.BM;
    const long long rounds = panels * perPanel / slots;
    if (rounds == 0) return 0;
    const long long bodyPanels = rounds * slots / perPanel;
    return bodyPanels >= panels ? M : (int)(bodyPanels * v.BM);
}

int ridge_gemm_launch_split(int body, int tail, int bodyRows, const void* A, const void* B, void* C, int M, int N,
                            int K, void* stream) {
    // Every check before the first launch: a refused call enqueues nothing.
    if (bodyRows <= 0 || bodyRows >= M) return (int)hipErrorInvalidValue;
    if (!ridge_gemm_divides(body, bodyRows, N, K) || !ridge_gemm_divides(tail, M - bodyRows, N, K))
        return (int)hipErrorInvalidValue;
    if (A == nullptr || B == nullptr || C == nullptr) return (int)hipErrorInvalidValue;
    if (((uintptr_t)A | (uintptr_t)B | (uintptr_t)C) & 15u) return (int)hipErrorInvalidValue;
    const char* tailA = static_cast<const char*>(A) + (size_t)bodyRows * K * 2;
    char* tailC = static_cast<char*>(C) + (size_t)bodyRows * N * 2;
    const int rc = ridge_gemm_launch(body, A, B, C, bodyRows, N, K, stream);
    if (rc != 0) return rc;
    return ridge_gemm_launch(tail, tailA, B, tailC, M - bodyRows, N, K, stream);
}

size_t ridge_gemm_variant_table_csv(char* buf, size_t cap) {
    std::string s = "idx,BM,BN,BK,WM,WN,stages,groupM,ldsBytes,threads,regsPerThread,waves,vgprs,agprs,sgprs,"
                    "scratchBytes,occupancy,pingPong,schedule\n";
    char line[256];
    for (int i = 0; i < kNumVariants; ++i) {
        ridge_gemm_variant_t v;
        ridge_gemm_get_variant(i, &v);
        std::snprintf(line, sizeof(line), "%d,%d,%d,%d,%d,%d,%d,%d,%d,%d,%d,%d,%d,%d,%d,%d,%d,%d,%d\n", i, v.BM,
                      v.BN, v.BK, v.WM, v.WN, v.stages, v.groupM, v.ldsBytes, v.threads, v.regsPerThread, v.waves,
                      v.vgprs, v.agprs, v.sgprs, v.scratchBytes, v.occupancy, v.pingPong, v.schedule);
        s += line;
    }
    if (buf != nullptr && cap > 0) {
        const size_t n = s.size() < cap - 1 ? s.size() : cap - 1;
        std::memcpy(buf, s.data(), n);
        buf[n] = '\0';
    }
    return s.size();
}

size_t ridge_gemm_variant_struct_size(void) { return sizeof(ridge_gemm_variant_t); }

const char* ridge_gemm_build_info(void) {
    return "ridge_gemm gfx950 mfma_f32_16x16x32_f16, direct-to-LDS ring, tr16 B reads, xcd+groupM order, "
           "ping-pong schedule for 8-wave rings of 3+ stages, persistent store-behind rows with loader waves";
}

}  // extern "C"
