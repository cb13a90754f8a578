// Device bytes of a render's buffers, shared by the code that allocates them
// (hip/integrator.hip, hip/guide.hip: each checks these sums against its own
// buffer types with static_asserts) and the render service, which reserves
// them before a job starts (host/service.cpp).
#pragma once
#include <stdint.h>

namespace dl_sizes {

// Path state, per path of a pass: ray origin and direction, hit record,
// shadow-ray direction (a shadow ray starts at the ray origin), throughput,
// radiance and pending NEE term (one 16-byte vector each), the aux word (8),
// the depth and record slot (8), the pcg32 state (8), the sample index (4),
// the film position (8), the scene index (1), two double-buffered material queues of kMatQueueSegs
// segments (4 bytes per path per segment each), and the ray and shadow
// queues (4 each).
constexpr int kMatQueueSegs = 8;
constexpr uint64_t kStateBytesPerPath = 7 * 16 + 8 + 8 + 8 + 4 + 8 + 1 + 2 * kMatQueueSegs * 4 + 2 * 4;  // 221

// Film: float4 accumulation (sum w L, sum w) + resolved RGB per pixel.
constexpr uint64_t kFilmBytesPerPixel = 16 + 12;

// Guided rendering (the learned proposal).
constexpr int kGuideMixFloats = 40;          // decoded mixture per queued shading point
constexpr int kGuideRecordFloats = 24;       // training record
constexpr uint32_t kGuideRecordSlots = 1u << 23;
constexpr uint32_t kGuideBatchRows = 1u << 18;  // records per Adam step
constexpr uint32_t kGuideTrainRows = 64;        // rows of a training tile
constexpr uint32_t kGuideTrainBlocks = 512;     // blocks of a training step (at most), a partial gradient each
// Blocks of a training step on n rows: a tile each until there are
// kGuideTrainBlocks, two for each of the MI355X's 256 CUs.  They depend on the
// rows alone, not on the device's CUs: the blocks' shares of the rows are the
// order of the gradient's sums, so a trained network is the same everywhere.
constexpr uint32_t guide_train_blocks(uint32_t n) {
    const uint32_t tiles = n / kGuideTrainRows + (n % kGuideTrainRows != 0 ? 1 : 0);
    return tiles < kGuideTrainBlocks ? tiles : kGuideTrainBlocks;
}
constexpr uint32_t kGuideSumBlocks = 64;        // partial sums of the training weights
constexpr uint32_t kGuideScanTile = 1024;       // records per prefix-sum tile
constexpr int kGuideParams = 21808;
constexpr int kGuideWSlot = 64 * 96;            // bfloat16 elements per layer copy

// network parameters, Adam moments, gradient, biases, bfloat16 copies
// (W in two orders, W^T), the step's loss and the partial sums
constexpr uint64_t kGuideNetBytes = 4ull * kGuideParams * 4 + 5 * 64 * 4 + 3ull * 5 * kGuideWSlot * 2 +
                                    (1 + kGuideSumBlocks + kGuideTrainBlocks) * 4;
// one training batch: its features (96), directions (3) and weights (1); the
// blocks' partial gradients
constexpr uint64_t kGuideTrainBytes =
    (uint64_t)kGuideBatchRows * (96 + 3 + 1) * 4 + (uint64_t)kGuideTrainBlocks * kGuideParams * 4;
// record weights and the prefix-sum tiles over every record slot
constexpr uint64_t kGuideResampleBytes =
    (uint64_t)kGuideRecordSlots * 4 + 2ull * (kGuideRecordSlots / kGuideScanTile + 1) * 4;

// Everything a guided render adds to a plain one whose passes hold `paths`
// paths.
constexpr uint64_t guide_bytes(uint64_t paths) {
    return paths * kGuideMixFloats * 4 + (uint64_t)kGuideRecordSlots * kGuideRecordFloats * 4 + kGuideNetBytes +
           kGuideTrainBytes + kGuideResampleBytes;
}

}  // namespace dl_sizes
