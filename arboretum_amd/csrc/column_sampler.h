// Column sampling of the trees of a booster.
#ifndef ARBORETUM_AMD_COLUMN_SAMPLER_H_
#define ARBORETUM_AMD_COLUMN_SAMPLER_H_

#include <algorithm>
#include <cstdint>
#include <cstring>
#include <random>
#include <vector>

#include "config.h"
#include "device_common.h"
#include "memory_pool.h"

namespace arb {

// The features a tree may split on at every level (InitGrowingTree / InitTreeLevel,
// garden.cu:126-165, and the `take` prefix of FindBestSplits, :249-253): the
// ids are shuffled per tree, the first floor(bytree * columns) of them again
// per level, and the first floor(bylevel * bytree * columns) are active.
//
// The draws depend on nothing but the seed, so the masks are made for several trees at a time and
// copied behind the kernels of the trees before: a copy per tree, which had to wait for them, left the
// device idle between trees for as long as the host takes to launch one (200,000 rows x 50: 293 -> 262 us a
// tree).
class ColumnSampler {
 public:
  ~ColumnSampler() { Release(); }

  void Init(const Configuration &cfg, size_t columns, int features, int levels) {
    rnd_.seed(cfg.internal.seed);  // garden.cu:87
    columns_ = columns;
    F_ = features;
    levels_ = levels;
    take_tree_ = (int)(cfg.tree.colsample_bytree * columns);
    take_level_ = (unsigned)(cfg.tree.colsample_bylevel * cfg.tree.colsample_bytree * columns);
    if (take_level_ >= columns) return;  // no sampling
    const size_t bytes = MaskBytes();
    most_ = std::max<size_t>(1, std::min<size_t>(64, ((size_t)1 << 20) / bytes));
    host_ = static_cast<unsigned char *>(PinnedPoolTake(most_ * bytes));
    device_ = static_cast<unsigned char *>(DevicePoolTake(most_ * bytes));
    HIP_OK(hipEventCreateWithFlags(&copied_, hipEventDisableTiming));
    made_ = at_ = std::min<size_t>(most_, 4);  // (the first batch: twice that)
  }
  // The caller has waited for the kernels that read the masks.
  void Release() noexcept {
    if (copied_) {
      (void)hipEventSynchronize(copied_);
      (void)hipEventDestroy(copied_);
    }
    PinnedPoolGive(host_);
    DevicePoolGive(device_);
    host_ = device_ = nullptr;
    copied_ = nullptr;
  }

  // To the next tree, whose kernels go to `stream` as those of the trees before.
  void NextTree(hipStream_t stream) {
    if (!device_) return;
    if (++at_ < made_) return;
    HIP_OK(hipEventSynchronize(copied_));  // (recorded a batch of trees ago)
    made_ = std::min(most_, 2 * made_);
    std::memset(host_, 0, made_ * MaskBytes());
    std::vector<unsigned> ids(columns_);
    for (size_t t = 0; t < made_; ++t) {
      unsigned char *mask = host_ + t * MaskBytes();
      for (size_t i = 0; i < columns_; ++i) ids[i] = (unsigned)i;
      std::shuffle(ids.begin(), ids.end(), rnd_);
      for (int level = 0; level < levels_; ++level, mask += F_) {
        std::shuffle(ids.begin(), ids.begin() + take_tree_, rnd_);
        for (unsigned j = 0; j < take_level_; ++j)
          if (ids[j] < (unsigned)F_) mask[ids[j]] = 1;
      }
    }
    HIP_OK(hipMemcpyAsync(device_, host_, made_ * MaskBytes(), hipMemcpyHostToDevice, stream));
    HIP_OK(hipEventRecord(copied_, stream));
    at_ = 0;
  }
  bool Samples() const { return device_ != nullptr; }
  // Mask of a level of the current tree, a byte per feature; null: every feature.
  const unsigned char *Active(int level) const {
    return device_ ? device_ + at_ * MaskBytes() + (size_t)level * F_ : nullptr;
  }

 private:
  size_t MaskBytes() const { return (size_t)levels_ * F_; }
  std::default_random_engine rnd_;
  size_t columns_ = 0, most_ = 0, made_ = 0, at_ = 0;
  int F_ = 0, levels_ = 0, take_tree_ = 0;
  unsigned take_level_ = 0;
  unsigned char *host_ = nullptr, *device_ = nullptr;
  hipEvent_t copied_ = nullptr;
};

}  // namespace arb
#endif  // ARBORETUM_AMD_COLUMN_SAMPLER_H_
