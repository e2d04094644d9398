/*
 * Which stream has which scratch slot of a device: plain C++, so that a host program can go through the cases. The
 * caller holds the lock.
 */
#ifndef MSHADOW_AMD_CSRC_SCRATCH_SLOTS_H_
#define MSHADOW_AMD_CSRC_SCRATCH_SLOTS_H_

namespace mshadow_abi {

const int kScratchDevices = 16;

template <int SLOTS>
struct ScratchSlots {
  bool used[kScratchDevices][SLOTS];
  const void *owner[kScratchDevices][SLOTS];

  /*! \brief the stream's slot, a free one where it has none yet, -1 where there is none */
  int Take(int dev, const void *stream) {
    for (int i = 0; i < SLOTS; ++i) {
      if (used[dev][i] && owner[dev][i] == stream) return i;
    }
    for (int i = 0; i < SLOTS; ++i) {
      if (used[dev][i]) continue;
      used[dev][i] = true;
      owner[dev][i] = stream;
      return i;
    }
    return -1;
  }
  bool Has(const void *stream) const {
    for (int d = 0; d < kScratchDevices; ++d) {
      for (int i = 0; i < SLOTS; ++i) {
        if (used[d][i] && owner[d][i] == stream) return true;
      }
    }
    return false;
  }
  /*! \brief the stream is going away. Its slots are free again if its work is done; where that is not known nobody
   *  gets them, nor does a later stream with the same handle. */
  void Release(const void *stream, bool done) {
    for (int d = 0; d < kScratchDevices; ++d) {
      for (int i = 0; i < SLOTS; ++i) {
        if (!used[d][i] || owner[d][i] != stream) continue;
        used[d][i] = !done;
        owner[d][i] = this;  // no stream's handle
      }
    }
  }
};

}  // namespace mshadow_abi

#endif  // MSHADOW_AMD_CSRC_SCRATCH_SLOTS_H_
