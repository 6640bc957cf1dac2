// pme_slots.hpp -- where the binning keeps an atom's records (host and device).
#pragma once
#include <cstddef>

#if defined(__HIP__)
#include <hip/hip_runtime.h>
#define PME_HOST_DEVICE __host__ __device__ __forceinline__
#else
#define PME_HOST_DEVICE inline
#endif

namespace pme {

// A slot of the record store.  The store holds 8 slots per atom, so from 2^28
// atoms on a slot does not fit 32 bits: every place that holds one has this type.
using RecordSlot = size_t;
constexpr RecordSlot kNoSlot = (RecordSlot)-1;

// slot of record `at` of chunk w, rec_stride slots per chunk
PME_HOST_DEVICE RecordSlot record_slot(int w, int rec_stride, int at) {
  return (RecordSlot)w * (RecordSlot)rec_stride + (RecordSlot)at;
}

// One element of the list in which a batch of records is reordered
using RecordList = RecordSlot;

}  // namespace pme
