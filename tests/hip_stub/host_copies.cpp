// host_copies UP DOWN [nopin]: one upload of UP bytes and, without a wait between them,
// one download of DOWN bytes through the same HostCopy (a submit whose results
// are read in the same call).  Ends with 0 if both arrived whole and no memory or
// event was given back while the stream still needed it.  nopin: there is no
// pinned memory.
#include <hip/hip_runtime.h>

#include <cstdio>

#include "../../hybridmantis_amd/csrc/fd2_hostcopy.h"

int main(int argc, char** argv) {
  if (argc != 3 && argc != 4) return 2;
  hipstub::no_pinned = argc == 4;
  const size_t up = strtoull(argv[1], nullptr, 10), down = strtoull(argv[2], nullptr, 10);
  std::vector<char> from(up), dev(up), results(down), to(down);
  for (size_t i = 0; i < up; ++i) from[i] = (char)(i * 31 + i / 251);
  for (size_t i = 0; i < down; ++i) results[i] = (char)(i * 17 + i / 253);
  int wrong = 0;
  {
    fd2::HostCopy copy;
    const int rc = copy.upload(0, 0, dev.data(), up, 1, [&](char* dst, size_t off, size_t len) {
      memcpy(dst, from.data() + off, len);
      return (int)FD2_OK;
    });
    if (rc != FD2_OK || copy.download(0, 0, to.data(), results.data(), down) != FD2_OK) wrong |= 1;
    hipStreamSynchronize(0);
    if (dev != from) wrong |= 2;
    if (to != results) wrong |= 4;
  }
  if (hipstub::faults) wrong |= 8;
  printf("wrong %d faults %d rings freed %d\n", wrong, hipstub::faults, hipstub::ring_frees);
  return wrong ? 1 : 0;
}
