// cz_scratch.h - grow-only device buffers of the forward's scratch.  Plain host
// C++ (no device code): the CPU sanitizer build of the host code compiles it
// as it is, with an allocator that refuses.
#pragma once

#include <cstddef>
#include <vector>

namespace cz {

// *p with room for `need` elements.  A buffer that grows is kept in `retired`
// (captured graphs and launched work may still point at it).  alloc(bytes)
// returns nullptr when there is no room: the call returns -1 and the buffer
// stays as it was, because a caller may go on without the growth (a layer past
// 8192 slots falls back) while another layer of the chain has been promised
// the present one.
template <typename T, typename Alloc>
int grow_buffer(T **p, size_t *cap, size_t need, std::vector<void *> &retired, Alloc alloc) {
    if (*cap >= need) return 0;
    void *q = alloc(need * sizeof(T));
    if (!q) return -1;
    if (*p) retired.push_back((void *)*p);
    *p = (T *)q;
    *cap = need;
    return 0;
}

// The same with room for `want` >= need elements where that fits, so that calls
// that grow a little at a time do not each retire a buffer.
template <typename T, typename Alloc>
int grow_stepped(T **p, size_t *cap, size_t need, size_t want, std::vector<void *> &retired, Alloc alloc) {
    if (*cap >= need || grow_buffer(p, cap, want, retired, alloc) == 0) return 0;
    return want > need ? grow_buffer(p, cap, need, retired, alloc) : -1;
}

}  // namespace cz
