// The arrival word of the grid-wide maximum (grid_max, ft_common.hpp), over
// whatever atomics it is given, so that the protocol also runs on host threads.
//
// The word is generation << 32 | arrivals. A launch's workgroups each add 1;
// the one that makes it nwg advances the generation and takes the nwg arrivals
// off in one add, the others poll until the generation moves.
//
// Launches that use one word must be ordered. Two that overlap mix their
// counts: workgroups go on too early, or at the end of their polls, and the
// arrivals need not add up to either launch's. So that only the overlapping
// calls are spoiled, no workgroup leaves arrivals in the word it last saw: in
// an ordered launch there are none once the generation has moved. Each arrival
// and each release is followed by its own workgroup's look, so none is left
// once the launches have ended. The polls' look is free; the releasing
// workgroup's is a load that it waits for while the others' polls are under way.
//
// W: add(x) returns the word before; and_(x); load(); pause() between polls.
#pragma once

#ifdef __HIPCC__
#define FT_WORD_FN __device__ __forceinline__
#else
#define FT_WORD_FN inline
#endif

namespace ft {

typedef unsigned long long grid_word_t;

// Arrive, and wait for the launch's last arrival or for `polls` polls.
template <typename W>
FT_WORD_FN void grid_arrive(W w, unsigned nwg, unsigned polls) {
    const grid_word_t old = w.add(1);
    const unsigned gen = (unsigned)(old >> 32);
    const bool last = (unsigned)old + 1u == nwg;
    if (last) w.add((1ull << 32) - nwg);
    grid_word_t cur = w.load();
    bool moved = last || (unsigned)(cur >> 32) != gen;
#pragma unroll 1
    for (unsigned i = 1; i < polls && !moved; ++i) {
        w.pause();
        cur = w.load();
        moved = (unsigned)(cur >> 32) != gen;
    }
    if (!moved || (unsigned)cur) w.and_(~0ull << 32);
}

}  // namespace ft
