// args_ahead.h — a kernel's arguments, asked for all at once.
//
// A launch finds its arguments in no cache: the first scalar load from each of their 64-byte lines goes to memory.  The compiler loads an argument where it is used, so a kernel of few loads whose
// arguments fill five lines and more waits for them line after line in front of its first weights: four times in stack_few_kernel, three in stack_rows_kernel.  One load from every
// line in front of a value that everything needs brings them together; what is loaded later comes from the scalar cache.  us a pass, so / not: keronex-batch (sixteen requests) 18380 / 18660, zakusun-serve
// (four) 10160 / 10280.  The vector kernels of one and two rows are slower with it (vitudra-chat 9720 / 9610): their groups' arguments fill fifteen lines, of which a workgroup uses five.
#pragma once

namespace tgx {

// v (a number, or a pointer that is only compared), which a first step of the kernel needs, once a dword of every line of `a` (up to eight lines) and `more` (of the launch's own sizes, say) have come
template <class T, class A>
__device__ __forceinline__ T args_ahead(T v, const A& a, int more = 0) {
  constexpr unsigned n = sizeof(A) / 4;
  static_assert(sizeof(A) % 4 == 0 && n > 0 && n <= 16 * 8, "whole dwords, eight lines");
  const int* p = reinterpret_cast<const int*>(&a);
  auto at = [&](unsigned l) { return p[16 * l < n ? 16 * l : n - 1]; };      // (past the end: its last dword, which may begin a line of its own)
  // (not volatile: it would count as a write of memory, and what kernels read by scalar loads behind it would take vector loads)
  asm("" : "+s"(v) : "s"(at(0)), "s"(at(1)), "s"(at(2)), "s"(at(3)), "s"(at(4)), "s"(at(5)), "s"(at(6)), "s"(at(7)), "s"(more));
  return v;
}

}  // namespace tgx
