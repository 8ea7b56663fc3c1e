// A HIP runtime for the CPU tests of the library's host code: what is enqueued on a stream is done when the stream (or an
// event) is waited for and not before, device memory is host memory, and calls can be made to fail.  No kernel runs, but the
// one that copies between device memory and a pinned slot, whose accesses are checked against the allocations, as are the outputs of
// the norm + quantizer.
#pragma once
#include <cstddef>
#include <string>
#include <vector>

namespace fake_hip {

extern thread_local int inside;  // this thread is in the runtime, not in the library's code
extern long launches;      // kernels enqueued so far
extern long other_device;  // kernels on a stream of another GPU than the calling thread's (there are two)
extern long out_of_range;  // accesses of the copy kernel outside every allocation (they are left out), and outputs of the norm + quantizer
size_t pending();          // enqueued and not done
size_t allocations();      // device allocations that are not freed
std::vector<std::string> kernels();  // names of the kernels enqueued since the last call of this, with their template arguments and grids, "(x x y)"
void fail_launch(long n);  // the n-th kernel launch from now fails (n = 1: the next one; 0: none)
void fail_copy(long n);    // the same for hipMemcpyAsync
void fail_pinned(bool on); // no pinned memory is to be had

}  // namespace fake_hip
