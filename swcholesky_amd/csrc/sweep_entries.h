// Entries of the sweeps' vectors as they pass between workgroups.  Included by
// sweep_kernels.h inside numeric.hip's anonymous namespace.

// Bits of an entry not yet computed: a signalling NaN that arithmetic does not return
// (it returns quiet ones); publish() keeps any result away from it.
constexpr unsigned long long kPending = 0x7ff4a5c35a3c4b21ull;
constexpr unsigned long long kQuietNan = 0x7ff8000000000000ull;

// The vectors are double arrays everywhere else: an access to their bits may alias those, or
// a mark could pass the load of the right-hand side it replaces.
typedef unsigned long long __attribute__((may_alias)) EntryBits;

// Entries pass between workgroups as relaxed agent-scope atomics: each is coherent by
// itself (written through to, and read from, memory beyond the XCDs' caches), and its own
// readiness, so no order between entries is needed.
__device__ inline unsigned long long load_entry(const double* p) {
  return __hip_atomic_load(reinterpret_cast<const EntryBits*>(p), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline void publish(double* p, double v) {
  unsigned long long b = __builtin_bit_cast(unsigned long long, v);
  if (b == kPending) b = kQuietNan;
  __hip_atomic_store(reinterpret_cast<EntryBits*>(p), b, __ATOMIC_RELAXED,
                     __HIP_MEMORY_SCOPE_AGENT);
}

// (For a later launch: a plain store.)
__device__ inline void mark_pending(double* p) {
  *reinterpret_cast<EntryBits*>(p) = kPending;
}
