// Which of the processes that share a GPU may launch kernels whose workgroups wait for each other.
// Such a launch needs all its workgroups on the chip at once.  Launches of one process are put in order
// (ResidentOrder in the backend); those of two processes are not: each could get part of the CUs and both would
// wait until their bounds.  So a process holds an advisory lock on the GPU while it may have one under way, and
// a session that does not get it runs its rounds as launches of their own for that step.  The lock
// is on a file the kernel keeps for every PCI device (nothing is written to it), so it needs no file of its
// own, is the same one in every container of the machine, and goes with a process that dies.
#ifndef CAVS_HOST_RESIDENT_H_
#define CAVS_HOST_RESIDENT_H_

namespace cavs {

class ResidentClaim {
 public:
  ResidentClaim() = default;
  ResidentClaim(const ResidentClaim &) = delete;
  ResidentClaim &operator=(const ResidentClaim &) = delete;
  ~ResidentClaim() { give(); }
  // Whether this process may (from now until every session of it has given its claim back).  Half a microsecond.
  bool take(int device);
  // No such launch of this session is under way any more.
  void give();

 private:
  int device_ = -1;
};

}  // namespace cavs
#endif
