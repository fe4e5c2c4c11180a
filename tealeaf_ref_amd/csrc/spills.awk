# Reads the compiler's kernel-resource-usage remarks of one source and fails if
# one of the kernels that KERNELS (a pattern) names spills registers in a way it
# must not, or if there is none of them.  None may use scratch memory;
#   VECTORS=1  nor move vector registers elsewhere: the compiler may place such a
#              move inside a region that only some lanes run, where it misses the
#              others (it has sent the on-chip loops' stores astray).  The
#              many-step passes have no such region where they move a few to
#              accumulation registers;
#   SCALARS=1  nor scalar registers to lanes: the many-step passes' coefficients
#              have come back wrong from there.
/remark: +Function Name:/ {
  name = $0
  sub(/.*Function Name: */, "", name)
  sub(/ .*/, "", name)
  watched = name ~ KERNELS
  if (watched) seen += 1
}
/remark: +(VGPRs Spill|ScratchSize \[bytes\/lane\]|SGPRs Spill):/ && watched {
  what = $0
  sub(/.*remark: */, "", what)
  sub(/ *\[-R.*/, "", what)
  n = what
  sub(/.*: */, "", n)
  if (n + 0 > 0 && (what ~ /^Scratch/ || (what ~ /^VGPRs/ ? VECTORS : SCALARS))) {
    print name ": " what
    bad = 1
  }
}
END {
  if (!seen) print "no kernel " KERNELS " in the compiler's report"
  exit (bad || !seen)
}
