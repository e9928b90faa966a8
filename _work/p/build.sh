# build.sh <names of objects to drop>: headers are not tracked
cd /root/repo
python3 - "$@" <<'P'
import sys, os, glob
for f in glob.glob('build/temp*/xllm_service_amd/csrc/*/*.o'):
    b = os.path.basename(f).replace('_hip.o','').replace('.o','')
    if b in sys.argv[1:]: os.remove(f); print('drop', b)
P
python -c "import __graft_entry__ as g; g.build()" > /tmp/build.log 2>&1; rc=$?
grep -n "error:" /tmp/build.log | head; echo rc $rc
